"""GEMM operands of any extent, alignment and leading dimension.

The kernels read and write 16-byte pieces at the element's own alignment,
clamp the rows and columns of edge tiles and guard the last partial k-stage.
Every matrix here is embedded in a larger buffer of NaN (row padding, the
elements before its first and after its last): a piece that read past a row
it owns, or an accumulator that took a clamped row's product, would carry a
NaN into the result; a store past an edge would replace a NaN around D.
Bar: the sum bound of K products in the data type, normwise (fp64 1e-12,
fp32 1e-5, the bar of the other kernel tests)."""

import pytest
import torch

from util import normwise

pytestmark = pytest.mark.gpu
TOL = {torch.float64: 1e-12, torch.float32: 1e-5}


def embed(x, ld, off, dt):
    """x (batch, rows, cols) in a NaN buffer: row pitch ld, first element at
    `off`, batches ld + 1 elements apart beyond their rows. Returns the
    buffer, the batch stride and a view of the data in it."""
    b, r, c = x.shape
    stride = r * ld + 1
    buf = torch.full((off + b * stride + 8,), float("nan"), dtype=dt, device="cuda")
    view = torch.as_strided(buf, (b, r, c), (stride, ld, 1), off)
    view.copy_(x.to("cuda", dt))
    return buf, stride, view


# (M, N, K): around the 32-, 64-, 128- and 256-wide tiles and the 16-, 64- and
# 128-deep stages; one row or column; fewer rows than a 16-byte piece holds.
SHAPES = [(65, 129, 17), (63, 127, 33), (130, 257, 64), (64, 256, 48), (1, 70, 40), (70, 1, 40), (3, 3, 19),
          (2, 131, 15), (129, 2, 16), (33, 31, 129), (150, 150, 55), (31, 33, 130), (200, 66, 1), (257, 513, 31)]


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_unaligned_ragged(hip, dt, ta, tb, M, N, K):
    from trntensor_amd.hip import engine

    g = torch.Generator().manual_seed(M * 5 + N * 3 + K)
    batch = 2
    for pad, off, with_c in ((1, 1, True), (0, 0, False), (2, 3, False)):
        A = torch.randn(batch, M, K, generator=g, dtype=torch.float64)
        B = torch.randn(batch, K, N, generator=g, dtype=torch.float64)
        C = torch.randn(batch, M, N, generator=g, dtype=torch.float64)
        sa = A.transpose(1, 2) if ta else A
        sb = B.transpose(1, 2) if tb else B
        lda, ldb, ldc, ldd = sa.shape[2] + pad, sb.shape[2] + pad, N + pad, N + 2 * pad
        Ab, sA, _ = embed(sa, lda, off, dt)
        Bb, sB, _ = embed(sb, ldb, off, dt)
        Cb, sC, _ = embed(C, ldc, off, dt)
        Db, sD, D = embed(torch.full((batch, M, N), float("nan")), ldd, off, dt)
        engine.gemm(ta, tb, M, N, K, Ab, lda, sA, Bb, ldb, sB, Db, ldd, sD, batch, 1.5, 0.5 if with_c else 0.0,
                    Cb[off:] if with_c else None, ldc, sC, a_off=off, b_off=off, d_off=off)
        ref = 1.5 * torch.bmm(A, B) + (0.5 * C if with_c else 0.0)
        torch.cuda.synchronize()
        assert normwise(D.cpu().double(), ref) <= TOL[dt], (pad, off)
        assert int(torch.isnan(Db).sum()) == Db.numel() - batch * M * N, (pad, off)


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(65, 129, 17), (64, 128, 32), (130, 255, 50), (5, 3, 40), (70, 2, 33), (3, 131, 16)])
def test_gemm_dot_unaligned_ragged(hip, dt, ta, tb, M, N, K):
    """The dot epilogue on ragged, unaligned operands: rows and columns past
    the matrix must not enter the sum."""
    from trntensor_amd.hip import engine

    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(1, M, K, generator=g, dtype=torch.float64)
    B = torch.randn(1, K, N, generator=g, dtype=torch.float64)
    E = torch.randn(1, M, N, generator=g, dtype=torch.float64)
    sa, sb = A.transpose(1, 2) if ta else A, B.transpose(1, 2) if tb else B
    lda, ldb = sa.shape[2] + 1, sb.shape[2] + 1
    Ab, sA, _ = embed(sa, lda, 1, dt)
    Bb, sB, _ = embed(sb, ldb, 1, dt)
    Eb, _, _ = embed(E, N + 1, 1, dt)
    out = torch.full((), float("nan"), dtype=dt, device="cuda")
    engine.gemm_dot(ta, tb, M, N, K, Ab, lda, sA, Bb, ldb, sB, 1, M, N, Eb[1:], [0, N + 1, 0, 1, 0], None, None,
                    1.0, 0.0, None, out, a_off=1, b_off=1)
    X = torch.bmm(A, B)
    scale = float((X.abs() * E.abs()).sum())
    assert abs(float(out) - float((X * E).sum())) <= TOL[dt] * scale


@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
@pytest.mark.parametrize("M,N", [(12 * 17, 9), (9, 12 * 17), (12 * 11, 10 * 13), (300, 6 * 7), (1, 130), (70, 1)])
@pytest.mark.parametrize("K", [5, 200])
def test_gemm_dot_orientation(hip, ta, tb, M, N, K):
    """fp64 dots run as given or exchanged, after their tiles and E's strides:
    E contiguous along n, along m, and as an outer product of two factors
    whose letters interleave (m = (a, b), n = (i, j), E = X[a, i] Y[b, j]),
    each against float64 torch."""
    from trntensor_amd.hip import engine

    dt = torch.float64
    g = torch.Generator().manual_seed(M + 7 * N + K)
    A = torch.randn(1, M, K, generator=g, dtype=dt)
    B = torch.randn(1, K, N, generator=g, dtype=dt)
    E = torch.randn(M, N, generator=g, dtype=dt)
    sa, sb = A.transpose(1, 2) if ta else A, B.transpose(1, 2) if tb else B
    Ad, Bd = sa.contiguous().cuda(), sb.contiguous().cuda()
    ml = next(d for d in (17, 11, 9, 1) if M % d == 0)
    nl = next(d for d in (13, 7, 1) if N % d == 0)
    X = torch.randn(M // ml, N // nl, generator=g, dtype=dt)
    Y = torch.randn(ml, nl, generator=g, dtype=dt)
    outer = (X[:, None, :, None] * Y[None, :, None, :]).reshape(M, N)
    forms = [(E, E, [0, N, 0, 1, 0], None, None, M, N), (E, E.t().contiguous(), [0, 1, 0, M, 0], None, None, M, N),
             (outer, X, [N // nl, 0, 1, 0, 0], Y, [0, nl, 0, 1, 0], ml, nl),
             (outer, X.t().contiguous(), [1, 0, M // ml, 0, 0], Y.t().contiguous(), [0, 1, 0, ml, 0], ml, nl)]
    P = torch.bmm(A, B)[0]
    for k, (full, e1, s1, e2, s2, m_lo, n_lo) in enumerate(forms):
        out = torch.full((), float("nan"), dtype=dt, device="cuda")
        engine.gemm_dot(ta, tb, M, N, K, Ad, sa.shape[2], 0, Bd, sb.shape[2], 0, 1, m_lo, n_lo, e1.cuda(), s1,
                        None if e2 is None else e2.cuda(), s2, 1.0, 0.0, None, out)
        assert abs(float(out) - float((P * full).sum())) <= TOL[dt] * float((P * full).abs().sum()), k


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(33, 47, 21), (500, 700, 37), (1030, 1025, 18), (2050, 2049, 17), (1, 1, 16), (17, 3, 100)])
def test_gemm_dd_tiles(hip, ta, tb, M, N, K):
    """The double-double GEMM's tiles (chosen by the grid they give): every
    shape against float64, and bitwise against the same rows computed in
    blocks of 40, whose grids take smaller tiles: the order of an output's
    sums does not depend on the tile."""
    from trntensor_amd.hip import engine

    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(1, M, K, generator=g, dtype=torch.float64)
    B = torch.randn(1, K, N, generator=g, dtype=torch.float64)
    dt = torch.float64
    sa, sb = A.transpose(1, 2) if ta else A, B.transpose(1, 2) if tb else B
    lda, ldb = sa.shape[2] + 1, sb.shape[2] + 1
    Ab, sA, _ = embed(sa, lda, 1, dt)
    Bb, sB, _ = embed(sb, ldb, 1, dt)
    with engine.accumulation("dd"):
        Db, sD, D = embed(torch.full((1, M, N), float("nan")), N + 1, 1, dt)
        engine.gemm(ta, tb, M, N, K, Ab, lda, sA, Bb, ldb, sB, Db, N + 1, sD, 1, 1.0, 0.0, None, 0, 0, a_off=1,
                    b_off=1, d_off=1)
        for m in range(0, min(M, 200), 40):
            h = min(40, M - m)
            P = torch.empty(h, N, dtype=dt, device="cuda")
            engine.gemm(ta, tb, h, N, K, Ab, lda, sA, Bb, ldb, sB, P, N, 0, 1, 1.0, 0.0, None, 0, 0,
                        a_off=1 + (m if ta else m * lda), b_off=1)
            assert torch.equal(P, D[0, m : m + h])
    assert normwise(D.cpu(), torch.bmm(A, B)) <= TOL[dt]
    assert int(torch.isnan(Db).sum()) == Db.numel() - M * N


# fp32 sizes whose grids take the 64 x 64, the pipelined 64 x 128 and the
# pipelined 128 x 128 tile, ragged in both extents and in K (also K below one
# stage, whole stages, and one element over).
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N", [(2061, 2051), (1999, 3001), (4001, 4003), (2048, 3072), (4096, 3968)])
@pytest.mark.parametrize("K", [31, 64, 65])
def test_gemm_f32_wide_tiles(hip, ta, tb, M, N, K):
    """Against float64 torch on the device, with C and alpha/beta, operands
    and D in NaN buffers; and bitwise against the last rows computed in a
    product of 40 rows (the 32 x 32 tiles)."""
    from trntensor_amd.hip import engine

    dt = torch.float32
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(1, M, K, generator=g, dtype=torch.float64, device="cuda").to(dt)
    B = torch.randn(1, K, N, generator=g, dtype=torch.float64, device="cuda").to(dt)
    C = torch.randn(1, M, N, generator=g, dtype=torch.float64, device="cuda").to(dt)
    sa, sb = A.transpose(1, 2) if ta else A, B.transpose(1, 2) if tb else B
    pad = M % 2  # aligned for the whole-tile shapes
    lda, ldb = sa.shape[2] + pad, sb.shape[2] + pad
    Ab, sA, _ = embed(sa, lda, pad, dt)
    Bb, sB, _ = embed(sb, ldb, pad, dt)
    Cb, sC, _ = embed(C, N + pad, pad, dt)
    Db, sD, D = embed(torch.full((1, M, N), float("nan")), N + pad, pad, dt)
    engine.gemm(ta, tb, M, N, K, Ab, lda, sA, Bb, ldb, sB, Db, N + pad, sD, 1, 1.5, 0.5, Cb[pad:], N + pad, sC,
                a_off=pad, b_off=pad, d_off=pad)
    ref = 1.5 * torch.matmul(A[0].double(), B[0].double()) + 0.5 * C[0].double()
    assert float((D[0].double() - ref).abs().max() / ref.abs().max()) <= TOL[dt]
    assert int(torch.isnan(Db).sum()) == Db.numel() - M * N
    m = M - 40
    P = torch.empty(40, N, dtype=dt, device="cuda")
    engine.gemm(ta, tb, 40, N, K, Ab, lda, sA, Bb, ldb, sB, P, N, 0, 1, 1.5, 0.5, C[0, m:], N, 0,
                a_off=pad + (m if ta else m * lda), b_off=pad)
    assert torch.equal(P, D[0, m:])


# fp64 sizes whose grids take 32-, 48- and 64-row direct-B tiles, ragged in the
# columns (odd: a lane's column pair straddles the edge) and in K.
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N", [(21, 60001), (17, 60030), (40, 60001), (47, 60033), (61, 60001), (150, 20003), (1000, 3001)])
@pytest.mark.parametrize("K,with_c", [(15, True), (33, False), (64, True)])
def test_gemm_f64_row_tiles(hip, ta, tb, M, N, K, with_c):
    """Against float64 torch on the device, operands and D in NaN buffers, and
    bitwise against the last columns computed in a product of 40 columns (the
    32 x 32 tiles)."""
    from trntensor_amd.hip import engine

    dt = torch.float64
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(1, M, K, generator=g, dtype=dt, device="cuda")
    B = torch.randn(1, K, N, generator=g, dtype=dt, device="cuda")
    C = torch.randn(1, M, N, generator=g, dtype=dt, device="cuda") if with_c else None
    sa, sb = A.transpose(1, 2) if ta else A, B.transpose(1, 2) if tb else B
    lda, ldb = sa.shape[2] + 1, sb.shape[2] + 1
    Ab, sA, _ = embed(sa, lda, 1, dt)
    Bb, sB, _ = embed(sb, ldb, 1, dt)
    Cb, sC, _ = embed(C, N + 1, 1, dt) if with_c else (None, 0, None)
    Db, sD, D = embed(torch.full((1, M, N), float("nan")), N + 1, 1, dt)
    beta = 0.5 if with_c else 0.0
    engine.gemm(ta, tb, M, N, K, Ab, lda, sA, Bb, ldb, sB, Db, N + 1, sD, 1, 1.5, beta, Cb[1:] if with_c else None,
                N + 1, sC, a_off=1, b_off=1, d_off=1)
    ref = 1.5 * torch.matmul(A[0], B[0]) + (0.5 * C[0] if with_c else 0.0)
    assert float((D[0] - ref).abs().max() / ref.abs().max()) <= TOL[dt]
    assert int(torch.isnan(Db).sum()) == Db.numel() - M * N
    n = N - 40
    P = torch.empty(M, 40, dtype=dt, device="cuda")
    Cp = C[0, :, n:].contiguous() if with_c else None
    engine.gemm(ta, tb, M, 40, K, Ab, lda, sA, Bb, ldb, sB, P, 40, 0, 1, 1.5, beta, Cp, 40, 0, a_off=1,
                b_off=1 + (n * ldb if tb else n))
    assert torch.equal(P, D[0, :, n:])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(33, 65, 63), (31, 129, 64), (1, 70, 40), (70, 1, 33), (7, 9, 130), (65, 63, 128),
                                   (700, 900, 65), (2001, 1999, 33), (130, 7, 1), (520, 4100, 70)])
def test_gemm16_unaligned_ragged(hip, dt, ta, tb, M, N, K):
    """16-bit operands of any alignment in NaN buffers. Products and sums in
    fp32, one rounding per output: half an ulp of the type plus the fp32 sum
    bound K 2^-24 on sum |a b|."""
    from trntensor_amd.hip import engine

    g = torch.Generator(device="cuda").manual_seed(M * 3 + N + K)
    for pad, with_c in ((1, True), (0, False), (3, False)):
        A = torch.randn(1, M, K, generator=g, device="cuda").to(dt)
        B = torch.randn(1, K, N, generator=g, device="cuda").to(dt)
        C = torch.randn(1, M, N, generator=g, device="cuda").to(dt)
        sa, sb = A.transpose(1, 2) if ta else A, B.transpose(1, 2) if tb else B
        lda, ldb = sa.shape[2] + pad, sb.shape[2] + pad
        Ab, sA, _ = embed(sa, lda, pad, dt)
        Bb, sB, _ = embed(sb, ldb, pad, dt)
        Cb, sC, _ = embed(C, N + pad, pad, dt)
        Db, sD, D = embed(torch.full((1, M, N), float("nan")), N + pad, pad, dt)
        engine.gemm(ta, tb, M, N, K, Ab, lda, sA, Bb, ldb, sB, Db, N + pad, sD, 1, 1.5, 0.5 if with_c else 0.0,
                    Cb[pad:] if with_c else None, N + pad, sC, a_off=pad, b_off=pad, d_off=pad)
        a, b = A[0].double(), B[0].double()
        ref = 1.5 * (a @ b) + (0.5 * C[0].double() if with_c else 0.0)
        mag = 1.5 * (a.abs() @ b.abs()) + (0.5 * C[0].double().abs() if with_c else 0.0)
        ulp = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
        err = (D[0].double() - ref).abs()
        assert bool((err <= ulp * ref.abs() + (K + 3) * 2.0 ** -24 * mag + 1e-7).all()), (pad, err.max().item())
        assert int(torch.isnan(Db).sum()) == Db.numel() - M * N


@pytest.mark.parametrize("kind,batch,M,N", [("f32", 2**23 + 5, 33, 1), ("f64", 2**23 + 5, 33, 1),
                                            ("dd", 2**23 + 5, 17, 1), ("bf16", 2**23 + 5, 33, 1),
                                            ("f64", 1, 2**29 + 40, 1), ("f32", 1, 1, 2**29 + 40)])
def test_gemm_more_tiles_than_a_grid(hip, kind, batch, M, N):
    """2^24 small tiles and more do not fit one launch: larger tiles or
    several launches take them. K = 1, so every output is one rounded product
    (the double-double sum included) and equals torch's."""
    import contextlib

    from trntensor_amd.hip import engine

    dt = {"f32": torch.float32, "bf16": torch.bfloat16}.get(kind, torch.float64)
    g = torch.Generator(device="cuda").manual_seed(batch + M)
    A = torch.randn(batch, M, 1, generator=g, dtype=torch.float32, device="cuda").to(dt)
    B = torch.randn(batch, 1, N, generator=g, dtype=torch.float32, device="cuda").to(dt)
    D = torch.full((batch, M, N), float("nan"), dtype=dt, device="cuda")
    with engine.accumulation("dd") if kind == "dd" else contextlib.nullcontext():
        # A one-row matrix is passed as its transpose (leading dimension M = 1).
        ta = M == 1
        engine.gemm(ta, False, M, N, 1, A, M if ta else 1, M, B, N, N, D, N, M * N, batch, 1.0, 0.0, None, 0, 0)
    assert torch.equal(D, A * B)


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("batch,M,N", [(2**24 + 5, 1, 1), (2**24 + 5, 1, 2), (1, 2**20 + 1, 2**18 + 1)])
def test_gemm_dot_more_tiles_than_a_grid(hip, dt, batch, M, N):
    """A dot of 2^24 tiles and more runs as several launches, each writing its
    own partials. K = 1 and small whole numbers: every partial and their sum
    (below 2^53, in double) are exact, so the result equals the closed form
    sum_b e_b (sum_m a_bm)(sum_n b_bn), rounded once to the data type. E is
    one value per batch entry, broadcast over rows and columns (stride 0)."""
    from trntensor_amd.hip import engine

    g = torch.Generator(device="cuda").manual_seed(batch + M + N)
    A, B, E = (torch.randint(1, 4, s, generator=g, device="cuda").to(dt) for s in ((batch, M), (batch, N), (batch,)))
    out = torch.full((), float("nan"), dtype=dt, device="cuda")
    engine.gemm_dot(False, False, M, N, 1, A, 1, M, B, N, N, batch, M, N, E, [0, 0, 0, 0, 1], None, None, 1.0, 0.0,
                    None, out)
    want = (E.double() * A.double().sum(1) * B.double().sum(1)).sum()
    assert float(out) == float(want.to(dt)), (float(out), float(want))


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K,batch", [(3701, 1179, 3, 1), (193, 161, 16, 150), (42, 50003, 13, 1),
                                         (90007, 5, 5, 1), (70001, 36, 1, 1), (243, 17, 15, 400),
                                         (61, 97, 104, 700), (67, 255, 128, 200), (130, 63, 17, 300)])
def test_gemm_f32_short_k(hip, ta, tb, M, N, K, batch):
    """Sums of at most 16 terms, for which wide tiles take the well-filled
    grids, and the tiles up to K = 128: against float64 torch, operands and D in
    NaN buffers, and bitwise against the last row computed by itself (32 x 32
    tiles)."""
    from trntensor_amd.hip import engine

    dt = torch.float32
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(batch, M, K, generator=g, dtype=torch.float64, device="cuda").to(dt)
    B = torch.randn(batch, K, N, generator=g, dtype=torch.float64, device="cuda").to(dt)
    sa, sb = A.transpose(1, 2) if ta else A, B.transpose(1, 2) if tb else B
    lda, ldb = sa.shape[2] + 1, sb.shape[2] + 1
    Ab, sA, _ = embed(sa, lda, 1, dt)
    Bb, sB, _ = embed(sb, ldb, 1, dt)
    C = torch.randn(batch, M, N, generator=g, dtype=torch.float64, device="cuda").to(dt)
    for with_c in (False, True):
        Db, sD, D = embed(torch.full((batch, M, N), float("nan")), N + 1, 1, dt)
        engine.gemm(ta, tb, M, N, K, Ab, lda, sA, Bb, ldb, sB, Db, N + 1, sD, batch, 1.5, 0.5 if with_c else 0.0,
                    C if with_c else None, N, M * N, a_off=1, b_off=1, d_off=1)
        ref = 1.5 * torch.bmm(A.double(), B.double()) + (0.5 * C.double() if with_c else 0.0)
        assert float((D.double() - ref).abs().max() / ref.abs().max()) <= TOL[dt]
        assert int(torch.isnan(Db).sum()) == Db.numel() - batch * M * N
        P = torch.empty(batch, 1, N, dtype=dt, device="cuda")
        engine.gemm(ta, tb, 1, N, K, Ab, lda, sA, Bb, ldb, sB, P, N, N, batch, 1.5, 0.5 if with_c else 0.0,
                    C[:, M - 1] if with_c else None, N, M * N, a_off=1 + (M - 1 if ta else (M - 1) * lda), b_off=1)
        assert torch.equal(P[:, 0], D[:, M - 1])
