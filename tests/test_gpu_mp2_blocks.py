"""DF-MP2 energy at the edges of the 64-row virtual blocks: every form a work
unit takes (full, at most 32 columns left, 16-row blocks within them), pair
counts on both sides of the unit order's group rule, any row alignment, and
the row-padded copy. Bars as in test_gpu_mp2 (relative 1e-10 fp64, 1e-5 fp32)."""

import pytest
import torch

import trntensor_amd as tt
from oracle import cpu_ref
from util import rel

pytestmark = pytest.mark.gpu
TOL = {torch.float64: 1e-10, torch.float32: 1e-5}


def inputs(nocc, nvir, naux, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    B = torch.randn(nocc, nvir, naux, generator=g, dtype=torch.float64) * 0.1
    eo = torch.sort(-20 + 19.7 * torch.rand(nocc, generator=g, dtype=torch.float64))[0]
    ev = torch.sort(0.1 + 4.9 * torch.rand(nvir, generator=g, dtype=torch.float64))[0]
    return B.to(dtype), eo.to(dtype), ev.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("nvir", [1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 80, 81, 96, 97, 128, 130, 150, 161])
def test_mp2_block_edges(hip, dtype, nvir):
    for nocc, naux in ((3, 37), (1, 16), (4, 5)):
        B, eo, ev = inputs(nocc, nvir, naux, dtype, nvir + naux)
        buf = torch.full((B.numel() + 2,), float("nan"), dtype=dtype, device="cuda")
        buf[1:-1] = B.reshape(-1).cuda()  # odd base address, NaN around
        got = tt.mp2_energy(buf[1:-1].view(nocc, nvir, naux), eo.cuda(), ev.cuda())
        assert rel(got, cpu_ref.mp2_energy(B.double(), eo.double(), ev.double())) <= TOL[dtype], (nocc, naux)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("nocc", [1, 7, 44, 45, 46])
def test_mp2_unit_order_covers_every_pair(hip, dtype, nocc):
    """44 occupied orbitals (990 pairs) are the last below 1024 pairs."""
    B, eo, ev = inputs(nocc, 70, 9, dtype, nocc)
    b, o, v = B.cuda(), eo.cuda(), ev.cuda()
    whole = tt.mp2_energy(b, o, v)
    assert rel(whole, cpu_ref.mp2_energy(B.double(), eo.double(), ev.double())) <= TOL[dtype]
    parts = sum(float(tt.mp2_energy_shard(b, o, v, r, 3)) for r in range(3))
    assert rel(parts, float(whole)) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("shape", [(70, 100, 33), (70, 99, 33), (110, 65, 17)])
def test_mp2_copy_rule(hip, dtype, shape):
    """Both sides of nocc * nvir = 7000: the full workspace (the row-padded
    copy is made from 7000 on) and the partials alone give one energy."""
    from trntensor_amd.hip import _lib, engine

    lib = _lib.load()
    nocc, nvir, naux = shape
    B, eo, ev = inputs(nocc, nvir, naux, dtype, sum(shape))
    b, o, v = B.cuda(), eo.cuda(), ev.cuda()
    code = engine.dtype_code(dtype)
    vals = []
    for n in (naux, (naux + 15) // 16 * 16):
        size = int(lib.tt_mp2_energy_workspace_bytes(code, nocc, nvir, n))
        ws = torch.full((size,), 255, dtype=torch.uint8, device="cuda")  # NaN bytes
        e = torch.full((), float("nan"), dtype=dtype, device="cuda")
        _lib.check(lib.tt_mp2_energy(code, nocc, nvir, naux, b.data_ptr(), o.data_ptr(), v.data_ptr(), e.data_ptr(),
                                     ws.data_ptr(), size, 1, engine._stream_ptr(b.device)), "tt_mp2_energy")
        vals.append(float(e))
    assert vals[0] == vals[1]
    assert rel(vals[0], cpu_ref.mp2_energy(B.double(), eo.double(), ev.double())) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("deterministic", [True, False])
def test_mp2_more_units_than_a_grid(hip, dtype, deterministic):
    """5793 occupied orbitals are 16782321 pairs, more workgroups than one
    launch may have: the units run as several launches. One virtual and one
    auxiliary function, so E = sum_ij (b_i b_j)^2 / (e_i + e_j - 2 e_a); the
    shards (each within one launch) sum to the same energy."""
    nocc = 5793
    B, eo, ev = (x.cuda() for x in inputs(nocc, 1, 1, dtype, 11))
    got = float(hip._hip_mp2_energy(B, eo, ev, deterministic=deterministic))
    b2, o = B.double().reshape(-1) ** 2, eo.double()
    want = float((b2[:, None] * b2[None, :] / (o[:, None] + o[None, :] - 2.0 * ev.double())).sum())
    assert rel(got, want) <= TOL[dtype]
    parts = sum(float(hip._hip_mp2_energy_shard(B, eo, ev, r, 3, deterministic=deterministic)) for r in range(3))
    assert rel(parts, want) <= TOL[dtype]
