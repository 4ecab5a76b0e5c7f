// Host-side interface of the MFMA GEMM core shared by the C-ABI sources.
#pragma once

#include "tt_common.hpp"

namespace tt {

struct GemmArgs {
    const void* A;
    const void* B;
    const void* C;
    void* D;
    int64_t M, N, K;
    int64_t lda, ldb, ldc, ldd;
    int64_t sA, sB, sC, sD;
    int64_t batch;
    int64_t tiles_m, tiles_n;
    double alpha, beta;
    // Dot epilogue: instead of storing D, each workgroup writes
    // sum_{m,n} D[m,n] * E(m,n) to partial[first + workgroup], with
    // E(m,n) = E1[off1] * (E2 ? E2[off2] : 1), off = m_hi*s[0] + m_lo*s[1] +
    // n_hi*s[2] + n_lo*s[3] + batch*s[4], (m_hi, m_lo) = divmod(m, mdiv.d),
    // (n_hi, n_lo) = divmod(n, ndiv.d).
    const void* E1;
    const void* E2;
    int64_t e1s[5], e2s[5];
    FastDiv mdiv, ndiv;
    double* partial;
    int64_t first;  // first tile of this launch (dot epilogue)
};

// A product with more tiles than a launch may have workgroups runs as two,
// lo and hi (both copies of it): halves of the batch, or of the longer side,
// at a multiple of `unit` rows or columns.
inline void split_gemm(size_t elem, bool ta, bool tb, int64_t unit, GemmArgs& lo, GemmArgs& hi) {
    const GemmArgs g = lo;
    const int64_t tm = (g.M + unit - 1) / unit, tn = (g.N + unit - 1) / unit;
    int64_t a = 0, b = 0, c = 0, d = 0;
    if (g.batch > 1) {
        lo.batch = g.batch / 2;
        hi.batch = g.batch - lo.batch;
        a = lo.batch * g.sA, b = lo.batch * g.sB, c = lo.batch * g.sC, d = lo.batch * g.sD;
    } else if (tm >= tn) {
        lo.M = tm / 2 * unit;
        hi.M = g.M - lo.M;
        a = ta ? lo.M : lo.M * g.lda, c = lo.M * g.ldc, d = lo.M * g.ldd;
    } else {
        lo.N = tn / 2 * unit;
        hi.N = g.N - lo.N;
        b = tb ? lo.N * g.ldb : lo.N, c = lo.N, d = lo.N;
    }
    auto at = [&](const void* p, int64_t n) { return p ? static_cast<const char*>(p) + n * (int64_t)elem : nullptr; };
    hi.A = at(g.A, a);
    hi.B = at(g.B, b);
    hi.C = at(g.C, c);
    hi.D = static_cast<char*>(g.D) + d * (int64_t)elem;
}

// Compute units of the current device (cached per device).
int device_cus();
// tt_gemm after argument checks (store epilogue).
int gemm_dispatch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st);
// Double-double GEMM (dtype TT_F64_DD) on the vector ALUs; same arguments.
int gemm_dd_dispatch(bool ta, bool tb, GemmArgs& g, hipStream_t st);
// 16-bit GEMM (dtype TT_BF16 / TT_F16) on the 16x16x32 MFMA; same arguments.
int gemm16_dispatch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st);
// Its direct-load variant: 16-byte aligned operands (A, B, lda, ldb and
// batch strides multiples of 8 elements), whole tiles of gemm16_dma_tile,
// K a multiple of 32. gemm16_dma_rows: the tile height for a layout and K.
int gemm16_dma_dispatch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st);
int gemm16_dma_rows(bool ta, bool tb, int64_t K);
// Its tile (bm x bn) for an M x N x K problem of `batch` products.
void gemm16_dma_tile(bool ta, bool tb, int64_t M, int64_t N, int64_t K, int64_t batch, int& bm, int& bn);
// fp32/fp64 on 32 x 32 tiles (tt_gemm_small.hip): any problem.
int gemm_small_launch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st);
// fp32 on pipelined 128 x 128 (tall) or 64 x 128 tiles (tt_gemm_mid.hip): K >= 1,
// and M >= 4 with A transposed, N >= 4 with B not transposed.
int gemm_mid_f32_launch(bool ta, bool tb, bool tall, GemmArgs& g, hipStream_t st);
// fp32 on 256 x 256 tiles (tt_gemm_big.hip): whether it takes the problem,
// and its launch.
bool gemm_big_f32_fits(bool ta, bool tb, const GemmArgs& g);
int gemm_big_f32_launch(GemmArgs& g, hipStream_t st);
// Dot epilogue; writes one double per workgroup to g.partial and returns the
// number of workgroups in *nparts.
int gemm_dot_dispatch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st, int64_t* nparts);

}  // namespace tt
