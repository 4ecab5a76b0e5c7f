// Double-double GEMM on the vector ALUs: the kernel behind precision="dd".
//   D[b][m, n] = alpha * dd_sum_k op(A)[m, k] op(B)[k, n]  (+ beta * C[b][m, n])
// Each product is formed exactly (TwoProduct) and summed into a (p, s) pair
// per output (Dot2, see tt_common.hpp), so an output is the dot product
// accumulated in about twice double precision and rounded to double once.
//
// Tile: 16 RM x 16 RN outputs per 256-thread workgroup, RM x RN per thread
// (rows RM ty + i, columns RN tx + j with tx = t % 16, ty = t / 16), K staged
// through LDS 16 at a time as As[k][m] and Bs[k][n], double-buffered with one
// barrier per stage. The work is VALU-bound
// (10 double-precision VALU operations per multiply-add; at 4 x 4 outputs per
// thread 2 LDS reads of 32 bytes per 16 multiply-adds), so the global loads
// are plain bounds-checked element loads: RM (RN) consecutive elements per
// thread along the operand's contiguous direction, the next stage prefetched
// into registers while the current one is computed. The order of an output's
// sums does not depend on the tile: results are bitwise equal.
#include "tt_gemm.hpp"

namespace tt {

namespace {

constexpr int kDdK = 16;

template <bool TA, bool TB, int RM, int RN>
__global__ __launch_bounds__(256) void gemm_dd_kernel(GemmArgs g) {
    constexpr int TM = 16 * RM, TN = 16 * RN;
    constexpr int UNR = RM * RN >= 16 ? 2 : 8;  // k unrolled as far as registers allow
    // Rows stay 32-byte aligned; k rows start on different banks.
    __shared__ __attribute__((aligned(32))) double As[2][kDdK][TM + 4];
    __shared__ __attribute__((aligned(32))) double Bs[2][kDdK][TN + 4];
    typedef typename VecN<double, RM>::type va_t;
    typedef typename VecN<double, RN>::type vb_t;
    const int t = threadIdx.x;
    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t w = blockIdx.x;
    const int64_t bat = w / tiles;
    const int64_t rem = w - bat * tiles;
    const int64_t tm = rem / g.tiles_n;
    const int64_t tn = rem - tm * g.tiles_n;
    const int64_t m0 = tm * TM, n0 = tn * TN;
    const double* A = static_cast<const double*>(g.A) + bat * g.sA;
    const double* B = static_cast<const double*>(g.B) + bat * g.sB;

    // op(A)[m, k] = TA ? A[k * lda + m] : A[m * lda + k]
    // op(B)[k, n] = TB ? B[n * ldb + k] : B[k * ldb + n]
    const int a_k = TA ? t / 16 : (t % (16 / RM)) * RM;
    const int a_m = TA ? (t % 16) * RM : t / (16 / RM);
    const int b_k = TB ? (t % (16 / RN)) * RN : t / 16;
    const int b_n = TB ? t / (16 / RN) : (t % 16) * RN;
    double ra[RM], rb[RN];

    auto load = [&](int64_t k0) {
#pragma unroll
        for (int e = 0; e < RM; ++e) {
            const int64_t m = m0 + a_m + (TA ? e : 0);
            const int64_t k = k0 + a_k + (TA ? 0 : e);
            const bool ok = m < g.M && k < g.K;
            const int64_t off = ok ? (TA ? k * g.lda + m : m * g.lda + k) : 0;
            const double v = A[off];
            ra[e] = ok ? v : 0.0;
        }
#pragma unroll
        for (int e = 0; e < RN; ++e) {
            const int64_t n = n0 + b_n + (TB ? 0 : e);
            const int64_t k = k0 + b_k + (TB ? e : 0);
            const bool ok = n < g.N && k < g.K;
            const int64_t off = ok ? (TB ? n * g.ldb + k : k * g.ldb + n) : 0;
            const double v = B[off];
            rb[e] = ok ? v : 0.0;
        }
    };
    auto stage = [&](int b) {
#pragma unroll
        for (int e = 0; e < RM; ++e) As[b][a_k + (TA ? 0 : e)][a_m + (TA ? e : 0)] = ra[e];
#pragma unroll
        for (int e = 0; e < RN; ++e) Bs[b][b_k + (TB ? e : 0)][b_n + (TB ? 0 : e)] = rb[e];
    };

    const int tx = t % 16, ty = t / 16;
    Dot2 acc[RM][RN];
    if (g.K > 0) {
        load(0);
        stage(0);
    }
    __syncthreads();
    int buf = 0;
    for (int64_t k0 = 0; k0 < g.K; k0 += kDdK) {
        const bool more = k0 + kDdK < g.K;
        if (more) load(k0 + kDdK);
#pragma unroll UNR
        for (int kk = 0; kk < kDdK; ++kk) {
            const va_t a = *reinterpret_cast<const va_t*>(&As[buf][kk][ty * RM]);
            const vb_t b = *reinterpret_cast<const vb_t*>(&Bs[buf][kk][tx * RN]);
#pragma unroll
            for (int i = 0; i < RM; ++i)
#pragma unroll
                for (int j = 0; j < RN; ++j) acc[i][j].add_prod(a[i], b[j]);
        }
        if (more) stage(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }

    double* D = static_cast<double*>(g.D) + bat * g.sD;
    const double* C = g.C ? static_cast<const double*>(g.C) + bat * g.sC : nullptr;
    // All C values are loaded (clamped addresses, branch-free) before the
    // first store: D may alias C, so loads placed between stores could not be
    // moved ahead of them and would each wait out a memory latency.
    double cv[RM][RN];
    if (C) {
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j) {
                const int64_t m = m0 + ty * RM + i, n = n0 + tx * RN + j;
                const bool ok = m < g.M && n < g.N;
                const double c = C[ok ? m * g.ldc + n : 0];
                cv[i][j] = ok ? c : 0.0;
            }
    }
#pragma unroll
    for (int i = 0; i < RM; ++i) {
        const int64_t m = m0 + ty * RM + i;
        if (m >= g.M) continue;
#pragma unroll
        for (int j = 0; j < RN; ++j) {
            const int64_t n = n0 + tx * RN + j;
            if (n >= g.N) continue;
            double v = acc[i][j].value();
            if (g.alpha != 1.0) v = g.alpha * v;
            if (C) v = v + g.beta * cv[i][j];
            D[m * g.ldd + n] = v;
        }
    }
}

template <int RM, int RN>
int launch_dd(bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    g.tiles_m = (g.M + 16 * RM - 1) / (16 * RM);
    g.tiles_n = (g.N + 16 * RN - 1) / (16 * RN);
    const int64_t total = g.tiles_m * g.tiles_n * g.batch;
    if (total > 0x7fffffffLL)
        return set_error(TT_UNSUPPORTED, "tt_gemm: %lld tiles exceed one launch", (long long)total);
    if (total > kMaxGrid) {
        GemmArgs lo = g, hi = g;
        split_gemm(sizeof(double), ta, tb, 64, lo, hi);
        const int rc = launch_dd<RM, RN>(ta, tb, lo, st);
        return rc == TT_OK ? launch_dd<RM, RN>(ta, tb, hi, st) : rc;
    }
    const dim3 grid((unsigned)total), block(256);
    if (!ta && !tb) hipLaunchKernelGGL((gemm_dd_kernel<false, false, RM, RN>), grid, block, 0, st, g);
    if (!ta && tb) hipLaunchKernelGGL((gemm_dd_kernel<false, true, RM, RN>), grid, block, 0, st, g);
    if (ta && !tb) hipLaunchKernelGGL((gemm_dd_kernel<true, false, RM, RN>), grid, block, 0, st, g);
    if (ta && tb) hipLaunchKernelGGL((gemm_dd_kernel<true, true, RM, RN>), grid, block, 0, st, g);
    return check_launch("tt_gemm (double-double)");
}

}  // namespace

int gemm_dd_dispatch(bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    // The tile with the least estimated time of the busiest CU: its tiles
    // times their outputs, times what a larger tile saves in LDS reads and
    // overhead per multiply-add (measured where every CU has many tiles, 2048^2
    // x 1024: 1.29, 1.32, 1.40, 1.48 ms at 4 x 4, 2 x 2, 1 x 2, 1 x 1 outputs
    // per thread), times what one or two workgroups on a CU lose because
    // nothing covers their latencies (1024^3: 0.422 ms at one 4 x 4 tile per
    // CU, 0.378 at four 2 x 2 tiles). us against 4 x 4 everywhere: 500 x 700 x
    // 900 164 against 377, 300^3 27 against 124, 97 x 643 x 1280 106 against
    // 514, 64^3 7 against 28, 900 x 1200 x 800 329 against 545, 1500^2 x 800
    // 604 against 768.
    const int64_t cus = device_cus();
    auto cost = [&](int64_t rm, int64_t rn, double per_mac) {
        const int64_t n = ((g.M + 16 * rm - 1) / (16 * rm)) * ((g.N + 16 * rn - 1) / (16 * rn)) * g.batch;
        const int64_t rounds = (n + cus - 1) / cus;
        return (double)rounds * rm * rn * per_mac * (rounds == 1 ? 1.25 : rounds == 2 ? 1.1 : 1.0);
    };
    const double c44 = cost(4, 4, 1.0), c22 = cost(2, 2, 1.03), c12 = cost(1, 2, 1.09), c11 = cost(1, 1, 1.16);
    if (c44 <= c22 && c44 <= c12 && c44 <= c11) return launch_dd<4, 4>(ta, tb, g, st);
    if (c22 <= c12 && c22 <= c11) return launch_dd<2, 2>(ta, tb, g, st);
    if (c12 <= c11) return launch_dd<1, 2>(ta, tb, g, st);
    return launch_dd<1, 1>(ta, tb, g, st);
}

}  // namespace tt
