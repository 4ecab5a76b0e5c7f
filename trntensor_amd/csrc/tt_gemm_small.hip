// fp32/fp64 GEMM on 32 x 32 tiles for grids too small to fill the chip with
// the wide tiles (tt_gemm; any layout, extent, alignment, batch).
//
// What bounds these launches is not the MFMA rate but the number of
// workgroups and the serial chain of stages in each (load, LDS store, barrier,
// fragment reads, 16 dependent MFMAs). So: 32 x 32 outputs per workgroup (four
// waves of one 16 x 16 MFMA block) and stages of 64 k, or 128 where one such
// stage holds all of K and the launch makes a single memory round trip; LDS
// single-buffered (17-37 KB: four and more workgroups per CU where the grid
// has that many), the next stage in flight in registers behind the MFMAs. The
// k order per output is that of every other kernel here (16-deep passes; MFMA
// step s gives lane group g the k index 16 t + 4 g + s): results are bitwise
// equal. Against the wide tiles, same box, us: fp64 21 x 150 x 150 x 555 NT
// 43.7 -> 24.2, 500^3 38.0 -> 12.3, 300 x 310 x 320 25 -> 8, 1000^3 73 -> 51;
// fp32 500^3 27.0 -> 10.1, 1000^3 54 -> 31, 12 x 200 x 200 x 1000 46 -> 21,
// 150 x 2000 x 3000 170 -> 55. Measured and left: two stages in flight in
// registers (5% slower; 47 us on the last shape), two LDS buffers and one
// barrier per stage (equal on one workgroup per CU, 5-15% slower on more),
// fragments loaded from memory straight into the MFMA registers without LDS
// (1.1-2.4x the time from 500^3 up), 32 x 64 tiles (5-45% slower below 128
// wide tiles).
#include "tt_gemm.hpp"
#include "tt_stage.hpp"

namespace tt {

namespace {

constexpr int kSmall = 32;    // tile rows and columns

// FULL: M and N are multiples of 32 (no row or column clamping).
template <typename T, bool TA, bool TB, bool FULL, int BK>
__global__ __launch_bounds__(kThreads) void gemm_small_kernel(GemmArgs g) {
    typedef Mfma<T> MF;
    typedef typename MF::acc_t acc_t;
    typedef Stage<T, kSmall, !TA, BK> SA;
    typedef Stage<T, kSmall, TB, BK> SB;
    __shared__ __attribute__((aligned(16))) T lds[SA::ELEMS + SB::ELEMS];
    T* const la = lds;
    T* const lb = lds + SA::ELEMS;

    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t id = xcd_remap(blockIdx.x, tiles * g.batch);
    const int64_t bat = id / tiles;
    const int64_t t = id - bat * tiles;
    // Grouped order: 8 tile-rows sweep each tile-column.
    constexpr int64_t GROUP = 8;
    const int64_t grp = t / (GROUP * g.tiles_n);
    const int64_t first_m = grp * GROUP;
    const int64_t gsize = min(g.tiles_m - first_m, GROUP);
    const int64_t rem = t - grp * GROUP * g.tiles_n;
    const int64_t m0 = (first_m + rem % gsize) * kSmall;
    const int64_t n0 = (rem / gsize) * kSmall;
    const T* A = static_cast<const T*>(g.A) + bat * g.sA;
    const T* B = static_cast<const T*>(g.B) + bat * g.sB;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm0 = (wave >> 1) * 16;
    const int wn0 = (wave & 1) * 16;

    acc_t acc = acc_t{0, 0, 0, 0};
    SA sa;
    SB sb;
    const int64_t nk = (g.K + BK - 1) / BK;
    // Stages 0 .. nfull-1 have all their k in range (a row-contiguous operand
    // with fewer rows than one vector takes the guarded loads throughout).
    const int64_t nfull = (!TA || g.M >= Vec16<T>::n) && (TB || g.N >= Vec16<T>::n) ? g.K / BK : 0;
    const bool edge_m = TA && !FULL && m0 + kSmall > g.M, edge_n = !TB && !FULL && n0 + kSmall > g.N;
    auto load = [&](int64_t s) __attribute__((always_inline)) {
        sa.template load<FULL>(A, g.lda, m0, g.M, s * BK);
        sb.template load<FULL>(B, g.ldb, n0, g.N, s * BK);
    };
    auto load_tail = [&](int64_t s) __attribute__((always_inline)) {
        sa.load_tail(A, g.lda, m0, g.M, s * BK, g.K);
        sb.load_tail(B, g.ldb, n0, g.N, s * BK, g.K);
    };
    auto store = [&]() __attribute__((always_inline)) {
        sa.store(la);
        sb.store(lb);
    };
    // Pieces that were clamped at the matrix edge (uniform: edge tiles only).
    auto align = [&]() __attribute__((always_inline)) {
        if (edge_m) sa.align(m0, g.M);
        if (edge_n) sb.align(n0, g.N);
    };
    auto pass = [&](int kk) __attribute__((always_inline)) {
        T fa[4], fb[4];
        SA::frag(la, wm0, lane, kk, fa);
        SB::frag(lb, wn0, lane, kk, fb);
#pragma unroll
        for (int st = 0; st < 4; ++st) acc = MF::mma(fa[st], fb[st], acc);
    };

    if (nfull > 0) {
        load(0);
        align();
        store();
    } else if (nk > 0) {
        load_tail(0);
        store();
    }
    __syncthreads();
    // The scheduling barrier keeps the LDS stores (and the wait for their
    // loads) behind this stage's MFMAs.
    auto compute = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) pass(kk);
        __builtin_amdgcn_sched_barrier(0);
    };
    int64_t kt = 0;
    for (; kt + 1 < nfull; ++kt) {
        load(kt + 1);
        compute();
        align();
        __syncthreads();
        store();
        __syncthreads();
    }
    for (; kt + 1 < nk; ++kt) {
        load_tail(kt + 1);
        compute();
        __syncthreads();
        store();
        __syncthreads();
    }
    // The last stage: only the 16-k passes that K reaches.
    if (nk > 0) {
        const int left = (int)(g.K - (nk - 1) * BK);
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk)
            if (16 * kk < left) pass(kk);
    }

    // D = alpha * acc (+ beta * C); D may alias C element for element, so the
    // lane's C values are loaded (clamped, branch-free) before its stores.
    const T alpha = (T)g.alpha;
    const T beta = (T)g.beta;
    const T* C = g.C ? static_cast<const T*>(g.C) + bat * g.sC : nullptr;
    T* D = static_cast<T*>(g.D) + bat * g.sD;
    const int64_t col = n0 + wn0 + (lane & 15);
    T cv[4];
    if (C) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = m0 + wm0 + MF::row(lane >> 4, r);
            cv[r] = C[row < g.M && col < g.N ? row * g.ldc + col : 0];
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int64_t row = m0 + wm0 + MF::row(lane >> 4, r);
        if (row < g.M && col < g.N) {
            T v = acc[r];
            if (g.alpha != 1.0) v = alpha * v;
            if (C) v = v + beta * cv[r];
            D[row * g.ldd + col] = v;
        }
    }
}

template <typename T>
int launch(bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    g.tiles_m = (g.M + kSmall - 1) / kSmall;
    g.tiles_n = (g.N + kSmall - 1) / kSmall;
    const int64_t total = g.tiles_m * g.tiles_n * g.batch;
    if (total > 0x7fffffffLL) return set_error(TT_UNSUPPORTED, "tt_gemm: %lld tiles exceed one launch", (long long)total);
    if (total > kMaxGrid) {
        GemmArgs lo = g, hi = g;
        split_gemm(sizeof(T), ta, tb, kSmall, lo, hi);
        const int rc = launch<T>(ta, tb, lo, st);
        return rc == TT_OK ? launch<T>(ta, tb, hi, st) : rc;
    }
    // One 128-deep fp32 stage holds K <= 128 (fp64: 64, as any stage).
    const bool deep = sizeof(T) == 4 && g.K > 64 && g.K <= 128;
    const bool full = g.M % kSmall == 0 && g.N % kSmall == 0;
    const dim3 grid((unsigned)total), block(kThreads);
#define TT_SMALL_CASE(TA, TB, F)                                                                          \
    if (ta == TA && tb == TB && full == F) {                                                              \
        if constexpr (sizeof(T) == 4)                                                                     \
            if (deep) hipLaunchKernelGGL((gemm_small_kernel<T, TA, TB, F, 128>), grid, block, 0, st, g);  \
        if (!deep) hipLaunchKernelGGL((gemm_small_kernel<T, TA, TB, F, 64>), grid, block, 0, st, g);      \
    }
    TT_SMALL_CASE(false, false, false)
    TT_SMALL_CASE(false, true, false)
    TT_SMALL_CASE(true, false, false)
    TT_SMALL_CASE(true, true, false)
    TT_SMALL_CASE(false, false, true)
    TT_SMALL_CASE(false, true, true)
    TT_SMALL_CASE(true, false, true)
    TT_SMALL_CASE(true, true, true)
#undef TT_SMALL_CASE
    return check_launch("tt_gemm");
}

}  // namespace

int gemm_small_launch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    return dtype == TT_F64 ? launch<double>(ta, tb, g, st) : launch<float>(ta, tb, g, st);
}

}  // namespace tt
