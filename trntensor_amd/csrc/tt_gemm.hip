// MFMA GEMM core for gfx950: batched, strided, transposed operands in place,
// fused alpha/beta epilogue. fp64 on v_mfma_f64_16x16x4f64, fp32 on
// v_mfma_f32_16x16x4f32.
//
// Workgroup: 256 threads = 4 wavefronts, output tile BM x BN, each wavefront
// a 64x64 sub-tile (4 x 4 MFMA blocks, 64 accumulators per lane).
// K advances in stages of 16 through two LDS buffers: while the MFMAs consume
// one stage, the next stage's global loads are in flight in registers and are
// written to the other buffer afterwards (one barrier per stage).
//
// LDS layouts follow the operand's contiguous direction so every global load
// and LDS store is a 16-byte vector:
//   k-contiguous operand   -> [row][k],  row pitch 16 + 16 B of padding
//   row-contiguous operand -> [k][row],  k-row pitch ROWS + 16 B of padding
// Inside a 16-wide stage, MFMA step s (0..3) gives lane-group g = lane / 16
// the k index 4 g + s for both operands, so a lane's four k values are
// adjacent in the [row][k] layout and one 32-byte read feeds four MFMAs.
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "tt_gemm.hpp"
#include "tt_stage.hpp"

namespace tt {

// FULL: M and N are multiples of the tile (no row or column clamping).
template <typename T, int BM, int BN, int FM, int FN, bool TA, bool TB, bool FULL, bool DOT, int NBUF, int BK>
__global__ __launch_bounds__(kThreads) void gemm_kernel(GemmArgs g) {
    typedef Mfma<T> MF;
    typedef typename MF::acc_t acc_t;
    // A rows are m: k-contiguous unless transposed. B rows are n: k-contiguous iff transposed.
    typedef Stage<T, BM, !TA, BK> SA;
    typedef Stage<T, BN, TB, BK> SB;
    // Each wavefront owns an (16 FM) x (16 FN) sub-tile: FM x FN MFMA blocks.
    constexpr int WM = 16 * FM, WN = 16 * FN;
    constexpr int WAVES_N = BN / WN;
    static_assert((BM / WM) * WAVES_N == 4, "four wavefront tiles per workgroup");

    static_assert(NBUF == 1 || NBUF == 2, "stage buffers");
    __shared__ __attribute__((aligned(16))) T lds[NBUF * (SA::ELEMS + SB::ELEMS)];
    // Stage buffers: A0 (A1) B0 (B1).
    auto bufA = [&](int b) -> T* { return lds + b * SA::ELEMS; };
    auto bufB = [&](int b) -> T* { return lds + NBUF * SA::ELEMS + b * SB::ELEMS; };

    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t total = tiles * g.batch;
    const int64_t id = DOT ? g.first + xcd_remap(blockIdx.x, gridDim.x) : xcd_remap(blockIdx.x, total);
    const int64_t bat = id / tiles;
    int64_t t = id - bat * tiles;
    // Grouped order: 8 tile-rows sweep each tile-column, so concurrently
    // running workgroups share A panels and B panels.
    constexpr int64_t GROUP = 8;
    const int64_t grp = t / (GROUP * g.tiles_n);
    const int64_t first_m = grp * GROUP;
    const int64_t gsize = min(g.tiles_m - first_m, GROUP);
    const int64_t rem = t - grp * GROUP * g.tiles_n;
    const int64_t tm = first_m + rem % gsize;
    const int64_t tn = rem / gsize;
    const int64_t m0 = tm * BM;
    const int64_t n0 = tn * BN;

    const T* A = static_cast<const T*>(g.A) + bat * g.sA;
    const T* B = static_cast<const T*>(g.B) + bat * g.sB;

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm0 = (wave / WAVES_N) * WM;
    const int wn0 = (wave % WAVES_N) * WN;

    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

    SA sa;
    SB sb;
    // The dot's few wide tiles often lie mostly past a ragged edge, and loading
    // clamped pieces there costs more than the branch: us, fp32, loaded / skipped /
    // under the guards before the clamped loads: 12288 x 72 x 892 NN 60 / 51 / 53, TT
    // 59 / 49 / 54, 5352 x 128 x 1243 x 3 TN 87 / 71 / 82. Not with both operands
    // k-contiguous (4100 x 4001 x 512 NT 201 / 251 / 204, 2000 x 3000 x 1001 117 / 130).
    constexpr bool SKIP = DOT && !FULL && (TA || !TB);
    if constexpr (SKIP) {
        sa.clear();
        sb.clear();
    }
    const int64_t nk = (g.K + BK - 1) / BK;
    // Stages 0 .. nfull-1 have all their k in range (a row-contiguous operand
    // with fewer rows than one vector takes the guarded loads throughout).
    const int64_t nfull = (!TA || g.M >= Vec16<T>::n) && (TB || g.N >= Vec16<T>::n) ? g.K / BK : 0;
    // The lambdas below are always inlined: left as calls (which the inliner
    // chose for 64-deep stages), they capture acc by reference and the
    // accumulators go to scratch memory.
    auto load = [&](int64_t k0) __attribute__((always_inline)) {
        sa.template load<FULL, SKIP>(A, g.lda, m0, g.M, k0);
        sb.template load<FULL, SKIP>(B, g.ldb, n0, g.N, k0);
    };
    auto load_tail = [&](int64_t k0) __attribute__((always_inline)) {
        sa.load_tail(A, g.lda, m0, g.M, k0, g.K);
        sb.load_tail(B, g.ldb, n0, g.N, k0, g.K);
    };
    // Pieces that were clamped at the matrix edge (uniform: edge tiles only).
    const bool edge_m = TA && !FULL && m0 + BM > g.M, edge_n = !TB && !FULL && n0 + BN > g.N;
    auto store = [&](int b) __attribute__((always_inline)) {
        sa.store(bufA(b));
        sb.store(bufB(b));
    };
    auto align = [&]() __attribute__((always_inline)) {
        if (edge_m) sa.align(m0, g.M);
        if (edge_n) sb.align(n0, g.N);
    };
    // The stage's 16-k passes, of which the last, partial stage of a deep-stage
    // kernel runs only those that K reaches.
    auto compute = [&](int buf, int64_t left) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) {
            if (kk > 0 && 16 * kk >= left) break;
            T fa[FM][4], fb[FN][4];
#pragma unroll
            for (int i = 0; i < FM; ++i) SA::frag(bufA(buf), wm0 + 16 * i, lane, kk, fa[i]);
#pragma unroll
            for (int j = 0; j < FN; ++j) SB::frag(bufB(buf), wn0 + 16 * j, lane, kk, fb[j]);
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] = MF::mma(fa[i][st], fb[j][st], acc[i][j]);
        }
    };
    if (nk > 0) {
        if (nfull > 0) {
            load(0);
            align();
        } else {
            load_tail(0);
        }
        store(0);
    }
    __syncthreads();

    // The scheduling barrier keeps the prefetch's LDS stores (and the wait for
    // its global loads) behind this stage's MFMAs. With two buffers the next
    // stage goes to the other buffer (one barrier per stage); with one, it
    // replaces the current stage after a second barrier (half the LDS, so
    // more workgroups per CU).
    auto next = [&](int64_t kt) -> int { return NBUF == 2 ? (int)((kt & 1) ^ 1) : 0; };
    auto cur = [&](int64_t kt) -> int { return NBUF == 2 ? (int)(kt & 1) : 0; };
    int64_t kt = 0;
    for (; kt + 1 < nfull; ++kt) {
        load((kt + 1) * BK);
        compute(cur(kt), BK);
        __builtin_amdgcn_sched_barrier(0);
        align();
        if (NBUF == 1) __syncthreads();
        store(next(kt));
        __syncthreads();
    }
    for (; kt < nk; ++kt) {
        const bool more = kt + 1 < nk;
        if (more) load_tail((kt + 1) * BK);
        compute(cur(kt), g.K - kt * BK);
        __builtin_amdgcn_sched_barrier(0);
        if (NBUF == 1) __syncthreads();
        if (more) store(next(kt));
        __syncthreads();
    }

    const int col_l = lane & 15;
    const int lgrp = lane >> 4;
    if (DOT) {
        // Dot epilogue: sum of D .* E over this tile, one double per workgroup.
        __shared__ double red[4];
        const T* E1 = static_cast<const T*>(g.E1) + bat * g.e1s[4];
        const T* E2 = g.E2 ? static_cast<const T*>(g.E2) + bat * g.e2s[4] : nullptr;
        double sum = 0.0;
        // Each 16x16 block's eight E loads (branch-free: rows and columns
        // outside the matrix read element (0, 0)) go out together before
        // its sums, which keep the order below. Loaded under the
        // per-element bounds branches, every load waited out a full
        // latency before its sum: 128 waits per lane at 128 x 128, and
        // config 5's greedy path took 69.4 ms against 68.4 ms this way
        // (results bitwise equal).
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int64_t col = n0 + wn0 + 16 * j + col_l;
            const bool cok = col < g.N;
            const uint32_t nh = fdiv((uint32_t)(cok ? col : 0), g.ndiv);
            const uint32_t nl = (uint32_t)(cok ? col : 0) - nh * g.ndiv.d;
            const int64_t o1n = nh * g.e1s[2] + nl * g.e1s[3];
            const int64_t o2n = nh * g.e2s[2] + nl * g.e2s[3];
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                T e1v[4], e2v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + wm0 + 16 * i + MF::row(lgrp, r);
                    const bool ok = cok && row < g.M;
                    const uint32_t mh = fdiv((uint32_t)(ok ? row : 0), g.mdiv);
                    const uint32_t ml = (uint32_t)(ok ? row : 0) - mh * g.mdiv.d;
                    e1v[r] = E1[ok ? mh * g.e1s[0] + ml * g.e1s[1] + o1n : 0];
                    if (E2) e2v[r] = E2[ok ? mh * g.e2s[0] + ml * g.e2s[1] + o2n : 0];
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + wm0 + 16 * i + MF::row(lgrp, r);
                    if (cok && row < g.M) {
                        T e = e1v[r];
                        if (E2) e = e * e2v[r];
                        sum += (double)(acc[i][j][r] * e);
                    }
                }
            }
        }
        const double tot = block256_sum(sum, red);
        if (threadIdx.x == 0) g.partial[g.first + blockIdx.x] = tot;
        return;
    }

    // Store epilogue: D = alpha * acc (+ beta * C), masked at the matrix edge.
    // D may alias C, so the compiler cannot move a load of C past a store of
    // D: loaded element by element, every element would wait out a full
    // memory latency before its store. Each 16-row block's C values are
    // therefore loaded (from clamped addresses, branch-free) before any of
    // its stores, which keeps FN * 4 loads in flight together.
    const T alpha = (T)g.alpha;
    const T beta = (T)g.beta;
    const T* C = g.C ? static_cast<const T*>(g.C) + bat * g.sC : nullptr;
    T* D = static_cast<T*>(g.D) + bat * g.sD;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        T cv[FN][4];
        if (C) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int64_t col = n0 + wn0 + 16 * j + col_l;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + wm0 + 16 * i + MF::row(lgrp, r);
                    const bool ok = row < g.M && col < g.N;
                    const T c = C[ok ? row * g.ldc + col : 0];
                    cv[j][r] = ok ? c : T(0);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int64_t col = n0 + wn0 + 16 * j + col_l;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = m0 + wm0 + 16 * i + MF::row(lgrp, r);
                if (row < g.M && col < g.N) {
                    T v = acc[i][j][r];
                    if (g.alpha != 1.0) v = alpha * v;
                    if (C) v = v + beta * cv[j][r];
                    D[row * g.ldd + col] = v;
                }
            }
        }
    }
}

// Store epilogue of the direct-B kernels: D = alpha * acc (+ beta * C) for
// the 64 x BN tile at rows m0.., column tile tn of batch entry bat.
// acc[a][b][r] is row m0 + 16 a + MF::row(lg, r), column col + b; a lane's NB
// columns are one 16-byte piece of D and of C. The lane indices are formed
// again here rather than held through the K loop.
// PLAIN: no C and the tile inside N (the caller checked), so every row is one
// unconditional 16-byte store per lane.
template <typename T, bool FULLM, bool PLAIN = false, int FM = 4>
__device__ __forceinline__ void directb_store(const GemmArgs& g, typename Mfma<T>::acc_t (&acc)[FM][16 / sizeof(T)],
                                              int64_t bat, int64_t m0, int64_t tn) {
    typedef Mfma<T> MF;
    constexpr int NB = 16 / sizeof(T);
    constexpr int BN = 64 * NB;
    typedef typename VecN<T, 16 / sizeof(T)>::type v16_t;
    typedef typename Mem16<T>::type mem_t;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lg = (tid & 63) >> 4;
    const int64_t col = tn * BN + (tid >> 6) * (16 * NB) + NB * (tid & 15);
    const T alpha = (T)g.alpha;
    const T beta = (T)g.beta;
    T* D = static_cast<T*>(g.D) + bat * g.sD;
    if constexpr (PLAIN) {
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v16_t v;
#pragma unroll
                for (int b = 0; b < NB; ++b) v[b] = g.alpha != 1.0 ? alpha * acc[a][b][r] : acc[a][b][r];
                *reinterpret_cast<mem_t*>(D + (m0 + 16 * a + MF::row(lg, r)) * g.ldd + col) = v;
            }
        return;
    }
    const T* C = g.C ? static_cast<const T*>(g.C) + bat * g.sC : nullptr;
    const bool colok = col + NB <= g.N;  // all NB columns inside
    if (C) {
        // A lane's NB columns of a row are one 16-byte piece of C and of D.
        // The C pieces of two row blocks (eight rows) go out together before
        // their stores: two memory round trips per tile instead of four, and
        // one load per row instead of NB. D may alias C exactly: every row's
        // C piece is loaded before that row's store. Same box, alternating,
        // bitwise equal: 64 x 512^3 with alpha/beta and C 0.1362-0.1366
        // against 0.1429-0.1432 ms fp32, 0.2615-0.2618 against 0.2646-0.2661
        // ms fp64; 4096^3 fp32 0.993 against 0.999 ms.
#pragma unroll
        for (int a2 = 0; a2 < FM; a2 += 2) {
            constexpr int H = 2;
            v16_t cv[2][4];
#pragma unroll
            for (int h = 0; h < H && a2 + h < FM; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + 16 * (a2 + h) + MF::row(lg, r);
                    const bool ok = (FULLM || row < g.M) && colok;
                    cv[h][r] = *reinterpret_cast<const mem_t*>(C + (ok ? row * g.ldc + col : 0));
                }
#pragma unroll
            for (int h = 0; h < H && a2 + h < FM; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + 16 * (a2 + h) + MF::row(lg, r);
                    if ((!FULLM && row >= g.M) || !colok) continue;
                    v16_t v;
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        v[b] = acc[a2 + h][b][r];
                        if (g.alpha != 1.0) v[b] = alpha * v[b];
                        v[b] = v[b] + beta * cv[h][r][b];
                    }
                    *reinterpret_cast<mem_t*>(D + row * g.ldd + col) = v;
                }
        }
    } else {
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = m0 + 16 * a + MF::row(lg, r);
                if ((!FULLM && row >= g.M) || !colok) continue;
                v16_t v;
#pragma unroll
                for (int b = 0; b < NB; ++b) v[b] = g.alpha != 1.0 ? alpha * acc[a][b][r] : acc[a][b][r];
                *reinterpret_cast<mem_t*>(D + row * g.ldd + col) = v;
            }
    }
    if (g.N % NB) {
        // The lane whose NB columns straddle N computed columns N - NB ..
        // N - 1 (its B column was clamped): it stores those from col up.
        if (col < g.N && !colok) {
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + 16 * a + MF::row(lg, r);
#pragma unroll
                    for (int b = 1; b < NB; ++b) {
                        const int64_t cb = g.N - NB + b;
                        if (cb < col || (!FULLM && row >= g.M)) continue;
                        T v = acc[a][b][r];
                        if (g.alpha != 1.0) v = alpha * v;
                        if (C) v = v + beta * C[row * g.ldc + cb];
                        D[row * g.ldd + cb] = v;
                    }
                }
        }
    }
}

// GEMM (or dot epilogue, DOT): fp64 on 64 x 128 tiles, fp32 on 64 x 256 tiles,
// four waves each; N at least NB (below), the last column tile may be partial.
// A (either layout) is staged through LDS one 64-row slab per workgroup,
// double-buffered, one barrier per 16-k stage; rows from M up and k from K up
// read as zero. B goes from memory straight into the MFMA operand registers:
// wave w owns all 64 rows and 16 NB columns (NB = 16 bytes / element: 2 for
// fp64, 4 for fp32), and lane (g, c) feeds MFMA block b (0 .. NB - 1) with
// column n0 + 16 NB w + NB c + b, so one 16-byte load per k-row gives it every
// block's operand and B never passes through LDS. With B k-contiguous (TB)
// the lane's 16-byte piece is NB consecutive k of one column instead, and its
// four pieces cover its NB columns over the stage's 4 k. MFMA step s of stage t gives
// lane group g the k index 16 t + 4 g + s, the order of gemm_kernel, whose
// results it reproduces bitwise. 118-128 VGPRs: four waves per SIMD. NT: B is
// read once (M <= 64, e.g. the AO->MO half transform), so its loads bypass the
// caches. AO->MO half transform (64 x 786432 x 512) against the LDS-staged
// small-M tile: 0.877-0.883 against 0.893-0.900 ms on one box and 0.885-0.886
// against 0.913-0.915 ms on another, alternating; M < 64 (48 x 65536 x 256,
// four batches) measured the same.
template <typename T, bool FULLM, bool TA, bool TB, bool NT, bool DOT, int FM = 4>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void gemm_directb_kernel(GemmArgs g) {
    typedef Mfma<T> MF;
    typedef typename MF::acc_t acc_t;
    constexpr int NB = 16 / sizeof(T);  // MFMA column blocks per wave: one 16-byte B piece per lane
    constexpr int BN = 64 * NB;         // tile columns: 128 (fp64), 256 (fp32)
    constexpr int SPL = TB ? 16 / sizeof(T) : 1;  // MFMA steps one B load feeds (TB: k-contiguous piece)
    typedef typename VecN<T, 16 / sizeof(T)>::type v16_t;
    typedef typename Mem16<T>::type mem_t;
    typedef Stage<T, FM == 2 ? 32 : 64, !TA, kBK> SA;  // A: a slab of at least 16 FM rows, [k][m] (TA) or [m][k] in LDS
    __shared__ __attribute__((aligned(16))) T lds[2 * SA::ELEMS];

    // Tile order: the 64-row slabs of one column tile are adjacent (they
    // share its B panel in L2). With more than 64 row tiles, the rows go in
    // groups of 16 slabs that sweep every column tile before the next group,
    // so a group's A slabs stay cached instead of A streaming from HBM once
    // per column tile. Config 5's fused GEMM (2500 x 128 tiles, A 1 GB):
    // 60.36 and 60.01 against 60.92 and 61.10 ms on one box (groups of 32:
    // 60.28 and 60.31 ms; of 64: 60.83 and 60.98 ms).
    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t id = DOT ? g.first + xcd_remap(blockIdx.x, gridDim.x) : xcd_remap(blockIdx.x, tiles * g.batch);
    const int64_t bat = id / tiles;
    const int64_t rem = id - bat * tiles;
    constexpr int64_t kRowGroup = 16;
    int64_t tn, tm;
    if (g.tiles_m > 4 * kRowGroup) {
        const int64_t grp = rem / (kRowGroup * g.tiles_n);
        const int64_t gm = min(kRowGroup, g.tiles_m - grp * kRowGroup);  // row tiles in this group
        const int64_t r = rem - grp * kRowGroup * g.tiles_n;
        tn = r / gm;
        tm = grp * kRowGroup + r % gm;
    } else {
        tn = rem / g.tiles_m;
        tm = rem - tn * g.tiles_m;
    }
    const int64_t m0 = tm * (16 * FM);
    const T* A = static_cast<const T*>(g.A) + bat * g.sA;
    const int64_t nk = (g.K + kBK - 1) / kBK;
    const int64_t nfull = g.K / kBK;

    acc_t acc[FM][NB];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = acc_t{0, 0, 0, 0};
    if (nk > 0) {
        const int lane = threadIdx.x & 63;
        const int lg = lane >> 4;
        const int c = lane & 15;
        // The lane's first column, clamped into the matrix: in a last, partial
        // column tile the lanes that pass N read column N - NB instead; of
        // their results only the columns a lane straddling N owns are stored
        // (a column of D depends on that column of B only).
        const int64_t col0 = min(tn * BN + (threadIdx.x >> 6) * (16 * NB) + NB * c, g.N - NB);
        // B row-major: piece p (0..3) is k-row 16 t + 4 g + p, all NB columns.
        // B k-contiguous: piece p is column col0 + p % NB, k 16 t + 4 g +
        // SPL (p / NB) .. + SPL - 1 (MFMA steps SPL (p / NB) ..).
        const T* B = TB ? static_cast<const T*>(g.B) + bat * g.sB + col0 * g.ldb + 4 * lg
                        : static_cast<const T*>(g.B) + bat * g.sB + col0 + (int64_t)(4 * lg) * g.ldb;
        auto bptr = [&](int64_t t, int p) __attribute__((always_inline)) -> const T* {
            return TB ? B + (int64_t)(p % NB) * g.ldb + 16 * t + SPL * (p / NB) : B + (16 * t + p) * g.ldb;
        };
        SA sa;
        v16_t rb[4];  // B pieces of the current stage
        auto bload = [&](int64_t t, int p) __attribute__((always_inline)) {
            const mem_t* q = reinterpret_cast<const mem_t*>(bptr(t, p));
            rb[p] = NT ? __builtin_nontemporal_load(q) : *q;
        };
        // Stage t's B where it may pass K: k from K up reads as zero.
        auto bload_tail = [&](int64_t t, int p) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 16 / (int)sizeof(T); ++e) {
                const int64_t k = 16 * t + 4 * lg + (TB ? SPL * (p / NB) + e : p);
                const bool ok = k < g.K;
                const T* q = TB ? bptr(t, p) + e : bptr(t, p) + e;
                const T x = *(ok ? q : static_cast<const T*>(g.B));
                rb[p][e] = ok ? x : T(0);
            }
        };
        // A's stage t: interior, or (K % 16 left over) the last one.
        auto aload = [&](int64_t t) __attribute__((always_inline)) { sa.template load<FULLM>(A, g.lda, m0, g.M, t * kBK); };
        auto aload_tail = [&](int64_t t) __attribute__((always_inline)) { sa.load_tail(A, g.lda, m0, g.M, t * kBK, g.K); };
        const bool edge_m = TA && !FULLM && m0 + (FM == 2 ? 32 : 64) > g.M;  // clamped pieces (uniform)
        auto astore = [&](int64_t t) __attribute__((always_inline)) {
            if (edge_m && t < nfull) sa.align(m0, g.M);
            sa.store(lds + (t & 1) * SA::ELEMS);
        };
        auto afrag = [&](const T* sbuf, int a, int s) __attribute__((always_inline)) -> T {
            return TA ? sbuf[(4 * lg + s) * SA::PITCH + 16 * a + c] : sbuf[(16 * a + c) * SA::PITCH + 4 * lg + s];
        };
        // The MFMAs piece p feeds. Every accumulator still takes MFMA steps
        // 0, 1, 2, 3 in order.
        T fa[FM][SPL];
        auto piece = [&](const T* sbuf, int p) __attribute__((always_inline)) {
            if (!TB) {
#pragma unroll
                for (int a = 0; a < FM; ++a) fa[a][0] = afrag(sbuf, a, p);
#pragma unroll
                for (int a = 0; a < FM; ++a)
#pragma unroll
                    for (int b = 0; b < NB; ++b) acc[a][b] = MF::mma(fa[a][0], rb[p][b], acc[a][b]);
            } else {
                const int h = p / NB, b = p % NB;
                if (b == 0) {
#pragma unroll
                    for (int a = 0; a < FM; ++a)
#pragma unroll
                        for (int e = 0; e < SPL; ++e) fa[a][e] = afrag(sbuf, a, SPL * h + e);
                }
#pragma unroll
                for (int e = 0; e < SPL; ++e)
#pragma unroll
                    for (int a = 0; a < FM; ++a) acc[a][b] = MF::mma(fa[a][e], rb[p][e], acc[a][b]);
            }
        };
        // A wave whose columns all lie past N (in a last, partial column tile)
        // only helps stage A: the same loads, stores and barriers as the
        // loop below, no B loads and no MFMAs, so its SIMD's MFMA pipe serves
        // the other workgroups. Its accumulators stay zero and are never
        // stored. (With DOT such a wave computes along: its columns are left out
        // of the sum below, and skipping it was not measured there.) Config 5's
        // optimal-order step 'jb,abP->jaP' (N = 800): 0.828 against 0.830 and
        // 0.836 ms for the whole path, 12% fewer executed MFMA FLOP there.
        const int wave_u = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (!DOT && tn * BN + (int64_t)wave_u * (16 * NB) >= g.N) {
            for (int64_t t = 0; t < nk; ++t) {
                if (t < nfull) aload(t);
                else aload_tail(t);
                astore(t);
                __syncthreads();
            }
        } else {
        if (nfull > 0) aload(0);
        else aload_tail(0);
        astore(0);
        int64_t t = 0;
        // Only the vector loads of B lead into the main loop: with the
        // element-wise tail loads joining them there, the compiler's wait at
        // the top of each stage covered every outstanding load (same box,
        // alternating, bitwise equal: 4096^3 fp32 1.0135 against 1.0172 ms,
        // 64 x 512^3 with alpha/beta 0.1441 against 0.1456 ms fp32 and 0.2639
        // against 0.2669 ms fp64).
        if (nfull == 0) {
#pragma unroll
            for (int p = 0; p < 4; ++p) bload_tail(0, p);
            __syncthreads();
        } else {  // the main loop below is this branch's (closed after it)
#pragma unroll
            for (int p = 0; p < 4; ++p) bload(0, p);
            __syncthreads();
        for (; t + 1 < nfull; ++t) {
            // Stage t + 1 of A goes to the other buffer; B piece p is reloaded
            // for stage t + 1 as soon as its MFMAs have issued. With B
            // k-contiguous the fp64 wave issuing the MFMAs runs at raised
            // priority for the burst (0.4-0.5% faster); with B row-major the
            // default priority is faster (same box, alternating, bitwise
            // equal: AO->MO half transform 0.865 against 0.890 ms, 4096^3 1.883
            // against 1.924 ms, 64 x 512^3 with alpha/beta 0.266 against 0.275
            // ms, the transform's batched GEMM 0.479 against 0.511 ms).
            aload(t + 1);
            const T* cur = lds + (t & 1) * SA::ELEMS;
            if (sizeof(T) == 8 && TB) __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                piece(cur, p);
                bload(t + 1, p);
            }
            if (sizeof(T) == 8 && TB) __builtin_amdgcn_s_setprio(0);
            if constexpr (sizeof(T) == 4 && !TB) {
                // A's loads, then each piece's MFMAs followed by its
                // next-stage B load; left to itself the compiler issued the
                // four B loads together near the end of the stage (same box,
                // alternating, bitwise equal: 4096^3 1.0036 against 1.0135
                // ms, 64 x 512^3 with alpha/beta 0.1437 against 0.1441 ms; in
                // fp64 4096^3 measured 1% slower with it).
                __builtin_amdgcn_sched_group_barrier(0x020, SA::NC, 0);
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    __builtin_amdgcn_sched_group_barrier(0x008, FM * NB, 0);
                    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            astore(t + 1);
            __syncthreads();
        }
        }  // nfull > 0
        if (t + 1 < nk) {
            // The partial last stage (K not a multiple of 16).
            aload_tail(t + 1);
            const T* cur = lds + (t & 1) * SA::ELEMS;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                piece(cur, p);
                bload_tail(t + 1, p);
            }
            astore(t + 1);
            __syncthreads();
            ++t;
        }
        const T* cur = lds + (t & 1) * SA::ELEMS;
#pragma unroll
        for (int p = 0; p < 4; ++p) piece(cur, p);
        }  // live wave
    }

    if constexpr (DOT) {
        // acc[a][b][r] is row m0 + 16 a + MF::row(lg, r), column col + b. The
        // lane indices are formed again here rather than held through the K
        // loop.
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lg = (tid & 63) >> 4;
        const int64_t col = tn * BN + (tid >> 6) * (16 * NB) + NB * (tid & 15);
        // Dot epilogue: sum of D .* E over this tile, one double per
        // workgroup (see gemm_kernel's), in a fixed order: column blocks,
        // row blocks, then rows; each block's eight E loads go out together.
        __shared__ double red[4];
        const T* E1 = static_cast<const T*>(g.E1) + bat * g.e1s[4];
        const T* E2 = g.E2 ? static_cast<const T*>(g.E2) + bat * g.e2s[4] : nullptr;
        double sum = 0.0;
        // E2 present or not, the tile inside the matrix or not: straight-line
        // copies of the loop below. Row blocks outside, a block's E loads of
        // all columns in flight together (up to 16): four round trips to
        // memory per tile.
        auto dot = [&](auto has_e2, auto inside) __attribute__((always_inline)) {
            constexpr bool HE2 = decltype(has_e2)::value, IN = decltype(inside)::value;
            // In a partial last column tile a lane that passes N computed
            // columns N - NB .. N - 1; it owns those from col up.
            const int64_t cw = IN ? col : min(col, g.N - NB);
            int64_t o1n[NB], o2n[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const uint32_t cb = (uint32_t)(IN || cw + b >= col ? cw + b : 0);
                const uint32_t nh = fdiv(cb, g.ndiv);
                const uint32_t nl = cb - nh * g.ndiv.d;
                o1n[b] = nh * g.e1s[2] + nl * g.e1s[3];
                if (HE2) o2n[b] = nh * g.e2s[2] + nl * g.e2s[3];
            }
#pragma unroll
            for (int a = 0; a < FM; ++a) {
                T e1v[4][NB], e2v[4][NB];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + 16 * a + MF::row(lg, r);
                    const uint32_t rr = (uint32_t)(IN || row < g.M ? row : 0);
                    const uint32_t mh = fdiv(rr, g.mdiv);
                    const uint32_t ml = rr - mh * g.mdiv.d;
                    const int64_t o1m = mh * g.e1s[0] + ml * g.e1s[1];
                    const int64_t o2m = HE2 ? mh * g.e2s[0] + ml * g.e2s[1] : 0;
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        e1v[r][b] = E1[o1m + o1n[b]];
                        if (HE2) e2v[r][b] = E2[o2m + o2n[b]];
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + 16 * a + MF::row(lg, r);
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        if (IN || (row < g.M && cw + b >= col)) {
                            T e = e1v[r][b];
                            if (HE2) e = e * e2v[r][b];
                            sum += (double)(acc[a][b][r] * e);
                        }
                }
                // One block's loads in flight at a time.
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        const bool inside = m0 + 16 * FM <= g.M && (tn + 1) * BN <= g.N;
        if (inside) {
            if (E2) dot(std::true_type{}, std::true_type{});
            else dot(std::false_type{}, std::true_type{});
        } else {
            if (E2) dot(std::true_type{}, std::false_type{});
            else dot(std::false_type{}, std::false_type{});
        }
        const double tot = block256_sum(sum, red);
        if (tid == 0) g.partial[g.first + blockIdx.x] = tot;
        return;
    } else {
        directb_store<T, FULLM, false, FM>(g, acc, bat, m0, tn);
    }
}

// Persistent form of gemm_directb_kernel (store epilogue, no C, whole 64-row and BN-column tiles, K a positive multiple of 16): each workgroup walks a list of tiles
// and the stages of consecutive tiles form one software pipeline. The next
// tile's first stage (A slab into LDS, B pieces into registers) is loaded
// during the current tile's last MFMAs, and the current tile's stores are
// issued while those loads are in flight, so no workgroup waits out a
// memory latency between tiles. Hardware workgroup w runs on XCD w % 8; the
// tiles are split into eight contiguous ranges, one per XCD, and the
// workgroups of an XCD take that range's tiles round-robin. The MFMA order
// per accumulator is gemm_directb_kernel's: results are bitwise equal.
template <typename T, bool TA, bool TB, bool NT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void gemm_directb_persistent_kernel(
    GemmArgs g) {
    typedef Mfma<T> MF;
    typedef typename MF::acc_t acc_t;
    constexpr int NB = 16 / sizeof(T);
    constexpr int BN = 64 * NB;
    constexpr int SPL = TB ? 16 / sizeof(T) : 1;
    typedef typename VecN<T, 16 / sizeof(T)>::type v16_t;
    typedef typename Mem16<T>::type mem_t;
    typedef Stage<T, 64, !TA, kBK> SA;
    __shared__ __attribute__((aligned(16))) T lds[2 * SA::ELEMS];

    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t total = tiles * g.batch;
    const int64_t x = blockIdx.x % kNumXcd;
    const int64_t per = gridDim.x / kNumXcd;  // the grid is a multiple of 8
    const int64_t hi = total * (x + 1) / kNumXcd;
    int64_t id = total * x / kNumXcd + blockIdx.x / kNumXcd;
    if (id >= hi) return;  // the whole workgroup: no barrier is left waiting
    const int64_t nk = g.K / kBK;

    const int lane = threadIdx.x & 63;
    const int lg = lane >> 4;
    const int c = lane & 15;
    // The lane's offset into a tile's B panel (N is a multiple of BN: no
    // column clamp), the same for every tile; the tile bases are uniform.
    const int64_t wcol = (threadIdx.x >> 6) * (16 * NB) + NB * c;
    const int64_t boff = TB ? wcol * g.ldb + 4 * lg : wcol + (int64_t)(4 * lg) * g.ldb;
    struct Tile {
        const T* A;
        const T* B;
        int64_t bat, tn, m0;
    };
    auto tile = [&](int64_t tid) __attribute__((always_inline)) -> Tile {
        Tile u;
        u.bat = tid / tiles;
        const int64_t rem = tid - u.bat * tiles;
        u.tn = rem / g.tiles_m;
        u.m0 = (rem - u.tn * g.tiles_m) * 64;
        u.A = static_cast<const T*>(g.A) + u.bat * g.sA;
        u.B = static_cast<const T*>(g.B) + u.bat * g.sB + (TB ? u.tn * BN * g.ldb : u.tn * BN);
        return u;
    };
    SA sa;
    v16_t rb[4];
    auto bload = [&](const T* B, int64_t t, int p) __attribute__((always_inline)) {
        const T* q = (TB ? B + (int64_t)(p % NB) * g.ldb + 16 * t + SPL * (p / NB) : B + (16 * t + p) * g.ldb) + boff;
        rb[p] = NT ? __builtin_nontemporal_load(reinterpret_cast<const mem_t*>(q)) : *reinterpret_cast<const mem_t*>(q);
    };
    auto afrag = [&](const T* sbuf, int a, int s) __attribute__((always_inline)) -> T {
        return TA ? sbuf[(4 * lg + s) * SA::PITCH + 16 * a + c] : sbuf[(16 * a + c) * SA::PITCH + 4 * lg + s];
    };
    acc_t acc[4][NB];
    T fa[4][SPL];
    auto piece = [&](const T* sbuf, int p) __attribute__((always_inline)) {
        if (!TB) {
#pragma unroll
            for (int a = 0; a < 4; ++a) fa[a][0] = afrag(sbuf, a, p);
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[a][b] = MF::mma(fa[a][0], rb[p][b], acc[a][b]);
        } else {
            const int h = p / NB, b = p % NB;
            if (b == 0) {
#pragma unroll
                for (int a = 0; a < 4; ++a)
#pragma unroll
                    for (int e = 0; e < SPL; ++e) fa[a][e] = afrag(sbuf, a, SPL * h + e);
            }
#pragma unroll
            for (int e = 0; e < SPL; ++e)
#pragma unroll
                for (int a = 0; a < 4; ++a) acc[a][b] = MF::mma(fa[a][e], rb[p][e], acc[a][b]);
        }
    };

    Tile cur = tile(id);
    sa.template load<true>(cur.A, g.lda, cur.m0, g.M, 0);
    sa.store(lds);
#pragma unroll
    for (int p = 0; p < 4; ++p) bload(cur.B, 0, p);
    __syncthreads();
    int buf = 0;
    for (;;) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[a][b] = acc_t{0, 0, 0, 0};
        for (int64_t t = 0; t + 1 < nk; ++t) {
            sa.template load<true>(cur.A, g.lda, cur.m0, g.M, (t + 1) * kBK);
            const T* sb = lds + buf * SA::ELEMS;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                piece(sb, p);
                bload(cur.B, t + 1, p);
            }
            __builtin_amdgcn_sched_barrier(0);
            sa.store(lds + (buf ^ 1) * SA::ELEMS);
            __syncthreads();
            buf ^= 1;
        }
        // Last stage: the next tile's first stage goes out behind its MFMAs.
        const int64_t nid = id + per;
        const bool more = nid < hi;
        const Tile nxt = tile(more ? nid : id);
        if (more) sa.template load<true>(nxt.A, g.lda, nxt.m0, g.M, 0);
        const T* sb = lds + buf * SA::ELEMS;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            piece(sb, p);
            if (more) bload(nxt.B, 0, p);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) sa.store(lds + (buf ^ 1) * SA::ELEMS);
        directb_store<T, true, true>(g, acc, cur.bat, cur.m0, cur.tn);
        if (!more) break;
        __syncthreads();
        buf ^= 1;
        id = nid;
        cur = nxt;
    }
}


// Streaming direct-B GEMM (fp64, A transposed, B row-major, no C, at most two
// 64-row tiles: the AO->MO half transform's shape, where B streams from HBM
// once and feeds at most 128 rows). Persistent like
// gemm_directb_persistent_kernel, but 64 x 256 tiles of four waves of 64 x 64
// (NB = 4 column blocks), two workgroups per CU (two waves per SIMD), so
// each A fragment read from LDS feeds 16 MFMAs instead of 8. Column block
// 2 j + e of a lane is column 32 j + 2 c + e of its wave's 64: every 16-byte
// B load and D store of a lane group covers 256 contiguous bytes. Per
// 16-k stage: the next piece's A fragments are read ahead, the next stage's B
// pieces are loaded one per 8 MFMAs, and the barrier comes before the last
// piece, whose MFMAs cover the next stage's first fragment reads. The stages
// of consecutive tiles form one pipeline (the next tile's first stage is
// loaded during the current tile's last). MFMA order per output as
// gemm_directb_kernel's: bitwise equal. Same box, alternating, against the
// persistent 64 x 128 kernel: 64 x 786432 x 512 0.842-0.851 against
// 0.880 ms, 64 x 393216 x 1024 0.819 against 0.855 ms, 128 x 393216 x 512
// 0.775 against 0.803 ms; with five row tiles (the transform's batched
// GEMM, 320 x 1536 x 512 x 64) it lost (0.490 against 0.483 ms), with 1.5
// tiles per workgroup it tied. One wave per SIMD with NB = 8 (AGPR
// accumulators) ran 0.951 against 0.914 ms on another box, and B two stages
// ahead (238 VGPRs) 0.907 against 0.852 ms.
template <bool NT>
__global__ __launch_bounds__(kThreads, 2) void gemm_directb_stream_kernel(GemmArgs g) {
    typedef Mfma<double> MF;
    typedef typename MF::acc_t acc_t;
    constexpr int NB = 4;
    constexpr int BN = 64 * NB;
    typedef typename Vec16<double>::type v16_t;
    typedef Mem16<double>::type mem_t;
    typedef Stage<double, 64, false, kBK> SA;
    __shared__ __attribute__((aligned(16))) double lds[2 * SA::ELEMS];

    // Hardware workgroup w runs on XCD w % 8; the tiles are split into eight
    // contiguous ranges, one per XCD, taken round-robin by its workgroups.
    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t total = tiles * g.batch;
    const int64_t x = blockIdx.x % kNumXcd;
    const int64_t per = gridDim.x / kNumXcd;  // the grid is a multiple of 8
    const int64_t hi = total * (x + 1) / kNumXcd;
    int64_t id = total * x / kNumXcd + blockIdx.x / kNumXcd;
    if (id >= hi) return;  // the whole workgroup: no barrier is left waiting
    const int64_t nk = g.K / kBK;

    const int lane = threadIdx.x & 63;
    const int lg = lane >> 4;
    const int c = lane & 15;
    const int64_t wcol = (threadIdx.x >> 6) * (16 * NB) + 2 * c;
    const int64_t boff = wcol + (int64_t)(4 * lg) * g.ldb;
    struct Tile {
        const double* A;
        const double* B;
        int64_t bat, tn, m0;
    };
    auto tile = [&](int64_t tid) __attribute__((always_inline)) -> Tile {
        Tile u;
        u.bat = tid / tiles;
        const int64_t rem = tid - u.bat * tiles;
        u.tn = rem / g.tiles_m;
        u.m0 = (rem - u.tn * g.tiles_m) * 64;
        u.A = static_cast<const double*>(g.A) + u.bat * g.sA;
        u.B = static_cast<const double*>(g.B) + u.bat * g.sB + u.tn * BN;
        return u;
    };
    SA sa;
    v16_t rb[4][NB / 2];  // [piece p][j]: k-row 16 t + 4 lg + p, columns 32 j + 2 c, + 1
    auto bload = [&](const double* B, int64_t t, int p) __attribute__((always_inline)) {
        const double* q = B + (16 * t + p) * g.ldb + boff;
#pragma unroll
        for (int j = 0; j < NB / 2; ++j) {
            const mem_t* qq = reinterpret_cast<const mem_t*>(q + 32 * j);
            rb[p][j] = NT ? __builtin_nontemporal_load(qq) : *qq;
        }
    };
    auto afrag = [&](const double* sbuf, int a, int s) __attribute__((always_inline)) -> double {
        return sbuf[(4 * lg + s) * SA::PITCH + 16 * a + c];
    };
    acc_t acc[4][NB];
    double fa[2][4];
    auto piece = [&](int p, const double (&f)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[a][b] = MF::mma(f[a], rb[p][b >> 1][b & 1], acc[a][b]);
    };
    // Scheduling groups: the piece's A reads first (0x100), then one B load
    // (0x020) after every 8 MFMAs (0x008).
    auto spread = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < NB / 2; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // One stage of the current tile from LDS buffer buf; stage tn1 of tile
    // nxt is loaded behind it when `more`.
    auto stage = [&](int buf, bool more, const Tile& nxt, int64_t tn1) __attribute__((always_inline)) {
        if (more) sa.template load<true>(nxt.A, g.lda, nxt.m0, g.M, tn1 * kBK);
        const double* sb = lds + buf * SA::ELEMS;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int a = 0; a < 4; ++a) fa[(p + 1) & 1][a] = afrag(sb, a, p + 1);
            piece(p, fa[p & 1]);
            if (more) bload(nxt.B, tn1, p);
            spread();
        }
        if (more) sa.store(lds + (buf ^ 1) * SA::ELEMS);
        __syncthreads();
        if (more) {
#pragma unroll
            for (int a = 0; a < 4; ++a) fa[0][a] = afrag(lds + (buf ^ 1) * SA::ELEMS, a, 0);
        }
        piece(3, fa[1]);
        if (more) bload(nxt.B, tn1, 3);
        spread();
    };
    // D is written once and not read here: non-temporal stores (64 x 786432
    // x 512, same box, alternating, three runs: 0.838-0.845 against
    // 0.844-0.849 ms; K 1024 with N / 2: 0.818 against 0.813 ms).
    auto store = [&](const Tile& u) __attribute__((always_inline)) {
        double* D = static_cast<double*>(g.D) + u.bat * g.sD;
        const int64_t col = u.tn * BN + wcol;
        const double alpha = g.alpha;
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = u.m0 + 16 * a + MF::row(lg, r);
#pragma unroll
                for (int j = 0; j < NB / 2; ++j) {
                    v16_t v;
                    v[0] = acc[a][2 * j][r];
                    v[1] = acc[a][2 * j + 1][r];
                    if (alpha != 1.0) v = v * alpha;
                    __builtin_nontemporal_store(v, reinterpret_cast<mem_t*>(D + row * g.ldd + col + 32 * j));
                }
            }
    };

    Tile cur = tile(id);
    sa.template load<true>(cur.A, g.lda, cur.m0, g.M, 0);
    sa.store(lds);
#pragma unroll
    for (int p = 0; p < 4; ++p) bload(cur.B, 0, p);
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; ++a) fa[0][a] = afrag(lds, a, 0);
    int buf = 0;
    for (;;) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[a][b] = acc_t{0, 0, 0, 0};
        for (int64_t t = 0; t + 1 < nk; ++t) {
            stage(buf, true, cur, t + 1);
            buf ^= 1;
        }
        const int64_t nid = id + per;
        const bool more = nid < hi;
        const Tile nxt = tile(more ? nid : id);
        stage(buf, more, nxt, 0);
        buf ^= 1;
        store(cur);
        if (!more) break;
        id = nid;
        cur = nxt;
    }
}

int device_cus() {
    static int cus[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cus[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

// Runs launch(workgroups) for `total` tiles. The dot epilogue takes more than a
// launch may have as several launches, each writing its own range of the
// partials from g.first up (a dot of 2^24 tiles in one launch left partials
// unwritten). Products that store D never get here with so many: the tile
// choice leaves them to kernels that split the product.
template <bool DOT, typename F>
static void launch_tiles(GemmArgs& g, int64_t total, F launch) {
    int64_t n = total;
    for (g.first = 0; g.first < total; g.first += n) {
        if (DOT) n = std::min(total - g.first, kMaxGrid);
        launch(dim3((unsigned)n));
    }
}

template <typename T, bool DOT>
static int launch_directb(GemmArgs& g, bool ta, bool tb, bool nt, hipStream_t st) {
    constexpr int BN = 64 * (16 / sizeof(T));
    g.tiles_m = (g.M + 63) / 64;
    g.tiles_n = (g.N + BN - 1) / BN;
    const int64_t total = g.tiles_m * g.tiles_n * g.batch;
    if (total > 0x7fffffffLL) return set_error(TT_UNSUPPORTED, "tt_gemm: %lld tiles exceed one launch", (long long)total);
    const bool full = g.M % 64 == 0;
    // Three or more rounds of tiles (four workgroups per CU) with A
    // transposed and B row-major (the AO->MO transform's two GEMMs): the
    // persistent kernel. Same box, alternating, bitwise equal: AO->MO half
    // transform (64 x 786432 x 512) 0.8646 against 0.8787 ms, the transform's
    // batched GEMM (64 x 320 x 1536 x 512) 0.4702 against 0.4830 ms. At two
    // rounds (4096^3, 64 x 512^3 without C) it measured 1-2% slower, and its
    // other layouts spill registers.
    const int64_t slots = (int64_t)device_cus() / kNumXcd * 4;
    // fp64 with at most two row tiles and at least three 64 x 256 tiles per
    // workgroup at two per CU: the streaming kernel.
    if constexpr (sizeof(T) == 8 && !DOT) {
        const int64_t stiles = g.tiles_m * (g.N / 256) * g.batch;
        const int64_t sgrid = (int64_t)device_cus() / kNumXcd * kNumXcd * 2;
        if (ta && !tb && full && !g.C && g.N % 256 == 0 && g.K >= kBK && g.K % kBK == 0 &&
            g.tiles_m <= 2 && stiles >= 3 * sgrid) {
            g.tiles_n = g.N / 256;
            const dim3 grid((unsigned)sgrid), block(kThreads);
            if (nt) hipLaunchKernelGGL((gemm_directb_stream_kernel<true>), grid, block, 0, st, g);
            else hipLaunchKernelGGL((gemm_directb_stream_kernel<false>), grid, block, 0, st, g);
            return check_launch("tt_gemm");
        }
    }
    if (!DOT && ta && !tb && full && !g.C && g.N % BN == 0 && g.K >= kBK && g.K % kBK == 0 &&
        total >= 3 * slots * kNumXcd) {
        const dim3 grid((unsigned)(slots * kNumXcd)), block(kThreads);
        if (nt) hipLaunchKernelGGL((gemm_directb_persistent_kernel<T, true, false, true>), grid, block, 0, st, g);
        else hipLaunchKernelGGL((gemm_directb_persistent_kernel<T, true, false, false>), grid, block, 0, st, g);
        return check_launch("tt_gemm");
    }
    const dim3 block(kThreads);
    launch_tiles<DOT>(g, total, [&](dim3 grid) {
#define TT_DIRECTB_CASE(F, A_T, B_T, N_T)                         \
    if (full == F && ta == A_T && tb == B_T && nt == N_T)         \
        hipLaunchKernelGGL((gemm_directb_kernel<T, F, A_T, B_T, N_T, DOT>), grid, block, 0, st, g);
#define TT_DIRECTB_NT(F, A_T, B_T) TT_DIRECTB_CASE(F, A_T, B_T, true) TT_DIRECTB_CASE(F, A_T, B_T, false)
#define TT_DIRECTB_A(B_T)                                            \
    TT_DIRECTB_NT(true, true, B_T) TT_DIRECTB_NT(false, true, B_T) \
    TT_DIRECTB_NT(true, false, B_T) TT_DIRECTB_NT(false, false, B_T)
    TT_DIRECTB_A(false)
    if constexpr (sizeof(T) == 8) {  // fp32 comes here with B row-major only
        TT_DIRECTB_A(true)
    }
#undef TT_DIRECTB_A
#undef TT_DIRECTB_NT
#undef TT_DIRECTB_CASE
    });
    return check_launch("tt_gemm");
}

// fp64 direct-B tiles of 16 FM = 32 or 48 rows (rows always clamped).
static int launch_directb_rows(GemmArgs& g, bool ta, bool tb, bool nt, int fm, hipStream_t st) {
    g.tiles_m = (g.M + 16 * fm - 1) / (16 * fm);
    g.tiles_n = (g.N + 127) / 128;
    const int64_t total = g.tiles_m * g.tiles_n * g.batch;
    if (total > 0x7fffffffLL) return set_error(TT_UNSUPPORTED, "tt_gemm: %lld tiles exceed one launch", (long long)total);
    const dim3 grid((unsigned)total), block(kThreads);
#define TT_ROWS_CASE(R, A_T, B_T, N_T)                 \
    if (fm == R && ta == A_T && tb == B_T && nt == N_T) \
        hipLaunchKernelGGL((gemm_directb_kernel<double, false, A_T, B_T, N_T, false, R>), grid, block, 0, st, g);
#define TT_ROWS_NT(R, A_T, B_T) TT_ROWS_CASE(R, A_T, B_T, true) TT_ROWS_CASE(R, A_T, B_T, false)
#define TT_ROWS(R) TT_ROWS_NT(R, true, true) TT_ROWS_NT(R, true, false) TT_ROWS_NT(R, false, true) TT_ROWS_NT(R, false, false)
    TT_ROWS(2)
    TT_ROWS(3)
#undef TT_ROWS
#undef TT_ROWS_NT
#undef TT_ROWS_CASE
    return check_launch("tt_gemm");
}

// fp64 products without the dot epilogue (all kernels bitwise equal): the tile
// with the least estimated time of the busiest CU: its tiles times their
// area (where a CU has several, a wave past the last column gives its share
// back, hence columns rounded up to 32), times the kernel's cost per output,
// times what a single direct-B tile on a CU loses because nothing covers the
// latencies of its 16-deep stages (21 x 150 x 150 x 555 NT on fresh operands: 29
// us on 32 x 128 tiles, 21 on 32 x 32 with 64-deep stages). us measured on 64 /
// 48 / 32 rows x 128 columns (direct-B) / 32 x 32: 21 x 94905 x 171 TN
// 46/38/29/40; 40 x 94905 x 171 47/40/58/67; 77 x 200000 x 300 TN
// 274/225/227/309; 110 x 200000 x 300 275/307/284/390; 77 x 223 x 900 x 300
// 199/198/187/246; 21 x 150 x 555 x 171 32/27/26/25; 60 x 100 x 100 x 1000 NT
// 72/59/49/48; 3000^2 x 1000 323/289/296/350; 1400^2 x 700 56/74/57/69; 1100 x
// 1200 x 500 41/-/-/39.5; 12 x 90 x 300 x 100 12.8/10.8/8.9/7.2.
static int gemm_f64(GemmArgs& g, bool ta, bool tb, hipStream_t st) {
    const bool nt = g.M <= 64 && (g.batch == 1 || g.sB != 0);  // B is read once
    const int64_t cus = device_cus();
    auto up = [](int64_t n, int64_t t) { return (n + t - 1) / t; };
    // A wave past the last column does not give all of its share back where K is
    // long. us on 32 x 128 / 32 x 32: 284545 x 7 x 222 NT 170 / 119, 137622 x 9 x 302
    // NT 104 / 75, 57 x 11 x 607 x 513 TN 55 / 43; but 34 x 19 x 447 x 1866 83 (48 rows)
    // / 96.
    double cols = (double)(up(g.N, 32) * 32) / (double)(up(g.N, 128) * 128);
    if (g.K > 32) cols = std::max(cols, g.N <= 32 ? 0.4 : 0.55);
    // Few rows and a long k-contiguous B: a direct-B lane reads its own column's
    // row, and nothing but the stage ahead covers that stream; the 32 x 32 tile
    // stages whole lines. us on 64 / 48 / 32 rows / 32 x 32: 60 x 69201 x 282 92 / 140 /
    // 119 / 59, 50 x 277167 x 330 403 / 702 / 638 / 276, 17 x 40746 x 654 105 / 101 / 97 /
    // 45; up to K = 80 level (37 x 78114 x 63 26 / 21 / 27 / 30).
    const double stream = tb && g.M <= 64 && g.K > 80 ? 1.5 : 1.0;
    auto direct = [&](int64_t fm, double per_output) {
        const int64_t n = up(g.M, 16 * fm) * up(g.N, 128) * g.batch;
        if (n > kMaxGrid) return 1e300;  // not one launch; the 32 x 32 tiles take several
        const int64_t rounds = up(n, cus);
        const double share = rounds == 1 ? 1.0 : rounds == 2 ? (1.0 + cols) / 2 : cols;
        return (double)(rounds * 16 * fm * 128) * share * per_output * (rounds == 1 ? 1.6 : 1.0) * stream;
    };
    const int64_t sr = up(up(g.M, 32) * up(g.N, 32) * g.batch, cus);
    // A short sum leaves most of a 64-deep stage empty: 318 x 3602 x 7 NT 7.7 us
    // on 32 x 32, 5.8 on 32 x 128; 8 x 68679 x 1 8.9 / 5.6.
    const bool empty = g.K <= 32 && g.N > 32 && sr > 4;
    const double small = (double)(sr * 32 * 32) * 1.4 * (sr <= 2 ? 1.1 : 1.0) * (empty ? 1.4 : 1.0);
    const double d4 = direct(4, 1.0), d3 = direct(3, 1.04), d2 = direct(2, 1.1);
    // A whole 16-byte piece along a row-contiguous operand, else 32 x 32 tiles
    // (100000 x 1 x 300 51 against 118 us on 256 x 64 LDS tiles).
    const bool direct_ok = g.N >= 2 && (!ta || g.M >= 2);
    // One 32 x 32 tile per batch entry, where the direct-B tiles have one live
    // wave: 12 x 32 x 32 x 1432 NT 6.6 us against 8.0 on 32 x 128.
    const bool one = g.M <= 32 && g.N <= 32 && g.K > 16;
    if (!direct_ok || one || (small < d4 && small < d3 && small < d2)) return gemm_small_launch(TT_F64, ta, tb, g, st);
    if (d2 < d4 && d2 < d3) return launch_directb_rows(g, ta, tb, nt, 2, st);
    if (d3 < d4) return launch_directb_rows(g, ta, tb, nt, 3, st);
    return launch_directb<double, false>(g, ta, tb, nt, st);
}

template <typename T, int BM, int BN, int FM, int FN, bool DOT, int NBUF = 2, int BK = kBK>
static int launch_tile(GemmArgs& g, bool ta, bool tb, hipStream_t st) {
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    const int64_t total = g.tiles_m * g.tiles_n * g.batch;
    if (total > 0x7fffffffLL) return set_error(TT_UNSUPPORTED, "tt_gemm: %lld tiles exceed one launch", (long long)total);
    const bool full = g.M % BM == 0 && g.N % BN == 0;
    const dim3 block(kThreads);
    launch_tiles<DOT>(g, total, [&](dim3 grid) {
#define TT_GEMM_CASE(TA, TB, F) \
    if (ta == TA && tb == TB && full == F) hipLaunchKernelGGL((gemm_kernel<T, BM, BN, FM, FN, TA, TB, F, DOT, NBUF, BK>), grid, block, 0, st, g);
    TT_GEMM_CASE(false, false, false)
    TT_GEMM_CASE(false, false, true)
    TT_GEMM_CASE(false, true, false)
    TT_GEMM_CASE(false, true, true)
    TT_GEMM_CASE(true, false, false)
    TT_GEMM_CASE(true, false, true)
    TT_GEMM_CASE(true, true, false)
    TT_GEMM_CASE(true, true, true)
#undef TT_GEMM_CASE
    });
    return check_launch("tt_gemm");
}

// fp32 products (all kernels bitwise equal).
static int gemm_f32(GemmArgs& g, bool ta, bool tb, hipStream_t st) {
    const int64_t cus = device_cus();
    // Both operands not transposed, whole 256 x 256 tiles in whole rounds of
    // one tile per CU (at least 95% of the last round busy), without C or with
    // K >= 1024: the 256 x 256 LDS tile (tt_gemm_big.hip). Same box,
    // alternating, fraction of the fp32 peak against the 64 x 256 direct-B tile:
    // 4096^3 with alpha/beta and C 0.93 against 0.88; 64 x 512^3 without C
    // 0.834 against 0.806, 16 x 1024^3 with C 0.866 against 0.845. A partial
    // last round loses (6144^2 x 2048, 2.25 rounds: 1.444 against 1.118 ms),
    // and so does a short K with C, whose epilogue one wave per SIMD cannot
    // hide (64 x 512^3 with C 0.785 against 0.801, 128 x 512^3 with C 0.760
    // against 0.799).
    if (gemm_big_f32_fits(ta, tb, g) && (!g.C || g.K >= 1024)) {
        const int64_t tiles = (g.M / 256) * (g.N / 256) * g.batch;
        const int64_t rounds = (tiles + cus - 1) / cus;
        if (tiles >= cus && 100 * tiles >= 95 * rounds * cus) return gemm_big_f32_launch(g, st);
    }
    // Otherwise the tile with the least estimated time of the busiest CU: its
    // tiles times their area, times the kernel's cost per output where every CU
    // has many tiles (from 4096^3, 6144^2 x 2048, 1999 x 3001 x 1201 in the
    // four layouts), times what one or two tiles on a CU lose because nothing
    // covers their latencies (least on the pipelined tiles). us measured on
    // direct-B 64 x 256 / 128 x 128 / 64 x 128 / 64 x 64 / 32 x 32: 2048 x 3072
    // x 1216 161/158/136/144/163; 3001^2 x 1201 -/230/206/204/250; 1999 x 1501
    // x 1201 NT -/81/84/72/81; 1400^2 x 3000 -/188/111/131/135; 30 x 300^2 x
    // 1000 -/135/76/68/73; 1500^2 x 300 -/28/27/24/23; 1000^3 -/68/39/32/29;
    // 150 x 2000 x 3000 -/186/105/86/52; 4000^2 x 1000 -/260/268/285/311; 64 x
    // 786432 x 512 TN 452/787/470/535/623; 80 x 200000 x 300 TN
    // -/156/150/170/160.
    const double never = 1e300;
    auto tiles = [&](int64_t bm, int64_t bn) { return ((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * g.batch; };
    auto cost = [&](int64_t bm, int64_t bn, double per_output, double one, double two) {
        const int64_t n = tiles(bm, bn);
        if (n > kMaxGrid && bm > 32) return never;  // not one launch; the 32 x 32 tiles take several
        const int64_t rounds = (n + cus - 1) / cus;
        return (double)(rounds * bm * bn) * per_output * (rounds == 1 ? one : rounds == 2 ? two : 1.0);
    };
    const bool rows_ok = !ta || g.M >= 4, cols_ok = tb || g.N >= 4;  // a 16-byte piece along a row-contiguous operand
    // Short sums do not pay for deep stages and their prologue. K of at most
    // one 16-deep stage: every tile costs about the same per workgroup, whatever
    // its area (32 x 32 2.1 ns, 64 x 128 with 16-deep stages 6 ns, chip-wide), so
    // the wide ones win where they are few and well filled. us, 64 x 128 / best of
    // the others (the 64-deep tiles had lost these to the kernels before them):
    // 3706 x 1179 x 3 9.0 / 14.3, 198 x 161 x 5 x 1356 61 / 76, 43 x 183720 x 3
    // 14.3 / 17.4, 72 x 234521 x 1 25 / 37; 256 x 64 / 32 x 32 without C: 169059 x
    // 5 x 5 8.9 / 12.2, 113627 x 36 x 3 9.6 / 12.0, 242 x 17 x 4 x 365 7.9 / 8.6.
    if (g.K <= 16) {
        const int64_t n32 = tiles(32, 32), wide = tiles(64, 128), tall = tiles(256, 64);
        if (g.N <= 64 && !g.C && n32 >= 2560 && n32 >= 7 * tall * ((g.N + 31) / 32) && tall <= kMaxGrid)
            return launch_tile<float, 256, 64, 4, 4, false>(g, ta, tb, st);
        // Half-empty tiles (M <= 32) that read C wait for more rounds: 20 x 71286 x
        // 8 with C 8.5 / 7.4 us, 16 x 163083 x 11 11.4 / 13.3.
        if (n32 >= (g.C && g.M <= 32 ? 4096 : 1280) && n32 >= 3 * wide && wide <= kMaxGrid)
            return launch_tile<float, 64, 128, 2, 4, false>(g, ta, tb, st);
    }
    // Up to K = 128 the 64 x 128 tile with 16-deep stages stays a candidate, and
    // the 32 x 32 tile's single 128-deep stage (K > 64) leaves fewer workgroups on
    // a CU: 60 x 96 x 104 x 704 NT with C 22 / 28 us.
    const double wide16 = g.K > 16 && g.K <= 128 ? cost(64, 128, 1.02, 1.3, 1.1) : never;
    const double direct = rows_ok && !tb && g.N % 256 == 0 ? cost(64, 256, 0.97, 1.1, 1.0) : never;
    const double tall = rows_ok && cols_ok && g.K > 0 ? cost(128, 128, 1.0, 1.05, 1.0) : never;
    const double mid = rows_ok && cols_ok && g.K > 0 ? cost(64, 128, 1.04, 1.05, 1.0) : never;
    const double square = cost(64, 64, 1.1, 1.25, 1.1);
    const bool deep = g.K > 64 && g.K <= 128 && tiles(32, 32) > 2 * cus;
    const double small = cost(32, 32, (ta && !tb ? 1.5 : tb && !ta ? 1.25 : 1.35) * (deep ? 1.2 : 1.0), 1.1, 1.1);
    const double best = std::min({direct, tall, mid, square, small, wide16});
    if (best == small) return gemm_small_launch(TT_F32, ta, tb, g, st);
    if (best == square) return launch_tile<float, 64, 64, 2, 2, false, 1, 64>(g, ta, tb, st);
    if (best == wide16) return launch_tile<float, 64, 128, 2, 4, false>(g, ta, tb, st);
    if (best == direct) return launch_directb<float, false>(g, ta, false, g.M <= 64 && (g.batch == 1 || g.sB != 0), st);
    return gemm_mid_f32_launch(ta, tb, best == tall, g, st);
}

template <typename T, bool DOT>
static int gemm_typed(GemmArgs& g, bool ta, bool tb, hipStream_t st) {
    constexpr int V = Vec16<T>::n;
    // fp64: A through LDS, B straight into the MFMA registers
    // (gemm_directb_kernel above), non-temporal when B is read once (M <= 64
    // and B not broadcast over the batch). Same box, alternating, bitwise
    // equal, against LDS-staged tiles: 4096^3 with alpha/beta 1.952 against
    // 2.082 ms (NN 1.944 against 2.069, TN 1.965 against 2.171, NT 2.026
    // against 2.130, TT 2.025 against 2.104), 4096^2 x 512 0.258 against
    // 0.274 ms, 64 x 512^3 with alpha/beta and C 0.275 against 0.292 ms, the
    // AO->MO transform's two GEMMs 0.885 against 0.914 and 0.492 against
    // 0.520 ms; partial column tiles (3000 x 3000 x 1000 with alpha/beta 0.331
    // against 0.438 ms, NT 0.382 against 0.426, 8192 x 200 x 2048 0.145 against
    // 0.186 ms). Odd N, leading dimensions and batch strides take it too
    // (2999 x 3001 x 1001 with alpha/beta 306 against 713 us on guarded,
    // element-wise LDS tiles, aligned 3000 x 3000 x 1000 311 us; 21 x 150 x
    // 150 x 555 NT 42 against 112 us). With the dot epilogue: config 5's GEMM
    // (160000 x 16384 x 800, B k-contiguous) 66.2-66.4 against 67.9-68.0 ms,
    // 16900 x 900 x 450 (both extents ragged) 0.31 against 0.35 ms, the sum
    // equal to 2e-15 (another order of the per-tile sums).
    // What is left for the dot (N = 1, or a transposed A of one row) runs on
    // the 64 x 128 LDS tiles.
    if constexpr (sizeof(T) == 8 && !DOT) {
        return gemm_f64(g, ta, tb, st);
    } else if constexpr (sizeof(T) == 8) {
        if (g.N >= V && (!ta || g.M >= V))
            return launch_directb<T, DOT>(g, ta, tb, g.M <= 64 && (g.batch == 1 || g.sB != 0), st);
        return launch_tile<T, 64, 128, 2, 4, DOT>(g, ta, tb, st);
    } else if constexpr (DOT) {
        if (g.M <= 64) return launch_tile<T, 64, 128, 2, 4, DOT>(g, ta, tb, st);
        if (g.N <= 64) return launch_tile<T, 256, 64, 4, 4, DOT>(g, ta, tb, st);
        // Fewer than 448 128 x 128 tiles leave CUs idle; 64 x 128 tiles double
        // the grid.
        if (((g.M + 127) / 128) * ((g.N + 127) / 128) * g.batch < 448)
            return launch_tile<T, 64, 128, 2, 4, DOT>(g, ta, tb, st);
        return launch_tile<T, 128, 128, 4, 4, DOT>(g, ta, tb, st);
    } else {
        return gemm_f32(g, ta, tb, st);
    }
}

int gemm_dispatch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    g.E1 = g.E2 = nullptr;
    g.partial = nullptr;
    if (dtype == TT_F64) return gemm_typed<double, false>(g, ta, tb, st);
    if (dtype == TT_F32) return gemm_typed<float, false>(g, ta, tb, st);
    if (dtype == TT_F64_DD) return gemm_dd_dispatch(ta, tb, g, st);
    if (dtype == TT_BF16 || dtype == TT_F16) return gemm16_dispatch(dtype, ta, tb, g, st);
    return set_error(TT_UNSUPPORTED, "tt_gemm: dtype %d (only TT_F32, TT_F64, TT_F64_DD, TT_BF16, TT_F16)", dtype);
}

int gemm_dot_dispatch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st, int64_t* nparts) {
    int rc;
    if (dtype == TT_F64) rc = gemm_typed<double, true>(g, ta, tb, st);
    else if (dtype == TT_F32) rc = gemm_typed<float, true>(g, ta, tb, st);
    else return set_error(TT_UNSUPPORTED, "tt_gemm_dot: dtype %d (only TT_F32, TT_F64)", dtype);
    *nparts = g.tiles_m * g.tiles_n * g.batch;
    return rc;
}

// out[0] = alpha * (fixed-order sum of the partials) (+ beta * C[0]).
template <typename T>
__global__ __launch_bounds__(256) void dot_finalize_kernel(const double* partial, int64_t n, double alpha, double beta,
                                                           const T* C, T* out) {
    __shared__ double red[4];
    const double s = strided_sum256(partial, n);
    const double tot = block256_sum(s, red);
    if (threadIdx.x == 0) {
        T v = (T)tot;
        if (alpha != 1.0) v = (T)alpha * v;
        if (C) v = v + (T)beta * C[0];
        out[0] = v;
    }
}

// A contiguous vector operand (one row of op(A), one column of op(B)) is
// k-contiguous in either form, and as such read in 16-byte pieces instead of
// element by element: dots 1 x 29 x 1332 x 24 TN fp64 152 -> 94 us, 47 x 1 x 1224 TN
// fp32 97 -> 60; products 1 x 77977 x 13 TT fp64 9.6 -> 5.3 us, 3000 x 1 x 3000
// 93 -> 45, fp32 62 -> 36, bf16 32 -> 18.
static void vector_operands(bool& ta, bool& tb, GemmArgs& g) {
    if (g.N == 1 && !tb && g.ldb == 1) tb = true, g.ldb = std::max<int64_t>(g.K, 1);
    if (g.M == 1 && ta && g.lda == 1) ta = false, g.lda = std::max<int64_t>(g.K, 1);
}

}  // namespace tt

extern "C" int tt_gemm(int dtype, int transA, int transB, int64_t M, int64_t N, int64_t K, double alpha,
                       const void* A, int64_t lda, int64_t strideA, const void* B, int64_t ldb, int64_t strideB,
                       double beta, const void* C, int64_t ldc, int64_t strideC, void* D, int64_t ldd,
                       int64_t strideD, int64_t batch, void* stream) {
    using namespace tt;
    if (M < 0 || N < 0 || K < 0 || batch < 0)
        return set_error(TT_INVALID, "tt_gemm: negative extent (M=%lld N=%lld K=%lld batch=%lld)", (long long)M,
                         (long long)N, (long long)K, (long long)batch);
    if (M == 0 || N == 0 || batch == 0) return TT_OK;
    if (!D) return set_error(TT_INVALID, "tt_gemm: D is NULL");
    if (K > 0 && (!A || !B)) return set_error(TT_INVALID, "tt_gemm: A or B is NULL");
    const int64_t rowsA = transA ? K : M, colsA = transA ? M : K;
    const int64_t rowsB = transB ? N : K, colsB = transB ? K : N;
    if (K > 0 && ((rowsA > 1 && lda < colsA) || (rowsB > 1 && ldb < colsB)))
        return set_error(TT_INVALID, "tt_gemm: leading dimension smaller than a row (lda=%lld ldb=%lld)",
                         (long long)lda, (long long)ldb);
    if ((M > 1 && ldd < N) || (C && M > 1 && ldc < N))
        return set_error(TT_INVALID, "tt_gemm: ldd/ldc smaller than N");
    GemmArgs g;
    g.A = A;
    g.B = B;
    g.C = C;
    g.D = D;
    g.M = M;
    g.N = N;
    g.K = K;
    g.lda = lda;
    g.ldb = ldb;
    g.ldc = ldc;
    g.ldd = ldd;
    g.sA = strideA;
    g.sB = strideB;
    g.sC = strideC;
    g.sD = strideD;
    g.batch = batch;
    g.alpha = alpha;
    g.beta = beta;
    bool ta = transA != 0, tb = transB != 0;
    vector_operands(ta, tb, g);
    return gemm_dispatch(dtype, ta, tb, g, static_cast<hipStream_t>(stream));
}

extern "C" int tt_gemm_packed(const int64_t* params, double alpha, double beta, const void* A, const void* B,
                              const void* C, void* D, void* stream) {
    if (!params) return tt::set_error(TT_INVALID, "tt_gemm_packed: params is NULL");
    const int64_t* p = params;
    return tt_gemm((int)p[0], (int)p[1], (int)p[2], p[3], p[4], p[5], alpha, A, p[6], p[7], B, p[8], p[9], beta, C,
                   p[10], p[11], D, p[12], p[13], p[14], stream);
}

extern "C" size_t tt_gemm_dot_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t batch) {
    (void)dtype;
    if (M <= 0 || N <= 0 || batch <= 0) return 256;
    // One double per workgroup; every tile configuration is at least 64 x 64.
    const size_t parts = (size_t)((M + 63) / 64) * (size_t)((N + 63) / 64) * (size_t)batch;
    return ((parts * sizeof(double) + 255) / 256) * 256;
}

extern "C" int tt_gemm_dot(int dtype, int transA, int transB, int64_t M, int64_t N, int64_t K, const void* A,
                           int64_t lda, int64_t strideA, const void* B, int64_t ldb, int64_t strideB, int64_t batch,
                           int64_t m_lo, int64_t n_lo, const void* E1, const int64_t* e1_strides, const void* E2,
                           const int64_t* e2_strides, double alpha, double beta, const void* C, void* out,
                           void* workspace, size_t workspace_bytes, void* stream) {
    using namespace tt;
    if (M < 0 || N < 0 || K < 0 || batch < 0)
        return set_error(TT_INVALID, "tt_gemm_dot: negative extent (M=%lld N=%lld K=%lld batch=%lld)", (long long)M,
                         (long long)N, (long long)K, (long long)batch);
    if (dtype != TT_F32 && dtype != TT_F64)
        return set_error(TT_UNSUPPORTED, "tt_gemm_dot: dtype %d (only TT_F32, TT_F64)", dtype);
    if (!out || !workspace) return set_error(TT_INVALID, "tt_gemm_dot: out or workspace is NULL");
    if (M >= (1LL << 31) || N >= (1LL << 31))
        return set_error(TT_UNSUPPORTED, "tt_gemm_dot: M or N reaches 2^31");
    const int64_t mlo = m_lo > 0 ? m_lo : 1, nlo = n_lo > 0 ? n_lo : 1;
    const size_t need = tt_gemm_dot_workspace_bytes(dtype, M, N, batch);
    if (workspace_bytes < need)
        return set_error(TT_INVALID, "tt_gemm_dot: workspace of %zu bytes, need %zu", workspace_bytes, need);
    hipStream_t st = static_cast<hipStream_t>(stream);
    int64_t nparts = 0;
    if (M > 0 && N > 0 && batch > 0) {
        if (K > 0 && (!A || !B)) return set_error(TT_INVALID, "tt_gemm_dot: A or B is NULL");
        if (!E1 || !e1_strides || (E2 && !e2_strides)) return set_error(TT_INVALID, "tt_gemm_dot: E1 is NULL");
        const int64_t rowsA = transA ? K : M, colsA = transA ? M : K;
        const int64_t rowsB = transB ? N : K, colsB = transB ? K : N;
        if (K > 0 && ((rowsA > 1 && lda < colsA) || (rowsB > 1 && ldb < colsB)))
            return set_error(TT_INVALID, "tt_gemm_dot: leading dimension smaller than a row (lda=%lld ldb=%lld)",
                             (long long)lda, (long long)ldb);
        GemmArgs g;
        memset(&g, 0, sizeof(g));
        g.A = A;
        g.B = B;
        g.M = M;
        g.N = N;
        g.K = K;
        g.lda = lda;
        g.ldb = ldb;
        g.sA = strideA;
        g.sB = strideB;
        g.batch = batch;
        g.alpha = 1.0;
        g.E1 = E1;
        g.E2 = E2;
        for (int k = 0; k < 5; ++k) {
            g.e1s[k] = e1_strides[k];
            g.e2s[k] = E2 ? e2_strides[k] : 0;
        }
        g.mdiv = make_fastdiv((uint32_t)mlo);
        g.ndiv = make_fastdiv((uint32_t)nlo);
        g.partial = static_cast<double*>(workspace);
        bool ta = transA != 0, tb = transB != 0;
        // fp64 runs on 64 x 128 tiles. X^T = op(B)^T op(A)^T is formed instead,
        // E read with its row and column parts exchanged, where that costs less:
        // the busiest CU's tiles times their K, plus 60 k for what a tile costs
        // besides, plus 50 k where the lanes, which run along the columns, read E
        // or E2 with a stride of more than 16 elements (a cache line); with equal
        // costs the fewer tiles. us, as given / exchanged: E and E2 an outer product
        // with strided lanes as given, not when exchanged: 16900 x 900 x 450 (2120 /
        // 1995 tiles) 273 / 238, 16384 x 1024 x 512 (2048 / 2048) 265 / 256, 40000 x
        // 256 x 100 (1250 / 1252) 65 / 54, 160000 x 16384 x 800 60.1 / 59.2 ms. E
        // contiguous along n: 4065 x 21285 x 4 (10688 / 10656) 262 / 469, 1605 x 19235
        // x 12 124 / 175, 128 x 20254 x 533 80 / 85, 27541 x 256 x 270 84 / 99; but
        // 19486 x 773 x 417 (9 tiles on a CU / 8) 255 / 224, 16501 x 9 x 70 18 / 13.
        const int64_t given = ((M + 63) / 64) * ((N + 127) / 128) * batch;
        const int64_t exch = ((N + 63) / 64) * ((M + 127) / 128) * batch;
        auto pen = [&](int lane) {
            auto strided = [&](const int64_t* s) { return s[lane] > 16 || s[lane] < -16; };
            return strided(g.e1s) || (E2 && strided(g.e2s)) ? 50 : 0;
        };
        bool exchange = false;
        if (dtype == TT_F64 && exch <= 0x7fffffffLL) {
            const int64_t kg = K + 60 + pen(n_lo > 1 ? 3 : 2), ke = K + 60 + pen(m_lo > 1 ? 1 : 0);
            double cg = (double)kg, ce = (double)ke;
            if (std::max(given, exch) > 64) {  // else one round of the CUs either way
                const int64_t cus = device_cus();
                cg *= (double)((given + cus - 1) / cus);
                ce *= (double)((exch + cus - 1) / cus);
            }
            exchange = ce < cg || (ce == cg && exch < given);
        }
        if (exchange) {
            std::swap(g.A, g.B);
            std::swap(g.M, g.N);
            std::swap(g.lda, g.ldb);
            std::swap(g.sA, g.sB);
            std::swap(g.mdiv, g.ndiv);
            for (int k = 0; k < 2; ++k) {
                std::swap(g.e1s[k], g.e1s[k + 2]);
                std::swap(g.e2s[k], g.e2s[k + 2]);
            }
            const bool t = !tb;
            tb = !ta;
            ta = t;
        }
        vector_operands(ta, tb, g);
        const int rc = gemm_dot_dispatch(dtype, ta, tb, g, st, &nparts);
        if (rc != TT_OK) return rc;
    }
    if (dtype == TT_F64)
        hipLaunchKernelGGL(dot_finalize_kernel<double>, dim3(1), dim3(256), 0, st, (const double*)workspace, nparts,
                           alpha, beta, static_cast<const double*>(C), static_cast<double*>(out));
    else
        hipLaunchKernelGGL(dot_finalize_kernel<float>, dim3(1), dim3(256), 0, st, (const double*)workspace, nparts,
                           alpha, beta, static_cast<const float*>(C), static_cast<float*>(out));
    return check_launch("tt_gemm_dot");
}
