// fp32 GEMM on software-pipelined 128 x 128 and 64 x 128 tiles (tt_gemm,
// TT_F32; any layout, extent, alignment and batch with at least four
// elements along a row-contiguous operand).
//
// MFMA-bound, with the grid's quantisation: a 256-CU chip runs a product of a
// few thousand rows in two to four tiles per CU, so the tile is small enough
// for the last round to matter little, and each tile keeps the MFMAs fed by
// itself. Four waves of 64 x 64 (32 x 64) outputs, two (three) workgroups per
// CU, stages of 32 k double-buffered in LDS with one barrier each; a 16-k
// chunk's fragments are read while the previous chunk multiplies, and the
// global loads, LDS stores and fragment reads are spread among the MFMAs by
// scheduling groups. Both operands are read in 16-byte LDS pieces in either
// layout: four k of one row, or four rows of one k, in which case row 4 c + b
// belongs to MFMA block b and D's columns come out as 16-byte pieces. KC rows
// are padded by 8 floats, row-contiguous k-rows not at all: at 1999 x 3001 x
// 1201 NN with C one in seven of the LDS's active cycles is a bank conflict and
// the MFMAs are busy 0.72 of the time (counters). The k order per output is that of every other kernel (bitwise
// equal). Same box, us, against the two-buffer tiles with 16-deep stages they
// replace: 1999 x 3001 x 1201 with alpha/beta and C 126 against 143 (224 with
// element-wise loads), 1400^2 x 3000 111 against 172, 2048 x 3072 x 1216 135
// against 160 (64 x 256 direct-B), 4096^3 NT 977 against 1018, 600 x 4000 x 900
// NT with C 57 against 83.
#include "tt_gemm.hpp"
#include "tt_stage.hpp"

namespace tt {

namespace {

constexpr int kMidK = 32;  // k per stage: two 16-k chunks

// One operand's fragments. KC: row block i of a wave is rows 16 i + lane % 16,
// one 16-byte LDS read gives its four MFMA steps. Row-contiguous: the wave's
// rows form sets of SW = 16 NB; a read of NB consecutive rows of one k gives
// step p of the set's NB blocks, block b of which is rows NB c + b.
template <bool KC, int ROWS, int WROWS>
struct MidFrag {
    static constexpr int SW = WROWS < 64 ? WROWS : 64;
    static constexpr int NB = SW / 16;
    static constexpr int BLOCKS = WROWS / 16;
    static constexpr int READS = KC ? BLOCKS : 4 * (WROWS / SW);  // LDS reads per 16-k chunk
    typedef typename VecN<float, NB>::type nb_t;
    f4_t v[KC ? BLOCKS : 1];
    nb_t w[KC ? 1 : WROWS / SW][KC ? 1 : 4];

    template <typename ST>
    __device__ __forceinline__ void read(const float* s, int row0, int h, int lg, int c) {
        if constexpr (KC) {
#pragma unroll
            for (int i = 0; i < BLOCKS; ++i)
                v[i] = *reinterpret_cast<const f4_t*>(s + (row0 + 16 * i + c) * ST::PITCH + 16 * h + 4 * lg);
        } else {
#pragma unroll
            for (int t = 0; t < WROWS / SW; ++t)
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    w[t][p] = *reinterpret_cast<const nb_t*>(s + (16 * h + 4 * lg + p) * ST::PITCH + row0 + SW * t + NB * c);
        }
    }
    __device__ __forceinline__ float get(int i, int p) const {
        if constexpr (KC) return v[i][p];
        else return w[i / NB][p][i % NB];
    }
    // Row (of the wave's WROWS) that index x (0..15) of block i is.
    __device__ __forceinline__ static int row(int i, int x) { return KC ? 16 * i + x : SW * (i / NB) + NB * x + i % NB; }
};

template <bool TA, bool TB, bool FULL, int BM, int BN>
__global__ __launch_bounds__(kThreads, BM == 128 ? 2 : 3) void gemm_mid_f32_kernel(GemmArgs g) {
    constexpr int BK = kMidK, WM = BM / 2, WN = BN / 2;
    typedef Stage<float, BM, !TA, BK, 8, 0> SA;
    typedef Stage<float, BN, TB, BK, 8, 0> SB;
    typedef MidFrag<!TA, BM, WM> FA;
    typedef MidFrag<TB, BN, WN> FB;
    constexpr int MB = FA::BLOCKS, NBK = FB::BLOCKS;
    constexpr int NR = FA::READS + FB::READS;  // LDS reads per chunk
    constexpr int NL = SA::NC + SB::NC;        // loads (and stores) per thread and stage
    constexpr int NM = MB * NBK;               // MFMAs per step
    constexpr int BUF = SA::ELEMS + SB::ELEMS;
    __shared__ __attribute__((aligned(16))) float lds[2 * BUF];

    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t id0 = xcd_remap(blockIdx.x, tiles * g.batch);
    const int64_t bat = id0 / tiles, id = id0 - bat * tiles;
    constexpr int64_t GROUP = BM == 128 ? 4 : 8;
    const int64_t grp = id / (GROUP * g.tiles_n);
    const int64_t gm = min(GROUP, g.tiles_m - grp * GROUP);
    const int64_t rr = id - grp * GROUP * g.tiles_n;
    const int64_t tn = rr / gm, tm = grp * GROUP + rr % gm;
    const int64_t m0 = tm * BM, n0 = tn * BN;
    const float* A = static_cast<const float*>(g.A) + bat * g.sA;
    const float* B = static_cast<const float*>(g.B) + bat * g.sB;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int lg = lane >> 4, c = lane & 15;
    const int wm0 = (wave >> 1) * WM, wn0 = (wave & 1) * WN;

    f4_t acc[MB][NBK];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NBK; ++j) acc[i][j] = f4_t{0, 0, 0, 0};

    SA sa;
    SB sb;
    auto load = [&](int64_t s) __attribute__((always_inline)) {
        sa.template load<FULL>(A, g.lda, m0, g.M, s * BK);
        sb.template load<FULL>(B, g.ldb, n0, g.N, s * BK);
    };
    auto load_tail = [&](int64_t s) __attribute__((always_inline)) {
        sa.load_tail(A, g.lda, m0, g.M, s * BK, g.K);
        sb.load_tail(B, g.ldb, n0, g.N, s * BK, g.K);
    };
    auto store = [&](int buf) __attribute__((always_inline)) {
        sa.store(lds + buf * BUF);
        sb.store(lds + buf * BUF + SA::ELEMS);
    };
    // Pieces that were clamped at the matrix edge (uniform: edge tiles only).
    const bool edge_m = TA && !FULL && m0 + BM > g.M, edge_n = !TB && !FULL && n0 + BN > g.N;
    auto align = [&]() __attribute__((always_inline)) {
        if (edge_m) sa.align(m0, g.M);
        if (edge_n) sb.align(n0, g.N);
    };
    auto reads = [&](int buf, int h, FA& fa, FB& fb) __attribute__((always_inline)) {
        fa.template read<SA>(lds + buf * BUF, wm0, h, lg, c);
        fb.template read<SB>(lds + buf * BUF + SA::ELEMS, wn0, h, lg, c);
    };
    auto mfma = [&](const FA& fa, const FB& fb, int p0, int p1) __attribute__((always_inline)) {
#pragma unroll
        for (int p = p0; p < p1; ++p)
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NBK; ++j) acc[i][j] = Mfma<float>::mma(fa.get(i, p), fb.get(j, p), acc[i][j]);
    };

    const int64_t nk = (g.K + BK - 1) / BK, nfull = g.K / BK;
    FA fa0, fa1;
    FB fb0, fb1;
    if (nfull > 0) {
        load(0);
        align();
    } else {
        load_tail(0);
    }
    store(0);
    __syncthreads();
    reads(0, 0, fa0, fb0);
    int64_t st = 0;
    // Scheduling-group masks: 0x008 MFMA, 0x020 global load, 0x100 LDS read,
    // 0x200 LDS write.
    for (; st + 1 < nfull; ++st) {
        const int buf = (int)(st & 1);
        load(st + 1);
        reads(buf, 1, fa1, fb1);
        mfma(fa0, fb0, 0, 4);
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            if (i < NR) __builtin_amdgcn_sched_group_barrier(0x100, (NR + NL - 1) / NL, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 4 * NM / NL, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        mfma(fa1, fb1, 0, 1);
        __builtin_amdgcn_sched_barrier(0);
        align();
        store(buf ^ 1);
        mfma(fa1, fb1, 1, 3);
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 2 * NM / NL, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        reads(buf ^ 1, 0, fa0, fb0);
        mfma(fa1, fb1, 3, 4);
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, NM / NR, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    for (; st + 1 < nk; ++st) {
        const int buf = (int)(st & 1);
        load_tail(st + 1);
        reads(buf, 1, fa1, fb1);
        mfma(fa0, fb0, 0, 4);
        mfma(fa1, fb1, 0, 4);
        __builtin_amdgcn_sched_barrier(0);
        store(buf ^ 1);
        __syncthreads();
        reads(buf ^ 1, 0, fa0, fb0);
    }
    reads((int)(st & 1), 1, fa1, fb1);
    mfma(fa0, fb0, 0, 4);
    mfma(fa1, fb1, 0, 4);

    // D = alpha acc (+ beta C). D may alias C element for element: a row
    // block's C values are loaded before its stores.
    const float alpha = (float)g.alpha, beta = (float)g.beta;
    float* D = static_cast<float*>(g.D) + bat * g.sD;
    const float* C = g.C ? static_cast<const float*>(g.C) + bat * g.sC : nullptr;
    typedef typename Mem16<float>::type mem_t;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        if constexpr (!TB) {
            // Blocks 4 s .. 4 s + 3 of a lane are four consecutive columns.
            static_assert(FB::NB == 4, "16-byte pieces of D");
            f4_t cv[4][NBK / 4];
            if (C) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int s = 0; s < NBK / 4; ++s) {
                        const int64_t row = m0 + wm0 + FA::row(i, 4 * lg + r), col = n0 + wn0 + FB::row(4 * s, c);
                        const bool ok = FULL || (row < g.M && col + 4 <= g.N);
                        cv[r][s] = *reinterpret_cast<const mem_t*>(C + (ok ? row * g.ldc + col : 0));
                    }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int s = 0; s < NBK / 4; ++s) {
                    const int64_t row = m0 + wm0 + FA::row(i, 4 * lg + r), col = n0 + wn0 + FB::row(4 * s, c);
                    if (!FULL && (row >= g.M || col >= g.N)) continue;
                    f4_t v;
#pragma unroll
                    for (int b = 0; b < 4; ++b) v[b] = g.alpha != 1.0 ? alpha * acc[i][4 * s + b][r] : acc[i][4 * s + b][r];
                    if (FULL || col + 4 <= g.N) {
                        if (C) {
#pragma unroll
                            for (int b = 0; b < 4; ++b) v[b] = v[b] + beta * cv[r][s][b];
                        }
                        *reinterpret_cast<mem_t*>(D + row * g.ldd + col) = v;
                    } else {
#pragma unroll
                        for (int b = 0; b < 3; ++b)
                            if (col + b < g.N) {
                                float x = v[b];
                                if (C) x = x + beta * C[row * g.ldc + col + b];
                                D[row * g.ldd + col + b] = x;
                            }
                    }
                }
        } else {
            float cv[NBK][4];
            if (C) {
#pragma unroll
                for (int j = 0; j < NBK; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int64_t row = m0 + wm0 + FA::row(i, 4 * lg + r), col = n0 + wn0 + FB::row(j, c);
                        const bool ok = FULL || (row < g.M && col < g.N);
                        cv[j][r] = C[ok ? row * g.ldc + col : 0];
                    }
            }
#pragma unroll
            for (int j = 0; j < NBK; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + wm0 + FA::row(i, 4 * lg + r), col = n0 + wn0 + FB::row(j, c);
                    if (!FULL && (row >= g.M || col >= g.N)) continue;
                    float v = acc[i][j][r];
                    if (g.alpha != 1.0) v = alpha * v;
                    if (C) v = v + beta * cv[j][r];
                    D[row * g.ldd + col] = v;
                }
        }
    }
}

template <int BM, int BN>
int launch(bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    const int64_t total = g.tiles_m * g.tiles_n * g.batch;
    if (total > 0x7fffffffLL) return set_error(TT_UNSUPPORTED, "tt_gemm: %lld tiles exceed one launch", (long long)total);
    const bool full = g.M % BM == 0 && g.N % BN == 0;
    const dim3 grid((unsigned)total), block(kThreads);
#define TT_MID_CASE(TA, TB, F)             \
    if (ta == TA && tb == TB && full == F) \
        hipLaunchKernelGGL((gemm_mid_f32_kernel<TA, TB, F, BM, BN>), grid, block, 0, st, g);
    TT_MID_CASE(false, false, false)
    TT_MID_CASE(false, true, false)
    TT_MID_CASE(true, false, false)
    TT_MID_CASE(true, true, false)
    TT_MID_CASE(false, false, true)
    TT_MID_CASE(false, true, true)
    TT_MID_CASE(true, false, true)
    TT_MID_CASE(true, true, true)
#undef TT_MID_CASE
    return check_launch("tt_gemm");
}

}  // namespace

int gemm_mid_f32_launch(bool ta, bool tb, bool tall, GemmArgs& g, hipStream_t st) {
    return tall ? launch<128, 128>(ta, tb, g, st) : launch<64, 128>(ta, tb, g, st);
}

}  // namespace tt
