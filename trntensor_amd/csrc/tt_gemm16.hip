// 16-bit GEMM for bf16 / fp16 operands (dtype TT_BF16 / TT_F16 of tt_gemm):
//   D = alpha * op(A) op(B) (+ beta * C), products and sums in fp32 on
//   v_mfma_f32_16x16x32_{bf16,f16}, alpha/beta applied in fp32, one rounding
//   to the 16-bit type at the store.
//
// Workgroup: 256 threads = 4 wavefronts in a 2 x 2 grid over a BM x BN
// output tile (32 x 64 to 256 x 128), each wave (BM / 2) x (BN / 2) of
// 16 x 16 MFMA blocks with fp32 accumulators. K advances BK (64 or 32) per
// stage through two LDS buffers (one barrier per stage), the next stage's
// global loads held in registers during the current stage's MFMAs.
//
// MFMA operand layout (16x16x32): lane l holds A[l % 16][8 (l / 16) + j] and
// B[8 (l / 16) + j][l % 16], j = 0..7; accumulator element r holds
// D[4 (l / 16) + r][l % 16].
//
// Each operand is staged in its memory order, so staging is a plain copy:
//   k-contiguous operand: LDS [row][k], row pitch BK + 8 elements; a lane's
//     MFMA operand (8 consecutive k of one row) is one 16-byte read;
//   row-contiguous operand: LDS [k][row], k-row pitch ROWS + 16 elements;
//     a lane's MFMA operand is gathered across k-rows by two transposing
//     reads h = 0, 1 (ds_read_b64_tr_b16: within each 16 lanes, lane
//     16 g + 4 j + a supplies
//     the address of rows 4 a .. 4 a + 3 of k-row 8 g + 4 h + j, and lane
//     16 g + 4 a + b receives element b of the blocks of lanes 16 g + 4 j + a,
//     j = 0..3, i.e. k 8 g + 4 h .. 8 g + 4 h + 3 of row 4 a + b).
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "tt_gemm.hpp"

namespace tt {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
// The same 16 bytes in memory at the element's own alignment (gfx950 serves a
// 16-byte global access at any element address).
typedef unsigned short u16x8_mem __attribute__((ext_vector_type(8), aligned(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma16;
template <>
struct Mfma16<__bf16> {
    static __device__ __forceinline__ f32x4 mma(u16x8 a, u16x8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       c, 0, 0, 0);
    }
};
template <>
struct Mfma16<_Float16> {
    static __device__ __forceinline__ f32x4 mma(u16x8 a, u16x8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                      0, 0, 0);
    }
};

// One operand's ROWS x BK stage: global -> registers -> LDS, plus MFMA operand
// reads. KC: element (row, k) at p[row * ld + k], LDS [row][k]; otherwise at
// p[k * ld + row], LDS [k][row]. Each of the 256 threads copies NP 16-byte
// pieces that are consecutive in memory.
template <bool KC, int ROWS, int BK>
struct Stage16 {
    static constexpr int PITCH = KC ? BK + 8 : ROWS + 16;  // elements (16-byte multiple)
    static constexpr int ELEMS = KC ? ROWS * PITCH : BK * PITCH;
    static constexpr int LINE = KC ? BK / 8 : ROWS / 8;    // 16-byte pieces per LDS line
    static constexpr int NP = ROWS * BK / 8 / 256;         // pieces per thread
    static constexpr int TPL = LINE / NP;                  // threads per line
    static_assert(NP >= 1 && LINE % NP == 0 && BK % 32 == 0 && ROWS % 32 == 0, "stage split");
    u16x8 reg[NP];

    // Line (row for KC, k-row otherwise) and first element along it for this thread.
    __device__ __forceinline__ static void place(int& line, int& off) {
        line = threadIdx.x / TPL;
        off = (threadIdx.x % TPL) * NP * 8;
    }

    // A stage whose BK k are all in range: unconditional vector loads.
    // INSIDE: the tile's rows are too; otherwise a KC row past the end reads
    // the last row again and an RC piece that would pass the end starts at
    // rows - 8 instead (rows >= 8; align() moves its elements into place):
    // what lands in rows past the end feeds only outputs that are never
    // stored.
    template <bool INSIDE>
    __device__ __forceinline__ void load(const unsigned short* __restrict__ p, int64_t ld, int64_t row0, int64_t rows,
                                         int64_t k0) {
        int line, off;
        place(line, off);
        if (INSIDE || KC) {
            const int64_t row = INSIDE ? row0 + line : min(row0 + line, rows - 1);
            const unsigned short* src = KC ? p + row * ld + k0 + off : p + (k0 + line) * ld + row0 + off;
#pragma unroll
            for (int c = 0; c < NP; ++c) reg[c] = *reinterpret_cast<const u16x8_mem*>(src + 8 * c);
        } else {
#pragma unroll
            for (int c = 0; c < NP; ++c) {
                const int64_t row = min(row0 + off + 8 * c, rows - 8);
                reg[c] = *reinterpret_cast<const u16x8_mem*>(p + (k0 + line) * ld + row);
            }
        }
    }

    // After a clamped load of an RC operand: each piece that was started early
    // is moved down by its overshoot.
    __device__ __forceinline__ void align(int64_t row0, int64_t rows) {
        if (KC) return;
        int line, off;
        place(line, off);
        typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int c = 0; c < NP; ++c) {
            const int64_t over = row0 + off + 8 * c + 8 - rows;  // <= 0: not clamped; >= 8: no row inside
            if (over <= 0 || over >= 8) continue;
            const int sh = 16 * (int)over;
            u64x2 x = __builtin_bit_cast(u64x2, reg[c]);
            if (sh < 64) {
                x[0] = (x[0] >> sh) | (x[1] << (64 - sh));
                x[1] = x[1] >> sh;
            } else {
                x[0] = x[1] >> (sh - 64);
                x[1] = 0;
            }
            reg[c] = __builtin_bit_cast(u16x8, x);
        }
    }

    // The stage that passes K (zero from there), and every stage when an RC
    // operand has fewer than 8 rows: a piece wholly inside is one vector load,
    // one wholly outside is zero without a load, and only a piece that
    // straddles the edge is loaded element by element from clamped addresses.
    __device__ __forceinline__ void load_tail(const unsigned short* __restrict__ p, int64_t ld, int64_t row0,
                                              int64_t rows, int64_t k0, int64_t kdim) {
        int line, off;
        place(line, off);
#pragma unroll
        for (int c = 0; c < NP; ++c) {
            // Piece start (gr, gk) and its extent along the contiguous direction.
            const int64_t gr = row0 + (KC ? line : off + 8 * c);
            const int64_t gk = k0 + (KC ? off + 8 * c : line);
            const bool inside = KC ? (gr < rows && gk + 8 <= kdim) : (gk < kdim && gr + 8 <= rows);
            const bool outside = gr >= rows || gk >= kdim;
            if (inside) {
                reg[c] = *reinterpret_cast<const u16x8_mem*>(KC ? p + gr * ld + gk : p + gk * ld + gr);
            } else if (outside) {
                reg[c] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int64_t r = gr + (KC ? 0 : e), k = gk + (KC ? e : 0);
                    const bool ok = r < rows && k < kdim;
                    const unsigned short x = *(ok ? (KC ? p + r * ld + k : p + k * ld + r) : p);
                    reg[c][e] = ok ? x : (unsigned short)0;
                }
            }
        }
    }

    __device__ __forceinline__ void store(unsigned short* s) const {
        int line, off;
        place(line, off);
        unsigned short* dst = s + line * PITCH + off;
#pragma unroll
        for (int c = 0; c < NP; ++c) *reinterpret_cast<u16x8*>(dst + 8 * c) = reg[c];
    }

    // This lane's MFMA operand for the 16 rows from rb, k step ks (k 32 ks .. 32 ks + 31).
    __device__ __forceinline__ static u16x8 frag(const unsigned short* s, int rb, int ks, int lane) {
        if (KC) return *reinterpret_cast<const u16x8*>(s + (rb + (lane & 15)) * PITCH + 32 * ks + 8 * (lane >> 4));
        const int g = lane >> 4, j = (lane & 15) >> 2, a = lane & 3;
        const unsigned short* base = s + (32 * ks + 8 * g + j) * PITCH + rb + 4 * a;
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(base));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(base + 4 * PITCH));
        return u16x8{(unsigned short)lo[0], (unsigned short)lo[1], (unsigned short)lo[2], (unsigned short)lo[3],
                     (unsigned short)hi[0], (unsigned short)hi[1], (unsigned short)hi[2], (unsigned short)hi[3]};
    }
};

template <typename T>
__device__ __forceinline__ float to_f32(unsigned short x) {
    return (float)__builtin_bit_cast(T, x);
}
template <typename T>
__device__ __forceinline__ unsigned short from_f32(float x) {
    return __builtin_bit_cast(unsigned short, (T)x);
}

// FULL: M and N are multiples of the tile (no row or column clamping).
template <typename T, bool TA, bool TB, bool FULL, int BM, int BN, int BK>
__global__ __launch_bounds__(256) void gemm16_kernel(GemmArgs g) {
    // A rows are m: k-contiguous unless transposed. B rows are n: k-contiguous iff transposed.
    typedef Stage16<!TA, BM, BK> SA;
    typedef Stage16<TB, BN, BK> SB;
    // Four wavefronts in a 2 x 2 grid, each FM x FN MFMA blocks of 16 x 16.
    constexpr int WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
    __shared__ __attribute__((aligned(16))) unsigned short lds[2 * (SA::ELEMS + SB::ELEMS)];
    auto bufA = [&](int b) -> unsigned short* { return lds + b * SA::ELEMS; };
    auto bufB = [&](int b) -> unsigned short* { return lds + 2 * SA::ELEMS + b * SB::ELEMS; };

    const int64_t tiles = g.tiles_m * g.tiles_n;
    const int64_t total = tiles * g.batch;
    const int64_t id = xcd_remap(blockIdx.x, total);
    const int64_t bat = id / tiles;
    const int64_t t = id - bat * tiles;
    constexpr int64_t GROUP = 8;
    const int64_t grp = t / (GROUP * g.tiles_n);
    const int64_t first_m = grp * GROUP;
    const int64_t gsize = min(g.tiles_m - first_m, GROUP);
    const int64_t rem = t - grp * GROUP * g.tiles_n;
    const int64_t m0 = (first_m + rem % gsize) * BM;
    const int64_t n0 = (rem / gsize) * BN;

    const unsigned short* A = static_cast<const unsigned short*>(g.A) + bat * g.sA;
    const unsigned short* B = static_cast<const unsigned short*>(g.B) + bat * g.sB;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm0 = (wave >> 1) * WM;
    const int wn0 = (wave & 1) * WN;
    const int lrow = lane & 15;
    const int lg = lane >> 4;

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0, 0, 0, 0};

    SA sa;
    SB sb;
    const int64_t nk = (g.K + BK - 1) / BK;
    // Stages 0 .. nfull-1 have all their k in range (a row-contiguous operand
    // with fewer rows than one vector takes the guarded loads throughout).
    const int64_t nfull = (!TA || g.M >= 8) && (TB || g.N >= 8) ? g.K / BK : 0;
    auto load = [&](int64_t k0) __attribute__((always_inline)) {
        sa.template load<FULL>(A, g.lda, m0, g.M, k0);
        sb.template load<FULL>(B, g.ldb, n0, g.N, k0);
    };
    auto load_tail = [&](int64_t k0) __attribute__((always_inline)) {
        sa.load_tail(A, g.lda, m0, g.M, k0, g.K);
        sb.load_tail(B, g.ldb, n0, g.N, k0, g.K);
    };
    // Pieces that were clamped at the matrix edge (uniform: edge tiles only).
    const bool edge_m = TA && !FULL && m0 + BM > g.M, edge_n = !TB && !FULL && n0 + BN > g.N;
    auto align = [&]() __attribute__((always_inline)) {
        if (edge_m) sa.align(m0, g.M);
        if (edge_n) sb.align(n0, g.N);
    };
    auto compute = [&](int buf) {
        const unsigned short* a = bufA(buf);
        const unsigned short* b = bufB(buf);
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks) {
            u16x8 fa[FM], fb[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[i] = SA::frag(a, wm0 + 16 * i, ks, lane);
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[j] = SB::frag(b, wn0 + 16 * j, ks, lane);
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = Mfma16<T>::mma(fa[i], fb[j], acc[i][j]);
        }
    };
    int64_t kt = 0;
    if (nk > 0) {
        if (nfull > 0) {
            load(0);
            align();
        } else {
            load_tail(0);
        }
        sa.store(bufA(0));
        sb.store(bufB(0));
    }
    __syncthreads();
    for (; kt + 1 < nfull; ++kt) {
        load((kt + 1) * BK);
        compute(kt & 1);
        __builtin_amdgcn_sched_barrier(0);
        align();
        sa.store(bufA((kt & 1) ^ 1));
        sb.store(bufB((kt & 1) ^ 1));
        __syncthreads();
    }
    // Buffer kt & 1 holds stage kt; the remaining stages load one ahead.
    for (; kt < nk; ++kt) {
        const bool more = kt + 1 < nk;
        if (more) load_tail((kt + 1) * BK);
        compute(kt & 1);
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
            sa.store(bufA((kt & 1) ^ 1));
            sb.store(bufB((kt & 1) ^ 1));
        }
        __syncthreads();
    }

    // Epilogue through LDS (free after the last barrier): each wave writes one
    // 16-row slab of its tile as fp32 with alpha applied, then each lane
    // finishes 8 consecutive columns of one row with a 16-byte load of C and a
    // 16-byte store of D (element-wise at ragged or unaligned edges).
    const unsigned short* C = g.C ? static_cast<const unsigned short*>(g.C) + bat * g.sC : nullptr;
    unsigned short* D = static_cast<unsigned short*>(g.D) + bat * g.sD;
    const float alpha = (float)g.alpha;
    const float beta = (float)g.beta;
    constexpr int SP = WN + 4;  // slab pitch in floats (16-byte multiple)
    static_assert(4 * 16 * SP * sizeof(float) <= sizeof(lds), "epilogue slabs fit in the stage buffers");
    float* slab = reinterpret_cast<float*>(lds) + wave * 16 * SP;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        // This slab's C chunks are loaded before any of its stores (and before the
        // slab exchange, whose barrier then covers their latency): D may
        // alias C, so the compiler cannot move a load of C past a store of D,
        // and chunk-by-chunk loads would each wait out a full memory latency.
        u16x8 cc[WN / 32];
#pragma unroll
        for (int h = 0; h < WN / 32; ++h) {
            const int v = lane + 64 * h;
            const int rr = v / (WN / 8), cb = v % (WN / 8);
            const int64_t row = m0 + wm0 + 16 * i + rr;
            const int64_t col = n0 + wn0 + 8 * cb;
            cc[h] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (C && row < g.M && col + 8 <= g.N) cc[h] = *reinterpret_cast<const u16x8_mem*>(C + row * g.ldc + col);
        }
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = acc[i][j][r];
                if (g.alpha != 1.0) v = alpha * v;
                slab[(4 * lg + r) * SP + 16 * j + lrow] = v;
            }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < WN / 32; ++h) {
            const int v = lane + 64 * h;
            const int rr = v / (WN / 8), cb = v % (WN / 8);
            const int64_t row = m0 + wm0 + 16 * i + rr;
            const int64_t col = n0 + wn0 + 8 * cb;
            const f32x4 lo = *reinterpret_cast<const f32x4*>(slab + rr * SP + 8 * cb);
            const f32x4 hi = *reinterpret_cast<const f32x4*>(slab + rr * SP + 8 * cb + 4);
            float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if (row < g.M) {
                if (col + 8 <= g.N) {
                    if (C) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) x[e] = x[e] + beta * to_f32<T>(cc[h][e]);
                    }
                    u16x8 d;
#pragma unroll
                    for (int e = 0; e < 8; ++e) d[e] = from_f32<T>(x[e]);
                    *reinterpret_cast<u16x8_mem*>(D + row * g.ldd + col) = d;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (col + e < g.N) {
                            float y = x[e];
                            if (C) y = y + beta * to_f32<T>(C[row * g.ldc + col + e]);
                            D[row * g.ldd + col + e] = from_f32<T>(y);
                        }
                }
            }
        }
        __syncthreads();
    }
}

template <typename T, int BM, int BN, int BK>
int launch16(bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    const int64_t total = g.tiles_m * g.tiles_n * g.batch;
    if (total > 0x7fffffffLL) return set_error(TT_UNSUPPORTED, "tt_gemm: %lld tiles exceed one launch", (long long)total);
    if (total > kMaxGrid) {
        GemmArgs lo = g, hi = g;
        split_gemm(2, ta, tb, 256, lo, hi);
        const int rc = launch16<T, BM, BN, BK>(ta, tb, lo, st);
        return rc == TT_OK ? launch16<T, BM, BN, BK>(ta, tb, hi, st) : rc;
    }
    const bool full = g.M % BM == 0 && g.N % BN == 0;
    const dim3 grid((unsigned)total), block(256);
#define TT_GEMM16_CASE(TA, TB, F)           \
    if (ta == TA && tb == TB && full == F) \
        hipLaunchKernelGGL((gemm16_kernel<T, TA, TB, F, BM, BN, BK>), grid, block, 0, st, g);
    TT_GEMM16_CASE(false, false, false)
    TT_GEMM16_CASE(false, false, true)
    TT_GEMM16_CASE(false, true, false)
    TT_GEMM16_CASE(false, true, true)
    TT_GEMM16_CASE(true, false, false)
    TT_GEMM16_CASE(true, false, true)
    TT_GEMM16_CASE(true, true, false)
    TT_GEMM16_CASE(true, true, true)
#undef TT_GEMM16_CASE
    return check_launch("tt_gemm (16-bit)");
}

int64_t up(int64_t n, int64_t t) { return (n + t - 1) / t; }

// Estimated time of the busiest CU (arbitrary units): its bm x bn tiles times
// their area, times the kernel's cost per output where every CU has many
// tiles, times what a single tile on a CU loses because nothing covers its
// latencies.
double cost16(const GemmArgs& g, int64_t bm, int64_t bn, double per_output, double one) {
    const int64_t rounds = up(up(g.M, bm) * up(g.N, bn) * g.batch, device_cus());
    return (double)(rounds * bm * bn) * per_output * (rounds == 1 ? one : 1.0);
}

// The register-staged kernel's tile: 0: 128 x 128, 1: 64 x 64, 2: 32 x 64. us
// measured (bf16): 787 x 423 x 3415 106/51/40 (336 with element-wise loads of
// the odd rows on 128 x 128), 4332 x 1643 x 1352 TT 48/59/86 (241), 2001 x 3003 x
// 1001 49/45/58 (172), 684 x 5650 x 287 22/13/16 (53), 1236 x 2965 x 167 TT
// 16/12/14 (32), 1672 x 194 x 241 TT 11.6/6.6/5.8 (27), 1024^3 17.6/10.8/10.7,
// 1591 x 225 x 5665 219/80/63 (527). 64 x 128 tiles were within 5% of the best of
// these or behind it, 128-deep stages 10% faster on 32 x 64 with B
// k-contiguous and few tiles, up to 1.6 times slower elsewhere.
double staged_cost(const GemmArgs& g, int* tile) {
    const double c[3] = {cost16(g, 128, 128, 1.0, 1.5), cost16(g, 64, 64, 1.3, 1.5), cost16(g, 32, 64, 1.8, 1.5)};
    *tile = (int)(std::min_element(c, c + 3) - c);
    return c[*tile];
}

// Register-staged kernel (any shape, alignment and K).
template <typename T>
int gemm16_staged(bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    // Many tiles with A row-contiguous: 256 x 128 tiles of depth 32 (4096^3,
    // bf16: 934-939 against 840-862 TFLOP/s on 128 x 128 x 64; 4095^3 TN 202
    // against 329 us).
    if (ta && up(g.M, 256) * up(g.N, 128) * g.batch >= 512) return launch16<T, 256, 128, 32>(ta, tb, g, st);
    int tile;
    staged_cost(g, &tile);
    if (tile == 2) return launch16<T, 32, 64, 64>(ta, tb, g, st);
    if (tile == 1) return launch16<T, 64, 64, 64>(ta, tb, g, st);
    return launch16<T, 128, 128, 64>(ta, tb, g, st);
}

template <typename T>
int gemm16_typed(bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    auto ok16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    bool vec = ok16(g.A) && ok16(g.B) && g.lda % 8 == 0 && g.ldb % 8 == 0;
    if (g.batch > 1) vec = vec && g.sA % 8 == 0 && g.sB % 8 == 0;
    // The direct-load kernel needs K deep enough to amortise its prologue and
    // epilogue. With its 128 x 256 tiles
    // it is level or ahead from K = 256 in every layout (bf16, 64 x 512^2 x 256:
    // NN 370-374 against 338-342 TFLOP/s, NT 389-409 against 338-346, TN
    // 398-403 against 400-401, TT 419 against 392-396; 64 x 512^3: 588-669
    // against 508-562).
    const int64_t kmin = 256;
    // The ragged strips run as separate, serial launches, so they are limited
    // to 1/64 of the outputs (2000 x 3000 x 320, 5.8% in strips: 42-48 against
    // 71-75 TFLOP/s on the register-staged kernel alone). On its 128 x 256 or 128
    // x 128 tiles the kernel costs 0.7 of the staged 128 x 128 tile's time per
    // output (4096^3 NN 120 against 172 us, 2048^3 33 against 44), so smaller
    // staged tiles take the grids that leave its CUs idle (2048^3 40 us on 64 x
    // 64; 1024^3 17.7 against 10.7 us).
    int bm_, bn_;
    gemm16_dma_tile(ta, tb, g.M, g.N, g.K, g.batch, bm_, bn_);
    const int64_t bm = bm_, bn = bn_;
    const int64_t Mi = g.M & ~(bm - 1), Ni = g.N & ~(bn - 1);
    const bool small_strips = (g.M - Mi) * g.N + Mi * (g.N - Ni) <= g.M * g.N / 64;
    if (!vec || g.M < bm || g.N < bn || g.K < kmin || g.K % 32 != 0 || !small_strips)
        return gemm16_staged<T>(ta, tb, g, st);
    int tile;
    if (cost16(g, bm, bn, 0.7, 1.5) > staged_cost(g, &tile)) return gemm16_staged<T>(ta, tb, g, st);
    // Whole bm x bn tiles by the direct-load kernel; the ragged row and
    // column strips (if any) by the register-staged kernel on sub-matrices.
    const unsigned short* A = static_cast<const unsigned short*>(g.A);
    const unsigned short* B = static_cast<const unsigned short*>(g.B);
    const unsigned short* C = static_cast<const unsigned short*>(g.C);
    unsigned short* D = static_cast<unsigned short*>(g.D);
    GemmArgs gi = g;
    gi.M = Mi;
    gi.N = Ni;
    int rc = gemm16_dma_dispatch(std::is_same<T, __bf16>::value ? TT_BF16 : TT_F16, ta, tb, gi, st);
    if (rc == TT_OK && Mi < g.M) {
        GemmArgs ge = g;
        ge.M = g.M - Mi;
        ge.A = ta ? A + Mi : A + Mi * g.lda;
        ge.C = C ? C + Mi * g.ldc : nullptr;
        ge.D = D + Mi * g.ldd;
        rc = gemm16_staged<T>(ta, tb, ge, st);
    }
    if (rc == TT_OK && Ni < g.N) {
        GemmArgs ge = g;
        ge.M = Mi;
        ge.N = g.N - Ni;
        ge.B = tb ? B + Ni * g.ldb : B + Ni;
        ge.C = C ? C + Ni : nullptr;
        ge.D = D + Ni;
        rc = gemm16_staged<T>(ta, tb, ge, st);
    }
    return rc;
}

}  // namespace

int gemm16_dispatch(int dtype, bool ta, bool tb, GemmArgs& g, hipStream_t st) {
    if (dtype == TT_BF16) return gemm16_typed<__bf16>(ta, tb, g, st);
    return gemm16_typed<_Float16>(ta, tb, g, st);
}

}  // namespace tt
