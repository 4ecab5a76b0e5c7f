// LDS staging of one GEMM operand: the piece of the fp32/fp64 kernels that
// copies a ROWS x BK stage from memory through registers into LDS and reads
// MFMA fragments from it.
#pragma once

#include "tt_common.hpp"

namespace tt {

constexpr int kBK = 16;
constexpr int kThreads = 256;


// 16 bytes of T in memory at T's own alignment. gfx950 serves a 16-byte global
// access at any element address, so operands, leading dimensions and batch
// strides of any parity take the vector loads and stores; an access that is
// not 16-byte aligned only touches one cache line more now and then.
template <typename T>
struct Mem16 {
    typedef T type __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
};

// One operand's ROWS x BK stage: global -> registers -> LDS, plus fragment reads.
// KC: element (row, k) at p[row * ld + k]; otherwise at p[k * ld + row].
// Each thread stages E = ROWS * BK / 256 elements as NC 16-byte pieces:
//   KC: row t / TPK; BK = 16: one contiguous chunk from k = (t % TPK) E; deeper
//       stages: pieces (t % TPK) + TPK c, so an instruction's lanes read
//       TPK * 16 contiguous bytes of each row;
//   RC: TPR threads per k-row, k-rows t / TPR + (256 / TPR) j; within a k-row a
//       thread's pieces are (t % TPR) + TPR c, so every instruction covers
//       TPR * 16 contiguous bytes of the k-row (coalesced loads,
//       conflict-free stores).
// RC k-rows are padded by 4 elements: the four lane groups of a fragment read
// (k-rows 4 g + s) then land on disjoint LDS banks.
template <typename T, int ROWS, bool KC, int BK, int KPAD = 16 / sizeof(T), int RPAD = 4>
struct Stage {
    static constexpr int V = Vec16<T>::n;
    static constexpr int E = ROWS * BK / kThreads;
    static constexpr int NC = E / V;                              // 16-byte pieces per thread
    static constexpr int TPK = BK / E;                            // KC: threads per row
    static constexpr int TPR = ROWS / V < 16 ? ROWS / V : 16;     // RC: threads per k-row
    static constexpr int NCR = KC ? NC : ROWS / (TPR * V);        // RC: pieces per k-row and thread
    static constexpr int PITCH = KC ? (BK + KPAD) : (ROWS + RPAD);
    static constexpr int ELEMS = KC ? ROWS * PITCH : BK * PITCH;
    static_assert(BK % 16 == 0 && E % V == 0 && (KC ? BK % E == 0 : (NC % NCR == 0 && NCR >= 1)), "stage split");
    typedef typename Vec16<T>::type vec_t;
    typedef typename Mem16<T>::type mem_t;

    vec_t reg[NC];

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < V; ++e) reg[c][e] = T(0);
    }

    __device__ __forceinline__ static void place(int& row, int& k) {
        const int t = threadIdx.x;
        if (KC) {
            row = t / TPK;
            k = (t % TPK) * (BK == 16 ? E : V);
        } else {
            k = t / TPR;
            row = (t % TPR) * V;
        }
    }
    // Offsets of piece c relative to piece 0: along the rows and along k.
    __device__ __forceinline__ static constexpr int prow(int c) { return KC ? 0 : (c % NCR) * TPR * V; }
    __device__ __forceinline__ static constexpr int pk(int c) {
        return KC ? (BK == 16 ? c * V : c * TPK * V) : (c / NCR) * (kThreads / TPR);
    }

    // A stage whose BK k are all in range: unconditional vector loads.
    // INSIDE: the tile's rows are too. Otherwise rows from `rows` up are
    // clamped: a KC row past the end reads the last row again, an RC piece
    // that would pass the end starts at rows - V instead (rows >= V) and
    // store() moves its elements into place; what lands in rows past the end
    // feeds only outputs that are never stored. Ragged matrices so run the
    // same branch-free loop as whole tiles; guarded piece by piece
    // and loaded element by element when unaligned, as before, the edge
    // tiles set the time of the launch (fp32 1999 x 3001 x 1201 with
    // alpha/beta and C, all odd: 150 us against 224).
    // SKIP: pieces wholly past the edge are not loaded and keep what the
    // registers held (clear() them first), for kernels with tiles that lie mostly
    // past it.
    template <bool INSIDE, bool SKIP = false>
    __device__ __forceinline__ void load(const T* __restrict__ p, int64_t ld, int64_t row0, int64_t rows, int64_t k0) {
        int r, k;
        place(r, k);
        if (!INSIDE && SKIP && KC && row0 + r >= rows) return;
        if (INSIDE || KC) {
            const int64_t row = INSIDE ? row0 + r : min(row0 + r, rows - 1);
            const T* src = KC ? p + row * ld + (k0 + k) : p + (k0 + k) * ld + row;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const mem_t* q = reinterpret_cast<const mem_t*>(KC ? src + pk(c) : src + pk(c) * ld + prow(c));
                reg[c] = *q;
            }
        } else {
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (SKIP && row0 + r + prow(c) >= rows) continue;
                const int64_t row = min(row0 + r + prow(c), rows - V);
                const mem_t* q = reinterpret_cast<const mem_t*>(p + (k0 + k + pk(c)) * ld + row);
                reg[c] = *q;
            }
        }
    }

    // The stage that passes K (zero from there), and every stage when an RC
    // operand has fewer than V rows: a piece wholly inside is one vector
    // load, one wholly outside is zero without a load, and only a piece
    // straddling the edge is loaded element-wise from clamped addresses.
    // Rows past `rows` are zero; store() must not move them.
    __device__ __forceinline__ void load_tail(const T* __restrict__ p, int64_t ld, int64_t row0, int64_t rows,
                                              int64_t k0, int64_t kdim) {
        int r, k;
        place(r, k);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int64_t pr = row0 + r + prow(c);
            const int64_t pkk = k0 + k + pk(c);
            const bool inside = KC ? (pr < rows && pkk + V <= kdim) : (pkk < kdim && pr + V <= rows);
            const bool outside = pr >= rows || pkk >= kdim;
            if (inside) {
                reg[c] = *reinterpret_cast<const mem_t*>(KC ? p + pr * ld + pkk : p + pkk * ld + pr);
            } else if (outside) {
#pragma unroll
                for (int e = 0; e < V; ++e) reg[c][e] = T(0);
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    const int64_t gr = pr + (KC ? 0 : e);
                    const int64_t gk = pkk + (KC ? e : 0);
                    const bool ok = gr < rows && gk < kdim;
                    const T x = *(ok ? (KC ? p + gr * ld + gk : p + gk * ld + gr) : p);
                    reg[c][e] = ok ? x : T(0);
                }
            }
        }
    }

    __device__ __forceinline__ void store(T* s) const {
        int r, k;
        place(r, k);
        T* dst = KC ? (s + r * PITCH + k) : (s + k * PITCH + r);
#pragma unroll
        for (int c = 0; c < NC; ++c)
            *reinterpret_cast<vec_t*>(KC ? dst + pk(c) : dst + pk(c) * PITCH + prow(c)) = reg[c];
    }

    // After a clamped load<false> of an RC operand: each piece that was
    // started early is moved down by its overshoot.
    __device__ __forceinline__ void align(int64_t row0, int64_t rows) {
        if (KC) return;
        int r, k;
        place(r, k);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int64_t over = row0 + r + prow(c) + V - rows;  // <= 0: not clamped; >= V: no row inside
            const int s = over > 0 ? (int)over : 0;
            vec_t x = reg[c];
            if constexpr (V == 4) {
                const vec_t y = (s & 2) ? vec_t{x[2], x[3], x[0], x[1]} : x;
                reg[c] = (s & 1) ? vec_t{y[1], y[2], y[3], y[0]} : y;
            } else {
                reg[c] = (s & 1) ? vec_t{x[1], x[0]} : x;
            }
        }
    }

    // The four k values (MFMA steps 0..3 of 16-k pass kk) this lane feeds for
    // the 16-row block at rb.
    __device__ __forceinline__ static void frag(const T* s, int rb, int lane, int kk, T out[4]) {
        const int r = rb + (lane & 15);
        const int g = lane >> 4;
        if (KC) {
            typedef typename VecN<T, 4>::type v4_t;
            const v4_t x = *reinterpret_cast<const v4_t*>(s + r * PITCH + 16 * kk + 4 * g);
#pragma unroll
            for (int st = 0; st < 4; ++st) out[st] = x[st];
        } else {
#pragma unroll
            for (int st = 0; st < 4; ++st) out[st] = s[(16 * kk + 4 * g + st) * PITCH + r];
        }
    }
};

}  // namespace tt
