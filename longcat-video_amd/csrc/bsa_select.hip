// Pooled-score GEMM (MFMA) and deterministic per-row top-k selection.
//
// score[bh, m, n] = sum_d q_cmp[bh, m, d] * k_cmp[bh, n, d]   (fp32 accumulate,
// one rounding to the storage type, no softmax scale).
//
// Top-k: each wavefront owns one score row and holds it in registers as
// order-preserving integer images of the scores.  The k-th largest score VALUE
// is found by a bitwise binary search whose counting step is a wavefront
// ballot + popcount; every column above it wins, and of the columns equal to it
// the lowest-indexed ones that are still needed ("larger score, or equal score
// and lower index").  Walking the registers in column order emits the list in
// ascending block order directly; the descending-score list (a total order
// through keys that append the inverted column index to the score image) is
// ranked in LDS only when it is asked for.  The CDF rule counts with the same
// value search over masked sums of softmax weights.
#include "bsa_gate.h"
#include "bsa_mfma.h"

namespace bsa {
namespace {

using mfma::f32x16;
using mfma::mfma32;
using mfma::Vec8;

// ---------------------------------------------------------------- score GEMM
// Workgroup = 4 wavefronts = 128 score rows x up to kScoreCols columns.  The pooled key rows of the workgroup's
// columns (64 KB) are staged in LDS once, with fully coalesced loads; each wavefront keeps its 32 pooled query rows
// (all 128 d, the A operand) in registers and walks the 32-column tiles, reading the B fragments from LDS (lane l:
// row l%32 of the tile, the 8 consecutive d values 16*s + 8*(l/32) .. +8 of k-step s).  Read from global memory
// fragment by fragment instead, every load instruction touches 32 rows for 32 bytes each and the four wavefronts
// ask for the same rows again: the L1 path, not the 17 GFLOP of arithmetic, then sets the time (0.107 ms at
// 1440 x 1440 x 32 heads).  A finished 32x32 tile goes through a wavefront-private LDS patch so that it leaves
// as 16-byte stores (half a row per lane) instead of 2-byte ones.
constexpr int kScoreCols = 256;
constexpr int kScorePitch = 128 + 8;     // elements: 272-byte rows keep 16-byte alignment and spread the banks
// key_norm[bh] = the largest entry of the head's tile norms (a NaN row has no bound), by one wavefront
__device__ inline void head_norm(const HeadNorms& n, int bh, int lane) {
    float best = 0.f;
    for (int i0 = lane; i0 < n.tiles; i0 += 8 * 64) {          // eight requests in flight: the workgroup waits for this wavefront
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = n.tile_norm[(int64_t)bh * n.tiles + min(i0 + 64 * j, n.tiles - 1)];
#pragma unroll
        for (int j = 0; j < 8; ++j) best = x[j] != x[j] ? INFINITY : fmaxf(best, x[j]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) best = fmaxf(best, __shfl_xor(best, off));
    if (lane == 0) n.key_norm[bh] = best;
}
template <typename T>
__global__ __launch_bounds__(256) void score_mfma_kernel(const T* __restrict__ qc,
                                                         const T* __restrict__ kc,
                                                         T* __restrict__ score, int nbq, int nbk, HeadNorms norms) {
    typedef typename Vec8<T>::type V8;
    constexpr int D = 128;
    __shared__ __attribute__((aligned(16))) T keys[kScoreCols * kScorePitch];
    __shared__ __attribute__((aligned(16))) T patch[4][32][40];      // 80-byte rows: 16-byte aligned, bank-spread
    const int bh = blockIdx.z;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int m0 = blockIdx.y * 128 + wave * 32;
    const int n_begin = blockIdx.x * kScoreCols;
    const int n_end = min(n_begin + kScoreCols, nbk);
    const int lr = lane & 31, lh = lane >> 5;
    // the key rows of this workgroup's columns: 16 pieces of 16 bytes per row, consecutive threads on consecutive pieces
    {
        const T* kb = kc + ((int64_t)bh * nbk) * D;
        uint4 piece[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int e = threadIdx.x + 256 * i, r = e >> 4, c = e & 15;
            piece[i] = *reinterpret_cast<const uint4*>(kb + (int64_t)min(n_begin + r, nbk - 1) * D + c * 8);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int e = threadIdx.x + 256 * i, r = e >> 4, c = e & 15;
            *reinterpret_cast<uint4*>(keys + r * kScorePitch + c * 8) = piece[i];
        }
    }
    const int mrow = min(m0 + lr, nbq - 1);   // clamp: rows past the end are computed, not stored
    const T* qa = qc + ((int64_t)bh * nbq + mrow) * D + lh * 8;
    V8 a[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) a[s] = *reinterpret_cast<const V8*>(qa + s * 16);
    __syncthreads();
    if (norms.tile_norm != nullptr && blockIdx.x == 0 && blockIdx.y == gridDim.y - 1 && wave == 3) head_norm(norms, bh, lane);
    if (m0 >= nbq) return;                    // whole wavefront out of range (no workgroup barrier below)
    T (*mine)[40] = patch[wave];
    const bool vec_ok = (nbk % 8) == 0;       // rows of the score matrix stay 16-byte aligned
    for (int n0 = n_begin; n0 < n_end; n0 += 32) {
        const T* kt = keys + (n0 - n_begin + lr) * kScorePitch + lh * 8;
        V8 b[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) b[s] = *reinterpret_cast<const V8*>(kt + s * 16);
        f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int s = 0; s < 8; ++s) acc = mfma32(a[s], b[s], acc);
        // accumulator i of lane l: row 8*(i/4) + 4*(l/32) + i%4, column l%32
#pragma unroll
        for (int i = 0; i < 16; ++i) mine[8 * (i / 4) + 4 * lh + (i % 4)][lr] = (T)acc[i];
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wavefront's LDS writes have landed
        __builtin_amdgcn_wave_barrier();
        const int r = lane >> 1, c0 = (lane & 1) * 16;
        const int m = m0 + r;
        if (m < nbq) {
            T* dst = score + ((int64_t)bh * nbq + m) * nbk + n0 + c0;
            if (vec_ok && n0 + c0 + 16 <= nbk) {
                *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(&mine[r][c0]);
                *reinterpret_cast<uint4*>(dst + 8) = *reinterpret_cast<const uint4*>(&mine[r][c0 + 8]);
            } else {
                for (int c = 0; c < 16 && n0 + c0 + c < nbk; ++c) dst[c] = mine[r][c0 + c];
            }
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);   // the patch is read before the next tile overwrites it
        __builtin_amdgcn_wave_barrier();
    }
}

__global__ __launch_bounds__(256) void score_f32_kernel(const float* __restrict__ qc, const float* __restrict__ kc,
                                                        float* __restrict__ score, int nbq, int nbk) {
    constexpr int D = 128;
    const int bh = blockIdx.z, lane = threadIdx.x & 63, n16 = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 64 + (threadIdx.x >> 6) * 16;
    if (n0 >= nbk) return;
    f32x4 a[8], b[8];
    score_row_f32(qc + ((int64_t)bh * nbq + min(m0 + n16, nbq - 1)) * D + 4 * g, a);
    score_row_f32(kc + ((int64_t)bh * nbk + min(n0 + n16, nbk - 1)) * D + 4 * g, b);
    const f32x4 acc = score_tile_f32(a, b);
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (m0 + 4 * g + i < nbq && n0 + n16 < nbk) score[((int64_t)bh * nbq + m0 + 4 * g + i) * nbk + n0 + n16] = acc[i];
}

// ---------------------------------------------------------------- top-k
// Top-k from a score matrix in memory: one wavefront per score row.
template <typename S, int NPL, bool SCORE_ORDER>
__global__ __launch_bounds__(256) void topk_kernel(const S* __restrict__ score,
                                                   int32_t* __restrict__ idx_out,
                                                   int32_t* __restrict__ idx_sorted_out,
                                                   int32_t* __restrict__ lens_out, int64_t rows,
                                                   int nbk, int k_all, const int32_t* __restrict__ k_rows,
                                                   int stride) {
    typedef typename KeyOf<S>::type K;
    extern __shared__ __attribute__((aligned(16))) unsigned char topk_keys[];    // SCORE_ORDER: 4 x stride keys
    __shared__ __attribute__((aligned(16))) uint32_t hist[4][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + wave;
    if (row >= rows) return;
    // the number of columns to keep: the same for every row, or one count per row (k_rows may be lens_out)
    const int k_sel = k_rows != nullptr ? k_rows[row] : k_all;
    if (lane == 0) lens_out[row] = k_sel;
    // unused tail of the row's lists
    for (int e = k_sel + lane; e < stride; e += 64) {
        if (idx_out) idx_out[row * stride + e] = -1;
        if (idx_sorted_out) idx_sorted_out[row * stride + e] = -1;
    }
    if (k_sel == 0) return;

    const S* srow = score + row * nbk;
    uint32_t val[NPL];                      // ord(score); 0 for columns past the end of the row
#pragma unroll
    for (int j = 0; j < NPL; ++j) {
        const int i = j * 64 + lane;
        const S raw = srow[min(i, nbk - 1)];               // unconditional load, masked afterwards
        val[j] = i < nbk ? ord_of(raw) : 0u;
    }
    select_row<S, NPL, SCORE_ORDER>(val, [&](int i) { return srow[i]; }, lane, nbk, k_sel,
                                    idx_out ? idx_out + row * stride : nullptr,
                                    idx_sorted_out ? idx_sorted_out + row * stride : nullptr,
                                    reinterpret_cast<K*>(topk_keys) + (SCORE_ORDER ? (size_t)wave * stride : 0), hist[wave]);
}

// Top-k of 16-bit scores when only the ascending-block-order list is wanted and rows are 16-byte aligned (nbk a
// multiple of 8): the same selection as select_row with another assignment of columns to lanes.  Lane l holds the
// columns 512 j + 8 l .. 8 l + 7 (one 16-byte load per j instead of eight 2-byte loads), so the ascending list
// position of a winner is (winners in earlier j) + (winners in lower lanes: one prefix sum per j) + (winners
// below it in its own lane) - one scan per 512 columns instead of two ballots per 64.
template <int NCH>
__global__ __launch_bounds__(256) void topk_blocked_kernel(const uint16_t* __restrict__ score,
                                                           int32_t* __restrict__ idx_sorted_out,
                                                           int32_t* __restrict__ lens_out, int64_t rows, int nbk, int k_all,
                                                           const int32_t* __restrict__ k_rows, int stride) {
    __shared__ __attribute__((aligned(16))) uint32_t hist[4][256];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + wave;
    if (row >= rows) return;
    const int k_sel = k_rows != nullptr ? k_rows[row] : k_all;
    if (lane == 0) lens_out[row] = k_sel;
    int32_t* out = idx_sorted_out + row * stride;
    for (int e = k_sel + lane; e < stride; e += 64) out[e] = -1;          // unused tail of the row's list
    if (k_sel == 0) return;

    const uint16_t* srow = score + row * nbk;
    uint32_t val[NCH * 8];                   // ord(score); 0 for columns past the end of the row
    bool in[NCH];
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
        const int col0 = 512 * j + 8 * lane;
        in[j] = col0 < nbk;
        const uint4 raw = *reinterpret_cast<const uint4*>(srow + (in[j] ? col0 : 0));   // unconditional load, masked afterwards
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint16_t r = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
            val[8 * j + e] = in[j] ? ord16(r) : 0u;
        }
    }
    uint32_t thr;
    int cnt_gt, cnt_eq;
    kth_value<16>(val, [&](int x) { return in[x >> 3]; }, lane, k_sel, hist[wave], thr, cnt_gt, cnt_eq);
    const int need_eq = k_sel - cnt_gt;
    const bool all_equal_win = need_eq >= cnt_eq;            // the same in every lane: no tie is cut

    int pos = 0, eq_seen = 0;                                  // winners / columns equal to t in the chunks before j
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
        if (512 * j >= nbk) break;
        uint32_t win = 0;                                      // bit e: column 512 j + 8 lane + e wins
        if (all_equal_win) {
#pragma unroll
            for (int e = 0; e < 8; ++e) win |= (val[8 * j + e] >= thr && in[j]) ? (1u << e) : 0u;
        } else {
            uint32_t gt = 0, eq = 0;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                gt |= (val[8 * j + e] > thr) ? (1u << e) : 0u;
                eq |= (val[8 * j + e] == thr && in[j]) ? (1u << e) : 0u;
            }
            // of the columns equal to t the first need_eq in column order win
            const int n_eq = __popc(eq);
            const int upto = wave_scan(n_eq);
            int take = min(max(need_eq - (eq_seen + upto - n_eq), 0), n_eq);
            eq_seen += __builtin_amdgcn_readlane(upto, 63);
            win = gt;
            while (take > 0) {
                const uint32_t low = eq & (0u - eq);
                win |= low;
                eq ^= low;
                --take;
            }
        }
        const int n_win = __popc(win);
        const int upto = wave_scan(n_win);
        int p = pos + upto - n_win;
        pos += __builtin_amdgcn_readlane(upto, 63);
        while (win != 0u) {
            out[p++] = 512 * j + 8 * lane + __builtin_ctz(win);
            win &= win - 1u;
        }
    }
}

// ---------------------------------------------------------------- visiting order
__global__ __launch_bounds__(64) void pace_order_kernel(const int32_t* in, int32_t* out, const int32_t* __restrict__ lens, int nbk, int stride, HalfLists halves,
                                                        ListBits bits, Divisor by_span) {
    extern __shared__ int32_t pace_lds[];
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int32_t* src = in + row * stride;
    int32_t* dst = out + row * stride;
    const int n = min(max(lens[row], 0), stride);
    if (bits.words != nullptr) {
        const int64_t bh = row / bits.rows;
        const int m = (int)(row - bh * bits.rows);
        for (int e = lane; e < n; e += 64)
            atomicOr(bits.words + (bh * nbk + min(max(src[e], 0), nbk - 1)) * bits.per_row + (m >> 5), 1u << (m & 31));
    }
    if (src != dst)
        for (int e = n + lane; e < stride; e += 64) dst[e] = src[e];
    if (n <= kPaceWidth && halves.lists == nullptr) {
        if (src != dst)
            for (int e = lane; e < n; e += 64) dst[e] = src[e];
        return;
    }
    for (int e = lane; e < n; e += 64) pace_lds[e] = min(max(src[e], 0), nbk - 1);
    wave_sync();
    const int32_t* order = pace_lds;
    if (n > kPaceWidth) order = pace_row(pace_lds, n, stride, nbk, lane, dst, by_span);
    else if (src != dst)
        for (int e = lane; e < n; e += 64) dst[e] = src[e];
    if (halves.lists != nullptr) expand_row(order, n, halves, row, lane);
}

// ---------------------------------------------------------------- the whole gating of a small call in one launch
// Scores, top-k and visiting order of kRows score rows per workgroup of 16 wavefronts: the scores go to LDS instead of
// memory (the same MFMA chain as score_mfma_kernel and the same rounding, so the same bits), a wavefront selects
// kRows / 16 of the rows from there and writes their lists in visiting order.  One launch instead of three: a launch of
// a few microseconds' work costs 4.4 us in a stream of dependent ones.  A workgroup takes most of a CU's LDS, so a call
// of many rows overlaps nothing and is better served by the separate kernels (kGateMaxGroups).
template <typename T> struct GateRows { static constexpr int kRows = 32; typedef uint16_t bits; };
template <> struct GateRows<float> { static constexpr int kRows = 16; typedef uint32_t bits; };
constexpr int kGateThreads = 1024;
constexpr int kGateMaxBlocks = 512;
// Row groups up to which a call gates in one launch: one per CU.  The whole operator, one launch against the separate
// kernels, us (480 blocks, by heads): bf16, lists of 30: 97.1 / 103.8 at 30 groups, 313 / 325 at 120, 646 / 651 at 255,
// 790 / 792 at 300, 952 / 952 at 360, 1 217 / 1 214 at 480; lists of 240, whose selection takes longer than a launch:
// 469 / 479 at 30, 1 733 / 1 729 at 120, 3 441 / 3 419 at 240.  fp32 gains where blocks are few: 15.4 / 17.6 with 4 blocks and
// 4 heads, 114 / 115 with 64, 386 / 386 with 128, 833 / 831 with 192; one head of 480 blocks loses 414 / 402.
constexpr int kGateMaxGroups = 256;
__host__ __device__ inline int gate_pitch(int nbk) { return (nbk + 31) / 32 * 32 + 8; }

template <typename T, int NPL>
__global__ __launch_bounds__(kGateThreads) void gate_kernel(const T* __restrict__ qc, const T* __restrict__ kc, int32_t* __restrict__ lists,
                                                            int32_t* __restrict__ lens, int nbq, int nbk, int k_sel, int paced, HeadNorms norms, HalfLists halves,
                                                            int counts_at, Divisor by_span) {
    typedef typename GateRows<T>::bits S;
    constexpr int D = 128, R = GateRows<T>::kRows;
    extern __shared__ __attribute__((aligned(16))) unsigned char gate_lds[];
    const int pitch = gate_pitch(nbk), words = gate_wave_words(k_sel);
    T* const scores = reinterpret_cast<T*>(gate_lds);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    uint32_t* const mine = reinterpret_cast<uint32_t*>(gate_lds + (size_t)R * pitch * sizeof(T)) + wave * words;
    touch_arguments<decltype(gate_kernel<T, NPL>)>();
    const int bh = blockIdx.y, m0 = blockIdx.x * R;
    // the keys of every tile, which the lists of halves ask for one after another at the end: looked up here, beside the scores
    uint8_t* const counts = counts_at > 0 ? gate_lds + counts_at : nullptr;
    if (counts_at > 0)
        for (int i = threadIdx.x; i < nbk * halves.nsub; i += kGateThreads) counts[i] = (uint8_t)__popcll(halves.valid[i]);
    if (norms.tile_norm != nullptr && wave == kGateThreads / 64 - 1 && blockIdx.x == 0 && blockIdx.z == 0) head_norm(norms, bh, lane);
    const T* qb = qc + (int64_t)bh * nbq * D;
    const T* kb = kc + (int64_t)bh * nbk * D;
    if constexpr (sizeof(T) == 2) {
        typedef typename Vec8<T>::type V8;
        const int lr = lane & 31, lh = lane >> 5;
        if (wave * 32 < nbk) {
            V8 a[8];
            const T* qa = qb + (int64_t)min(m0 + lr, nbq - 1) * D + lh * 8;
#pragma unroll
            for (int s = 0; s < 8; ++s) a[s] = *reinterpret_cast<const V8*>(qa + s * 16);
            for (int n0 = wave * 32; n0 < nbk; n0 += 32 * (kGateThreads / 64)) {
                const T* kt = kb + (int64_t)min(n0 + lr, nbk - 1) * D + lh * 8;
                V8 b[8];
#pragma unroll
                for (int s = 0; s < 8; ++s) b[s] = *reinterpret_cast<const V8*>(kt + s * 16);
                f32x16 acc;
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
                for (int s = 0; s < 8; ++s) acc = mfma32(a[s], b[s], acc);
#pragma unroll
                for (int i = 0; i < 16; ++i) scores[(8 * (i / 4) + 4 * lh + (i % 4)) * pitch + n0 + lr] = (T)acc[i];
            }
        }
    } else {
        const int n16 = lane & 15, g = lane >> 4;
        if (wave * 16 < nbk) {
            f32x4 a[8], b[8];
            score_row_f32(qb + (int64_t)min(m0 + n16, nbq - 1) * D + 4 * g, a);
            for (int n0 = wave * 16; n0 < nbk; n0 += 16 * (kGateThreads / 64)) {
                score_row_f32(kb + (int64_t)min(n0 + n16, nbk - 1) * D + 4 * g, b);
                const f32x4 acc = score_tile_f32(a, b);
#pragma unroll
                for (int i = 0; i < 4; ++i) scores[(4 * g + i) * pitch + n0 + n16] = acc[i];
            }
        }
    }
    __syncthreads();
    // with gridDim.z == 2 two workgroups compute the same scores and select half of the rows each
    for (int r = wave + (kGateThreads / 64) * blockIdx.z; r < R; r += (kGateThreads / 64) * gridDim.z) {
        const int m = m0 + r;
        if (m >= nbq) break;
        const int64_t row = (int64_t)bh * nbq + m;
        if (lane == 0) lens[row] = k_sel;
        if (k_sel == 0) {
            if (halves.lists != nullptr && lane == 0) halves.lens[row] = 0;
            continue;
        }
        const S* srow = reinterpret_cast<const S*>(scores + r * pitch);
        uint32_t val[NPL];
#pragma unroll
        for (int j = 0; j < NPL; ++j) {
            const int i = j * 64 + lane;
            const S raw = srow[min(i, nbk - 1)];
            val[j] = i < nbk ? ord_of(raw) : 0u;
        }
        int32_t* const list = reinterpret_cast<int32_t*>(mine);
        select_row<S, NPL, false>(val, [&](int i) { return srow[i]; }, lane, nbk, k_sel, nullptr, list, nullptr, mine);
        wave_sync();
        int32_t* const dst = lists + row * k_sel;
        const int32_t* order = list;
        if (paced && k_sel > kPaceWidth) order = pace_row(list, k_sel, k_sel, nbk, lane, dst, by_span);
        else
            for (int e = lane; e < k_sel; e += 64) dst[e] = list[e];
        if (halves.lists != nullptr) expand_row(order, k_sel, halves, row, lane, counts);
        wave_sync();
    }
}

// What a kernel that wants more than 64 KB of LDS is allowed: all of it, whatever this call needs, so that host threads with
// calls of different sizes do not lower each other's limit between its setting and the launch.
constexpr size_t kLdsLimit = 160 * 1024;

template <typename T>
size_t gate_lds_bytes(int nbk, int k_sel) {
    return (size_t)GateRows<T>::kRows * gate_pitch(nbk) * sizeof(T) + (size_t)(kGateThreads / 64) * gate_wave_words(k_sel) * 4;
}

template <typename T>
hipError_t launch_gate_t(const T* qc, const T* kc, int32_t* lists, int32_t* lens, int BH, int nbq, int nbk, int k_sel, bool paced,
                         hipStream_t st, HeadNorms norms, HalfLists halves) {
    size_t lds = gate_lds_bytes<T>(nbk, k_sel);
    const int64_t tiles = (int64_t)nbk * halves.nsub;
    int counts_at = 0;
    if (halves.lists != nullptr && tiles <= (int64_t)(kLdsLimit - lds)) {
        counts_at = (int)lds;
        lds += (size_t)tiles;
    }
    const int blocks = (nbq + GateRows<T>::kRows - 1) / GateRows<T>::kRows;
    const int parts = GateRows<T>::kRows > kGateThreads / 64 && blocks * BH <= kGateMaxGroups / 2 ? 2 : 1;
    const dim3 grid(blocks, BH, parts), block(kGateThreads);
    const Divisor by_span = pace_divisor(nbk, k_sel);
#define BSA_GATE(N)                                                                                                          \
    do {                                                                                                                     \
        if (lds > 64 * 1024) {                                                                                               \
            const hipError_t ea = hipFuncSetAttribute((const void*)gate_kernel<T, N>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsLimit); \
            if (ea != hipSuccess) return ea;                                                                                 \
        }                                                                                                                    \
        hipLaunchKernelGGL((gate_kernel<T, N>), grid, block, lds, st, qc, kc, lists, lens, nbq, nbk, k_sel, paced ? 1 : 0, norms, halves, counts_at, by_span);  \
    } while (0)
    if (nbk <= 64) BSA_GATE(1);
    else if (nbk <= 128) BSA_GATE(2);
    else if (nbk <= 256) BSA_GATE(4);
    else BSA_GATE(8);
#undef BSA_GATE
    return hipGetLastError();
}

// ---------------------------------------------------------------- CDF rule
// One wavefront per row: cdf_row.
template <typename S, int NPL>
__global__ __launch_bounds__(256) void cdf_count_kernel(const S* __restrict__ score, int32_t* __restrict__ lens_out,
                                                        int64_t rows, int nbk, float threshold, float scale, int k_min,
                                                        int cap, int dtype) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + wave;
    if (row >= rows) return;
    const S* srow = score + row * nbk;
    uint32_t val[NPL];
    float e[NPL];
#pragma unroll
    for (int j = 0; j < NPL; ++j) {
        const int i = j * 64 + lane;
        const S raw = srow[min(i, nbk - 1)];
        val[j] = i < nbk ? ord_of(raw) : 0u;
        e[j] = i < nbk ? score_value(raw, dtype) : -INFINITY;
    }
    const int n = cdf_row<8 * (int)sizeof(S)>(val, e, lane, nbk, threshold, scale, k_min, cap);
    if (lane == 0) lens_out[row] = n;
}

template <typename S>
hipError_t launch_cdf_count_t(const S* score, int32_t* lens, int64_t rows, int nbk, float threshold, float scale,
                              int k_min, int cap, int dtype, hipStream_t st) {
    dim3 grid((unsigned)((rows + 3) / 4)), block(256);
    // bound by the sixteen masked sums of doubles over a lane's columns, past the row's end too: many widths
#define BSA_CDF(N) hipLaunchKernelGGL((cdf_count_kernel<S, N>), grid, block, 0, st, score, lens, rows, nbk, threshold, scale, k_min, cap, dtype)
    if (nbk <= 4 * 64) BSA_CDF(4);
    else if (nbk <= 6 * 64) BSA_CDF(6);
    else if (nbk <= 8 * 64) BSA_CDF(8);
    else if (nbk <= 10 * 64) BSA_CDF(10);
    else if (nbk <= 12 * 64) BSA_CDF(12);
    else if (nbk <= 16 * 64) BSA_CDF(16);
    else if (nbk <= 24 * 64) BSA_CDF(24);
    else if (nbk <= 32 * 64) BSA_CDF(32);
    else BSA_CDF(64);
#undef BSA_CDF
    return hipGetLastError();
}

template <typename S>
hipError_t launch_topk_t(const S* score, int32_t* idx, int32_t* idx_sorted, int32_t* lens, int64_t rows,
                         int nbk, int k_sel, const int32_t* k_rows, int stride, hipStream_t st) {
    dim3 grid((unsigned)((rows + 3) / 4)), block(256);
    if (sizeof(S) == 2 && idx == nullptr && idx_sorted != nullptr && nbk % 8 == 0 && (reinterpret_cast<uintptr_t>(score) & 15) == 0) {
        const uint16_t* sc = reinterpret_cast<const uint16_t*>(score);
#define BSA_TOPK_BLOCKED(N) hipLaunchKernelGGL((topk_blocked_kernel<N>), grid, block, 0, st, sc, idx_sorted, lens, rows, nbk, k_sel, k_rows, stride)
        if (nbk <= 512) BSA_TOPK_BLOCKED(1);
        else if (nbk <= 1024) BSA_TOPK_BLOCKED(2);
        else if (nbk <= 1536) BSA_TOPK_BLOCKED(3);
        else if (nbk <= 2048) BSA_TOPK_BLOCKED(4);
        else if (nbk <= 3072) BSA_TOPK_BLOCKED(6);
        else BSA_TOPK_BLOCKED(8);
#undef BSA_TOPK_BLOCKED
        return hipGetLastError();
    }
    // the score-order ranking keeps the winners of the workgroup's four rows in LDS
    const size_t lds = idx != nullptr ? (size_t)4 * stride * sizeof(typename KeyOf<S>::type) : 0;
    const size_t most = (size_t)4 * kMaxSel * sizeof(typename KeyOf<S>::type);      // allowed for every call alike, as in launch_gate_t
#define BSA_TOPK(N)                                                                                \
    do {                                                                                           \
        if (idx != nullptr) {                                                                      \
            if (lds > 64 * 1024) {                                                                 \
                const hipError_t ea = hipFuncSetAttribute((const void*)topk_kernel<S, N, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most); \
                if (ea != hipSuccess) return ea;                                                   \
            }                                                                                      \
            hipLaunchKernelGGL((topk_kernel<S, N, true>), grid, block, lds, st, score, idx, idx_sorted, lens, rows, nbk, k_sel, k_rows, stride);  \
        } else {                                                                                   \
            hipLaunchKernelGGL((topk_kernel<S, N, false>), grid, block, 0, st, score, idx, idx_sorted, lens, rows, nbk, k_sel, k_rows, stride); \
        }                                                                                          \
    } while (0)
    if (nbk <= 4 * 64) BSA_TOPK(4);
    else if (nbk <= 8 * 64) BSA_TOPK(8);
    else if (nbk <= 16 * 64) BSA_TOPK(16);
    else if (nbk <= 24 * 64) BSA_TOPK(24);
    else if (nbk <= 32 * 64) BSA_TOPK(32);
    else BSA_TOPK(64);
#undef BSA_TOPK
    return hipGetLastError();
}

}  // namespace

hipError_t launch_score(const void* q_cmp, const void* k_cmp, void* score, int BH, int nbq, int nbk,
                        int D, int dtype, hipStream_t st, HeadNorms norms) {
    if (dtype == BSA_F32) {
        dim3 grid((nbk + 63) / 64, (nbq + 15) / 16, BH);
        hipLaunchKernelGGL(score_f32_kernel, grid, dim3(256), 0, st, (const float*)q_cmp,
                           (const float*)k_cmp, (float*)score, nbq, nbk);
    } else {
        dim3 grid((nbk + kScoreCols - 1) / kScoreCols, (nbq + 127) / 128, BH);
        if (dtype == BSA_BF16)
            hipLaunchKernelGGL((score_mfma_kernel<__bf16>), grid, dim3(256), 0, st,
                               (const __bf16*)q_cmp, (const __bf16*)k_cmp, (__bf16*)score, nbq, nbk, norms);
        else
            hipLaunchKernelGGL((score_mfma_kernel<_Float16>), grid, dim3(256), 0, st,
                               (const _Float16*)q_cmp, (const _Float16*)k_cmp, (_Float16*)score, nbq, nbk, norms);
    }
    return hipGetLastError();
}

hipError_t launch_topk(const void* score, int32_t* idx, int32_t* idx_sorted, int32_t* lens, int64_t rows,
                       int nbk, int k_sel, int dtype, hipStream_t st, const int32_t* k_rows, int stride) {
    if (stride <= 0) stride = k_sel;
    if (dtype == BSA_F32)
        return launch_topk_t<uint32_t>((const uint32_t*)score, idx, idx_sorted, lens, rows, nbk, k_sel, k_rows, stride, st);
    return launch_topk_t<uint16_t>((const uint16_t*)score, idx, idx_sorted, lens, rows, nbk, k_sel, k_rows, stride, st);
}

bool gate_fits(int BH, int nbq, int nbk, int k_sel, int dtype) {
    if (nbk > kGateMaxBlocks) return false;
    const int rows = dtype == BSA_F32 ? GateRows<float>::kRows : GateRows<__bf16>::kRows;
    const size_t lds = dtype == BSA_F32 ? gate_lds_bytes<float>(nbk, k_sel) : gate_lds_bytes<__bf16>(nbk, k_sel);
    return lds <= kLdsLimit && (int64_t)BH * ((nbq + rows - 1) / rows) <= kGateMaxGroups;
}

hipError_t launch_gate(const void* q_cmp, const void* k_cmp, int32_t* lists, int32_t* lens, int BH, int nbq, int nbk, int k_sel,
                       bool paced, int dtype, hipStream_t st, HeadNorms norms, HalfLists halves) {
    if (dtype == BSA_F32) return launch_gate_t<float>((const float*)q_cmp, (const float*)k_cmp, lists, lens, BH, nbq, nbk, k_sel, paced, st, norms, halves);
    if (dtype == BSA_BF16) return launch_gate_t<__bf16>((const __bf16*)q_cmp, (const __bf16*)k_cmp, lists, lens, BH, nbq, nbk, k_sel, paced, st, norms, halves);
    return launch_gate_t<_Float16>((const _Float16*)q_cmp, (const _Float16*)k_cmp, lists, lens, BH, nbq, nbk, k_sel, paced, st, norms, halves);
}

hipError_t launch_pace_order(const int32_t* in, int32_t* out, const int32_t* lens, int64_t rows, int nbk, int stride,
                             hipStream_t st, HalfLists halves, ListBits bits) {
    if (rows <= 0 || stride <= 0) return hipSuccess;
    const int groups = (stride + kPaceWidth - 1) / kPaceWidth;
    const size_t lds = ((size_t)3 * stride + groups) * sizeof(int32_t);
    if (lds > 64 * 1024 || rows > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(pace_order_kernel, dim3((unsigned)rows), dim3(64), lds, st, in, out, lens, nbk, stride, halves, bits, pace_divisor(nbk, stride));
    return hipGetLastError();
}

hipError_t launch_cdf_count(const void* score, int32_t* lens, int64_t rows, int nbk, float threshold, float scale,
                            int k_min, int cap, int dtype, hipStream_t st) {
    if (dtype == BSA_F32)
        return launch_cdf_count_t<uint32_t>((const uint32_t*)score, lens, rows, nbk, threshold, scale, k_min, cap, dtype, st);
    return launch_cdf_count_t<uint16_t>((const uint16_t*)score, lens, rows, nbk, threshold, scale, k_min, cap, dtype, st);
}

}  // namespace bsa
