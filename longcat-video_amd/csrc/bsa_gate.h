// One score row's selection and visiting order by a wavefront: what the gating kernels (bsa_select.hip) and the attention kernel
// of small calls, which selects for itself (bsa_frag.h), have in common.
#pragma once
#include "bsa_common.h"

namespace bsa {
namespace {

// fp32 storage type: v_mfma_f32_16x16x4, a wavefront per 16 x 16 scores.  Step (j, e) contracts d = 16 j + 4 (lane / 16) + e,
// so that a lane reads its row in 16-byte pieces.  Every kernel that
// scores runs score_tile_f32: the same bits.
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void score_row_f32(const float* row, f32x4 (&x)[8]) {       // row + 4 (lane / 16)
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = *reinterpret_cast<const f32x4*>(row + 16 * j);
}
__device__ __forceinline__ f32x4 score_tile_f32(const f32x4 (&a)[8], const f32x4 (&b)[8]) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][e], b[j][e], acc, 0, 0, 0);
    return acc;                              // accumulator i of lane l: row 4 (l / 16) + i, column l % 16
}

// Order-preserving maps to unsigned integers (NaN with the sign bit clear sorts
// above +inf, as torch.topk orders NaN).
// -0 is folded onto +0 first: the two compare equal, so they must tie.
__device__ inline uint32_t ord16(uint16_t u) {
    if (u == 0x8000u) u = 0;
    return (u & 0x8000u) ? (uint16_t)~u : (u | 0x8000u);
}
__device__ inline uint32_t ord32(uint32_t u) {
    if (u == 0x80000000u) u = 0;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

template <typename T> struct KeyOf;
template <> struct KeyOf<uint16_t> {   // bf16 / fp16 bit patterns (fp16 orders like its bits too)
    typedef uint32_t type;
    static constexpr int kBits = 32;
    __device__ static uint32_t make(uint16_t s, int idx) { return (ord16(s) << 16) | (0xFFFFu - idx); }
    __device__ static int index(uint32_t k) { return 0xFFFF - (int)(k & 0xFFFFu); }
};
template <> struct KeyOf<uint32_t> {   // fp32 bit patterns
    typedef uint64_t type;
    static constexpr int kBits = 64;
    __device__ static uint64_t make(uint32_t s, int idx) {
        return ((uint64_t)ord32(s) << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)idx);
    }
    __device__ static int index(uint64_t k) { return (int)(0xFFFFFFFFu - (uint32_t)k); }
};

constexpr int kMaxSel = 4096;   // longest list: the score-order ranking keeps a row's winners in LDS

// Order-preserving image of a score alone (ties stay ties).
__device__ inline uint32_t ord_of(uint16_t s) { return ord16(s); }
__device__ inline uint32_t ord_of(uint32_t s) { return ord32(s); }

// The k-th largest score value t of a row that a wavefront holds as val[N] per lane (order-preserving images;
// in_range(x): element x of this lane is a column of the row): every column above t wins, and of the columns equal
// to t the first k_sel - cnt_gt in column order.  thr = t, cnt_gt = columns above t, cnt_eq = columns equal to t.
// For 16-bit scores t is first looked for in a histogram of the codes just below the row maximum, otherwise (and for
// rows whose winners reach further down) by a bitwise binary search whose counting step is a ballot + popcount.
// h: 256 words of LDS of this wavefront.
template <int kValueBits, int N, typename InRange>
__device__ inline void kth_value(const uint32_t (&val)[N], InRange in_range, int lane, int k_sel, uint32_t* h,
                                 uint32_t& thr, int& cnt_gt, int& cnt_eq) {
    thr = 0;
    cnt_gt = 0;
    cnt_eq = 0;
    bool found = false;
    if (kValueBits == 16) {
        // 16-bit scores: the winners of a row usually lie within a few hundred codes of the row maximum, so one
        // histogram of (maximum - ord) over 255 bins, built with LDS atomics by the columns that fall into it,
        // and one scan find t.  Rows whose k_sel largest values reach further down take the search below.
        uint32_t mx = 0;
#pragma unroll
        for (int j = 0; j < N; ++j) mx = max(mx, val[j]);
        mx = wave_max(mx);
        *reinterpret_cast<uint4*>(h + 4 * lane) = make_uint4(0u, 0u, 0u, 0u);
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint32_t d = mx - val[j];
            if (in_range(j) && d < 255u) atomicAdd(h + d, 1u);
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_wave_barrier();
        const uint4 c = *reinterpret_cast<const uint4*>(h + 4 * lane);
        const int own = (int)(c.x + c.y + c.z + c.w);
        const int upto = wave_scan(own);                   // columns within bins 0 .. 4 lane + 3
        const int before = upto - own;
        const uint64_t holder = __ballot(before < k_sel && k_sel <= upto);
        if (holder != 0) {
            int bin = 4 * lane, run = before, in_bin = (int)c.x;
            if (run + (int)c.x < k_sel) { run += (int)c.x; ++bin; in_bin = (int)c.y;
                if (run + (int)c.y < k_sel) { run += (int)c.y; ++bin; in_bin = (int)c.z;
                    if (run + (int)c.z < k_sel) { run += (int)c.z; ++bin; in_bin = (int)c.w; } } }
            const int src = __builtin_ctzll(holder);
            thr = mx - (uint32_t)__builtin_amdgcn_readlane(bin, src);
            cnt_gt = __builtin_amdgcn_readlane(run, src);
            cnt_eq = __builtin_amdgcn_readlane(in_bin, src);
            found = true;
        }
    }
    if (!found) {
        // Largest t with count(ord >= t) >= k_sel, t = 0 if there is none above, by a bitwise binary search
        // whose counting step is a ballot + popcount.  Every candidate is at least 1, so the zeros past the end
        // of the row never count.  Leaving early with exactly k_sel columns at or above t is fine: the winners
        // are then all columns at or above t.
        for (int bit = kValueBits - 1; bit >= 0; --bit) {
            const uint32_t cand = thr | (1u << bit);
            int cnt = 0;
#pragma unroll
            for (int j = 0; j < N; ++j) cnt += __popcll(__ballot(val[j] >= cand));
            if (cnt >= k_sel) {
                thr = cand;
                if (cnt == k_sel) break;
            }
        }
        cnt_gt = 0;
        cnt_eq = 0;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            cnt_gt += __popcll(__ballot(val[j] > thr));
            cnt_eq += __popcll(__ballot(val[j] == thr && in_range(j)));      // thr may be 0, like the padding of val
        }
    }
}

// Selection of one score row by one wavefront; lane l holds the order-preserving images of columns l, l + 64,
// ... in registers (0 for columns past the end of the row).
//   1. the k-th largest score value t (kth_value);
//   2. every score above t wins, and of the scores equal to t the ones with the lowest column
//      index, as many as are still needed; walking the registers in column order hands out the
//      positions of the ascending-block-order list at the same time (no sort);
//   3. only when the score-order list is wanted: rank the winners by (score desc, index asc).
// raw_at(i): the stored score of column i.  mine: one key of LDS per list entry (SCORE_ORDER only); h: 256 words of LDS.
template <typename S, int NPL, bool SCORE_ORDER, typename RawAt>
__device__ inline void select_row(const uint32_t (&val)[NPL], RawAt raw_at, int lane, int nbk, int k_sel,
                                  int32_t* __restrict__ idx_row, int32_t* __restrict__ idx_sorted_row,
                                  typename KeyOf<S>::type* mine, uint32_t* h) {
    typedef typename KeyOf<S>::type K;
    uint32_t thr;
    int cnt_gt, cnt_eq;
    kth_value<8 * (int)sizeof(S)>(val, [&](int j) { return j * 64 + lane < nbk; }, lane, k_sel, h, thr, cnt_gt, cnt_eq);
    const int need_eq = k_sel - cnt_gt;

    int pos = 0, eq_seen = 0;
    const uint64_t lt = ((uint64_t)1 << lane) - 1;
#pragma unroll
    for (int j = 0; j < NPL; ++j) {
        const int i = j * 64 + lane;
        const bool eq = val[j] == thr && i < nbk;          // thr may be 0, like the padding of val
        const uint64_t meq = __ballot(eq);
        const bool win = val[j] > thr || (eq && eq_seen + __popcll(meq & lt) < need_eq);
        const uint64_t m = __ballot(win);
        if (win) {
            const int p = pos + __popcll(m & lt);
            if (idx_sorted_row) idx_sorted_row[p] = i;                        // column order = ascending block order
            if (SCORE_ORDER) mine[p] = KeyOf<S>::make(raw_at(i), i);
        }
        pos += __popcll(m);
        eq_seen += __popcll(meq);
    }
    if (!SCORE_ORDER) return;
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): LDS writes of this wavefront landed
    __builtin_amdgcn_wave_barrier();
    // descending score, ties towards the lowest index: the order of the combined keys
    for (int e = lane; e < k_sel; e += 64) {
        const K me = mine[e];
        int rank = 0;
        for (int o = 0; o < k_sel; ++o) rank += mine[o] > me;
        idx_row[rank] = KeyOf<S>::index(me);
    }
}

// ---------------------------------------------------------------- CDF rule
__device__ inline float score_value(uint16_t s, int dtype) {
    if (dtype == BSA_F16) return (float)__builtin_bit_cast(_Float16, s);
    return __uint_as_float((uint32_t)s << 16);
}
__device__ inline float score_value(uint32_t s, int) { return __uint_as_float(s); }
// The sum over the lanes l, l ^ 32, l ^ 16, ... of a butterfly, by moves between registers: the halves of the wavefront and of its
// rows trade, and inside a row a rotation by 8 (4, 2, 1) reaches lane l ^ 8 (a lane that holds what l ^ 4 does, ...).  A sum of
// doubles by __shfl is twelve round trips to LDS, and the search below makes sixteen of them (cdf_count_kernel, 16 heads of
// 20x30x52: 34 us that way).
__device__ __forceinline__ double wave_sum(double x) {
    auto halves = [](double y, uint32_t& lo, uint32_t& hi) {
        const uint64_t b = (uint64_t)__double_as_longlong(y);
        lo = (uint32_t)b; hi = (uint32_t)(b >> 32);
    };
    auto whole = [](uint32_t lo, uint32_t hi) { return __longlong_as_double((long long)((uint64_t)hi << 32 | lo)); };
    uint32_t lo, hi;
    halves(x, lo, hi);
    {
        const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false), b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        x = whole(a[0], b[0]) + whole(a[1], b[1]);
    }
    halves(x, lo, hi);
    {
        const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false), b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        x = whole(a[0], b[0]) + whole(a[1], b[1]);
    }
#define BSA_ROTATED(N)                                                                                  \
    halves(x, lo, hi);                                                                                  \
    x += whole((uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, 0x120 + N, 0xf, 0xf, false), (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, 0x120 + N, 0xf, 0xf, false))
    BSA_ROTATED(8);
    BSA_ROTATED(4);
    BSA_ROTATED(2);
    BSA_ROTATED(1);
#undef BSA_ROTATED
    return x;
}

// How many columns the CDF rule keeps per row: with the columns sorted by descending score (ties towards
// the lowest index) and weights softmax(score * scale), the number of leading columns whose running sum
// of weights stays at or below `threshold`; never fewer than k_min (the "cdf + top-k" rule) and never
// more than `cap`.  Sums run in double precision on the unnormalised weights
// e_i = exp((s_i - max) * scale): sum_top(e) <= threshold * sum_all(e).  The columns at or above a score
// value t form a prefix of the sorted order, so a bitwise binary search over t finds the value group in
// which the running sum crosses the threshold; inside that group every column weighs the same.
// val: the order-preserving images of the row's columns l, l + 64, ... in lane l, 0 past its end; e: the scores.
template <int kValueBits, int NPL>
__device__ inline int cdf_row(const uint32_t (&val)[NPL], float (&e)[NPL], int lane, int nbk, float threshold, float scale, int k_min, int cap) {
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < NPL; ++j) mx = fmaxf(mx, e[j]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    double total = 0.0;
#pragma unroll
    for (int j = 0; j < NPL; ++j) {
        e[j] = j * 64 + lane < nbk ? expf((e[j] - mx) * scale) : 0.f;
        total += (double)e[j];
    }
    total = wave_sum(total);
    const double budget = (double)threshold * total;
    // largest t whose columns at or above t outweigh the budget (t = 0: all columns, if even that holds)
    auto mass_ge = [&](uint32_t t) {
        double m = 0.0;
#pragma unroll
        for (int j = 0; j < NPL; ++j) m += val[j] >= t ? (double)e[j] : 0.0;     // padding has e = 0
        return wave_sum(m);
    };
    int n;
    // NaN by its bits: a file may be built without regard for them
    const bool nan = ((uint64_t)__double_as_longlong(total) << 1) > 0xffe0000000000000ull;
    if (nan || !(total > budget)) {
        n = nbk;                                  // threshold >= 1: everything
    } else {
        uint32_t thr = 0;
        for (int bit = kValueBits - 1; bit >= 0; --bit) {
            const uint32_t cand = thr | (1u << bit);
            if (mass_ge(cand) > budget) thr = cand;
        }
        // columns above thr fit; the group equal to thr crosses: take as many of it as still fit
        double above = 0.0, one = 0.0;
        int cnt_gt = 0, cnt_eq = 0;
#pragma unroll
        for (int j = 0; j < NPL; ++j) {
            const bool real = j * 64 + lane < nbk;
            above += val[j] > thr ? (double)e[j] : 0.0;
            cnt_gt += __popcll(__ballot(val[j] > thr));
            const bool eq = real && val[j] == thr;
            cnt_eq += __popcll(__ballot(eq));
            if (eq) one = (double)e[j];
        }
        above = wave_sum(above);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) one = fmax(one, __shfl_xor(one, o));
        int fit = one > 0.0 ? (int)floor((budget - above) / one) : cnt_eq;
        fit = max(0, min(fit, cnt_eq));
        n = cnt_gt + fit;
    }
    return __builtin_amdgcn_readfirstlane(min(max(n, k_min), min(cap, nbk)));
}

// The order in which the attention kernel visits one row's selected KV blocks.  Softmax attention does not
// depend on it beyond rounding, so it is chosen for the L2 cache: the query tiles that run side by side walk
// the KV sequence together when slot s of every list holds a block near s/n of the sequence, and then share
// the K/V tiles they have in common while those are still cached.  A plain ascending list drifts from that
// pace wherever it holds more or fewer blocks than the average in a stretch of the sequence.
//
// One wavefront per row.  in: n = lens[row] blocks in ascending order.  Visit slots are cut into groups of
// kPaceWidth; group g belongs to the blocks b with g == min(b * n / (nbk * kPaceWidth), groups - 1).  A group
// takes its own blocks in ascending order up to its number of slots; the blocks over that number (ascending
// over the whole list) fill the slots left empty (ascending); every group's slots are then put in ascending
// block order.  in == out is allowed.  A malformed list (unsorted, repeated or out-of-range blocks) still
// gives a permutation of the blocks clamped to the valid range.
constexpr int kPaceWidth = 8;
// Orders this wavefront's LDS accesses on both sides of it, for the compiler and the hardware; no other wavefront waits.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// A visiting list of n blocks (LDS, visible to the wavefront) as the halves that hold keys, for the attention kernel's
// kHalves walk: half of the (batch, head) | real keys << 20.  An odd number is made even with a repeat that holds no key.
// keys_of(tile): its number of keys, which come first in it.  Returns the number of halves without such a repeat.
template <typename Keys>
__device__ inline int expand_list(const int32_t* list, int n, int nsub, int32_t* out, int lane, Keys keys_of) {
    const uint64_t below = ((uint64_t)1 << lane) - 1;
    const int tiles = n * nsub;
    int total = 0, last_at = -1, last = 0;
    for (int base = 0; base < tiles; base += 64) {
        const int e = base + lane;
        int keys = 0, tile = 0;
        if (e < tiles) {
            const int j = nsub == 1 ? e : e / nsub;
            tile = list[j] * nsub + (e - j * nsub);
            keys = keys_of(tile);
        }
        const uint64_t one = __ballot(keys > 0), two = __ballot(keys > 32);
        const int at = total + __popcll(one & below) + __popcll(two & below);
        if (keys > 0) {
            last = 2 * tile; last_at = at;
            out[at] = last | (min(keys, 32) << 20);
        }
        if (keys > 32) {
            last = 2 * tile + 1; last_at = at + 1;
            out[at + 1] = last | ((keys - 32) << 20);
        }
        total += __popcll(one) + __popcll(two);
    }
    if ((total & 1) && last_at == total - 1) out[total] = last;
    return total;
}
// The same into the row's place in memory.  counts: the keys of every tile, in LDS; null: from the validity words.
__device__ inline void expand_row(const int32_t* list, int n, const HalfLists& h, int64_t row, int lane, const uint8_t* counts = nullptr) {
    int32_t* const out = h.lists + row * h.stride;
    const int total = counts != nullptr ? expand_list(list, n, h.nsub, out, lane, [&](int tile) { return (int)counts[tile]; })
                                        : expand_list(list, n, h.nsub, out, lane, [&](int tile) { return (int)__popcll(h.valid[tile]); });
    if (lane == 0) h.lens[row] = total;
}

// 32-bit words of LDS that pace_row needs for lists of n entries
__host__ __device__ inline int pace_words(int n) { return 3 * n + (n + kPaceWidth - 1) / kPaceWidth; }
// nbk * kPaceWidth, where the products that pace_row divides by it fit 31 bits, otherwise m = 0.
inline Divisor pace_divisor(int nbk, int stride) {
    return (int64_t)nbk * (stride > kPaceWidth ? stride : kPaceWidth) <= 0x7fffffff ? divisor(nbk * kPaceWidth) : Divisor{0, 0};
}
// work[0 .. n): the ascending list, clamped to the valid range; dst (may be null): where its visiting order goes.  Returns the visiting
// order in LDS.
__device__ inline const int32_t* pace_row(int32_t* work, int n, int cap, int nbk, int lane, int32_t* __restrict__ dst, const Divisor& by_span) {
    int32_t* const lst = work;                   // [cap] the row, ascending
    int32_t* const slots = lst + cap;            // [cap] block per visit slot, -1 = empty
    int32_t* const spare = slots + cap;          // [cap] blocks over their group's room, ascending
    int32_t* const first = spare + cap;          // [groups] position of a group's first block in lst
    const int groups = (n + kPaceWidth - 1) / kPaceWidth;
    // n < 2^13 (the LDS that the callers ask for bounds it) and b < nbk: 32-bit products and quotients
    const uint32_t span = (uint32_t)nbk * kPaceWidth;
    auto group_of = [&](int32_t b) {
        const uint32_t x = (uint32_t)b * (uint32_t)n;
        return (int)min(by_span.m != 0u ? (uint32_t)((int)x / by_span) : x / span, (uint32_t)groups - 1u);
    };
    for (int e = lane; e < n; e += 64) slots[e] = -1;
    for (int g = lane; g < groups; g += 64) first[g] = 0;
    wave_sync();
    for (int e = lane; e < n; e += 64) {
        const int g = group_of(lst[e]);
        if (e == 0 || group_of(lst[e - 1]) != g) first[g] = e;
    }
    wave_sync();
    const uint64_t below = ((uint64_t)1 << lane) - 1;
    int taken = 0;
    for (int base = 0; base < n; base += 64) {
        const int e = base + lane;
        bool over = false;
        if (e < n) {
            const int g = group_of(lst[e]), rank = e - first[g];
            const int room = min(kPaceWidth, n - g * kPaceWidth);
            if (rank >= 0 && rank < room) slots[g * kPaceWidth + rank] = lst[e];
            else over = true;
        }
        const uint64_t m = __ballot(over);
        if (over) spare[taken + __popcll(m & below)] = lst[e];
        taken += __popcll(m);
    }
    wave_sync();
    taken = 0;
    for (int base = 0; base < n; base += 64) {
        const int s = base + lane;
        const bool empty = s < n && slots[s] < 0;
        const uint64_t m = __ballot(empty);
        if (empty) slots[s] = spare[taken + __popcll(m & below)];
        taken += __popcll(m);
    }
    wave_sync();
    for (int s = lane; s < n; s += 64) {
        const int lo = s / kPaceWidth * kPaceWidth, hi = min(lo + kPaceWidth, n);
        const int32_t b = slots[s];
        int rank = 0;
        for (int t = lo; t < hi; ++t) rank += (slots[t] < b || (slots[t] == b && t < s)) ? 1 : 0;
        if (dst != nullptr) dst[lo + rank] = b;
        spare[lo + rank] = b;
    }
    wave_sync();
    return spare;
}
// words of LDS a wavefront selects and orders in: its histogram, later the row's list
__host__ __device__ inline int gate_wave_words(int k_sel) { const int w = pace_words(k_sel); return ((w > 256 ? w : 256) + 3) / 4 * 4; }

}  // namespace
}  // namespace bsa
