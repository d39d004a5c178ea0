// What the two attention kernels on fragment-order K and V (bsa_fwd_frag.hip; bsa_fwd_few.hip: calls that leave SIMDs
// idle) have in common: their items, how the keys of an item are listed, items in parts, and a list made in front of its walk.
#pragma once
#include "bsa_gate.h"
#include "bsa_mfma.h"

#include <type_traits>
#include <utility>

namespace bsa {

struct FragLayout {
    const int32_t* q_rows;        // token row of every blocked-order query slot, -1 = padding; null: q, o in blocked order
    int64_t q_st[3], o_st[3];     // element strides: batch, head, row
    // The query tiles of one (batch, head) that hold real rows, n_live numbers (null: every tile): work item u is then tile
    // tiles[u % n_live] of (batch, head) u / n_live.
    const int32_t* tiles;
    int n_live;
    Divisor by_live, by_tiles, by_block, by_heads, by_sub;       // n_live; query tiles of a (batch, head), of a block; heads; tiles of a KV block
};

// An item in parts: `count` wavefronts walk a share of its pairs each and leave the sums of their share (unnormalised
// accumulators in register order, running maximum and row sum per query) in `buf`, kPartFloats per part; merge_parts_kernel
// puts them together.  Part p of the launch's item i is its work item p * items + i.  count 1: whole items.
constexpr int kPartFloats = mfma::kTile * mfma::kD + 2 * mfma::kTile;
struct Parts {
    float* buf;
    int count, items;
    Divisor by_count, by_items;
};

// kGate: the item's list does not exist yet.  The workgroup makes it from the chunk means, as gate_kernel does (the same products and
// roundings, the same lists), in front of its walk: the scores of its block against every key block, a share of 32 of them to a
// wavefront at a time, then the first wavefront selects and orders.  Instead of another launch, its start and its end.
// Whole operator, us, with gate_kernel in front / like this: 2 heads of 16x22x12 23.0 / 19.9, 4 of 9x13x10 30.2 / 26.3, two prompts of
// 13 heads of 7x8x8 24.2 / 21.6, of 8 heads of 7x15x26 40.3 / 38.2.  The lists ([BH][nbq][width]) and
// their lengths also go to memory where they are wanted.
struct FragGate {
    const uint16_t *qc, *kc;         // chunk means, 16-bit storage; k's in operand order (operand_mean_at)
    int nbk, width;                  // entries of a list: the top-k rule's count, the most of the CDF rule's
    float threshold, scale;          // of the CDF rule, as cdf_count_kernel's; threshold 0: top-k
    int k_min;
    Divisor by_span;
};

// A call of launch_fwd_frag as far as its kernels see it.
struct FragCall {
    const void *q, *kf, *vf;
    const int32_t *idx, *lens;
    const uint64_t* tile_valid;
    void* o;
    float* lse;
    int64_t Sq, Sk, lse_rows;
    int bs_k, idx_stride, Hn, dtype;
    float qk_scale;
    bool halves;
    hipStream_t st;
};
// `items` work items at once, `team` wavefronts each (bsa_fwd_few.hip); gate: their lists are made in front of the walk.
hipError_t launch_fwd_few(const FragCall& c, const FragLayout& L, const Parts& parts, int items, int team, const FragGate* gate, int32_t* lists, uint32_t* list_lens,
                            uint32_t kv_bytes);

namespace {

using namespace mfma;

constexpr int kHalfBytes = 8192;      // 32 keys of a fragment-order K (or V) tile
constexpr int kListEntries = 4096;    // longest list a work item can walk (its staging area in LDS: 17 KB)
constexpr int kHalfEntries = 4096;    // ... of halves

// The tile number (over all heads) of work item u.  The table was written by an earlier kernel and is read through the scalar
// cache: the wait for it is its own, not one for every load of the wavefront, and all that is derived from it stays scalar.
// (Asked for an item ahead with vector loads, at every turn of every call, it cost grids without such a table 70 of 8 500 us
// at 32 heads of 720p.)
__device__ __forceinline__ int item_at(const FragLayout& L, int u, int nqt) {
    if (L.tiles == nullptr) return u;
    const int bh = u / L.by_live;
    return bh * nqt + *(const __attribute__((address_space(4))) int32_t*)(L.tiles + (u - bh * L.n_live));
}

// How an item's keys are listed (kWalk).  The walk goes in pairs of 32-key halves:
//   kTiles:  idx holds KV blocks of one 64-key tile (bs_k == 64; no division in the walk), a pair is a tile;
//   kBlocks: KV blocks of several tiles;
//   kHalves: idx holds the halves themselves, empty ones left out: half of the (batch, head) | real keys << 20, an even
//            number of entries (the last may repeat a half with no key), lens counts them without such a repeat.
// The real keys of a tile come first (prepare_kernel), so its validity is a count.  Leaving out a half whose
// probabilities would all be 0 changes no bit of the result: the sums run over the same numbers in the same order.
enum { kTiles, kBlocks, kHalves };
constexpr uint32_t kHalfId = 0xfffff;     // of a kHalves entry: the half; above it: its number of real keys
constexpr int kHalfCountShift = 20;

template <int kTeam>
constexpr int kTeamBytes = kTeam * (kTile * kD + 2 * kTile) * 4;      // the sums, maxima and row sums of every wavefront
static_assert(kTeamBytes<4> <= 160 * 1024 && 2 * (kTeamBytes<2> + 512) <= 160 * 1024, "LDS of a compute unit with four wavefronts");

constexpr int kGateWaveBlocks = 256, kGateMostBlocks = 512;      // key blocks that one wavefront scores, that a team does
// LDS of the selection: the list of halves; scores; keys of every tile; where the first wavefront works; the list's length
__host__ __device__ inline int gate_list_words(int width, int nsub, bool halves) { return halves ? (2 * width * nsub + 3) / 4 * 4 : 0; }
__host__ __device__ inline int gate_here_bytes(int nbk, int width, int nsub, bool halves) {
    return (gate_list_words(width, nsub, halves) + gate_wave_words(width) + 4) * 4 + (nbk + 31) / 32 * 64 + (halves ? (nbk * nsub + 15) / 16 * 16 : 0);
}

// The list of an item, of block row `row`, in LDS (`work`, gate_here_bytes), its length in `length`.  By all threads of the workgroup, with a
// barrier at the end.
template <typename T, int kTeam, bool kHalfLists>
__device__ __forceinline__ const uint32_t* make_list(const FragGate& G, char* work, int64_t row, int bh, int nsub, const uint64_t* tile_valid, int32_t* lists,
                                                     uint32_t* lens, int lane, int wave, int& length) {
    typedef typename Vec8<T>::type V8;
    const int words = gate_list_words(G.width, nsub, kHalfLists);
    int32_t* const halves_list = reinterpret_cast<int32_t*>(work);
    uint32_t* const mine = reinterpret_cast<uint32_t*>(work) + words;
    int* const total_at = reinterpret_cast<int*>(mine + gate_wave_words(G.width));
    T* const scores = reinterpret_cast<T*>(total_at + 4);
    uint8_t* const counts = reinterpret_cast<uint8_t*>(scores + (G.nbk + 31) / 32 * 32);
    if (kHalfLists)
        for (int i = threadIdx.x; i < G.nbk * nsub; i += 64 * kTeam) counts[i] = (uint8_t)__popcll(tile_valid[i]);
    const int lr = lane & 31, lh = lane >> 5;
    const T* const qm = reinterpret_cast<const T*>(G.qc) + row * kD + lh * 8;      // its mean as every row of the product
    // k's means in whole kilobytes; as rows of 256 bytes a load took 32 bytes of each of 32
    const T* const km = reinterpret_cast<const T*>(G.kc) + operand_mean_at(bh, G.nbk, 0, 0) + lane * 8;
    V8 qa[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) qa[c] = *reinterpret_cast<const V8*>(qm + 16 * c);
    // four of this wavefront's blocks of 32 are on their way at a time
    for (int n_first = 32 * wave; n_first < G.nbk; n_first += 4 * 32 * kTeam) {
        V8 kr[4][8];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int n0 = n_first + 32 * kTeam * t;
            if (n0 < G.nbk) {
                const T* const kt = km + n0 / 32 * 4096;
#pragma unroll
                for (int c = 0; c < 8; ++c) kr[t][c] = *reinterpret_cast<const V8*>(kt + 512 * c);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int n0 = n_first + 32 * kTeam * t;
            if (n0 < G.nbk) {
                f32x16 acc;
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
                for (int c = 0; c < 8; ++c) acc = mfma32(qa[c], kr[t][c], acc);
                if (lh == 0) scores[n0 + lr] = (T)acc[0];
            }
        }
    }
    __syncthreads();
    if (wave == 0) {
        const uint16_t* const raw = reinterpret_cast<const uint16_t*>(scores);
        int32_t* const list = reinterpret_cast<int32_t*>(mine);
        auto select = [&](auto n_c) -> int {                 // by columns to a lane
            constexpr int kPerLane = decltype(n_c)::value;
            uint32_t val[kPerLane];
#pragma unroll
            for (int j = 0; j < kPerLane; ++j) {
                const int i = j * 64 + lane;
                const uint16_t x = raw[min(i, G.nbk - 1)];
                val[j] = i < G.nbk ? ord_of(x) : 0u;
            }
            int n = G.width;
            if (G.threshold > 0.f) {
                float e[kPerLane];
#pragma unroll
                for (int j = 0; j < kPerLane; ++j) e[j] = j * 64 + lane < G.nbk ? (float)scores[min(j * 64 + lane, G.nbk - 1)] : -INFINITY;
                n = cdf_row<16>(val, e, lane, G.nbk, G.threshold, G.scale, G.k_min, G.width);
            }
            if (n > 0) select_row<uint16_t, kPerLane, false>(val, [&](int i) { return raw[i]; }, lane, G.nbk, n, nullptr, list, nullptr, mine);
            return n;
        };
        int k_sel;
        if (G.nbk <= 64) k_sel = select(std::integral_constant<int, 1>{});
        else if (G.nbk <= 128) k_sel = select(std::integral_constant<int, 2>{});
        else if (kTeam == 1 || G.nbk <= 256) k_sel = select(std::integral_constant<int, 4>{});
        else k_sel = select(std::integral_constant<int, 8>{});
        int32_t* const dst = lists != nullptr ? lists + row * G.width : nullptr;
        wave_sync();
        const int32_t* order_here = list;
        if (k_sel > kPaceWidth) order_here = pace_row(list, k_sel, k_sel, G.nbk, lane, dst, G.by_span);
        else if (dst != nullptr)
            for (int e = lane; e < k_sel; e += 64) dst[e] = list[e];
        if (dst != nullptr)
            for (int e = k_sel + lane; e < G.width; e += 64) dst[e] = -1;
        if (lens != nullptr && lane == 0) lens[row] = (uint32_t)k_sel;
        int total = k_sel;
        if constexpr (kHalfLists) total = expand_list(order_here, k_sel, nsub, halves_list, lane, [&](int tile) { return (int)counts[tile]; });
        if (lane == 0) {
            total_at[0] = total;
            total_at[1] = (int)(order_here - list);
        }
    }
    __syncthreads();
    length = total_at[0];
    return kHalfLists ? reinterpret_cast<const uint32_t*>(halves_list) : mine + __builtin_amdgcn_readfirstlane(total_at[1]);
}

}  // namespace
}  // namespace bsa
