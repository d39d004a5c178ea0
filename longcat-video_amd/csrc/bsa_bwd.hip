// Block-sparse flash-attention backward for gfx950 (bf16 / fp16 MFMA).  The kernels walk q and dO in blocked order.  The caller's
// tensors are either in blocked order too (launch_bwd without `thw`: small passes make delta, M2 and k_s) or in (T, H, W) token
// order, where one pass (bwd_prepare_kernel) makes what they need of the tensors where these lie, the real rows of a ragged chunk
// in front of its padding, and the kernels store every gradient row at its token (BwdThw, BwdStore).
//
// Follows the reference's backward (bsa_interface.py:341-461; kernels flash_attn_bsa_varlen_mask.py:288-360
// for dK/dV and :428-462 for dQ, wrappers :630-642 and :943-945) with the same rounding points:
//   M2 = lse * log2(e);  k_s = k * (sm_scale * log2(e)) rounded once to the storage type;
//   delta = rowsum(o * do) in fp32;
//   per (query block, selected KV block): s = q . k_s^T, p = exp2(s - M2), dp = do . v^T (all fp32),
//   ds = p * (dp - delta) rounded to the storage type, p rounded to the storage type for dV;
//   dV = sum p^T do,  dK = sm_scale * sum ds^T q,  dQ = ln 2 * sum ds k_s  (fp32 accumulators, one final rounding).
//
// Data movement.  dK / dV: k and v rows from where the caller has them (BwdLoad) into registers, scaled there; q and dO in blocked order
// through LDS (global_load_lds_dwordx4): row fragments (A operand whose rows are tokens) come out of it with ds_read_b128,
// transposed ones (A operand whose rows are head-dim columns, contraction over 16 tokens in accumulator order) with
// ds_read_b64_tr_b16.  dQ from kept dS: k_s as transposed fragments, written once by the pass in front, straight into registers.
// dQ from scratch: k_s and v in blocked order through LDS, q and dO rows in registers.
//
// dQ from scratch: one wavefront per 64 query rows (two halves of 32, so that every K_s and V fragment feeds two MFMAs).
// S^T = K_s Q^T and dP^T = V dO^T (Q and dO rows in registers as B operands) put one query per lane, so M2 and
// delta are one scalar per lane and dS^T in the accumulator registers is already the B operand of
// dQ^T += K_s^T dS^T.
// dK, dV: one kernel, a workgroup of two wavefronts per 64 keys.  S = Q K_s^T and dP = dO V^T (K_s and V rows in
// registers as B operands) put one key per lane; P and dS in the accumulator registers are the B operands of
// dV^T += dO^T P and dK^T += Q^T dS.
// Where its dS fits in memory the dK / dV kernel runs first and keeps it, and dQ is one product instead of three
// (bwd_dq_from_ds_kernel).
// The query blocks of a KV block come from a bit matrix [KV block][query block] that a small kernel fills from
// the forward's lists (ascending order for free).  Lists are expected to name a block at most once, as a
// selection does; for a repeated block dQ follows the list (as the forward does) and dK / dV the bit matrix, like
// the reference.
#include "bsa_mfma.h"
#include "bsa_slots.h"

#include <algorithm>
#include <atomic>

namespace bsa {
namespace {

using namespace mfma;

constexpr float kRcpLn2 = 1.4426950408889634f;
constexpr int kBwdHalfTileBytes = kTileBytes / 2;            // 32 rows of 256 B

// ------------------------------------------------------------------ small passes
// the sum of products of a lane's eight values, the same instructions in every kernel: fp16 pairs in one (what the compiler makes
// of the plain loop in one kernel and not in the next), bf16 one by one
__device__ __forceinline__ float dot8(const f16x8& a, const f16x8& b) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e += 2) s = __builtin_amdgcn_fdot2(f16x2{a[e], a[e + 1]}, f16x2{b[e], b[e + 1]}, s, false);
    return s;
}
__device__ __forceinline__ float dot8(const bf16x8& a, const bf16x8& b) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s = fmaf((float)a[e], (float)b[e], s);
    return s;
}

// Per query row, both negated because the kernels below add them (as the start value of an MFMA chain):
// delta[row] = -sum_d o * do (fp32), m2[row] = -lse * log2(e), -inf for rows without any key (their p is then 0).
// One 16-lane group per row.
template <typename T>
__global__ __launch_bounds__(256) void bwd_rows_kernel(const T* __restrict__ o, const T* __restrict__ dout,
                                                       const float* __restrict__ lse, float* __restrict__ delta,
                                                       float* __restrict__ m2, int64_t rows) {
    typedef typename Vec8<T>::type V8;
    const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    const int c = threadIdx.x & 15;
    float s = 0.f;
    if (row < rows) {
        const V8 a = *reinterpret_cast<const V8*>(o + row * kD + c * 8);
        const V8 b = *reinterpret_cast<const V8*>(dout + row * kD + c * 8);
        s = dot8(a, b);
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (row < rows && c == 0) {
        delta[row] = -s;
        const float l = lse[row];
        m2[row] = l == -INFINITY ? -INFINITY : -(l * kRcpLn2);
    }
}

// k_s = k * c, rounded once to the storage type (the product is formed in fp32, as torch does for a tensor times
// a Python scalar).  Padded keys' rows (bits of tile_valid, optional, a word for 64 of a head's Sk keys) become zeros, whatever k
// holds there: the kernels start their products from -inf, and an infinite product would make a NaN of that.
template <typename T>
__global__ __launch_bounds__(256) void bwd_scale_kernel(const T* __restrict__ k, T* __restrict__ ks, float c, int64_t n8,
                                                        const uint64_t* __restrict__ tile_valid, uint32_t Sk) {
    typedef typename Vec8<T>::type V8;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    uint4 raw = *reinterpret_cast<const uint4*>(k + i * 8);
    if (tile_valid != nullptr) {
        const uint32_t key = (uint32_t)(i >> 4) % Sk;              // all heads' rows fit 32 bits: 2^32 of them would be a terabyte
        keep_if(raw, (tile_valid[key / kTile] >> (key % kTile)) & 1ull);
    }
    V8 x = __builtin_bit_cast(V8, raw);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (T)((float)x[e] * c);
    *reinterpret_cast<V8*>(ks + i * 8) = x;
}

// Transposed fragments of k_s, what the dQ product takes as its A operand: per 64-key tile (16 KB) [half kh][key step st][d tile
// t][lane l][8 elements], element j of lane l = k_s[key 32 kh + 16 st + 8 (j >> 2) + 4 (l >> 5) + (j & 3)][d = 32 t + (l & 31)], the
// keys of a step in accumulator order.  A workgroup of 256 turns its tile in 16 KB of LDS: row r of a half lies there with unit
// p ^ f(r) at its 16-byte slot p, f(r) = ((r & 3) << 2) | ((r >> 2) & 3), as transposing reads want it.
__device__ __forceinline__ void put_turned_row(char* lds, int row, int c16, const uint4& x) {
    const int r = row & 31, f = ((r & 3) << 2) | ((r >> 2) & 3);
    *reinterpret_cast<uint4*>(lds + (row >> 5) * kBwdHalfTileBytes + r * 256 + ((c16 ^ f) << 4)) = x;
}
// The lane's offset of the first (hi: second) four rows of a transposed fragment of d tile t in a half that lies like this; 4096
// further per step of 16 rows.
__device__ __forceinline__ uint32_t turned_offset(int lane, int t, int hi) {
    const int lh = lane >> 5, s16 = lane & 15, g1 = (lane >> 4) & 1, tx = s16 >> 2, ty = (s16 & 3) >> 1, tz = s16 & 1;
    return (uint32_t)((4 * lh + tx + 8 * hi) * 256) + ((((uint32_t)(4 * t + 2 * g1 + ty)) ^ (uint32_t)((4 * tx) | (lh + 2 * hi))) << 4) +
           (uint32_t)(tz * 8);
}
__device__ __forceinline__ void store_turned_tile(const char* lds, char* out, int halves) {
    const int lane = threadIdx.x & 63, t = threadIdx.x >> 6;                 // a wavefront per d tile
    const uint32_t lo_at = turned_offset(lane, t, 0), hi_at = turned_offset(lane, t, 1);
    for (int x = 0; x < 2 * halves; ++x) {                                   // 16-key steps
        const s16x4 lo = lds_read_tr16(lds + x * 4096 + lo_at), hi = lds_read_tr16(lds + x * 4096 + hi_at);
        *reinterpret_cast<s16x8*>(out + x * 4096 + t * 1024 + lane * 16) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
}
// k_s as bwd_scale_kernel makes it, in transposed fragments: a workgroup per tile of 64 rows.
template <typename T>
__global__ __launch_bounds__(256) void bwd_scale_turned_kernel(const T* __restrict__ k, char* __restrict__ ks_turned, float c,
                                                               const uint64_t* __restrict__ tile_valid, int tiles) {
    typedef typename Vec8<T>::type V8;
    __shared__ __attribute__((aligned(16))) char turned[kTileBytes];
    const int c16 = threadIdx.x & 15, rg = threadIdx.x >> 4;
    const int64_t tile = blockIdx.x;
    const uint64_t word = tile_valid != nullptr ? tile_valid[tile % tiles] : ~0ull;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        V8 x = *reinterpret_cast<const V8*>(k + (tile * kTile + rg + 16 * i) * kD + c16 * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (T)((float)x[e] * c);
        uint4 raw = __builtin_bit_cast(uint4, x);
        keep_if(raw, (word >> (rg + 16 * i)) & 1ull);
        put_turned_row(turned, rg + 16 * i, c16, raw);
    }
    __syncthreads();
    store_turned_tile(turned, ks_turned + tile * kTileBytes, 2);
}

// Where a gradient row goes when the caller's tensors are in token order: the token of every blocked-order slot of one
// (batch, head) (-1: padding, nothing is stored) and the element strides of the destination.  rows null: blocked order.
struct BwdStore {
    const int32_t* rows;
    int64_t sB, sH, sS;
    int Hn;
};
// Where the dK / dV kernel reads k and v: element strides; rows by token or, with rows_by_slot, by slot (the same where no row table is
// stored through).
struct BwdLoad {
    const void* p;
    int64_t sB, sH, sS;
};

// What the kernels below need of tensors in token order, in one launch (HBM-bound): q and dO in blocked order, k_s in transposed
// fragments (where dS is kept) or in blocked order beside v (for dQ from scratch), delta and M2 per slot (padded slots: zero rows, delta -0, M2 -inf, so that their p is 0), the row tables of both grids, the validity
// words of the keys, and the bit matrix cleared.  A workgroup per 64-slot tile; workgroups 0 .. wg_q - 1 take tiles of the
// queries, the next wg_k tiles of the keys, the rest words of the matrix.  delta and M2 as bwd_rows_kernel takes them.
// On a padded grid the real rows of a chunk come first, so that the halves of 32 slots behind them hold none: these are neither
// written nor walked by the kernels, which take from `q_live` and `k_live` how many halves of a block to walk.  Forward and
// backward with slots as they lie / packed: 6 heads of 9x17x30 (a third of the halves are empty) 266.6 / 235.1 us, 32 heads of
// 24x30x52 (an eighth of the tiles have one half) 7 895 / 7 793.
// Five launches less in front of a small backward, at 4 us each; at 32 heads of 24x30x52 it takes what the separate passes took.
struct BwdPrep {
    Grid3 gq, gk;
    int Hn;
    const uint16_t *q, *o, *dout, *k, *v;
    int64_t q_st[3], o_st[3], do_st[3], k_st[3], v_st[3];      // element strides {batch, head, token}
    const float* lse;                                          // [B * Hn][tokens]
    int64_t q_tokens;
    uint16_t *q_blocked, *dout_blocked, *ks, *v_blocked;      // v_blocked null: k_s in transposed fragments
    float *delta, *m2;
    int32_t *q_rows, *k_rows;
    uint64_t* valid;
    uint32_t* bits;
    int64_t n_bits;
    float c;                                                   // of k_s
    int32_t *q_live, *k_live;                                  // of the grid's blocks; null: no padding, slots as they lie
    uint32_t* planes;                                          // with q_live: LiveHalves::planes
    int n_planes, plane_words;
};
template <typename T>
__global__ __launch_bounds__(256) void bwd_prepare_kernel(BwdPrep a, int wg_q, int wg_k) {
    typedef typename Vec8<T>::type V8;
    __shared__ __attribute__((aligned(16))) char turned[kTileBytes];
    const int lane = threadIdx.x & 63, c16 = threadIdx.x & 15, rg = threadIdx.x >> 4;
    const int w = blockIdx.x;
    if (w >= wg_q + wg_k) {
        const int64_t i = (int64_t)(w - wg_q - wg_k) * 256 + threadIdx.x;
        if (i < a.n_bits) a.bits[i] = 0u;
        if (a.k_live != nullptr && i < a.gk.blocks()) a.k_live[i] = live_halves(a.gk, (int)i);
        if (a.q_live != nullptr && (i & ~63ll) < a.gq.blocks()) {              // whole wavefronts
            const int n = i < a.gq.blocks() ? live_halves(a.gq, (int)i) : 0;
            if (i < a.gq.blocks()) a.q_live[i] = n;
            for (int p = 0; p < a.n_planes; ++p) {
                const uint64_t bit = __ballot((n >> p) & 1);
                if (lane < 2) a.planes[p * a.plane_words + (i >> 6) * 2 + lane] = (uint32_t)(bit >> (32 * lane));
            }
        }
        return;
    }
    const bool queries = w < wg_q, packed = (queries ? a.q_live : a.k_live) != nullptr;
    const Grid3& g = queries ? a.gq : a.gk;
    const int per_chunk = g.chunk() / kTile, tiles = g.blocks() * per_chunk;
    const int id = queries ? w : w - wg_q, bh = id / tiles, tile = id - bh * tiles;
    const int batch = bh / a.Hn, head = bh - batch * a.Hn;
    const Slots s = packed ? packed_slots_of(g, tile / per_chunk, tile % per_chunk, lane) : slots_of(g, tile / per_chunk, tile % per_chunk, lane);
    if (bh == 0 && threadIdx.x < 64) {
        (queries ? a.q_rows : a.k_rows)[(int64_t)tile * kTile + lane] = s.token;
        if (!queries && lane == 0) a.valid[tile] = s.word;
    }
    // 16-row sweeps: of both halves, of the first alone, none
    const int sweeps = !packed || (s.word >> 32) != 0ull ? 4 : s.word != 0ull ? 2 : 0;
    const int64_t row0 = (int64_t)id * kTile + rg;             // of the blocked tensors
    int token[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) token[i] = max(__shfl(s.token, rg + 16 * i), 0);
    auto at = [&](const uint16_t* p, const int64_t (&st)[3], int i) -> uint4 {
        return *reinterpret_cast<const uint4*>(p + batch * st[0] + head * st[1] + (int64_t)token[i] * st[2] + c16 * 8);
    };
    auto put = [&](uint16_t* p, int i, const uint4& x) { *reinterpret_cast<uint4*>(p + (row0 + 16 * i) * kD + c16 * 8) = x; };
    if (queries) {
        uint4 q[4], o[4], d[4];
        float l[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < sweeps) { q[i] = at(a.q, a.q_st, i); o[i] = at(a.o, a.o_st, i); d[i] = at(a.dout, a.do_st, i); }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < sweeps) l[i] = a.lse[bh * a.q_tokens + token[i]];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i >= sweeps) break;
            const bool real = (s.word >> (rg + 16 * i)) & 1ull;
            keep_if(q[i], real); keep_if(o[i], real); keep_if(d[i], real);
            float sum = dot8(__builtin_bit_cast(V8, o[i]), __builtin_bit_cast(V8, d[i]));
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
            put(a.q_blocked, i, q[i]);
            put(a.dout_blocked, i, d[i]);
            if (c16 == 0) {
                a.delta[row0 + 16 * i] = -sum;
                a.m2[row0 + 16 * i] = !real || l[i] == -INFINITY ? -INFINITY : -(l[i] * kRcpLn2);
            }
        }
    } else {
        const bool rows = a.v_blocked != nullptr;
        uint4 k[4], v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < sweeps) {
                k[i] = at(a.k, a.k_st, i);
                if (rows) v[i] = at(a.v, a.v_st, i);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i >= sweeps) break;
            const bool real = (s.word >> (rg + 16 * i)) & 1ull;
            V8 x = __builtin_bit_cast(V8, k[i]);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = (T)((float)x[e] * a.c);
            uint4 ks = __builtin_bit_cast(uint4, x);
            keep_if(ks, real);
            if (rows) {
                keep_if(v[i], real);
                put(a.ks, i, ks);
                put(a.v_blocked, i, v[i]);
            } else {
                put_turned_row(turned, rg + 16 * i, c16, ks);
            }
        }
        if (rows) return;
        __syncthreads();
        store_turned_tile(turned, reinterpret_cast<char*>(a.ks) + (int64_t)id * kTileBytes, sweeps / 2);
    }
}

__global__ void bwd_zero_kernel(uint32_t* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// The halves (32 slots) of a block that hold rows.  live null: all of them, `full`.
struct LiveHalves {
    const int32_t* live;             // per block of the grid
    // Of the query blocks also bit by bit: bit m % 32 of word p * plane_words + m / 32 is bit p of live[m], so that the halves of a
    // set of query blocks, a row of the bit matrix, are counted a word at a time.
    const uint32_t* planes;
    int n_planes, plane_words, full;
};
// halves of the query blocks of `bits`, word w of a row of the bit matrix
__device__ __forceinline__ int halves_of(const LiveHalves& q, uint32_t bits, int w) {
    if (q.live == nullptr) return q.full * __popc(bits);
    int n = 0;
    for (int p = 0; p < q.n_planes; ++p) n += __popc(bits & q.planes[p * q.plane_words + w]) << p;
    return n;
}

// counts[bh * nbk + j] = number of query halves that KV block j meets (those of the blocks set in its row of the bit matrix); with
// `base` also the number of dS units (kDsUnitBytes) of the head's blocks in front of j; order: the head's KV tiles by descending
// count in whole blocks, a counting sort (tiles of one count in no particular order).  One workgroup per head.  LDS: a bin per
// count, 0 .. nbq, and a word per wavefront at least.
constexpr int kCountThreads = 1024;      // of 256 where there are no more blocks
__global__ __launch_bounds__(kCountThreads) void bwd_count_kernel(const uint32_t* __restrict__ bits, int32_t* __restrict__ counts,
                                                        int32_t* __restrict__ base, int32_t* __restrict__ order, int words, int nbk, int nbq,
                                                        int tiles_per_block, LiveHalves q, Divisor by_full) {
    extern __shared__ int bins[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), threads = blockDim.x;
    const int64_t head = (int64_t)blockIdx.x * nbk;
    int before = 0;
    for (int j0 = 0; j0 < nbk; j0 += threads) {
        const int j = j0 + threadIdx.x;
        int c = 0;
        if (j < nbk) {
            const uint32_t* row = bits + (head + j) * words;
            for (int w0 = 0; w0 < words; w0 += 8) {                // eight words on their way
                uint32_t x[8];
#pragma unroll
                for (int w = 0; w < 8; ++w) x[w] = row[min(w0 + w, words - 1)];
#pragma unroll
                for (int w = 0; w < 8; ++w)
                    if (w0 + w < words) c += halves_of(q, x[w], w0 + w);
            }
        }
        if (j < nbk) counts[head + j] = c;
        if (base == nullptr) continue;
        int upto = wave_scan(c);
        if (lane == 63) bins[wave] = upto;
        __syncthreads();
        const int sums = wave_scan(lane < threads / 64 ? bins[lane] : 0);         // the wavefronts in front, then all of them
        upto += wave > 0 ? __builtin_amdgcn_readlane(sums, wave - 1) : 0;
        if (j < nbk) base[head + j] = (before + upto - c) * tiles_per_block;
        before += __builtin_amdgcn_readlane(sums, 63);
        __syncthreads();
    }
    for (int i = threadIdx.x; i <= nbq; i += threads) bins[i] = 0;
    __syncthreads();
    auto bin = [&](int j) -> int { return (counts[head + j] + q.full - 1) / by_full; };
    for (int j = threadIdx.x; j < nbk; j += threads) atomicAdd(&bins[bin(j)], tiles_per_block);       // this thread's own counts
    __syncthreads();
    // offsets in descending count: lane l of the first wavefront takes the l-th share of the bins, from the top
    if (wave == 0) {
        const int per = (nbq + 64) / 64, top = nbq - lane * per;
        int mine = 0;
        for (int i = 0; i < per; ++i)
            if (top - i >= 0) mine += bins[top - i];
        int run = wave_scan(mine) - mine;
        for (int i = 0; i < per; ++i)
            if (top - i >= 0) { const int n = bins[top - i]; bins[top - i] = run; run += n; }
    }
    __syncthreads();
    const int first_tile = (int)blockIdx.x * nbk * tiles_per_block;
    for (int j = threadIdx.x; j < nbk; j += threads) {
        const int to = atomicAdd(&bins[bin(j)], tiles_per_block);
        for (int i = 0; i < tiles_per_block; ++i) order[first_tile + to + i] = first_tile + j * tiles_per_block + i;
    }
}

// place[row * stride + e] = the first dS unit of list entry e in the order in which the dK / dV kernel walks its head: KV blocks
// ascending, inside a block its query blocks ascending (the halves of the query blocks in front of this one among the bits of
// the block's row).  zeros: kDsUnitBytes to clear.
__global__ __launch_bounds__(256) void bwd_place_kernel(const int32_t* __restrict__ idx, const int32_t* __restrict__ lens,
                                                        const uint32_t* __restrict__ bits, const int32_t* __restrict__ base,
                                                        int32_t* __restrict__ place, int nbq, int nbk, int stride, int words,
                                                        int tiles_per_block, int64_t rows, LiveHalves q, uint4* __restrict__ zeros) {
    if (blockIdx.x == 0) zeros[threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int64_t bh = row / nbq;
    const int m = (int)(row - bh * nbq);
    const int n = min(max(lens[row], 0), stride);
    for (int e = threadIdx.x & 63; e < n; e += 64) {
        const int64_t j = bh * nbk + min(max(idx[row * stride + e], 0), nbk - 1);
        const uint32_t* r = bits + j * words;
        int rank = halves_of(q, r[m >> 5] & ((1u << (m & 31)) - 1u), m >> 5);
        for (int w = 0; w < (m >> 5); ++w) rank += halves_of(q, r[w], w);
        place[row * stride + e] = base[j] + rank * tiles_per_block;
    }
}

template <typename T, typename V8>
__device__ __forceinline__ V8 pack8(const f32x16& x, int s) {
    V8 r;
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = (T)x[8 * s + j];
    return r;
}

// ------------------------------------------------------------------ dQ
// One wavefront per 64 query rows, as two halves of 32 so that every K_s and V fragment feeds two MFMAs.  The K_s and
// V rows of a half tile (32 keys x 256 B each, as they lie in memory - no fragment-order copies) go from global
// memory straight into the wavefront's own LDS (global_load_lds_dwordx4, two stages of 16 KB: one being read, one on
// its way, completion counted by hand), the row fragments come from there with ds_read_b128 and the transposed K_s
// fragments with ds_read_b64_tr_b16 (slot p of row r holds 16-byte unit p ^ f(r), f(r) = ((r & 3) << 2) | ((r >> 2) & 3),
// applied on the global side of the DMA, so that neither kind of read collides on a bank).  That leaves the registers
// for two sets of S^T / dP^T accumulators, so the products of the next half are issued between the exponentials of
// this one: the wavefront has its SIMD to itself and nothing else fills the MFMA pipe while it computes
// exponentials.  S^T and dP^T accumulate in ordinary registers (MFMAs from inline assembly, Q and dO named in the
// accumulation registers they are kept in); the compiler adds no wait states behind such an MFMA and moves no LDS
// read across it, so a set is first read a whole group of MFMAs after it was written and the row fragments are
// requested a group ahead by hand.
// First MFMA of a chain that starts from a block of registers instead of zero (B operand in an accumulation
// register): S^T - M2 comes out of the products, and the exponentials need no subtraction.
__device__ inline void mfma_from(f32x16& acc, bf16x8 a, bf16x8 b, const f32x16& init) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(acc) : "v"(a), "a"(b), "v"(init));
}
__device__ inline void mfma_from(f32x16& acc, f16x8 a, f16x8 b, const f32x16& init) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %3" : "=&v"(acc) : "v"(a), "a"(b), "v"(init));
}
// An MFMA reads its C operand for as long as its passes run, and nothing holds back a VALU write to those registers meanwhile
// (fifteen wait states; the compiler adds them behind its own MFMAs, not behind an assembly statement, where it sees the
// registers free at once).  The blocks that start a chain stay allocated up to here, at least two MFMAs on.
__device__ __forceinline__ void keep_start(const f32x16& a, const f32x16& b) { asm volatile("" :: "v"(a), "v"(b)); }

constexpr int kDqStage = 2 * kBwdHalfTileBytes;              // K_s rows and V rows of 32 keys
constexpr int kDqRingLds = 2 * kDqStage;

// kMasked: the caller has a validity word per KV tile (padding keys exist); they cost nothing per P element (see
// start_block below), only the look-up of the word per half tile.
// what the dQ kernels would divide by
struct DqSizes {
    int tiles;                       // query tiles of a (batch, head)
    Divisor by_tiles, by_block, by_sub, by_round;      // ... of a query block; tiles of a KV block; items of a round
};
// Halves with rows of query tile `item`, tile `sub` of its block: 2 where nothing is padded.
__device__ __forceinline__ int query_halves(const int32_t* q_live, int item, int head, const DqSizes& sz, int tiles_per_block) {
    if (q_live == nullptr) return 2;
    const int tile = item - head * sz.tiles, block = tile / sz.by_block;
    return min(max(__builtin_amdgcn_readfirstlane(q_live[block]) - 2 * (tile - block * tiles_per_block), 0), 2);
}
// Sixteen values of a lane's row, accumulator i <-> column 8 (i / 4) + 4 lh + i % 4, rounded and stored as 16-byte pieces: lanes l
// and l + 32, which hold one row, trade so that each has eight columns in a row of two of the four groups.
template <typename T>
__device__ __forceinline__ void store_columns(T* row, bool real, const float (&x)[16], int lane) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    uint2 p[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) p[g] = __builtin_bit_cast(uint2, T4{(T)x[4 * g], (T)x[4 * g + 1], (T)x[4 * g + 2], (T)x[4 * g + 3]});
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
        const auto a = __builtin_amdgcn_permlane32_swap(p[g].x, p[g + 1].x, false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(p[g].y, p[g + 1].y, false, false);
        if (real) *reinterpret_cast<uint4*>(row + 8 * g + 8 * (lane >> 5)) = make_uint4(a[0], b[0], a[1], b[1]);
    }
}
// dQ of a wavefront's 64 rows: accumulator i of d tile t <-> d = 32 t + 8 (i / 4) + 4 lh + i % 4, query lr (+ 32), row `rows` of the
// destination (negative: a padded slot of a token-order destination)
template <typename T>
__device__ __forceinline__ void store_dq(const f32x16 (&acc)[4][2], T* dq, const BwdStore& w, int64_t bh, int64_t Sq, const int64_t (&rows)[2], int lane) {
    T* const base = w.rows == nullptr ? dq + bh * Sq * kD : dq + (bh / w.Hn) * w.sB + (bh % w.Hn) * w.sH;
    const int64_t pitch = w.rows == nullptr ? kD : w.sS;
#pragma unroll
    for (int qq = 0; qq < 2; ++qq)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float x[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) x[i] = acc[t][qq][i] * kLn2;
            store_columns(base + rows[qq] * pitch + 32 * t, rows[qq] >= 0, x, lane);
        }
}
__device__ __forceinline__ int wave_sum(int x) {
    return __builtin_amdgcn_readlane(wave_scan(x), 63);
}
template <typename T, bool kMasked>
__global__ __launch_bounds__(64) void bwd_dq_lds_kernel(const T* __restrict__ q, const T* __restrict__ dout,
                                                        const T* __restrict__ ks, const T* __restrict__ v,
                                                        const float* __restrict__ m2, const float* __restrict__ delta,
                                                        const int32_t* __restrict__ idx, const int32_t* __restrict__ lens,
                                                        const uint64_t* __restrict__ tile_valid, T* __restrict__ dq,
                                                        int64_t Sq, int64_t Sk, int bs_q, int bs_k, int stride, int item_begin,
                                                        int item_end, int round, BwdStore dq_to, DqSizes sz, const int32_t* __restrict__ q_live,
                                                        const int32_t* __restrict__ k_live) {
    typedef typename Vec8<T>::type V8;
    extern __shared__ __attribute__((aligned(1024))) char dq_ring[];
    const int lane = threadIdx.x, lr = lane & 31, lh = lane >> 5;
    int item;
    {
        const int local = blockIdx.x, r0 = local / sz.by_round * round;
        const int n = min(round, item_end - item_begin - r0), w = local - r0, x = w & 7;
        item = item_begin + r0 + x * (n >> 3) + min(x, n & 7) + (w >> 3);
    }
    const int head = item / sz.by_tiles;
    const int64_t bh = head, qrow0 = (int64_t)(item - head * sz.tiles) * kTile, lrow = item / sz.by_block;      // the tiles of a block lie next to each other
    const int nbk = (int)(Sk / kTile) / sz.by_sub, nsub = bs_k / kTile;
    if (query_halves(q_live, item, head, sz, bs_q / kTile) == 0) return;
    const int n = __builtin_amdgcn_readfirstlane(min(max(lens[lrow], 0), stride));
    const int32_t* list = idx + lrow * stride;
    const char* k_src = reinterpret_cast<const char*>(ks) + bh * Sk * (int64_t)(kD * 2);
    const char* v_src = reinterpret_cast<const char*>(v) + bh * Sk * (int64_t)(kD * 2);

    V8 qreg[2][8], doreg[2][8];
    float m_row[2], d_row[2];
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
        const int64_t row = bh * Sq + qrow0 + 32 * qq + lr;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            qreg[qq][c] = *reinterpret_cast<const V8*>(q + row * kD + 16 * c + 8 * lh);
            doreg[qq][c] = *reinterpret_cast<const V8*>(dout + row * kD + 16 * c + 8 * lh);
        }
        m_row[qq] = m2[row];
        d_row[qq] = delta[row];
    }
    f32x16 acc[4][2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int qq = 0; qq < 2; ++qq)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][qq][i] = 0.f;
    f32x16 neg_m[2];                             // what the S^T accumulators of a query half start from
#pragma unroll
    for (int qq = 0; qq < 2; ++qq)
#pragma unroll
        for (int i = 0; i < 16; ++i) neg_m[qq][i] = m_row[qq];       // m2 and delta come negated

    // the walk: the halves with keys of one listed block after another
    auto block_at = [&](int e) -> int { return __builtin_amdgcn_readfirstlane(min(max(list[min(e, n - 1)], 0), nbk - 1)); };
    auto halves_of_block = [&](int block) -> int { return k_live != nullptr ? __builtin_amdgcn_readfirstlane(k_live[block]) : 2 * nsub; };
    int nhalves = 2 * n * nsub;
    if (k_live != nullptr) {
        int mine = 0;
        for (int e = lane; e < n; e += 64) mine += k_live[min(max(list[e], 0), nbk - 1)];
        nhalves = wave_sum(mine);
    }
    // halves come in pairs: an odd number of them ends with the last one again, all of its keys masked
    const int n_real = nhalves;
    nhalves = (nhalves + 1) & ~1;
    int entry = 0, next_block = 0, block_half = 0, half = 0, halves = 0;
    if (n > 0) next_block = block_at(0);
    // ---- global -> LDS: 16 loads of 1 KB per half
    const uint32_t lds0 = lds_address(dq_ring);
    uint32_t voff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = 4 * i + (lane >> 4);                                     // + 16 j
        const int f = ((row & 3) << 2) | ((row >> 2) & 3);
        voff[i] = (uint32_t)((row - 4 * i) * 256 + (((lane & 15) ^ f) << 4));    // load i adds 1 KB on both sides
    }
    uint32_t hv_ahead = ~0u;                     // validity of the keys of the half tile requested last
    auto issue = [&](int hp) {
        if (hp >= nhalves) return;
        if (hp < n_real) {
            if (half == halves) {
                block_half = next_block * 2 * nsub;
                halves = halves_of_block(next_block);
                half = 0;
                next_block = block_at(++entry);
            }
            ++half;
        }
        const int at = block_half + half - 1;
        if (kMasked) hv_ahead = hp < n_real ? (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(tile_valid[at >> 1] >> (32 * (at & 1)))) : 0u;
        const int64_t off = (int64_t)at * kBwdHalfTileBytes;
        const uint32_t dst = lds0 + (hp & 1) * kDqStage;
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
            load_to_lds_4x16(k_src + off + j * 4096, voff, dst + j * 4096);
            load_to_lds_4x16(v_src + off + j * 4096, voff, dst + kBwdHalfTileBytes + j * 4096);
        }
    };
    // ---- LDS -> fragments
    const uint32_t fl = (uint32_t)(((lr & 3) << 2) | ((lr >> 2) & 3));
    uint32_t roff[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) roff[c] = (uint32_t)(lr * 256) + ((((uint32_t)(2 * c + lh)) ^ fl) << 4);
    const int s16 = lane & 15, g1 = (lane >> 4) & 1, tx = s16 >> 2, ty = (s16 & 3) >> 1, tz = s16 & 1;
    uint32_t toff[4][2];                         // turned_offset, written out: as a call the kernels came out 0.3 % slower in small clips
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int hi = 0; hi < 2; ++hi)
            toff[t][hi] = (uint32_t)((4 * lh + tx + 8 * hi) * 256) + ((((uint32_t)(4 * t + 2 * g1 + ty)) ^ (uint32_t)((4 * tx) | (lh + 2 * hi))) << 4) +
                          (uint32_t)(tz * 8);
    V8 kt[8];                                    // the transposed K_s fragments of the half whose dQ products come next
    auto take_transposed = [&](int hp) {
        const char* part = dq_ring + (hp & 1) * kDqStage;
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            const char* base = part + (16 * (x >> 2)) * 256;
            const s16x4 lo = lds_read_tr16(base + toff[x & 3][0]), hi = lds_read_tr16(base + toff[x & 3][1]);
            kt[x] = __builtin_bit_cast(V8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };
    // accumulator i <-> key 8 (i / 4) + 4 lh + i % 4 of the half, query lr (+ 32)
    auto exponentials = [&](f32x16 (&s)[2], f32x16 (&dp)[2], int qq, int i0, int count) {
#pragma unroll
        for (int i = i0; i < i0 + count; ++i) {
            const float p = __builtin_amdgcn_exp2f(s[qq][i]);        // s holds S^T - M2, -inf for a padded key
            s[qq][i] = p * (dp[qq][i] + d_row[qq]);
        }
    };
    // Padded keys: the chain of a half tile that holds any starts from -inf in their accumulators instead of -M2, so
    // their p is exp2(-inf) = 0 and the exponentials test nothing.  Such half tiles are the few at the upper edges of
    // the grid; the start block is rebuilt only when the validity of the half in hand differs from all-valid or the
    // one before did.
    bool start_masked = false;
    auto start_block = [&](uint32_t hv) {
        if (!kMasked) return;
        const bool edge = hv != ~0u;
        if (!edge && !start_masked) return;
        start_masked = edge;
        const uint32_t mine = hv >> (4 * lh);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const bool ok = (mine >> (8 * (i / 4) + (i % 4))) & 1u;
            neg_m[0][i] = ok ? m_row[0] : -INFINITY;
            neg_m[1][i] = ok ? m_row[1] : -INFINITY;
        }
    };
    // S^T and dP^T of half hp (both query halves) into (s, dp); between its groups of four MFMAs the exponentials of
    // the half before, on (ps, pdp), eight accumulators per group.
    auto products = [&](int hp, f32x16 (&s)[2], f32x16 (&dp)[2], auto&& behind_requests, auto&& between) {
        const char* kp = dq_ring + (hp & 1) * kDqStage;
        const char* vp = kp + kBwdHalfTileBytes;
        V8 fk[2], fv[2];
        fk[0] = *reinterpret_cast<const V8*>(kp + roff[0]);
        fv[0] = *reinterpret_cast<const V8*>(vp + roff[0]);
        behind_requests();                       // the DMA set-up runs while the first LDS reads are on their way
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int b = c & 1;
            if (c < 7) {
                fk[b ^ 1] = *reinterpret_cast<const V8*>(kp + roff[c + 1]);
                fv[b ^ 1] = *reinterpret_cast<const V8*>(vp + roff[c + 1]);
            }
            if (c == 0) {
                mfma_from(s[0], fk[b], qreg[0][0], neg_m[0]);
                mfma_s<true, true>(dp[0], fv[b], doreg[0][0]);
                mfma_from(s[1], fk[b], qreg[1][0], neg_m[1]);
                mfma_s<true, true>(dp[1], fv[b], doreg[1][0]);
            } else {
                mfma_s<false, true>(s[0], fk[b], qreg[0][c]);
                mfma_s<false, true>(dp[0], fv[b], doreg[0][c]);
                mfma_s<false, true>(s[1], fk[b], qreg[1][c]);
                mfma_s<false, true>(dp[1], fv[b], doreg[1][c]);
            }
            between(c);
        }
    };
    auto gradients = [&](const f32x16 (&s)[2]) {
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            const V8 ds0 = pack8<T, V8>(s[0], st), ds1 = pack8<T, V8>(s[1], st);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                acc[t][0] = mfma32(kt[4 * st + t], ds0, acc[t][0]);
                acc[t][1] = mfma32(kt[4 * st + t], ds1, acc[t][1]);
            }
        }
    };
    // (s, dp): this half, products done; (ns, ndp): the next half
    auto step = [&](int hp, f32x16 (&s)[2], f32x16 (&dp)[2], f32x16 (&ns)[2], f32x16 (&ndp)[2]) {
        start_block(hv_ahead);                   // validity of half hp + 1, looked up when its rows were requested
        // The next half's rows must have landed; the stage that this half was read from (rows and transposed
        // fragments are in registers) takes half hp + 2.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        products(hp + 1, ns, ndp, [&]() { issue(hp + 2); }, [&](int c) { exponentials(s, dp, c >> 2, 4 * (c & 3), 4); });
        __builtin_amdgcn_sched_barrier(0);
        gradients(s);
        __builtin_amdgcn_sched_barrier(0);
        take_transposed(hp + 1);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // the chains into (ns, ndp) end here, sixteen MFMAs behind their last one
        mfma_chain_end(ns[0]); mfma_chain_end(ns[1]); mfma_chain_end(ndp[0]); mfma_chain_end(ndp[1]);
    };
    if (nhalves > 0) {
        f32x16 sa[2], dpa[2], sb[2], dpb[2];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // the Q / dO rows: from here on the DMA loads are counted by hand
        issue(0);
        const uint32_t hv_first = hv_ahead;
        issue(1);
        asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        start_block(hv_first);
        products(0, sa, dpa, [&]() {}, [&](int) {});
        take_transposed(0);
        asm volatile("s_nop 15\n\ts_nop 7\n\ts_waitcnt lgkmcnt(0)" ::: "memory");
        mfma_chain_end(sa[0]); mfma_chain_end(sa[1]); mfma_chain_end(dpa[0]); mfma_chain_end(dpa[1]);
        for (int hp = 0; hp < nhalves; hp += 2) {                                // halves come in pairs
            step(hp, sa, dpa, sb, dpb);
            step(hp + 1, sb, dpb, sa, dpa);
        }
    }
    int64_t rows[2] = {qrow0 + lr, qrow0 + 32 + lr};
    if (dq_to.rows != nullptr) { rows[0] = dq_to.rows[rows[0]]; rows[1] = dq_to.rows[rows[1]]; }
    store_dq<T>(acc, dq, dq_to, bh, Sq, rows, lane);
}

// ------------------------------------------------------------------ dQ from kept dS
// Where the dK / dV kernel keeps the dS it rounds for its own product (kDsUnitBytes per 32 queries and tile), dQ^T += K_s^T dS^T
// is all that is left to do: one product of three and no exponentials.  A wavefront walks the list of its 64 query rows as in
// bwd_dq_lds_kernel.  Per half tile (32 keys) the transposed fragments of K_s (8 KB) come straight into the registers of the A
// operand; the dS of its 64 queries (4 KB) come into registers too and go through 4 KB of LDS, out of which transposing reads make
// the B operand.  kDsqAhead halves are on their way: a wavefront has its SIMD and all of its registers to itself, and what a
// half needs is dealt out behind the sixteen MFMAs of the one before.  (Both through three stages of LDS, 36 KB a wavefront: the
// loads could only be issued once the reads before them were done, in front of the products: 1.75 ms for 32 heads of 24x30x52,
// 1.50 with everything in L2.)
//   dS in units of 32 queries against a 64-key tile, in the order in which the dK / dV kernel walks them (the tiles of a KV block next
//   to one another): [key half][16-query step st][lane][8 elements], lane = 32 lh + key: the queries 16 st + 4 lh .. + 3 and 8
//   further (the accumulator order of the dK / dV kernel), 1 KB per store instruction.
//   In LDS: unit (key, lh, st) at 16-byte slot 4 key + ((2 lh + st) ^ (key >> 1 & 3)) of its 2 KB block: the 32 lanes of a pass of
//   a transposing read (4 keys x 16 queries, two groups) cover 256 consecutive bytes, and eight lanes that write lie on different
//   banks.  (The order of the slots on the global side instead, as the LDS DMA needs it, gives every lane of a load a cache
//   line of its own: 64 clocks of the address unit for 16, and 1.81 ms.)
constexpr int kDsPairBytes = kTile * kTile * 2, kDsUnitBytes = kDsPairBytes / 2;
constexpr int kDsqAhead = 4;

// kTeam: wavefronts of a workgroup that share the list of its query rows, a contiguous share of the entries each; their sums are
// put together in LDS, in the order of the shares, 4 / kTeam tiles of d to a wavefront.  For calls whose query tiles would leave
// most SIMDs without one (launch_bwd).
template <typename T, int kTeam>
__global__ __launch_bounds__(64 * kTeam, 1) void bwd_dq_from_ds_kernel(const char* __restrict__ ks_turned, const char* __restrict__ ds, const char* __restrict__ zeros,
                                                            const int32_t* __restrict__ idx, const int32_t* __restrict__ place,
                                                            const int32_t* __restrict__ lens, T* __restrict__ dq, int64_t Sq,
                                                            int64_t Sk, int bs_q, int bs_k, int stride, int item_begin, int item_end,
                                                            int round, int64_t pairs_per_head, BwdStore dq_to, DqSizes sz,
                                                            const int32_t* __restrict__ q_live, const int32_t* __restrict__ k_live) {
    typedef typename Vec8<T>::type V8;
    constexpr int kTurnBytes = 2 * 2048, kSumFloats = kTile * kD;
    __shared__ __attribute__((aligned(16))) char turns[kTeam > 1 ? kTeam * kSumFloats * 4 : kTurnBytes];      // a team's sums lie where its dS was
    const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
    const int wave = kTeam > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
    char* const turn = turns + wave * kTurnBytes;
    touch_arguments<decltype(bwd_dq_from_ds_kernel<T, kTeam>)>();
    int item;
    {
        const int local = blockIdx.x, r0 = local / sz.by_round * round;
        const int n = min(round, item_end - item_begin - r0), w = local - r0, x = w & 7;
        item = item_begin + r0 + x * (n >> 3) + min(x, n & 7) + (w >> 3);
    }
    const int head = item / sz.by_tiles, lrow_n = item / sz.by_block;          // the tiles of a block lie next to each other
    const int64_t bh = head, qrow0 = (int64_t)(item - head * sz.tiles) * kTile, lrow = lrow_n;
    const int nbk = (int)(Sk / kTile) / sz.by_sub, nsub = bs_k / kTile, sub_q = item - lrow_n * (bs_q / kTile);
    // the list, 64 entries at a time in a register each, an entry per lane: block, dS unit, halves with keys
    const int n_all = __builtin_amdgcn_readfirstlane(min(max(lens[lrow], 0), stride));
    const int e_begin = n_all * wave / kTeam, n = n_all * (wave + 1) / kTeam - e_begin;      // this wavefront's share
    int list_j = 0, list_p = 0, list_n = 2 * nsub;
    auto take_entries = [&](int e0) {
        const int e = max(min(e_begin + e0 + lane, e_begin + n - 1), 0);
        list_j = min(max(idx[lrow * stride + e], 0), nbk - 1);
        list_p = place[lrow * stride + e];
        if (k_live != nullptr) list_n = k_live[list_j];
    };
    // waited for where they are loaded: the compiler would otherwise wait for them, and with them for every load before, at each half
    auto entries_there = [&]() { asm volatile("" : "+v"(list_j), "+v"(list_p), "+v"(list_n)); };
    take_entries(0);
    const int q_halves = query_halves(q_live, item, head, sz, bs_q / kTile);
    // the tokens of this lane's two rows; the epilogue stores through them
    int64_t rows[2] = {qrow0 + lr, qrow0 + 32 + lr};
    if (dq_to.rows != nullptr) { rows[0] = dq_to.rows[rows[0]]; rows[1] = dq_to.rows[rows[1]]; }
    if (q_halves == 0) return;
    int n_real = 2 * n * nsub;
    if (k_live != nullptr) {
        int mine = lane < n ? list_n : 0;
        for (int e = 64 + lane; e < n; e += 64) mine += k_live[min(max(idx[lrow * stride + e_begin + e], 0), nbk - 1)];
        n_real = wave_sum(mine);
    }
    entries_there();
    const char* k_src = ks_turned + bh * Sk * (int64_t)(kD * 2);
    const char* ds_src = ds + bh * pairs_per_head * kDsPairBytes;
    f32x16 acc[4][2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int qq = 0; qq < 2; ++qq)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][qq][i] = 0.f;

    // ---- the walk: where half hp's fragments and its dS lie, for hp = 0, 1, 2, ...; behind the last half its fragments again, with
    // zeros for dS.  A tile with rows in its first half alone takes that half's dS twice (the second sums are not stored).
    const int second_half = q_halves == 2 ? nsub * kDsUnitBytes : 0;
    int entry = 0, half = 0, walked = 0;
    int64_t k_at = 0;
    struct At { const char *k, *d0, *d1; };
    auto next = [&]() -> At {
        const bool more = walked < n_real;
        const int j = __builtin_amdgcn_readlane(list_j, entry & 63), p = __builtin_amdgcn_readlane(list_p, entry & 63);
        const int of_block = __builtin_amdgcn_readlane(list_n, entry & 63);
        k_at = more ? ((int64_t)j * (2 * nsub) + half) * kBwdHalfTileBytes : k_at;
        const char* d0 = more ? ds_src + ((int64_t)p + 2 * sub_q * nsub + (half >> 1)) * kDsUnitBytes + (half & 1) * 2048 : zeros;
        const char* d1 = more ? d0 + second_half : zeros;
        ++walked;
        const bool done = more && half + 1 == of_block;
        half = done ? 0 : half + 1;
        entry += done ? 1 : 0;
        if (done && (entry & 63) == 0 && entry < n) {
            take_entries(entry);
            entries_there();
        }
        return {k_src + k_at, d0, d1};
    };
    // dS i: query half i >> 1, 16-query step i & 1
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    auto load_ds = [&](const At& a, int i) -> u32x4 {
        return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>((i < 2 ? a.d0 : a.d1) + (i & 1) * 1024 + lane * 16));
    };
    auto load_k = [&](const At& a, int f) -> V8 { return *reinterpret_cast<const V8*>(a.k + f * 1024 + lane * 16); };      // f = 4 st + t

    const int s16 = lane & 15, g1 = (lane >> 4) & 1, tx = s16 >> 2, ty = (s16 & 3) >> 1, tz = s16 & 1;
    const uint32_t turn0 = lds_address(turn);
    const int turn_x = (lr >> 1) & 3;            // of the writing lane's key
    const uint32_t put_at[2] = {turn0 + (uint32_t)((4 * lr + ((2 * lh) ^ turn_x)) * 16), turn0 + (uint32_t)((4 * lr + ((2 * lh + 1) ^ turn_x)) * 16)};
    // chunk s16 & 3: lh' = its bit 0, the unit's half its bit 1; the keys 8 and 16 further have the same two bits
    const uint32_t take_at = turn0 + (uint32_t)((4 * (4 * lh + tx) + ((2 * tz + g1) ^ ((2 * lh + (tx >> 1)) & 3))) * 16 + 8 * ty);
    auto put = [&](int i, const u32x4& x) { *(__attribute__((address_space(3))) u32x4*)(uintptr_t)(put_at[i & 1] + (i >> 1) * 2048) = x; };
    V8 k[kDsqAhead][8], d[2][2][2];              // fragments by half; the B operand [half & 1][query half][16-key step]
    u32x4 raw[kDsqAhead][4];
    s16x4 lo = {};
    auto turn_read = [&](V8 (&to)[2][2], int i) {                // i = 4 st + 2 qq + which four keys
        const s16x4 x = lds_read_tr16_at(take_at + ((i >> 1) & 1) * 2048 + (i >> 2) * 1024 + (i & 1) * 512);
        if ((i & 1) == 0) lo = x;
        else to[(i >> 1) & 1][i >> 2] = __builtin_bit_cast(V8, (s16x8)__builtin_shufflevector(lo, x, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // Half hp, ring slot r, in sixteen slots of an MFMA each.  Its fragments are replaced by those of half hp + kDsqAhead as soon as
    // their second MFMA is out; the dS of half hp + 1 goes into LDS and out of it, its registers take half hp + 1 + kDsqAhead.
    auto step = [&](auto r_c, const At& a, At& ahead) {
        constexpr int r = decltype(r_c)::value, r1 = (r + 1) % kDsqAhead;
        ahead = next();
        __builtin_amdgcn_sched_barrier(0);
        static_for<16>([&](auto slot_c) {
            constexpr int i = decltype(slot_c)::value, st = i >> 3, t = (i >> 1) & 3, qq = i & 1;
            acc[t][qq] = mfma32(k[r][4 * st + t], d[r & 1][qq][st], acc[t][qq]);
            if constexpr (i < 4) put(i, raw[r1][i]);
            else if constexpr (i < 12) turn_read(d[r1 & 1], i - 4);
            if constexpr (qq == 1) k[r][4 * st + t] = load_k(a, 4 * st + t);
            if constexpr (i >= 4 && i < 12 && qq == 0) raw[r1][(i - 4) >> 1] = load_ds(ahead, (i - 4) >> 1);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    if (n_real > 0) {
        At at[kDsqAhead];
#pragma unroll
        for (int r = 0; r < kDsqAhead; ++r) at[r] = next();
#pragma unroll
        for (int r = 0; r < kDsqAhead; ++r) {
#pragma unroll
            for (int f = 0; f < 8; ++f) k[r][f] = load_k(at[r], f);
#pragma unroll
            for (int i = 0; i < 4; ++i) raw[r][i] = load_ds(at[r], i);
        }
        // the first half's dS, whose registers take half kDsqAhead
        At a = next(), ahead;
#pragma unroll
        for (int i = 0; i < 4; ++i) put(i, raw[0][i]);
#pragma unroll
        for (int i = 0; i < 8; ++i) turn_read(d[0], i);
#pragma unroll
        for (int i = 0; i < 4; ++i) raw[0][i] = load_ds(a, i);
        static_assert(kDsqAhead % 2 == 0, "d alternates");
        for (int hp = 0; hp < n_real; hp += kDsqAhead) {
            static_for<kDsqAhead>([&](auto r_c) {
                step(r_c, a, ahead);
                a = ahead;
            });
        }
    }
    if constexpr (kTeam > 1) {
        float* const sums = reinterpret_cast<float*>(turns);
        __syncthreads();                          // every wavefront is through with its dS
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int qq = 0; qq < 2; ++qq)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<float4*>(sums + wave * kSumFloats + (((t * 2 + qq) * 4 + g) * 64 + lane) * 4) =
                        make_float4(acc[t][qq][4 * g], acc[t][qq][4 * g + 1], acc[t][qq][4 * g + 2], acc[t][qq][4 * g + 3]);
        __syncthreads();
        constexpr int kOwn = 4 / kTeam;
        T* const base = dq_to.rows == nullptr ? dq + bh * Sq * kD : dq + (bh / dq_to.Hn) * dq_to.sB + (bh % dq_to.Hn) * dq_to.sH;
        const int64_t pitch = dq_to.rows == nullptr ? kD : dq_to.sS;
#pragma unroll
        for (int qq = 0; qq < 2; ++qq)
#pragma unroll
            for (int own = 0; own < kOwn; ++own) {
                const int t = wave * kOwn + own;
                float x[16];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                    for (int w = 0; w < kTeam; ++w) {
                        const float4 part = *reinterpret_cast<const float4*>(sums + w * kSumFloats + (((t * 2 + qq) * 4 + g) * 64 + lane) * 4);
                        sum.x += part.x; sum.y += part.y; sum.z += part.z; sum.w += part.w;
                    }
                    x[4 * g] = sum.x * kLn2; x[4 * g + 1] = sum.y * kLn2; x[4 * g + 2] = sum.z * kLn2; x[4 * g + 3] = sum.w * kLn2;
                }
                store_columns(base + rows[qq] * pitch + 32 * t, rows[qq] >= 0, x, lane);
            }
        return;
    }
    store_dq<T>(acc, dq, dq_to, bh, Sq, rows, lane);
}

// ------------------------------------------------------------------ dK and dV in one kernel, Q and dO through LDS
// One workgroup of two wavefronts per 64 keys; wavefront w owns keys 32 w .. 32 w + 31 and both of their gradients
// (128 accumulator registers).  The Q and dO tiles of a query tile (64 rows x 256 B each, as they lie in memory)
// go from global memory straight into LDS once per workgroup (global_load_lds_dwordx4; wavefront 0 brings Q and
// the queries' M2 and delta, wavefront 1 brings dO), in halves of 32 queries, four stages deep (two in use, two on
// their way), and both wavefronts take every operand from there: the row fragments (the A operands of S = Q K_s^T and
// dP = dO V^T) with ds_read_b128, the transposed
// ones (the A operands of dV^T += dO^T P and dK^T += Q^T dS) with ds_read_b64_tr_b16.  Per tile pair 32 KB leave
// the caches instead of the 80 KB of fragment-order copies that separate dK and dV kernels stream, S is computed
// once instead of twice (128 MFMAs per tile pair instead of 160), and no fragment-order copy of q or dO is made.
// The LDS side of the DMA is linear in the lane index, so the swizzle that keeps both kinds of read free of bank
// conflicts is applied on the global side: the 16-byte slot p of row r receives unit p ^ f(r),
// f(r) = ((r & 3) << 2) | ((r >> 2) & 3): 16 consecutive rows, and the 4 rows x 4 units of a transposing read's 32 lanes,
// land on different banks.
constexpr int kBwdHalfTile = kTileBytes / 2;                 // 32 query rows of Q or of dO
constexpr int kBwdStats = 1024;                              // M2 (128 B), delta (128 B), -inf (128 B, for padded keys and repeated halves)
constexpr int kBwdStage = 2 * kBwdHalfTile + kBwdStats;      // one half tile of queries: Q rows, dO rows, M2, delta
constexpr int kBwdStages = 4;                                // two in use (this half, the next half's rows), two on their way
constexpr int kBwdLoads = 9;                                 // DMA loads of a wavefront per half: its rows, 8 KB, and the numbers
// The Q parts of all stages, then their dO parts, then their numbers: every LDS read of the loop is a lane's offset, which changes
// with the pair of stages by one bit, and a constant below 2^16, which the instruction holds.
constexpr int kBwdDout = kBwdStages * kBwdHalfTile, kBwdNumbers = 2 * kBwdStages * kBwdHalfTile;
// The list of a KV block's query blocks, in LDS: the block, and above kBlockBits its halves with rows (where any are padded).
constexpr int kBlockBits = 15, kMostLiveHalves = (1 << (32 - kBlockBits)) - 1;
constexpr int kPlanesAtHand = 4;                             // chunks of less than 512 tokens

// What bounds it: with every instruction in a slot behind an MFMA (see the step) the matrix pipes are busy 54 % of the clocks at
// 1.59 GHz, which is what the board's power limit leaves; a wavefront waits 22 % of its time, a quarter of that for LDS.  3.13 ms at 32
// heads of 24x30x52 with dS kept (3.69 before the slots, 4.01 with 337 instructions a half beside the products, 249 since addresses are
// scalars, lists are walked without divisions and padded keys start their chains from -inf).
// kMasked: as in the dQ kernel - without validity words no key is padding and the test is compiled out.
// kKeep: dS, rounded as for the product, is also written out for bwd_dq_from_ds_kernel (pair_base: bwd_count_kernel's base).
// what the dK / dV kernel would divide by or divide to get
struct DkdvSizes {
    int tiles, nbq, nsub;            // key tiles of a (batch, head), query blocks, tiles of a KV block
    Divisor by_tiles, by_block, by_round;
};
// kGroups: pairs of wavefronts that share a tile's list of query blocks, a half of its entries each, every pair with stages of its
// own; at the end one adds up dK and the other dV, through LDS.  2 for calls of no more key tiles than there are compute units,
// which leave two of four SIMDs without a wavefront: see launch_bwd.
template <typename T, bool kMasked, bool kKeep, int kGroups>
__global__ __launch_bounds__(128 * kGroups, 1) void bwd_dkdv_kernel(const T* __restrict__ q, const T* __restrict__ dout,
                                                       BwdLoad k_from, BwdLoad v_from,
                                                       const float* __restrict__ m2, const float* __restrict__ delta,
                                                       const uint32_t* __restrict__ bits,
                                                       const uint64_t* __restrict__ tile_valid, T* __restrict__ dk,
                                                       T* __restrict__ dv, int64_t Sq, int64_t Sk, int words, float ks_scale,
                                                       float dk_scale, int rows_by_slot, const int32_t* __restrict__ order, int n_items, int round,
                                                       BwdStore dk_to, BwdStore dv_to, char* __restrict__ ds_out,
                                                       char* __restrict__ ds_spare, const int32_t* __restrict__ unit_base, int64_t pairs_per_head, DkdvSizes sz,
                                                       LiveHalves q_live, const int32_t* __restrict__ k_live,
                                                       const int32_t* __restrict__ counts) {
    typedef typename Vec8<T>::type V8;
    extern __shared__ __attribute__((aligned(1024))) char bwd_lds[];
    const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) & 1);
    const int group = kGroups > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 7)) : 0;
    touch_arguments<decltype(bwd_dkdv_kernel<T, kMasked, kKeep, kGroups>)>();
    // items longest list first, every XCD on a contiguous run of each group of `round` (see launch_bwd); a scalar, and with it
    // all that is derived from it (left to the compiler, addresses of the loop were made scalars half by half)
    int item;
    {
        const int local = blockIdx.x, r0 = local / sz.by_round * round;
        const int n = min(round, n_items - r0), w = local - r0, x = w & 7;
        item = __builtin_amdgcn_readfirstlane(order[r0 + x * (n >> 3) + min(x, n & 7) + (w >> 3)]);
    }
    const int head = item / sz.by_tiles, block = item / sz.by_block;          // the tiles of a block lie next to each other, over all heads
    const int64_t bh = head;
    const int64_t krow0 = (int64_t)(item - head * sz.tiles) * kTile;
    const int nbq = sz.nbq, nsub = sz.nsub;
    const uint32_t* mask_row = bits + (int64_t)block * words;
    // halves of this tile that hold keys: the second wavefront of a tile with one half brings its share of the rows, no more
    int key_halves = 2;
    if (k_live != nullptr) key_halves = __builtin_amdgcn_readfirstlane(k_live[block - head * (sz.tiles / sz.by_block)]) - 2 * (item - block * nsub);
    // halves come in pairs: an odd number of them ends with the last one again, whose p are 0 (M2 = -inf)
    int n_real = __builtin_amdgcn_readfirstlane(counts[block]), nhalves = (n_real + 1) & ~1;
    // the row of this lane's key: its token, or in blocked order its slot
    int64_t key_row = krow0 + 32 * wave + lr;
    if (dk_to.rows != nullptr) key_row = dk_to.rows[key_row];
    bool key_ok = true;
    if (kMasked) key_ok = (tile_valid[krow0 / kTile] >> (32 * wave + lr)) & 1ull;
    f32x16 acc_dk[4], acc_dv[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) { acc_dk[t][i] = 0.f; acc_dv[t][i] = 0.f; }

    // behind every stage's numbers: M2 for padded keys
    char* const stages = bwd_lds + group * (kBwdStages * kBwdStage);
    *reinterpret_cast<float*>(stages + kBwdNumbers + ((threadIdx.x >> 5) & 3) * kBwdStats + 256 + (threadIdx.x & 31) * 4) = -INFINITY;
    // the query blocks of this KV block, ascending, from the bit matrix into LDS (behind the stages)
    int32_t* qlist = reinterpret_cast<int32_t*>(bwd_lds + kGroups * kBwdStages * kBwdStage);
    uint32_t word_now = 0, plane[kPlanesAtHand] = {};
    auto take_words = [&](int w) {
        word_now = w < words ? mask_row[w] : 0u;
        if (q_live.live != nullptr) {
#pragma unroll
            for (int p = 0; p < kPlanesAtHand; ++p)
                if (p < q_live.n_planes && w < words) plane[p] = q_live.planes[p * q_live.plane_words + w];
        }
    };
    take_words(lane);
    if (key_halves <= 0) return;
    // Resident: K_s and V rows of this wavefront's 32 keys, as B operands (lane = key lr, 8 consecutive d), from where the caller's
    // rows lie.  Asked for here, behind the look-up of their token and in front of the list's: what is waited for before the first
    // product is one chain of dependent loads, not two.
    V8 k_rows[8], v_rows[8];
    {
        const int64_t at_row = rows_by_slot ? krow0 + 32 * wave + lr : max(key_row, (int64_t)0);
        const int batch = head / dk_to.Hn, in_batch = head - batch * dk_to.Hn;
        const T* kp = static_cast<const T*>(k_from.p) + batch * k_from.sB + in_batch * k_from.sH + at_row * k_from.sS + 8 * lh;
        const T* vp = static_cast<const T*>(v_from.p) + batch * v_from.sB + in_batch * v_from.sH + at_row * v_from.sS + 8 * lh;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            k_rows[c] = *reinterpret_cast<const V8*>(kp + 16 * c);
            v_rows[c] = *reinterpret_cast<const V8*>(vp + 16 * c);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    int count = 0;
    for (int w0 = 0; w0 < words; w0 += 64) {
        const int w = w0 + lane;
        if (w0 > 0) take_words(w);
        uint32_t word = word_now;
        if (w == words - 1 && (nbq & 31)) word &= (1u << (nbq & 31)) - 1u;
        const int mine = __popc(word), upto = wave_scan(mine);
        int pos = count + upto - mine;
        if (wave == 0 && group == 0)
            while (word != 0u) {
                const int b = __builtin_ctz(word);
                uint32_t n = 0;
                if (q_live.live != nullptr) {
                    if (q_live.n_planes <= kPlanesAtHand) {
#pragma unroll
                        for (int p = 0; p < kPlanesAtHand; ++p) n |= ((plane[p] >> b) & 1u) << p;
                    } else {
                        n = (uint32_t)q_live.live[32 * w + b];
                    }
                }
                qlist[pos++] = (int32_t)((uint32_t)(32 * w + b) | n << kBlockBits);
                word &= word - 1u;
            }
        count += __builtin_amdgcn_readlane(upto, 63);
    }
    __syncthreads();
    int count_u = __builtin_amdgcn_readfirstlane(count);          // the same in every lane; the compiler cannot tell
    // This pair's share of the list: entries, halves, and the halves in front of it.  Both pairs walk as many as the one that has more:
    // the barriers are the workgroup's.
    int halves_before = 0;
    if constexpr (kGroups > 1) {
        const int all = n_real, middle = count_u >> 1;
        int mine = 0;
        for (int e = lane; e < middle; e += 64) mine += q_live.live != nullptr ? (int)((uint32_t)qlist[e] >> kBlockBits) : q_live.full;
        const int first_share = wave_sum(mine);
        halves_before = group == 0 ? 0 : first_share;
        n_real = group == 0 ? first_share : all - first_share;
        nhalves = (max(first_share, all - first_share) + 1) & ~1;
        qlist += group == 0 ? 0 : middle;
        count_u = group == 0 ? middle : count_u - middle;
    }
    // the walk's halves one after another, without a branch; the entry of the next block is read from LDS a half before it is used
    int next_block = 0, next_entry = 0, block_half = 0, half = 0, halves = 0;
    if (nhalves > 0) next_block = qlist[0];
    if (kGroups > 1 && n_real == 0) {            // an empty share: the other pair's only block, all of it a repeat
        block_half = (int)((uint32_t)__builtin_amdgcn_readfirstlane(next_block) & ((1u << kBlockBits) - 1u)) * q_live.full;
        half = halves = 1;
    }
    auto next_half = [&](bool more) -> int {                     // !more: the last one again
        const uint32_t entry = (uint32_t)__builtin_amdgcn_readfirstlane(next_block);
        const bool fresh = more && half == halves;
        block_half = fresh ? (int)(entry & ((1u << kBlockBits) - 1u)) * q_live.full : block_half;
        halves = fresh ? (q_live.live != nullptr ? (int)(entry >> kBlockBits) : q_live.full) : halves;
        half = (fresh ? 0 : half) + (more ? 1 : 0);
        next_entry = min(next_entry + (fresh ? 1 : 0), kGroups > 1 ? max(count_u - 1, 0) : count_u - 1);
        next_block = qlist[next_entry];
        return block_half + half - 1;
    };

    // ---- global -> LDS
    const uint32_t lds0 = lds_address(bwd_lds) + (uint32_t)(group * (kBwdStages * kBwdStage));
    uint32_t voff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = 4 * i + (lane >> 4);                                     // + 16 j
        const int f = ((row & 3) << 2) | ((row >> 2) & 3);
        voff[i] = (uint32_t)((row - 4 * i) * 256 + (((lane & 15) ^ f) << 4));    // load i adds 1 KB on both sides
    }
    const uint32_t stat_gap = (uint32_t)(reinterpret_cast<const char*>(m2) - reinterpret_cast<const char*>(delta));
    const uint32_t voff_stats = (lane < 32 ? stat_gap : 0u) + (uint32_t)((lane & 31) * 4);      // 32 x M2, 32 x delta
    const char* tile_src = reinterpret_cast<const char*>(wave == 0 ? q : dout) + bh * Sq * (int64_t)(kD * 2);
    const char* stat_src = reinterpret_cast<const char*>(delta) + bh * Sq * 4;
    // half hp of the walk into stage hp % kBwdStages; called for hp = 0, 1, 2, ...  Behind the last half come copies of it, so that
    // every half has kBwdLoads loads behind it to count; both wavefronts bring the numbers.
    const char *src_now = nullptr, *stat_now = nullptr;
    uint32_t dst_now = 0, stat_dst = 0;
    auto issue_begin = [&](int hp) {
        const int64_t at = next_half(hp < n_real);
        const uint32_t stage = (uint32_t)hp & (kBwdStages - 1);
        src_now = tile_src + at * kBwdHalfTile;
        stat_now = stat_src + at * 128;
        dst_now = lds0 + wave * kBwdDout + stage * kBwdHalfTile;
        stat_dst = lds0 + kBwdNumbers + stage * kBwdStats;
    };
    auto issue_piece = [&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        if constexpr (i < 8) load_to_lds_16_at<1024 * (i & 3)>(src_now + (i >> 2) * 4096, voff[i & 3], dst_now + (i >> 2) * 4096);
        else load_to_lds_4(stat_now, voff_stats, stat_dst);
    };
    auto issue = [&](int hp) {
        issue_begin(hp);
        static_for<kBwdLoads>([&](auto i_c) { issue_piece(i_c); });
    };

    // ---- LDS -> fragments
    const uint32_t fl = (uint32_t)(((lr & 3) << 2) | ((lr >> 2) & 3));
    uint32_t roff[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) roff[c] = lds0 + (uint32_t)(lr * 256) + ((((uint32_t)(2 * c + lh)) ^ fl) << 4);
    const int s16 = lane & 15, g1 = (lane >> 4) & 1, tx = s16 >> 2, ty = (s16 & 3) >> 1, tz = s16 & 1;
    uint32_t toff[4][2];                         // turned_offset, written out
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int hi = 0; hi < 2; ++hi)
            toff[t][hi] = lds0 + (uint32_t)((4 * lh + tx + 8 * hi) * 256) + ((((uint32_t)(4 * t + 2 * g1 + ty)) ^ (uint32_t)((4 * tx) | (lh + 2 * hi))) << 4) +
                          (uint32_t)(tz * 8);
    // the queries' M2 as this lane's key sees them: -inf for a padded key, whose chains (its row of k_s is zeros) then give
    // p = exp2(-inf) = 0
    uint32_t numbers = lds0 + (uint32_t)(kBwdNumbers + 16 * lh), m2_at = numbers + (kMasked && !key_ok ? 256u : 0u);
    char* ds_item = !kKeep ? nullptr
        : ds_out + bh * pairs_per_head * kDsPairBytes + ((int64_t)__builtin_amdgcn_readfirstlane(unit_base[block]) + (item - block * nsub) + (int64_t)halves_before * nsub) * kDsUnitBytes + wave * 2048;
    // P and dS of a half as B operands, and the transposed fragments of its rows (dO and Q of d tile t at 2 t and 2 t + 1): its first
    // and its last 16 queries
    V8 p_ab[2], ds_ab[2], tr_ab[2][8];
    V8 fq[4], fd[4];                                             // row fragments c & 3
    // One half tile of queries (32) against this wavefront's 32 keys is 32 MFMAs, and a wavefront has a SIMD to itself: what it
    // does besides has to stand between them, and what they read has to be asked for long before.  A step issues, in slots of one
    // MFMA each, with half hp's S - M2 and dP - delta complete (s, dp):
    //    0 ..  7   dV, dK += the last 16 queries of half hp - 1 (their operands are in registers: nothing is waited for behind the barrier)
    //    8 .. 23   S, dP of half hp + 1, into (s_next, dp_next)
    //   24 .. 31   dV, dK += the first 16 queries of half hp
    // and behind the MFMA of a slot its share of the rest: the chains' start values and row fragments of half hp + 1 four to eight
    // slots before their MFMA, the transposed fragments of half hp sixteen, its exponentials, products and roundings, the DMA
    // loads of half hp + 3.  (Left to the compiler, the transposed reads stood right in front of their MFMAs, four round trips to
    // LDS a half, and the exponentials in bunches: 2 150 clocks a half beside 1 024 of products.)
    // S and dP accumulate in ordinary registers, where the exponentials read them: MFMAs from inline assembly, behind which the
    // compiler adds no wait states - a pair is first read nine MFMAs after its last product.
    V8 kreg[8], vreg[8];
    auto step = [&](auto odd_c, int hp, f32x16& s, f32x16& dp, f32x16& s_next, f32x16& dp_next) {
        constexpr int odd = decltype(odd_c)::value;                  // hp & 1
        constexpr uint32_t qn = (odd ^ 1) * kBwdHalfTile, dn = qn + kBwdDout;      // rows of half hp + 1, in its pair of stages
        constexpr uint32_t qt = odd * kBwdHalfTile, dt = qt + kBwdDout;            // rows of half hp
        // the halves with an odd number alone may be the one that repeats (with two pairs, all behind this one's share)
        const uint32_t m2_here = (odd && kGroups == 1) || hp + 1 < n_real ? m2_at : numbers + 256;
        char* const ds_to = (!odd && kGroups == 1) || hp < n_real ? ds_item : ds_spare;
        auto exponential = [&](int e) {
            s[e] = __builtin_amdgcn_exp2f(s[e]);                     // S - M2 -> P
            asm volatile("" : "+v"(s[e]));
        };
        auto product = [&](int e) {
            dp[e] = s[e] * dp[e];                                    // dP - delta -> dS
            asm volatile("" : "+v"(dp[e]));
        };
        auto round_pair = [&](V8& to, const f32x16& x, int e) {
            to[e & 7] = (T)x[e];
            to[(e + 1) & 7] = (T)x[e + 1];
            asm volatile("" : "+v"(to));
        };
        s16x4 lo[2];                                                 // first halves of transposed fragments on their way
        auto read_transposed = [&](auto n_c) {                       // n = 0 .. 31: 16 st2 + 4 t + 2 (Q or dO) + which half
            constexpr int n = decltype(n_c)::value, st2 = n >> 4, t = (n >> 2) & 3, of_q = (n >> 1) & 1;
            constexpr uint32_t base = (of_q ? qt : dt) + 16 * st2 * 256;
            if constexpr ((n & 1) == 0) {
                lo[st2] = lds_read_tr16_at(toff[t][0] + base);
            } else {
                const s16x4 hi = lds_read_tr16_at(toff[t][1] + base);
                tr_ab[st2][2 * t + of_q] = __builtin_bit_cast(V8, (s16x8)__builtin_shufflevector(lo[st2], hi, 0, 1, 2, 3, 4, 5, 6, 7));
            }
        };
        __builtin_amdgcn_sched_barrier(0);
        static_for<32>([&](auto slot_c) {
            constexpr int i = decltype(slot_c)::value;
            // ---- the MFMA
            if constexpr (i < 8 || i >= 24) {
                constexpr int st2 = i < 8 ? 1 : 0, x = i & 7, t = x >> 1;
                if constexpr ((x & 1) == 0) acc_dv[t] = mfma32(tr_ab[st2][x], p_ab[st2], acc_dv[t]);
                else acc_dk[t] = mfma32(tr_ab[st2][x], ds_ab[st2], acc_dk[t]);
            } else {
                constexpr int c = (i - 8) >> 1;
                if constexpr ((i & 1) == 0) mfma_s<false, true>(s_next, fq[c & 3], kreg[c]);
                else mfma_s<false, true>(dp_next, fd[c & 3], vreg[c]);
            }
            // ---- LDS
            if constexpr (i < 4) {                                   // accumulator e <-> query 8 (e / 4) + 4 lh + e % 4 of the half, key lr
                const f32x4_ mm = lds_read_at<f32x4_>(m2_here + ((odd ^ 1) * kBwdStats + 32 * i));
                const f32x4_ dd = lds_read_at<f32x4_>(numbers + ((odd ^ 1) * kBwdStats + 128 + 32 * i));
                s_next[4 * i] = mm.x; s_next[4 * i + 1] = mm.y; s_next[4 * i + 2] = mm.z; s_next[4 * i + 3] = mm.w;
                dp_next[4 * i] = dd.x; dp_next[4 * i + 1] = dd.y; dp_next[4 * i + 2] = dd.z; dp_next[4 * i + 3] = dd.w;
            } else if constexpr (i < 8) {
                fq[i - 4] = lds_read_at<V8>(roff[i - 4] + qn);
                fd[i - 4] = lds_read_at<V8>(roff[i - 4] + dn);
            } else if constexpr (i < 16) {
                constexpr int c = 4 + ((i - 8) >> 1);
                if constexpr ((i & 1) == 0) fq[c & 3] = lds_read_at<V8>(roff[c] + qn);
                else fd[c & 3] = lds_read_at<V8>(roff[c] + dn);
            }
            if constexpr (i >= 8 && i < 24) read_transposed(std::integral_constant<int, i - 8>{});
            if constexpr (i >= 16 && i < 24) read_transposed(std::integral_constant<int, i>{});
            if constexpr (i >= 24 && i < 28) {
                read_transposed(std::integral_constant<int, 24 + 2 * (i - 24)>{});
                read_transposed(std::integral_constant<int, 25 + 2 * (i - 24)>{});
            }
            // ---- the DMA loads of half hp + 3, into the stage that half hp - 1 was read from: both wavefronts are past the barrier behind it
            if constexpr (i == 0) issue_begin(hp + 3);
            if constexpr (i >= 1 && i <= kBwdLoads) issue_piece(std::integral_constant<int, i - 1>{});
            // ---- exponentials behind slots 0, 1, 3, 4, 6, 7, ..., each product a slot later
            if constexpr (i < 24 && i % 3 != 2) exponential(i / 3 * 2 + i % 3);
            if constexpr (i < 24 && i % 3 != 0) product(i / 3 * 2 + i % 3 - 1);
            // ---- roundings: the first 16 queries' elements are there behind slot 11, all behind slot 23
            if constexpr (i == 12 || i == 15 || i == 18 || i == 21) {
                constexpr int e = 2 * ((i - 12) / 3);
                round_pair(p_ab[0], s, e);
                round_pair(ds_ab[0], dp, e);
            }
            if constexpr (i >= 24 && i < 28) {
                constexpr int e = 8 + 2 * (i - 24);
                round_pair(p_ab[1], s, e);
                round_pair(ds_ab[1], dp, e);
            }
            if constexpr (kKeep && (i == 24 || i == 28))
                __builtin_nontemporal_store(ds_ab[i == 24 ? 0 : 1], reinterpret_cast<V8*>(ds_to + (i == 24 ? 0 : 1024) + lane * 16));
            // ---- The stages come in two pairs; a lane's offsets point into the pair that is read next and go over to the other one
            // with a bit, the rows' behind the even half (whose successor's successor lies there), the transposed reads' behind the odd.
            if constexpr (!odd && i >= 24) roff[i - 24] ^= 2 * kBwdHalfTile;
            if constexpr (!odd && i == 30) { numbers ^= 2 * kBwdStats; m2_at ^= 2 * kBwdStats; }
            if constexpr (odd && i >= 28) { toff[i - 28][0] ^= 2 * kBwdHalfTile; toff[i - 28][1] ^= 2 * kBwdHalfTile; }
            __builtin_amdgcn_sched_barrier(0);
        });
        if (kKeep) ds_item += (int64_t)nsub * kDsUnitBytes;
        // the chains into (s_next, dp_next) end here, eight MFMAs behind their last one
        mfma_chain_end(s_next); mfma_chain_end(dp_next);
        // The loads of half hp + 2 must have landed; behind them are on their way those of half hp + 3 and, with kKeep, the two stores
        // of this half and those of the one before: a store is acknowledged later than a load (waiting for those of the half before
        // cost 0.4 of 4.2 ms at 480p).
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kKeep ? kBwdLoads + 4 : kBwdLoads) : "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);                          // lgkmcnt(0): this half's stage has been read
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
    };
    if (nhalves > 0) {
        issue(0);
        issue(1);
        // k_s = k * c, rounded once to the storage type (as bwd_scale_kernel); padded keys' rows are zeros, whatever lies there: their
        // products start from -inf, and an infinite one would make a NaN of that.  (The wait for the rows is one for all that is
        // on its way; the first two halves have to be there as well.)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            V8 x = k_rows[c];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = (T)((float)x[e] * ks_scale);
            uint4 kr = __builtin_bit_cast(uint4, x), vr = __builtin_bit_cast(uint4, v_rows[c]);
            if (kMasked) { keep_if(kr, key_ok); keep_if(vr, key_ok); }
            // read by assembly MFMAs from accumulation registers
            asm volatile("" : "=a"(kreg[c]) : "0"(__builtin_bit_cast(V8, kr)));
            asm volatile("" : "=a"(vreg[c]) : "0"(__builtin_bit_cast(V8, vr)));
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        issue(2);
        if (kKeep) {                             // as many stores as a half before the first would have left on their way
            const V8 none = {};
            __builtin_nontemporal_store(none, reinterpret_cast<V8*>(ds_spare + lane * 16));
            __builtin_nontemporal_store(none, reinterpret_cast<V8*>(ds_spare + 1024 + lane * 16));
        }
        if (wave >= key_halves) {                // no keys: the rows alone
            for (int hp = 0; hp < nhalves; ++hp) {
                issue(hp + 3);
                asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kBwdLoads) : "memory");      // (the stores in front of the first count for nothing)
                __builtin_amdgcn_s_barrier();
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may land in LDS that is no longer this workgroup's
            if (kGroups > 1) { __syncthreads(); __syncthreads(); }       // where the others put their sums together
            return;
        }
        f32x16 s0, dp0, s1, dp1;
        V8 first_q[8], first_d[8];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4_ mm = lds_read_at<f32x4_>((kGroups == 1 || n_real > 0 ? m2_at : numbers + 256) + 32 * g), dd = lds_read_at<f32x4_>(numbers + (128 + 32 * g));
            s0[4 * g] = mm.x; s0[4 * g + 1] = mm.y; s0[4 * g + 2] = mm.z; s0[4 * g + 3] = mm.w;
            dp0[4 * g] = dd.x; dp0[4 * g + 1] = dd.y; dp0[4 * g + 2] = dd.z; dp0[4 * g + 3] = dd.w;
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            first_q[c] = lds_read_at<V8>(roff[c]);
            first_d[c] = lds_read_at<V8>(roff[c] + kBwdDout);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            mfma_s<false, true>(s0, first_q[c], kreg[c]);
            mfma_s<false, true>(dp0, first_d[c], vreg[c]);
        }
        asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
        mfma_chain_end(s0); mfma_chain_end(dp0);
        // nothing lies in front of the first half
#pragma unroll
        for (int e = 0; e < 8; ++e) { p_ab[1][e] = (T)0.f; ds_ab[1][e] = (T)0.f; }
#pragma unroll
        for (int x = 0; x < 8; ++x) tr_ab[1][x] = p_ab[1];
        for (int hp = 0; hp < nhalves; hp += 2) {                                // halves come in pairs
            step(std::integral_constant<int, 0>{}, hp, s0, dp0, s1, dp1);
            step(std::integral_constant<int, 1>{}, hp + 1, s1, dp1, s0, dp0);
        }
        // the last 16 queries of the last half
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            acc_dv[t] = mfma32(tr_ab[1][2 * t], p_ab[1], acc_dv[t]);
            acc_dk[t] = mfma32(tr_ab[1][2 * t + 1], ds_ab[1], acc_dk[t]);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // nothing may land in LDS that is no longer this workgroup's
    }
    if constexpr (kGroups > 1) {
        // The first pair leaves its dV, the second its dK, 16 KB a wavefront, and takes the other: first pair's sum plus second's.
        if (nhalves > 0) {
            __syncthreads();
            float* const mine = reinterpret_cast<float*>(bwd_lds) + (2 * group + wave) * (32 * kD);
            const float* const theirs = reinterpret_cast<const float*>(bwd_lds) + (2 * (group ^ 1) + wave) * (32 * kD);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x16& x = group == 0 ? acc_dv[t] : acc_dk[t];
                    *reinterpret_cast<float4*>(mine + ((t * 4 + g) * 64 + lane) * 4) = make_float4(x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]);
                }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float4 y = *reinterpret_cast<const float4*>(theirs + ((t * 4 + g) * 64 + lane) * 4);
                    f32x16& x = group == 0 ? acc_dk[t] : acc_dv[t];
                    x[4 * g] += y.x; x[4 * g + 1] += y.y; x[4 * g + 2] += y.z; x[4 * g + 3] += y.w;
                }
        }
    }
    // accumulator i of d tile t <-> d = 32 t + 8 (i / 4) + 4 lh + i % 4, key lr
    {
        const int batch = head / dk_to.Hn, in_batch = head - batch * dk_to.Hn;
        const bool blocked = dk_to.rows == nullptr;
        T* out_k = dk + (blocked ? (bh * Sk + key_row) * kD : batch * dk_to.sB + in_batch * dk_to.sH + key_row * dk_to.sS);
        T* out_v = dv + (blocked ? (bh * Sk + key_row) * kD : batch * dv_to.sB + in_batch * dv_to.sH + key_row * dv_to.sS);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float xk[16], xv[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                // padded keys' sums are replaced before the product, which fp16 would otherwise round with the conversion
                xk[i] = (kMasked && !key_ok ? 0.f : acc_dk[t][i]) * dk_scale;
                xv[i] = kMasked && !key_ok ? 0.f : acc_dv[t][i];
            }
            if (kGroups == 1 || group == 0) store_columns(out_k + 32 * t, key_row >= 0, xk, lane);
            if (kGroups == 1 || group == 1) store_columns(out_v + 32 * t, key_row >= 0, xv, lane);
        }
    }
}

}  // namespace

constexpr size_t kBwdLdsLimit = 160 * 1024;
// LDS of the dK / dV kernel for nbq query blocks: its stages, then the list of a KV block's query blocks
size_t bwd_dkdv_lds_bytes(int nbq, int groups = 1) { return (size_t)groups * kBwdStages * kBwdStage + (size_t)nbq * sizeof(int32_t); }
static_assert((kBwdLdsLimit - (size_t)kBwdStages * kBwdStage) / sizeof(int32_t) < ((size_t)1 << kBlockBits), "a list entry holds the block");
int bwd_max_query_blocks() { return (int)((kBwdLdsLimit - (size_t)kBwdStages * kBwdStage) / sizeof(int32_t)); }

// dS is kept between the two kernels where all of it (every list full) fits kDsBytes: 6.4 GB for 32 heads of 480p, where the
// backward took 6.28 ms instead of 6.61 when both were timed (dQ 1.81 instead of 2.58 ms, dK / dV 3.99 instead of 3.59 with the
// stores; 1.75 and 3.74 ms now).  Beyond
// that dQ is computed from scratch: in groups of heads that fit, each with the tail of its longest lists, nothing is left of
// the gain (32 heads of 720p in groups of seven 31.2 ms, of four 32.1, from scratch 31.3).  Nor is it kept when the caller's
// workspace has no room for it: the pieces that it needs are the last ones.
constexpr size_t kDsBytes = (size_t)8 << 30;
struct KeptDs {
    bool keep;
    int64_t pairs_per_head;
};
static KeptDs plan_ds(int64_t bh, int64_t Sq, int64_t Sk, int bs_q, int bs_k, int idx_stride) {
    const int64_t pairs = (Sq / kTile) * idx_stride * (bs_k / kTile);
    return {pairs <= (int64_t)(kDsBytes / kDsPairBytes) / bh, pairs};
}

// The pieces of the backward's workspace.
struct BwdWs {
    size_t ks, delta, m2, bits, paced, counts, order;      // k_s, with kept dS in transposed fragments, otherwise in blocked order; delta and M2; the bit matrix; the lists in the dQ
                                                           // kernel's visiting order; per KV block its number of query halves; the KV
                                                           // tiles of every head by that number
    size_t q_live, k_live, planes;                         // LiveHalves of both grids (token order, where they are padded)
    size_t base, place, ds, ds_spare, ds_zeros;                      // with kept dS: units in front of a KV block, the first unit of a list entry, dS,
                                                           // where a repeated half's goes, a unit of zeros
    size_t total;
};
static int plane_words(int64_t blocks) { return (int)((blocks + 63) / 64 * 2); }
static int plane_count(int chunk) {
    int bits = 0;
    while ((chunk / 32) >> bits) ++bits;
    return bits;
}
static BwdWs bwd_ws(const KeptDs& kept, int64_t bh, int64_t Sq, int64_t Sk, int bs_q, int bs_k, int idx_stride) {
    BwdWs w;
    size_t off = 0;
    auto take = [&](size_t n) { const size_t at = off; off += (n + 255) / 256 * 256; return at; };
    const size_t words = (size_t)((Sq / bs_q + 31) / 32), nbq = (size_t)(Sq / bs_q), nbk = (size_t)(Sk / bs_k);
    w.ks = take(bh * Sk * kD * 2);
    w.delta = take(bh * Sq * 4);
    w.m2 = take(bh * Sq * 4);
    w.bits = take(bh * nbk * words * 4);
    w.paced = take(bh * nbq * (size_t)idx_stride * 4);
    w.counts = take(bh * nbk * 4);
    w.order = take(bh * (size_t)(Sk / kTile) * 4);
    w.q_live = take(nbq * 4);
    w.k_live = take(nbk * 4);
    w.planes = take((size_t)plane_count(bs_q) * plane_words((int64_t)nbq) * 4);
    w.base = take(kept.keep ? bh * nbk * 4 : 0);
    w.place = take(kept.keep ? bh * nbq * (size_t)idx_stride * 4 : 0);
    w.ds = take(kept.keep ? (size_t)bh * (size_t)kept.pairs_per_head * kDsPairBytes : 0);
    w.ds_spare = take(kept.keep ? kDsUnitBytes : 0);
    w.ds_zeros = take(kept.keep ? kDsUnitBytes : 0);
    w.total = off;
    return w;
}
size_t bwd_workspace_bytes(int B, int Hn, int64_t Sq, int64_t Sk, int bs_q, int bs_k, int idx_stride, bool least) {
    const int64_t bh = (int64_t)B * Hn;
    KeptDs kept = plan_ds(bh, Sq, Sk, bs_q, bs_k, idx_stride);
    if (least) kept.keep = false;
    return bwd_ws(kept, bh, Sq, Sk, bs_q, bs_k, idx_stride).total;
}

hipError_t launch_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout, const float* lse,
                      const int32_t* idx, const int32_t* lens, const uint64_t* tile_valid, void* dq, void* dk, void* dv,
                      int B, int Hn, int64_t Sq, int64_t Sk, int bs_q, int bs_k, int idx_stride, float sm_scale, int dtype,
                      void* workspace, size_t workspace_bytes, hipStream_t st, const BwdThw* thw, bool unequal, bool read_copies) {
    const size_t bh = (size_t)B * Hn;
    KeptDs kept = plan_ds((int64_t)bh, Sq, Sk, bs_q, bs_k, idx_stride);
    kept.keep = kept.keep && !read_copies && bwd_ws(kept, (int64_t)bh, Sq, Sk, bs_q, bs_k, idx_stride).total <= workspace_bytes;
    const BwdWs at = bwd_ws(kept, (int64_t)bh, Sq, Sk, bs_q, bs_k, idx_stride);
    char* ws = static_cast<char*>(workspace);
    char* ks = ws + at.ks;
    float* delta = reinterpret_cast<float*>(ws + at.delta);
    float* m2 = reinterpret_cast<float*>(ws + at.m2);
    const int nbq = (int)(Sq / bs_q), nbk = (int)(Sk / bs_k);
    const int words = (nbq + 31) / 32;
    uint32_t* bits = reinterpret_cast<uint32_t*>(ws + at.bits);
    int32_t* paced = reinterpret_cast<int32_t*>(ws + at.paced);
    int32_t* counts = reinterpret_cast<int32_t*>(ws + at.counts);
    int32_t* order = reinterpret_cast<int32_t*>(ws + at.order);
    int32_t* base = reinterpret_cast<int32_t*>(ws + at.base);
    int32_t* place = reinterpret_cast<int32_t*>(ws + at.place);
    const int nsub = bs_k / kTile;
    // On a padded grid the real rows of a chunk come first, and the halves behind them are left out
    auto packs = [](const Grid3& g) { return (g.T % g.t || g.H % g.h || g.W % g.w) && g.chunk() / 32 <= kMostLiveHalves; };
    LiveHalves q_live = {nullptr, nullptr, 0, 0, bs_q / 32};
    int32_t* k_live = nullptr;
    if (thw != nullptr && packs(thw->gq))
        q_live = {reinterpret_cast<int32_t*>(ws + at.q_live), reinterpret_cast<uint32_t*>(ws + at.planes), plane_count(bs_q), plane_words(nbq), bs_q / 32};
    if (thw != nullptr && packs(thw->gk)) k_live = reinterpret_cast<int32_t*>(ws + at.k_live);

    // the dK / dV kernel's LDS: four stages of half a Q tile, half a dO tile and the queries' M2 / delta, then a KV block's query
    // blocks; bwd_count_kernel has a bin for each of their numbers, less than that
    const size_t lds = bwd_dkdv_lds_bytes(nbq);
    if (lds > kBwdLdsLimit) return hipErrorInvalidValue;          // the C-ABI layer has rejected such a shape already
    const size_t count_lds = (size_t)(nbq + 1 > kCountThreads / 64 ? nbq + 1 : kCountThreads / 64) * sizeof(int);
    // Per device, once: the dK / dV instantiations and bwd_count_kernel may use all of the LDS, and the number of compute units.
    static std::atomic<int> device_cus[64];
    int dev = 0;
    hipError_t e;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    int cus = device_cus[dev].load(std::memory_order_acquire);
    if (cus == 0) {
#define BSA_KERNELS(T, G)                                                                                                                   \
    reinterpret_cast<const void*>(bwd_dkdv_kernel<T, true, false, G>), reinterpret_cast<const void*>(bwd_dkdv_kernel<T, false, false, G>),  \
    reinterpret_cast<const void*>(bwd_dkdv_kernel<T, true, true, G>), reinterpret_cast<const void*>(bwd_dkdv_kernel<T, false, true, G>)
        const void* kernels[] = {reinterpret_cast<const void*>(bwd_count_kernel), BSA_KERNELS(__bf16, 1), BSA_KERNELS(__bf16, 2),
                                 BSA_KERNELS(_Float16, 1), BSA_KERNELS(_Float16, 2)};
#undef BSA_KERNELS
        for (const void* kf : kernels)
            if ((e = hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kBwdLdsLimit)) != hipSuccess) return e;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
        device_cus[dev].store(cus, std::memory_order_release);   // threads racing here set the same attributes
    }
    const int64_t qrows = (int64_t)bh * Sq, krows = (int64_t)bh * Sk, nwords = (int64_t)bh * nbk * words;
    const float c = sm_scale * kRcpLn2;
    BwdStore dq_to = {nullptr, 0, 0, 0, Hn}, dk_to = dq_to, dv_to = dq_to;
    BwdLoad k_from = {k, Hn * Sk * kD, Sk * kD, kD}, v_from = {v, Hn * Sk * kD, Sk * kD, kD};
    float rows_scale = c;            // what makes k_s of the rows at k_from
    if (thw != nullptr) {
        dq_to = {thw->q_rows, thw->dq_st[0], thw->dq_st[1], thw->dq_st[2], Hn};
        dk_to = {thw->k_rows, thw->dk_st[0], thw->dk_st[1], thw->dk_st[2], Hn};
        dv_to = {thw->k_rows, thw->dv_st[0], thw->dv_st[1], thw->dv_st[2], Hn};
        dq = thw->dq; dk = thw->dk; dv = thw->dv;
        k_from = {thw->k, thw->k_st[0], thw->k_st[1], thw->k_st[2]};
        v_from = {thw->v, thw->v_st[0], thw->v_st[1], thw->v_st[2]};
        if (read_copies) v_from = {thw->v_blocked, Hn * Sk * kD, Sk * kD, kD};
        q = thw->q_blocked; v = thw->v_blocked; dout = thw->dout_blocked;
        BwdPrep a = {};
        a.gq = thw->gq; a.gk = thw->gk; a.Hn = Hn;
        a.q = (const uint16_t*)thw->q; a.o = (const uint16_t*)thw->o; a.dout = (const uint16_t*)thw->dout; a.k = (const uint16_t*)thw->k;
        a.v = (const uint16_t*)thw->v;
        for (int i = 0; i < 3; ++i) {
            a.q_st[i] = thw->q_st[i]; a.o_st[i] = thw->o_st[i]; a.do_st[i] = thw->do_st[i]; a.k_st[i] = thw->k_st[i]; a.v_st[i] = thw->v_st[i];
        }
        a.lse = thw->lse; a.q_tokens = (int64_t)thw->gq.T * thw->gq.H * thw->gq.W;
        a.q_blocked = (uint16_t*)thw->q_blocked; a.dout_blocked = (uint16_t*)thw->dout_blocked; a.ks = (uint16_t*)ks;
        a.v_blocked = kept.keep ? nullptr : (uint16_t*)thw->v_blocked;
        a.delta = delta; a.m2 = m2; a.q_rows = thw->q_rows; a.k_rows = thw->k_rows; a.valid = thw->valid;
        a.bits = bits; a.n_bits = nwords; a.c = c;
        a.q_live = const_cast<int32_t*>(q_live.live); a.k_live = k_live;
        a.planes = const_cast<uint32_t*>(q_live.planes); a.n_planes = q_live.n_planes; a.plane_words = q_live.plane_words;
        const int64_t wg_q = qrows / kTile, wg_k = krows / kTile;
        const int64_t last = std::max(nwords, (int64_t)std::max(q_live.live != nullptr ? nbq : 0, k_live != nullptr ? nbk : 0)), wg_bits = (last + 255) / 256;
        if (wg_q + wg_k + wg_bits > 0x7fffffff) return hipErrorInvalidValue;
        const dim3 grid((unsigned)(wg_q + wg_k + wg_bits)), blk(256);
        if (dtype == BSA_BF16) hipLaunchKernelGGL((bwd_prepare_kernel<__bf16>), grid, blk, 0, st, a, (int)wg_q, (int)wg_k);
        else hipLaunchKernelGGL((bwd_prepare_kernel<_Float16>), grid, blk, 0, st, a, (int)wg_q, (int)wg_k);
    } else if (dtype == BSA_BF16) {
        hipLaunchKernelGGL((bwd_rows_kernel<__bf16>), dim3((unsigned)((qrows + 15) / 16)), dim3(256), 0, st, (const __bf16*)o,
                           (const __bf16*)dout, lse, delta, m2, qrows);
        if (kept.keep) hipLaunchKernelGGL((bwd_scale_turned_kernel<__bf16>), dim3((unsigned)(krows / kTile)), dim3(256), 0, st, (const __bf16*)k, ks, c, tile_valid, (int)(Sk / kTile));
        else hipLaunchKernelGGL((bwd_scale_kernel<__bf16>), dim3((unsigned)((krows * 16 + 255) / 256)), dim3(256), 0, st,
                                (const __bf16*)k, (__bf16*)ks, c, krows * 16, tile_valid, (uint32_t)Sk);
    } else {
        hipLaunchKernelGGL((bwd_rows_kernel<_Float16>), dim3((unsigned)((qrows + 15) / 16)), dim3(256), 0, st, (const _Float16*)o,
                           (const _Float16*)dout, lse, delta, m2, qrows);
        if (kept.keep) hipLaunchKernelGGL((bwd_scale_turned_kernel<_Float16>), dim3((unsigned)(krows / kTile)), dim3(256), 0, st, (const _Float16*)k, ks, c, tile_valid, (int)(Sk / kTile));
        else hipLaunchKernelGGL((bwd_scale_kernel<_Float16>), dim3((unsigned)((krows * 16 + 255) / 256)), dim3(256), 0, st,
                                (const _Float16*)k, (_Float16*)ks, c, krows * 16, tile_valid, (uint32_t)Sk);
    }
    if (read_copies) {
        k_from = {ks, Hn * Sk * kD, Sk * kD, kD};
        rows_scale = 1.f;
    }
    if (thw == nullptr) hipLaunchKernelGGL(bwd_zero_kernel, dim3((unsigned)((nwords + 255) / 256)), dim3(256), 0, st, bits, nwords);
    const int64_t lrows = (int64_t)bh * nbq;
    // dQ walks every list in the forward kernel's visiting order when the list is ascending (a selection in block
    // order); any other order is walked as given.  The order only moves fp32 roundings of the dQ sum.
    if ((e = launch_pace_order(idx, paced, lens, lrows, nbk, idx_stride, st, {}, {bits, nbq, words})) != hipSuccess) return e;
    hipLaunchKernelGGL(bwd_count_kernel, dim3((unsigned)bh), dim3(nbk <= 256 ? 256 : kCountThreads), count_lds, st, bits, counts, kept.keep ? base : nullptr, order, words, nbk, nbq,
                       nsub, q_live, divisor(q_live.full));

    const dim3 block(64);
    const bool masked = tile_valid != nullptr;
    // dQ from scratch: rounds of as many wavefronts as the device runs at once (one per SIMD), two rounds per launch.  The dK / dV
    // kernel runs as one grid, longest list first: its lists (the query blocks of a KV block) differ in length, and
    // rounds that wait for the longest list cost more than they bring.
    const int round = 4 * cus;
    const DqSizes dq_sizes = {(int)(Sq / kTile), divisor((int)(Sq / kTile)), divisor(bs_q / kTile), divisor(bs_k / kTile), divisor(round)};
    const DkdvSizes sizes = {(int)(Sk / kTile), nbq, nsub, divisor((int)(Sk / kTile)), divisor(bs_k / kTile), divisor(round)};
    const int total_q = (int)(bh * (Sq / kTile)), total_k = (int)(bh * (Sk / kTile));
#define BSA_DKDV(T, M, K, G)                                                                                                           \
    hipLaunchKernelGGL((bwd_dkdv_kernel<T, M, K, G>), dim3((unsigned)total_k), dim3(128 * G), bwd_dkdv_lds_bytes(nbq, G), st, (const T*)q, (const T*)dout, k_from, v_from,  \
                       m2, delta, bits, tile_valid, (T*)dk, (T*)dv, Sq, Sk, words, rows_scale, sm_scale, read_copies ? 1 : 0, order, total_k, round,  \
                       dk_to, dv_to, ws + at.ds, ws + at.ds_spare, base, kept.pairs_per_head, sizes, q_live, k_live, counts)
#define BSA_DQ(T, M)                                                                                                                   \
    hipLaunchKernelGGL((bwd_dq_lds_kernel<T, M>), dim3(end - first), block, kDqRingLds, st, (const T*)q, (const T*)dout, (const T*)ks, (const T*)v,  \
                       m2, delta, paced, lens, tile_valid, (T*)dq, Sq, Sk, bs_q, bs_k, idx_stride, first, end, round, dq_to, dq_sizes, q_live.live, k_live)
#define BSA_DQ_DS(T, TEAM)                                                                                                             \
    hipLaunchKernelGGL((bwd_dq_from_ds_kernel<T, TEAM>), dim3(end - first), dim3(64 * TEAM), 0, st, ks, ws + at.ds, ws + at.ds_zeros, paced, place, lens,  \
                       (T*)dq, Sq, Sk, bs_q, bs_k, idx_stride, first, end, round, kept.pairs_per_head, dq_to, dq_sizes, q_live.live, k_live)
#define BSA_BY_TYPE(F, ...)                                     \
    do {                                                        \
        if (dtype == BSA_BF16) F(__bf16, ##__VA_ARGS__);        \
        else F(_Float16, ##__VA_ARGS__);                        \
    } while (0)
    // Two pairs of wavefronts to a key tile where there are no more tiles than compute units (a workgroup's stages then fill a unit's LDS) and its
    // list has blocks to share: us, one pair / two, 252 tiles of 2 heads of 28x8x34 136 / 107, 240 of 13x8x58 75 / 61, 180 of 3
    // heads of 11x17x16 71 / 53.
    const bool two_pairs = total_k <= cus && bwd_dkdv_lds_bytes(nbq, 2) <= kBwdLdsLimit && (int64_t)nbq * idx_stride >= 4 * (int64_t)nbk;
#define BSA_DKDV_OF(K)                                                     \
    do {                                                                   \
        if (masked && two_pairs) BSA_BY_TYPE(BSA_DKDV, true, K, 2);        \
        else if (two_pairs) BSA_BY_TYPE(BSA_DKDV, false, K, 2);            \
        else if (masked) BSA_BY_TYPE(BSA_DKDV, true, K, 1);                \
        else BSA_BY_TYPE(BSA_DKDV, false, K, 1);                           \
    } while (0)
    if (kept.keep) {
        hipLaunchKernelGGL(bwd_place_kernel, dim3((unsigned)((lrows + 3) / 4)), dim3(256), 0, st, paced, lens, bits, base, place, nbq, nbk, idx_stride,
                           words, nsub, lrows, q_live, reinterpret_cast<uint4*>(ws + at.ds_zeros));
        BSA_DKDV_OF(true);
    }
    // One launch for lists that the caller declares unequal, since rounds would wait for their longest list: the whole backward by
    // rounds / at once, us, smooth inputs, from kept dS 8 heads of 12x32x48 at threshold 0.75 (28 to 89 of 288 blocks) 1 027 / 982,
    // at 0.5 (28 to 42) 607 / 600, from scratch 8 heads of 24x30x52 at 0.5 (62 to 185 of 624) 3 438 / 2 848; random inputs (141
    // and 142 of 288) 2 329 / 2 378 and (307 to 309) 10 227 / 10 286.
    // From kept dS, whose stream is read once whatever the walks' pace, also up to half of the blocks (dQ alone, ms, density 1/16, 32
    // heads of 24x30x52: 1.81 by two rounds, 1.76 at once; 1/4, 24 heads of 12x30x52: 1.32 and 1.31; 1/2, 12 heads: 1.27 and 1.28);
    // equal lists of every block keep their rounds (8 heads of 12x32x48 4 655 / 4 793, of 4 heads 2 789 / 2 770).  From scratch a list
    // as wide as the blocks may be of any length, and where all are full it makes no difference (24 heads of 12x32x48 13 576 /
    // 13 463, 2 of 24x45x80 27 916 / 27 980).
    const bool once = unequal || (kept.keep ? 2 * idx_stride < nbk : idx_stride >= nbk);
    const int span = once ? total_q : 2 * round, list_tiles = idx_stride * nsub;
    // As many wavefronts to a list as SIMDs would be left without one, while each has tiles: us, one / four, 252 query tiles of 2
    // heads of 28x8x34 77 / 52, 240 of 13x8x58 30 / 23, 180 of 3 heads of 11x17x16 29 / 20.
    for (int first = 0; first < total_q; first += span) {
        const int end = first + span < total_q ? first + span : total_q;
        if (kept.keep && 4 * total_q <= round && list_tiles >= 8) BSA_BY_TYPE(BSA_DQ_DS, 4);
        else if (kept.keep && 2 * total_q <= round && list_tiles >= 2) BSA_BY_TYPE(BSA_DQ_DS, 2);
        else if (kept.keep) BSA_BY_TYPE(BSA_DQ_DS, 1);
        else if (masked) BSA_BY_TYPE(BSA_DQ, true);
        else BSA_BY_TYPE(BSA_DQ, false);
    }
    if (!kept.keep) {
        BSA_DKDV_OF(false);
    }
#undef BSA_DKDV_OF
#undef BSA_DKDV
#undef BSA_DQ
#undef BSA_DQ_DS
#undef BSA_BY_TYPE
    return hipGetLastError();
}

}  // namespace bsa
