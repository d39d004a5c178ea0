// What the fragment-order attention kernel needs besides the selection, in one launch (HBM-bound): k and v in fragment
// order (the layouts are described in bsa_fwd_frag.hip and bsa_fwd_few.hip), the chunk means of q and k, the row table of q, the validity
// words of the KV tiles, the largest key norm per tile; with a row transform also the per-head RMSNorm and the 3-D RoPE of
// q and k on their way through.
//
// A small call runs the three parts (workgroups 0 .. wg_k - 1 take chunks of k, the next wg_v tiles of v, the rest chunks of
// q) in one launch instead of six: its parts take a few microseconds each, and a launch in a stream of dependent ones
// costs 4.4.  There q goes the way of k, which needs half of the registers: with query_part's sixteen loads in flight per lane
// in it the launch had half of the wavefronts (two prompts of 8 heads, 7x15x26: 16.3 -> 13.4 us).  A large call runs one launch per
// part, each with the form and the registers that suit it (kOneLaunchGroups).
#include "bsa_mfma.h"
#include "bsa_rope.h"
#include "bsa_slots.h"

#include <type_traits>

namespace bsa {
namespace {

using namespace mfma;

template <int kCtrl>
__device__ __forceinline__ float dpp_f32(float x) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), kCtrl, 0xf, 0xf, true));
}

template <bool kBf16>
__device__ __forceinline__ void widen(uint32_t w, float& lo, float& hi) {
    if (kBf16) { lo = __uint_as_float(w << 16); hi = __uint_as_float(w & 0xffff0000u); }
    else { lo = (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xffffu)); hi = (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)); }
}
template <bool kBf16>
__device__ __forceinline__ uint16_t narrow(float x) {
    return kBf16 ? __builtin_bit_cast(uint16_t, (__bf16)x) : __builtin_bit_cast(uint16_t, (_Float16)x);
}
template <bool kBf16>
__device__ __forceinline__ void add_row(float (&acc)[8], const uint4& x) {
    const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float lo, hi;
        widen<kBf16>(w[e], lo, hi);
        acc[2 * e] += lo;
        acc[2 * e + 1] += hi;
    }
}

// what is derived from x is not worked out ahead of this place
__device__ __forceinline__ void opaque(uint4& x) { asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w)); }

// key_norm[batch * heads + head] = the largest entry of the head's tile norms
__global__ __launch_bounds__(256) void head_norm_kernel(const float* __restrict__ tile_norm, float* __restrict__ key_norm, int tiles) {
    __shared__ float part[4];
    float best = 0.f;
    for (int i = threadIdx.x; i < tiles; i += 256) {
        const float x = tile_norm[(int64_t)blockIdx.x * tiles + i];
        best = x != x ? INFINITY : fmaxf(best, x);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) best = fmaxf(best, __shfl_xor(best, off));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) key_norm[blockIdx.x] = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
}

// Where a slot of a tile goes: the real ones (bits of `word`) to the front, both groups in slot order.  The keys of a tile
// may come in any order, so a tile with n real keys costs the attention kernel ceil(n / 32) steps instead of two.
__device__ __forceinline__ int front_place(uint64_t word, int slot) {
    if (word == ~0ull) return slot;
    const int before = __popcll(word & (((uint64_t)1 << slot) - 1));
    return (word >> slot) & 1ull ? before : __popcll(word) + slot - before;
}

// The row table of one tile of q (row_table_ints): the real slots of a chunk to its front, and the numbers of the tiles that
// hold any.  before: real slots in the chunk's earlier tiles.
__device__ __forceinline__ void write_row_table(const Grid3& g, int32_t* rows, int blk, int sub, int lane, const Slots& s, int before) {
    const int nw = blk % g.Nw, nh = (blk / g.Nw) % g.Nh, nt = blk / (g.Nw * g.Nh);
    const int real = chunk_rows(g, nt, nh, nw);
    const int ahead = __popcll(s.word & (((uint64_t)1 << lane) - 1));
    const int place = (s.word >> lane) & 1ull ? before + ahead : real + (sub * kTile - before) + lane - ahead;
    rows[(int64_t)blk * g.chunk() + place] = s.token;
    if (lane == 0 && sub * kTile < real)
        rows[(int64_t)g.blocks() * g.chunk() + live_tiles_before(g, nt, nh, nw) + sub] = blk * (g.chunk() / kTile) + sub;
}

// the row of token t: before `split` from the cache, from there on from src
__device__ __forceinline__ const uint16_t* row_at(const uint16_t* src, int64_t sS, const uint16_t* old, int64_t cS, int split, int t) {
    if (old == nullptr) return src + (int64_t)t * sS;
    return t < split ? old + (int64_t)t * cS : src + (int64_t)(t - split) * sS;
}

// workgroup -> (tile or chunk, batch * head).  For a token-major source (the heads of a token next to each other, as a QKV
// projection leaves them) the heads of one chunk run side by side, so that the 256-byte rows they fetch share DRAM pages
// and cache lines' neighbourhoods; otherwise the chunks of one head do.
// `heads`: heads of a batch, or groups of them.
__device__ __forceinline__ void place(int id, int per_head, int heads, int head_fastest, int& chunk, int& bh) {
    if (head_fastest) {
        const int per_batch = per_head * heads, b = id / per_batch, rest = id - b * per_batch;
        chunk = rest / heads;
        bh = b * heads + (rest - chunk * heads);
    } else {
        bh = id / per_head;
        chunk = id - bh * per_head;
    }
}

constexpr int kPitchK = kD + 4;      // elements: 264-byte rows, read and written in 8-byte pieces (with rows of 272, whose pieces could be 16, the kernel has eight registers more, a wavefront a SIMD less, and a preview's launch takes 13.9 us for 13.2)
constexpr int kPitchV = kD + 16;     // 288-byte rows: the transposing reads fetch 4 keys x 16 d per 16 lanes, and with rows 72 banks apart the four keys fall on different banks

// kMode: rows as they are; with norm and rotation; and with a cache in front of k and v, or their rows written out.
enum { kPlain, kNorm, kCached };

// k (or q, when it has a row transform): a workgroup per chunk of x.heads heads, tile by tile.  The chunk mean keeps permute_kernel's order
// of summation - a thread adds its rows rg, rg + 16, ... of the chunk, then the 16 partial sums of a column are added in
// ascending rg, one rounding at the end - so every route gives the same bits.
template <bool kBf16, int kMode, bool kIsK>
__device__ __forceinline__ void row_part(const PrepRows& x, const Grid3& g, int Hn, int id, const float* tab, int tab_T, float eps,
                                         uint16_t* tile, float2* cs) {
    constexpr bool kTransform = kMode != kPlain, kCache = kMode == kCached;
    typedef typename std::conditional<kBf16, __bf16, _Float16>::type T;
    const int per_chunk = g.chunk() / kTile, tiles = g.blocks() * per_chunk;
    const int units = (Hn + x.heads - 1) / x.heads;               // groups of heads of a batch
    int blk, unit;
    place(id, g.blocks(), units, x.head_fastest, blk, unit);
    const int batch = unit / units, head0 = (unit - batch * units) * x.heads, heads = min(x.heads, Hn - head0);
    const int lane = threadIdx.x & 63;
    const int c16 = threadIdx.x & 15, rg = threadIdx.x >> 4;      // 16 pieces of 16 B per row, 16 rows at a time
    const uint16_t* src = x.p + (int64_t)batch * x.sB + (int64_t)head0 * x.sH + c16 * 8;
    const uint16_t* old = kCache && x.cached != nullptr ? x.cached + (int64_t)batch * x.cB + (int64_t)head0 * x.cH + c16 * 8 : nullptr;
    // The rows of the first tile are asked for before anything else, those of a later one as soon as the tile before it is in
    // LDS: the loads of a tile are under way while the workgroup writes out, meets and stages.
    Slots s;
    uint4 xs[4];
    int token[4], loc[4];
    auto locate = [&](int sub) {
        s = slots_of(g, blk, sub, lane);
        if (x.valid_in != nullptr) s.word = x.valid_in[blk * per_chunk + sub];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            token[i] = __shfl(s.token, rg + 16 * i);
            if (kTransform) loc[i] = __shfl(s.loc, rg + 16 * i);
        }
    };
    auto load = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            xs[i] = *reinterpret_cast<const uint4*>(kCache ? row_at(src, x.sS, old, x.cS, x.split, max(token[i], 0)) : src + (int64_t)max(token[i], 0) * x.sS);
    };
    locate(0);
    load();
    // Rotation: a chunk spans at most 8 positions per axis, and a rotation pair turns with one axis only, so the
    // (cos, sin) the rows of the chunk need are 8 x 64 table entries, fetched once per workgroup instead of per row and head.
    int turn[4];                          // where the position that turns this lane's pair jj stands in Slots::loc
    if (kTransform) {
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const int pr = c16 * 4 + jj;
            turn[jj] = pr < kRopePairsT ? 0 : pr < kRopePairsT + kRopePairsH ? 8 : 16;
        }
        const int nw = blk % g.Nw, nh = (blk / g.Nw) % g.Nh, nt = blk / (g.Nw * g.Nh);
        for (int e = threadIdx.x; e < 8 * 64; e += 256) {
            const int a = e >> 6, pr = e & 63;
            int at, dsin;
            if (pr < kRopePairsT) {
                at = min(x.t0 + nt * g.t + a, tab_T - 1) * kRopePairsT + pr;
                dsin = tab_T * kRopePairsT;
            } else if (pr < kRopePairsT + kRopePairsH) {
                at = 2 * tab_T * kRopePairsT + min(nh * g.h + a, g.H - 1) * kRopePairsH + pr - kRopePairsT;
                dsin = g.H * kRopePairsH;
            } else {
                at = 2 * tab_T * kRopePairsT + 2 * g.H * kRopePairsH + min(nw * g.w + a, g.W - 1) * kRopePairsW + pr - kRopePairsT - kRopePairsH;
                dsin = g.W * kRopePairsW;
            }
            cs[e] = make_float2(tab[at], tab[at + dsin]);
        }
        __syncthreads();
    }
    for (int hi = 0; hi < heads; ++hi) {
    const int head = head0 + hi, bh = batch * Hn + head;
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    int rows_before = 0;
    for (int sub = 0; sub < per_chunk; ++sub) {
        const int tile_id = blk * per_chunk + sub;
        // What follows from the thread's number is worked out in every turn: kept over all of them, the LDS addresses and bit
        // positions of four rows would cost a wavefront a SIMD.
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int rg = tid >> 4, c16 = tid & 15;
        if (s.word != ~0ull) {
#pragma unroll
            for (int i = 0; i < 4; ++i) keep_if(xs[i], (s.word >> (rg + 16 * i)) & 1ull);
        }
        if (bh == 0 && threadIdx.x < 64) {
            if (x.valid != nullptr && lane == 0) x.valid[tile_id] = s.word;
            if (x.rows != nullptr) {
                write_row_table(g, x.rows, blk, sub, lane, s, rows_before);
                rows_before += __popcll(s.word);
            }
        }
        if (kTransform) {
            const uint4 wraw = *reinterpret_cast<const uint4*>(x.norm_w + c16 * 8);
            uint16_t* rows = x.rows_out == nullptr ? nullptr : x.rows_out + (int64_t)batch * x.rB + (int64_t)head * x.rH + c16 * 8;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (token[i] < 0) continue;                         // the 16 lanes of a row go together
                opaque(xs[i]);
                float c[4], sn[4];
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const float2 a = cs[((loc[i] >> turn[jj]) & 255) * 64 + c16 * 4 + jj];
                    c[jj] = a.x;
                    sn[jj] = a.y;
                }
                if (!kCache) {
                    xs[i] = norm_rope_piece<T>(xs[i], wraw, true, true, c, sn, eps);
                    if (!kIsK) *reinterpret_cast<uint4*>(rows + (int64_t)token[i] * x.rS) = xs[i];
                } else {
                    const int at = old == nullptr ? token[i] : token[i] - x.split;       // of p; below 0: cached (the cache holds normalised rows)
                    if (at >= 0) {
                        xs[i] = norm_rope_piece<T>(xs[i], wraw, true, false, c, sn, eps);
                        if (rows != nullptr) *reinterpret_cast<uint4*>(rows + (int64_t)at * x.rS) = xs[i];
                    }
                    xs[i] = norm_rope_piece<T>(xs[i], wraw, false, true, c, sn, eps);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // Of k also the largest Euclidean norm of a row of this tile as it is stored (after the transform), a little above the
        // exact value: the attention kernel bounds q . k by |q| |k| with the largest of a head.  The sixteen lanes of
        // a row add their squares (butterfly over the row's lanes with DPP moves), then the maximum over the rows.
        // Piece by piece: widened all at once, the 32 values of a lane's rows cost a wavefront a SIMD.
        float best = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            opaque(xs[i]);
            const uint32_t w[4] = {xs[i].x, xs[i].y, xs[i].z, xs[i].w};
            float sq = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float lo, hi;
                widen<kBf16>(w[e], lo, hi);
                acc[2 * e] += lo;
                acc[2 * e + 1] += hi;
                if (kIsK) sq = fmaf(lo, lo, fmaf(hi, hi, sq));
            }
            if (kIsK) {
                sq += dpp_f32<0xB1>(sq);         // quad_perm [1, 0, 3, 2]
                sq += dpp_f32<0x4E>(sq);         // quad_perm [2, 3, 0, 1]
                sq += dpp_f32<0x141>(sq);        // row_half_mirror
                sq += dpp_f32<0x140>(sq);        // row_mirror
                best = fmaxf(best, sq);          // NaN squares drop out here; such a row has no bound (below)
                if (sq != sq) best = INFINITY;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(acc[e]));      // added here, not where the sums are used
            __builtin_amdgcn_sched_barrier(0);
        }
        if (kIsK && x.tile_norm != nullptr) {
#pragma unroll
            for (int off = 32; off >= 16; off >>= 1) best = fmaxf(best, __shfl_xor(best, off));
            __shared__ float wave_best[4];
            if (lane == 0) wave_best[threadIdx.x >> 6] = best;
            __syncthreads();
            if (threadIdx.x == 0) {
                best = fmaxf(fmaxf(wave_best[0], wave_best[1]), fmaxf(wave_best[2], wave_best[3]));
                x.tile_norm[(int64_t)bh * tiles + tile_id] = __builtin_sqrtf(best) * 1.001f;
            }
        }
        if (x.frag != nullptr) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint16_t* row = tile + front_place(s.word, rg + 16 * i) * kPitchK + c16 * 8;
                *reinterpret_cast<uint2*>(row) = make_uint2(xs[i].x, xs[i].y);
                *reinterpret_cast<uint2*>(row + 4) = make_uint2(xs[i].z, xs[i].w);
            }
        }
        if (sub + 1 < per_chunk || hi + 1 < heads) {
            if (sub + 1 == per_chunk) {
                src += x.sH;
                if (kCache && old != nullptr) old += x.cH;
            }
            if (per_chunk > 1) locate(sub + 1 < per_chunk ? sub + 1 : 0);
            load();
        }
        if (x.frag != nullptr) {
            __syncthreads();
            char* out = x.frag + ((int64_t)bh * tiles + tile_id) * kTileBytes;
            // 16-byte piece tid + 256 i of the output: lane l of fragment w + 4 i, which is key half i / 2 and, of 16 keys x 32 d, d chunk
            // w / 2 + 2 (i % 2), its keys w % 2; of 32 keys x 16 d (few) d chunk w + 4 (i % 2)
            const int l = tid & 63, w = tid >> 6;
            const uint16_t* p = tile + (x.few ? (l & 31) * kPitchK + 16 * w + 8 * (l >> 5) : (16 * (w & 1) + (l & 15)) * kPitchK + 32 * (w >> 1) + 8 * (l >> 4));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint16_t* at = p + 32 * (i >> 1) * kPitchK + 64 * (i & 1);
                const uint2 lo = *reinterpret_cast<const uint2*>(at), hi = *reinterpret_cast<const uint2*>(at + 4);
                *reinterpret_cast<uint4*>(out + (int64_t)(tid + 256 * i) * 16) = make_uint4(lo.x, lo.y, hi.x, hi.y);
            }
            __syncthreads();                      // the next tile, or the sums below, may have the memory
        }
    }
    if (x.pooled != nullptr) {
        float* red = reinterpret_cast<float*>(tile);
#pragma unroll
        for (int e = 0; e < 8; ++e) red[rg * kD + c16 * 8 + e] = acc[e];
        __syncthreads();
        if (threadIdx.x < kD) {
            float sum = 0.f;
            for (int i = 0; i < 16; ++i) sum += red[i * kD + threadIdx.x];
            const int64_t at = x.pooled_operand ? operand_mean_at(bh, g.blocks(), blk, threadIdx.x) : ((int64_t)bh * g.blocks() + blk) * kD + threadIdx.x;
            x.pooled[at] = narrow<kBf16>(sum * (1.0f / g.chunk()));
        }
        __syncthreads();                          // the next head may have the memory
    }
    }   // heads
}

// v: a workgroup per tile, gathered into LDS and read transposed: a piece holds 8 keys of one d
template <bool kCache>
__device__ __forceinline__ void value_part(const PrepRows& x, const Grid3& g, int Hn, int id, uint16_t* tile) {
    const int per_chunk = g.chunk() / kTile, tiles = g.blocks() * per_chunk;
    int tile_id, bh;
    place(id, tiles, Hn, x.head_fastest, tile_id, bh);
    const int lane = threadIdx.x & 63;
    const int c16 = threadIdx.x & 15, rg = threadIdx.x >> 4;
    const uint16_t* src = x.p + (int64_t)(bh / Hn) * x.sB + (int64_t)(bh % Hn) * x.sH + c16 * 8;
    const uint16_t* old = kCache && x.cached != nullptr ? x.cached + (int64_t)(bh / Hn) * x.cB + (int64_t)(bh % Hn) * x.cH + c16 * 8 : nullptr;
    Slots s = slots_of(g, tile_id / per_chunk, tile_id % per_chunk, lane);
    if (x.valid_in != nullptr) s.word = x.valid_in[tile_id];
    uint4 xs[4];
    int token[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        token[i] = __shfl(s.token, rg + 16 * i);
        xs[i] = *reinterpret_cast<const uint4*>(kCache ? row_at(src, x.sS, old, x.cS, x.split, max(token[i], 0)) : src + (int64_t)max(token[i], 0) * x.sS);
    }
    if (s.word != ~0ull) {
#pragma unroll
        for (int i = 0; i < 4; ++i) keep_if(xs[i], (s.word >> (rg + 16 * i)) & 1ull);
    }
    if (kCache && x.rows_out != nullptr) {
        uint16_t* rows = x.rows_out + (int64_t)(bh / Hn) * x.rB + (int64_t)(bh % Hn) * x.rH + c16 * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int at = old == nullptr ? token[i] : token[i] - x.split;
            if (at >= 0) *reinterpret_cast<uint4*>(rows + (int64_t)at * x.rS) = xs[i];
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint4*>(tile + front_place(s.word, rg + 16 * i) * kPitchV + c16 * 8) = xs[i];
    __syncthreads();
    char* out = x.frag + ((int64_t)bh * tiles + tile_id) * kTileBytes;
    // ds_read_b64_tr_b16: the 16 lanes of a group point at a 4-key x 16-d patch (lane s at key s / 4,
    // d 4 (s % 4) .. + 4) and each receives the 4 keys of one d.  Piece threadIdx.x + 256 i: lane l of fragment w + 4 i, key half i / 2,
    // d tile w + 4 (i % 2) of 16, or (few) key step i % 2, d tile w of 32
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    auto write = [&](const uint16_t* from, auto odd, auto upper) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint16_t* at = from + 32 * (i >> 1) * kPitchV + (i & 1) * odd;
            const s16x4 lo = lds_read_tr16(at), hi = lds_read_tr16(at + upper);
            typedef short s16x8_ __attribute__((ext_vector_type(8)));
            *reinterpret_cast<s16x8_*>(out + (int64_t)(threadIdx.x + 256 * i) * 16) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    const int key = (l & 15) >> 2, d = 4 * (l & 3);
    if (x.few) write(tile + (4 * (l >> 5) + key) * kPitchV + 32 * w + 16 * (l >> 4 & 1) + d, std::integral_constant<int, 16 * kPitchV>{}, std::integral_constant<int, 8 * kPitchV>{});
    else write(tile + (4 * (l >> 4) + key) * kPitchV + 16 * w + d, std::integral_constant<int, 64>{}, std::integral_constant<int, 16 * kPitchV>{});
}

// Chunk means and row table of q, nothing else of it: a wavefront per chunk, no LDS, all of a lane's sixteen 16-byte loads
// of a tile in flight at once.  Lane = (c16, r4): 16-byte piece c16 of the rows rg = 4 r4 .. 4 r4 + 3 and their likes 16, 32,
// 48, ... slots on, summed in permute_kernel's order.
template <bool kBf16>
__device__ __forceinline__ void query_part(const PrepRows& x, const Grid3& g, int Hn, int64_t id, int64_t total) {
    if (id >= total) return;
    int blk, bh;
    place((int)id, g.blocks(), Hn, x.head_fastest, blk, bh);
    const int lane = threadIdx.x & 63, c16 = lane & 15, r4 = lane >> 4;
    const char* src = reinterpret_cast<const char*>(x.p + (int64_t)(bh / Hn) * x.sB + (int64_t)(bh % Hn) * x.sH);
    const int per_chunk = g.chunk() / kTile;
    float part[4][8];                       // this lane's rows rg = 4 r4 + u
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) part[u][e] = 0.f;
    int rows_before = 0;
    for (int sub = 0; sub < per_chunk; ++sub) {
        const Slots s = slots_of(g, blk, sub, lane);
        if (bh == 0 && x.rows != nullptr) {
            write_row_table(g, x.rows, blk, sub, lane, s, rows_before);
            rows_before += __popcll(s.word);
        }
        // every row unconditionally (a padded slot reads token 0 and is cleared afterwards): sixteen independent loads
        // per lane, no branch between them
        uint4 xs[4][4];
        const int slot0 = 4 * r4;
        if (x.offsets_32) {                 // one register per address instead of two
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t at = (uint32_t)max(__shfl(s.token, slot0 + u + 16 * i), 0) * (uint32_t)(x.sS * 2) + (uint32_t)c16 * 16u;
                    xs[u][i] = *reinterpret_cast<const uint4*>(src + at);
                }
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    xs[u][i] = *reinterpret_cast<const uint4*>(src + (int64_t)max(__shfl(s.token, slot0 + u + 16 * i), 0) * (x.sS * 2) + c16 * 16);
        }
        if (s.word != ~0ull) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) keep_if(xs[u][i], (s.word >> (slot0 + u + 16 * i)) & 1ull);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) add_row<kBf16>(part[u], xs[u][i]);
    }
    // the sixteen partial sums of a column in ascending rg: four per lane, handed from r4 to r4 + 1
    float sum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sum[e] = 0.f;
#pragma unroll
    for (int stage = 0; stage < 4; ++stage) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float below = stage == 0 ? 0.f : __shfl_up(sum[e], 16);
            if (r4 == stage) sum[e] = (((below + part[0][e]) + part[1][e]) + part[2][e]) + part[3][e];
        }
    }
    if (r4 == 3) {
        const float inv = 1.0f / g.chunk();
        uint32_t out[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = narrow<kBf16>(sum[2 * e] * inv) | ((uint32_t)narrow<kBf16>(sum[2 * e + 1] * inv) << 16);
        *reinterpret_cast<uint4*>(x.pooled + ((int64_t)bh * g.blocks() + blk) * kD + c16 * 8) = make_uint4(out[0], out[1], out[2], out[3]);
    }
}

// Workgroups (counted as the separate launches have them) up to which the three parts go in one launch.  The whole operator, one
// launch against three, us: rows as they are, 4x4x4 chunks, 8 heads of 24x30x52 (11 232 groups) 471 / 482, 4 heads of 24x45x80
// (12 960) 1 106 / 1 120, 16 heads of 24x30x52 (22 464) 933 / 931, 32 (44 928) 1 845 / 1 825; 16 heads of 13x30x53 in 4x4x8
// (11 648) 751 / 765; a block with norm, rotation and a cache, 16 + 5 frames of 30x52, 6 heads (9 984) 504 / 519, 12 (19 968) 986 /
// 1 005.
constexpr int64_t kOneLaunchGroups = 20480;

// Heads of a chunk that a workgroup with a row transform takes, one after another: where the rows lie and the rotation angles are
// the same for all of them, and a head's rows are on their way while the one before it is transformed and written.  By heads to a
// workgroup (32 heads of 24x45x80, k / q, us): 1 445 / 392 (a workgroup's loads behind its look-up of the angles), then with
// the loads in front and by 2 404 / 337, 4 362 / 307, 8 352 / 295, 16 354 / 297; with fewer registers (row_part) 8 317 / 275 = 4.6 and
// 5.1 TB/s.  Rows as they are gain nothing (229 by one head, 253 by four).  Calls of fewer chunks than kGroupedChunks keep the
// workgroups instead; the whole operator at that line, sparsity 0.985, us by one head / by eight, which also brings more calls into
// one launch: 4 160 chunks of k 181 / 174, 6 656 267 / 252, 8 320 422 / 394, 9 984 492 / 453, 13 312 642 / 605, 19 968 1 128 / 1 089; behind four
// cached frames 4 160 136 / 136, 6 656 270 / 260, 8 320 360 / 320, 13 312 555 / 513.
// The launch of k is held to the registers of five wavefronts a SIMD, but not the form with a cache, which would spill three: held /
// as it is, this launch takes 179 / 169 us for 32 heads of 24x30x52 behind 4 cached frames, 140 / 142 for 16 behind 5, where five
// wavefronts fit the call's workgroups into two whole rounds; the whole call 1 094 / 1 086 and 720 / 720, of 24x45x80 3 992 / 3 974.
constexpr int kHeadsPerGroup = 8;
constexpr int64_t kGroupedChunks = 8192;

enum { kAllParts, kKeys, kValues, kQueries };
template <bool kBf16, int kMode, int kPart>
__global__ __launch_bounds__(256, kPart == kKeys && kMode == kNorm ? 5 : 1) void prepare_kernel(PrepArgs a, int wg_k, int wg_v, int64_t chunks_q) {
    constexpr bool kTransform = kMode != kPlain;
    __shared__ __attribute__((aligned(16))) uint16_t tile[kPart == kQueries && !kTransform ? 8 : kTile * kPitchV];
    __shared__ float2 cs[kTransform && kPart != kValues ? 8 * 64 : 1];
    const int w = blockIdx.x;
    if (kPart <= kKeys && w == 0 && threadIdx.x == 0 && a.zero != nullptr) *a.zero = 0u;
    if (kPart == kKeys || (kPart == kAllParts && w < wg_k)) {
        row_part<kBf16, kMode, true>(a.k, a.gk, a.Hn, w, a.tab, a.tab_T, a.eps, tile, cs);
        return;
    }
    if (kPart == kValues || (kPart == kAllParts && w < wg_k + wg_v)) {
        value_part<kMode == kCached>(a.v, a.gk, a.Hn, kPart == kValues ? w : w - wg_k, tile);
        return;
    }
    const int wq = kPart == kQueries ? w : w - wg_k - wg_v;
    if (kTransform || kPart == kAllParts) row_part<kBf16, kTransform ? kNorm : kPlain, false>(a.q, a.gq, a.Hn, wq, a.tab, a.tab_T, a.eps, tile, cs);
    else query_part<kBf16>(a.q, a.gq, a.Hn, (int64_t)wq * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), chunks_q);
}

// the row table of q alone (the selection is the caller's): one workgroup per four tiles
__global__ __launch_bounds__(256) void row_table_kernel(Grid3 g, int32_t* __restrict__ rows, int tiles) {
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, per_chunk = g.chunk() / kTile;
    if (tile >= tiles) return;
    const int blk = tile / per_chunk, mine = tile % per_chunk;
    int before = 0;
    for (int sub = 0; sub < mine; ++sub) before += __popcll(slots_of(g, blk, sub, lane).word);
    write_row_table(g, rows, blk, mine, lane, slots_of(g, blk, mine, lane), before);
}

}  // namespace

hipError_t launch_prepare(const PrepArgs& args, int B, int dtype, hipStream_t st) {
    PrepArgs a = args;
    for (PrepRows* x : {&a.q, &a.k, &a.v}) x->head_fastest = x->sH < x->sS ? 1 : 0;
    a.q.offsets_32 = ((int64_t)a.gq.T * a.gq.H * a.gq.W + 1) * a.q.sS * 2 < ((int64_t)1 << 32) ? 1 : 0;
    const int64_t bh = (int64_t)B * a.Hn;
    const bool transform = a.tab != nullptr;                    // norm and rotation come together, q's rows are always wanted
    if (transform && (a.q.norm_w == nullptr || a.k.norm_w == nullptr || a.q.rows_out == nullptr)) return hipErrorInvalidValue;
    const bool cached = a.k.cached != nullptr || a.k.rows_out != nullptr || a.v.rows_out != nullptr;      // comes with a transform
    for (PrepRows* x : {&a.q, &a.k}) {
        const bool many = transform && bh * (x == &a.q ? a.gq : a.gk).blocks() >= kGroupedChunks;
        const int units = many ? (a.Hn + kHeadsPerGroup - 1) / kHeadsPerGroup : a.Hn;      // evenly: 9 heads are 5 and 4
        x->heads = (a.Hn + units - 1) / units;
    }
    auto groups = [&](const PrepRows& x, const Grid3& g) { return (int64_t)B * ((a.Hn + x.heads - 1) / x.heads) * g.blocks(); };
    const int64_t wg_k = a.k.p != nullptr ? groups(a.k, a.gk) : 0;
    const int64_t wg_v = a.v.p != nullptr ? bh * a.gk.blocks() * (a.gk.chunk() / kTile) : 0;
    const int64_t chunks_q = a.q.p != nullptr ? bh * a.gq.blocks() : 0;
    const int64_t wg_q = transform ? (a.q.p != nullptr ? groups(a.q, a.gq) : 0) : (chunks_q + 3) / 4;
    const int64_t total = wg_k + wg_v + wg_q;
    if (total <= 0 || total > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 block(256);
#define BSA_PREPARE(PART, N)                                                                                                        \
    do {                                                                                                                            \
        const dim3 grid((unsigned)(N));                                                                                             \
        if (dtype == BSA_BF16) {                                                                                                    \
            if (cached) hipLaunchKernelGGL((prepare_kernel<true, kCached, PART>), grid, block, 0, st, a, (int)wg_k, (int)wg_v, chunks_q);         \
            else if (transform) hipLaunchKernelGGL((prepare_kernel<true, kNorm, PART>), grid, block, 0, st, a, (int)wg_k, (int)wg_v, chunks_q);   \
            else hipLaunchKernelGGL((prepare_kernel<true, kPlain, PART>), grid, block, 0, st, a, (int)wg_k, (int)wg_v, chunks_q);   \
        } else {                                                                                                                    \
            if (cached) hipLaunchKernelGGL((prepare_kernel<false, kCached, PART>), grid, block, 0, st, a, (int)wg_k, (int)wg_v, chunks_q);        \
            else if (transform) hipLaunchKernelGGL((prepare_kernel<false, kNorm, PART>), grid, block, 0, st, a, (int)wg_k, (int)wg_v, chunks_q);  \
            else hipLaunchKernelGGL((prepare_kernel<false, kPlain, PART>), grid, block, 0, st, a, (int)wg_k, (int)wg_v, chunks_q);  \
        }                                                                                                                           \
    } while (0)
    if (total <= kOneLaunchGroups) {      // a workgroup per chunk of q here as well
        BSA_PREPARE(kAllParts, wg_k + wg_v + (transform ? wg_q : chunks_q));
    } else {
        if (wg_q > 0) BSA_PREPARE(kQueries, wg_q);
        if (wg_k > 0) BSA_PREPARE(kKeys, wg_k);
        if (wg_v > 0) BSA_PREPARE(kValues, wg_v);
    }
#undef BSA_PREPARE
    return hipGetLastError();
}

hipError_t launch_row_table(const Grid3& g, int32_t* rows, hipStream_t st) {
    const int tiles = g.blocks() * (g.chunk() / kTile);
    hipLaunchKernelGGL(row_table_kernel, dim3((tiles + 3) / 4), dim3(256), 0, st, g, rows, tiles);
    return hipGetLastError();
}

hipError_t launch_head_norm(const float* tile_norm, float* key_norm, int BH, int tiles, hipStream_t st) {
    hipLaunchKernelGGL(head_norm_kernel, dim3((unsigned)BH), dim3(256), 0, st, tile_norm, key_norm, tiles);
    return hipGetLastError();
}

// floats of the key norms: one per (batch, head), then (from a 256-byte boundary) one per tile
size_t key_norm_floats(int B, int Hn, int64_t tiles) { return tile_norm_offset(B, Hn) + (size_t)B * Hn * (size_t)tiles; }

}  // namespace bsa
