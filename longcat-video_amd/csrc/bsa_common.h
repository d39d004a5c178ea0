// Shared declarations of the gfx950 block-sparse attention engine.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>
#include "bsa_mi355x.h"

namespace bsa {

// Geometry of a (T,H,W) token grid cut into (t,h,w) chunks, padded high.
struct Grid3 {
    int T, H, W;      // real grid
    int t, h, w;      // chunk shape
    int Nt, Nh, Nw;   // chunks per axis (ceil)
    __host__ __device__ int chunk() const { return t * h * w; }
    __host__ __device__ int blocks() const { return Nt * Nh * Nw; }
};

inline Grid3 make_grid(int T, int H, int W, int t, int h, int w) {
    Grid3 g;
    g.T = T; g.H = H; g.W = W; g.t = t; g.h = h; g.w = w;
    g.Nt = (T + t - 1) / t; g.Nh = (H + h - 1) / h; g.Nw = (W + w - 1) / w;
    return g;
}

// A chunk's real rows come first in the row table of q, so that its 64-slot tiles behind the first ceil(rows / 64) hold none
// and drop out of the attention kernel's work.  Real rows of chunk (nt, nh, nw):
__host__ __device__ inline int chunk_rows(const Grid3& g, int nt, int nh, int nw) {
    auto extent = [](int n, int N, int size, int all) { return n < N - 1 ? size : all - (N - 1) * size; };
    return extent(nt, g.Nt, g.t, g.T) * extent(nh, g.Nh, g.h, g.H) * extent(nw, g.Nw, g.w, g.W);
}
// Tiles with real rows in the chunks in front of (nt, nh, nw); all of them for (Nt, 0, 0).  Chunks differ only in whether they
// are the last of an axis: 8 kinds.
__host__ __device__ inline int live_tiles_before(const Grid3& g, int nt, int nh, int nw) {
    auto chunk = [&](int t, int h, int w) { return (chunk_rows(g, t, h, w) + 63) / 64; };
    auto row = [&](int t, int h) { return (g.Nw - 1) * chunk(t, h, 0) + chunk(t, h, g.Nw - 1); };
    auto plane = [&](int t) { return (g.Nh - 1) * row(t, 0) + row(t, g.Nh - 1); };
    if (nt >= g.Nt) return (g.Nt - 1) * plane(0) + plane(g.Nt - 1);
    return nt * plane(0) + nh * row(nt, 0) + nw * chunk(nt, nh, 0);      // (.., 0) stands for every one but the last
}
__host__ __device__ inline int live_query_tiles(const Grid3& g) { return live_tiles_before(g, g.Nt, 0, 0); }
// int32 entries of the row table of q for `slots` padded slots: token row of every slot (-1: padding), then the numbers of the
// tiles that hold real rows, ascending.
inline size_t row_table_ints(int64_t slots) { return (size_t)(slots + slots / 64); }

// n / d for 0 <= n < 2^31 by a product: m = ceil(2^p / d) with p = 31 + ceil(log2 d), so m d - 2^p < d <= 2^(p - 31) and the error
// n (m d - 2^p) / (d 2^p) of the quotient stays below 1 / d.  A division by a number that the compiler does not know costs
// 25 (32 bits) to 120 instructions (64), one after another.
struct Divisor {
    uint32_t m, p;
};
inline Divisor divisor(int d) {
    uint32_t l = 0;
    while (((int64_t)1 << l) < d) ++l;
    const uint32_t p = 31 + l;
    return {(uint32_t)((((unsigned __int128)1 << p) + d - 1) / d), p};
}
__device__ __forceinline__ int operator/(int n, const Divisor& d) { return (int)(((uint64_t)(uint32_t)n * d.m) >> d.p); }

// Over a wavefront whose lanes all take part, by DPP moves: a few clocks a step, where a __shfl is a round trip to LDS.  Lanes that
// a move leaves without a source add 0.
__device__ __forceinline__ int wave_scan(int x) {                // the sum over lanes 0 .. lane
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);      // row_shr:1, 2, 4, 8: inside rows of 16 lanes
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);      // row_bcast:15 into rows 1 and 3, row_bcast:31 into 2 and 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    return x;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t x) {       // the same in every lane, a scalar
    auto step = [&](uint32_t y) { x = x > y ? x : y; };
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false));
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

// The bytes of a kernel's arguments, laid out one after another, each at its alignment.
template <typename Kernel>
struct ArgumentBytes;
template <typename... A>
struct ArgumentBytes<void(A...)> {
    static constexpr int count() {
        size_t at = 0;
        ((at = (at + alignof(A) - 1) / alignof(A) * alignof(A) + sizeof(A)), ...);
        return (int)((at + 3) / 4 * 4);
    }
};

// The compiler loads a kernel's arguments where it first needs them, a wait for memory for every cache line of them in front of
// the first useful load of a launch.  Asked for together they cost one.  Kernel: the type of the kernel, of 384 bytes at most.
template <typename Kernel>
__device__ __forceinline__ void touch_arguments() {
    constexpr int kBytes = ArgumentBytes<Kernel>::count();
    static_assert(kBytes >= 4 && kBytes <= 384, "six cache lines are asked for");
    uint32_t a, b, c, d, e, f;
    constexpr int last = kBytes - 4;
    asm volatile("s_load_dword %0, %6, %7\n\ts_load_dword %1, %6, %8\n\ts_load_dword %2, %6, %9\n\ts_load_dword %3, %6, %10\n\t"
                 "s_load_dword %4, %6, %11\n\ts_load_dword %5, %6, %12\n\ts_waitcnt lgkmcnt(0)"
                 : "=&s"(a), "=&s"(b), "=&s"(c), "=&s"(d), "=&s"(e), "=&s"(f)
                 : "s"(__builtin_amdgcn_kernarg_segment_ptr()), "i"(0), "i"(64 < last ? 64 : last), "i"(128 < last ? 128 : last),
                   "i"(192 < last ? 192 : last), "i"(256 < last ? 256 : last), "i"(last));
}

// Where the rows of the attention operands live.  Blocked order: tile i of a (batch, head) is rows
// 64*i .. 64*i+63 of a contiguous [B, Hn, S, D] tensor.  THW order: tile i is (a 64-slot part of)
// chunk i of the grid and its slots are gathered from / scattered to token positions, so the
// separate permute and unpermute passes over that tensor disappear.  Strides are in elements:
// batch, head, token.
struct FwdLayout {
    // token row of every blocked-order query slot, -1 for padding ([Sq]); null: q and o are in
    // blocked order themselves
    const int32_t* q_rows;
    // per 64-slot kv tile: token row of its first slot (< 2^24) when the tile is read where it
    // lies, or 2^24 + index of the tile in the edge copies ([Sk / 64]); null: k and v are in
    // blocked order themselves
    const uint32_t* k_tiles;
    int64_t q_st[3], o_st[3], k_st[3], v_st[3];   // k_st[2] == v_st[2]
    // blocked-order, zero-padded copies of the chunks that touch the padded high edge of the kv
    // grid, [B*Hn][edge_count][chunk][D]; every other chunk is read where it lies
    const void* k_edge;
    const void* v_edge;
    int kw, kh, kH, kW;        // kv tile geometry: runs of kw slots, kh runs per plane, grid H and W
};

// Chunks with padded slots ("edge chunks") are numbered densely: first the whole last t layer if
// T is ragged, then the last h row of the remaining layers if H is ragged, then the last w column
// of what is left if W is ragged.  Returns -1 for a chunk without padding.
__host__ __device__ inline int edge_index(const Grid3& g, int blk) {
    const int nw = blk % g.Nw, nh = (blk / g.Nw) % g.Nh, nt = blk / (g.Nw * g.Nh);
    const bool rt = g.T % g.t != 0, rh = g.H % g.h != 0, rw = g.W % g.w != 0;
    const int Nt1 = g.Nt - (rt ? 1 : 0), Nh1 = g.Nh - (rh ? 1 : 0);
    int base = 0;
    if (rt) {
        if (nt == g.Nt - 1) return nh * g.Nw + nw;
        base += g.Nh * g.Nw;
    }
    if (rh) {
        if (nh == g.Nh - 1) return base + nt * g.Nw + nw;
        base += Nt1 * g.Nw;
    }
    if (rw && nw == g.Nw - 1) return base + nt * Nh1 + nh;
    return -1;
}
inline int edge_count(const Grid3& g) {
    const bool rt = g.T % g.t != 0, rh = g.H % g.h != 0, rw = g.W % g.w != 0;
    const int Nt1 = g.Nt - (rt ? 1 : 0), Nh1 = g.Nh - (rh ? 1 : 0);
    return (rt ? g.Nh * g.Nw : 0) + (rh ? Nt1 * g.Nw : 0) + (rw ? Nt1 * Nh1 : 0);
}

// k and v tiles can be gathered from THW order when a 64-slot tile is a whole number of (h, w)
// planes of its chunk, built from runs of at least 4 tokens along w, and when all offsets inside
// a tile fit 32 bits.
inline bool kv_direct_ok(const Grid3& g, int64_t token_stride_bytes) {
    auto pow2 = [](int x) { return x > 0 && (x & (x - 1)) == 0; };
    if (!pow2(g.w) || !pow2(g.h) || g.w < 4 || g.w > 64) return false;
    if ((64 / g.w) % g.h != 0) return false;
    if ((int64_t)g.T * g.H * g.W >= (1 << 24)) return false;
    const int64_t planes = 64 / (g.w * g.h);
    return token_stride_bytes > 0 && planes * g.H * g.W * token_stride_bytes < ((int64_t)1 << 32);
}

inline int dtype_size(int dtype) {
    switch (dtype) {
        case BSA_BF16: case BSA_F16: return 2;
        case BSA_F32: return 4;
        default: return 0;
    }
}

// Records the message returned by bsa_last_error() and passes `code` through.
int set_error(int code, const char* fmt, ...);
bool gemm_serves_linear(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* residual, const void* out, int64_t ldo,
                        int64_t M, int N, int K);      // bsa_gemm.hip

// Kernel launchers (one per source file); all validate nothing and assume the
// C-ABI layer has checked shapes.  Each returns a hipError_t from the launch.
// edge_only: dst is [B*Hn][edge_count(g)][chunk][D] and only chunks with padded slots are copied
// row_table ([S_padded] int32): token row of every blocked-order slot, -1 for padding.
// tile_table ([S_padded/64] uint32): FwdLayout::k_tiles.  Both optional.
// src2 / dst2 (edge_only): a second tensor on the same grid whose edge chunks are copied as well.
hipError_t launch_permute(const void* src, const int64_t strides[3], void* dst, void* pooled,
                          uint64_t* tile_valid, int B, int Hn, const Grid3& g, int D, int dtype,
                          hipStream_t st, bool edge_only = false, int32_t* row_table = nullptr,
                          uint32_t* tile_table = nullptr, const void* src2 = nullptr,
                          const int64_t* strides2 = nullptr, void* dst2 = nullptr);
hipError_t launch_unpermute(const void* src, void* dst, const int64_t strides[3], int B, int Hn,
                            const Grid3& g, int D, int dtype, hipStream_t st);
hipError_t launch_mean_pool(const void* x, void* out, int B, int Hn, int64_t S, int block, int D,
                            int dtype, hipStream_t st);
// The kernels that score can also take the largest key norm of every (batch, head) from those of its tiles on the way
struct HeadNorms {
    const float* tile_norm;      // [BH][tiles]; null: not wanted
    float* key_norm;             // [BH]
    int tiles;
};
hipError_t launch_score(const void* q_cmp, const void* k_cmp, void* score, int BH, int nbq, int nbk,
                        int D, int dtype, hipStream_t st, HeadNorms norms = {nullptr, nullptr, 0});
// idx: descending score order; idx_sorted: ascending block index; either may be null
// k_rows: one count per row instead of k_sel (may alias lens); stride: row pitch of idx / idx_sorted
// (default k_sel), entries past a row's count are set to -1
hipError_t launch_topk(const void* score, int32_t* idx, int32_t* idx_sorted, int32_t* lens, int64_t rows,
                       int nbk, int k_sel, int dtype, hipStream_t st, const int32_t* k_rows = nullptr,
                       int stride = 0);
// Lists of 32-key halves for the attention kernel's walk over a padded grid (launch_fwd_frag, halves), written next to the
// visiting order: rows of `stride` entries (even, at least twice the tiles of a list), lens = entries in use.
struct HalfLists {
    const uint64_t* valid;       // validity words of the KV tiles
    int nsub;                    // tiles per KV block
    int32_t* lists;              // null: not wanted
    int32_t* lens;
    int stride;
};
// Scores, top-k and (with `paced`) visiting order of a small call in one launch: lists [BH][nbq][k_sel], ascending or in
// visiting order, lens = k_sel.  The same lists as launch_score, launch_topk and launch_pace_order; gate_fits says for
// which sizes it is built and the better choice.
bool gate_fits(int BH, int nbq, int nbk, int k_sel, int dtype);
// A selection that launch_fwd_frag and launch_fwd_f32 let the attention kernel make, or has made in front of it by make(ctx).
struct GateCall {
    const void *q_cmp, *k_cmp;       // chunk means
    int32_t *lists, *lens;           // where the lists go ([BH][nbq][width]), null: they are not read behind the attention
    const uint64_t* valid;           // validity words of the key tiles
    int nbk, width;                  // width: the top-k rule's count, the most of the CDF rule's
    float threshold, scale;          // CDF rule (launch_cdf_count), threshold 0: top-k
    int k_min;
    bool inside;                     // launch_fwd_frag: the attention kernel makes it (frag_selects)
    hipError_t (*make)(void* ctx);
    void* ctx;
};
hipError_t launch_gate(const void* q_cmp, const void* k_cmp, int32_t* lists, int32_t* lens, int BH, int nbq, int nbk, int k_sel,
                       bool paced, int dtype, hipStream_t st, HeadNorms norms = {nullptr, nullptr, 0}, HalfLists halves = {});
// lens[row] = number of columns the CDF rule keeps, clamped to [k_min, cap]
hipError_t launch_cdf_count(const void* score, int32_t* lens, int64_t rows, int nbk, float threshold,
                            float scale, int k_min, int cap, int dtype, hipStream_t st);
hipError_t launch_fwd(const void* q, const void* k, const void* v, const int32_t* idx,
                      const int32_t* lens, const uint64_t* tile_valid, void* o, float* lse,
                      int B, int Hn, int64_t Sq, int64_t Sk, int bs_q, int bs_k, int idx_stride,
                      float sm_scale, int dtype, hipStream_t st, const FwdLayout* layout = nullptr,
                      int64_t layout_lse_rows = 0, int64_t layout_edge_bytes = 0, const int32_t* order = nullptr,
                      uint32_t* queue = nullptr);
// fp32 (bsa_f32.hip).  Chunk means and row tables (token of every blocked-order slot of one (batch, head), -1 = padding) of
// q and k in one launch, and the attention kernel; layout null: q, k, v, o in blocked order.
struct F32Layout {
    const int32_t *q_rows, *k_rows;
    int64_t q_st[3], k_st[3], v_st[3], o_st[3];      // element strides {batch, head, token}
    int64_t lse_rows;
};
hipError_t launch_pool_f32(const void* q, const int64_t q_st[3], const Grid3& gq, float* q_pooled, int32_t* q_rows, const void* k,
                           const int64_t k_st[3], const Grid3& gk, float* k_pooled, int32_t* k_rows, int B, int Hn, hipStream_t st);
hipError_t launch_fwd_f32(const void* q, const void* k, const void* v, const int32_t* idx, const int32_t* lens,
                          const uint64_t* tile_valid, void* o, float* lse, int B, int Hn, int64_t Sq, int64_t Sk, int bs_q, int bs_k,
                          int idx_stride, float sm_scale, hipStream_t st, const F32Layout* layout = nullptr, const GateCall* gate_call = nullptr);

// Rewrites every row's ascending list of KV blocks into the order the attention kernel visits them in (see
// pace_order_kernel).  rows of `stride` entries, lens[row] of them in use; in == out allowed; stride <= 5000.
// With `bits` the lists are also written down the other way: words[bh][block][row / 32] gets bit row % 32 of every block in
// row `row` of (batch, head) bh, `rows` rows each (cleared by the caller).
struct ListBits {
    uint32_t* words;
    int rows, per_row;
};
hipError_t launch_pace_order(const int32_t* in, int32_t* out, const int32_t* lens, int64_t rows, int nbk, int stride,
                             hipStream_t st, HalfLists halves = {}, ListBits bits = {});
// order: for every (batch, head) its 64-row query tiles by descending list length (lens is per query
// block of tiles_per_block tiles, clamped to [0, max_len]); with `order` and a two-word `queue`
// launch_fwd enqueues the 16-bit kernel both as rounds and as one launch whose workgroups draw items
// from a counter, and a kernel that compares the list lengths decides on the device which of them runs
hipError_t launch_order_by_length(const int32_t* lens, int32_t* order, int BH, int nbq, int tiles_per_block, int max_len,
                                  hipStream_t st);

// For launch_fwd: queue[0] = 0 (the counter work items are drawn with) and queue[1] = the choice between rounds (0) and the
// longest-first queue (1), made on the device from the list lengths (see choose_schedule_kernel)
void launch_schedule_choice(const int32_t* lens, int nbq, int tiles_per_block, int total, int round, int resident,
                            int max_len, uint32_t* queue, hipStream_t st);

// One tensor on its way through launch_prepare (bsa_prepare.hip).  16-bit types as raw bits; strides in elements.
struct PrepRows {
    const uint16_t* p;               // null: this part is left out
    int64_t sB, sH, sS;              // batch, head, token
    const uint16_t* cached;          // k, v, optional: the tokens before `split` come from here, already normalised, and p holds the rest
    int64_t cB, cH, cS;
    int split;
    int heads;                       // set by launch_prepare: heads of a chunk that a workgroup takes
    char* frag;                      // k, v: [B*Hn][padded slots / 64][16 KB] in fragment order (bsa_fwd_frag.hip, bsa_fwd_few.hip), the real slots of a tile first, zeros behind
    uint16_t* pooled;                // q, k: chunk means [B*Hn][blocks][128], the bits launch_permute's pooling gives; optional for k
    int pooled_operand;              // k: ... in operand order instead (operand_mean_at)
    int few;                         // k, v: the order is that of 32x32x16 products (frag_few)
    int32_t* rows;                   // q: row_table_ints() entries; the real slots of a chunk come first
    uint64_t* valid;                 // k, optional: bit s of word i = slot 64 i + s holds a real token
    const uint64_t* valid_in;        // k, v, optional: the real slots of every tile as the caller has them (instead of the grid's)
    float* tile_norm;                // k, optional: largest Euclidean norm of a row of every tile, a part in a thousand above
    const uint16_t* norm_w;          // q, k, with a rotation table: 128 weights of the per-head RMSNorm in front of the rotation
    int t0;                          // q, k: frame offset of the grid inside the rotation table
    uint16_t* rows_out;              // optional: the rows of p at their token positions; q after the transform, k before the rotation
    int64_t rB, rH, rS;              // ... element strides
    int head_fastest;                // set by launch_prepare: the order in which workgroups take (chunk, head)
    int offsets_32;                  // set by launch_prepare: the rows of a (batch, head) lie within 4 GB
};
// Chunk means of k as the attention kernel's products take them where it selects itself, 32 blocks of a (batch, head) to a group: a product's
// fragment (16 of the 128 d) is 1 KB in lane order, lane l block l % 32 and d 8 (l / 32) .. + 8.  The last group is filled up.
__host__ __device__ inline int64_t operand_mean_at(int64_t bh, int blocks, int blk, int d) {
    return ((bh * ((blocks + 31) / 32) + blk / 32) * 8 + d / 16) * 512 + (d >> 3 & 1) * 256 + (blk & 31) * 8 + (d & 7);
}
struct PrepArgs {
    PrepRows q, k, v;
    Grid3 gq, gk;
    int Hn;
    const float* tab;                // rotation table (the layout bsa_norm_rope reads) for q and k; null: rows as they are
    int tab_T;                       // ... its frames
    float eps;
    uint32_t* zero;                  // optional: a word to clear
};
hipError_t launch_prepare(const PrepArgs& a, int B, int dtype, hipStream_t st);
hipError_t launch_row_table(const Grid3& g, int32_t* rows, hipStream_t st);
// Key norms: one per (batch, head), the largest of its tiles', then (from a 256-byte boundary) one per tile.
inline size_t tile_norm_offset(int B, int Hn) { return ((size_t)B * Hn + 63) & ~(size_t)63; }
size_t key_norm_floats(int B, int Hn, int64_t tiles);
hipError_t launch_head_norm(const float* tile_norm, float* key_norm, int BH, int tiles, hipStream_t st);
// The attention kernel on fragment-order K and V.  q_rows (optional): token row of every blocked-order query
// slot, -1 for padding; q_st / o_st: element strides {batch, head, row}; lse_rows: rows per (batch, head) of lse.
hipError_t launch_fwd_frag(const void* q, const void* kf, const void* vf, const int32_t* idx, const int32_t* lens,
                           const uint64_t* tile_valid, void* o, float* lse, int B, int Hn, int64_t Sq, int64_t Sk,
                           int bs_q, int bs_k, int idx_stride, float sm_scale, int dtype, hipStream_t st,
                           const int32_t* q_rows, const int64_t q_st[3], const int64_t o_st[3], int64_t lse_rows,
                           const Grid3* q_grid = nullptr, int32_t* order = nullptr, uint32_t* queue = nullptr, const float* key_norm = nullptr,
                           int32_t* fallback = nullptr, bool fallback_cleared = false, const Grid3* halves_of = nullptr, float* part_buf = nullptr,
                           const GateCall* gate_call = nullptr);
// order (B * Hn * Sq / 64 int32) and queue (kFragQueueWords), both or none: scratch for the schedule of lists of unequal length,
// enqueued besides the rounds; which of the two runs is decided on the device.
constexpr int kFragQueueWords = 16;
// fallback (optional, frag_fallback_ints(B * Hn * Sq / 64) int32): with it and key_norm the bf16 rounds run the kernel that
// takes no row maxima and list here the items whose logits it cannot bound; a last launch computes those.  Its first word
// counts them: fallback_cleared says that it is zero already.
// q_grid (optional, with q_rows): the grid whose row table (row_table_ints) q_rows is; tiles without real rows are then left out.
// part_buf (optional, frag_part_floats() floats, lists of one length): the last, partial round may be cut into parts, merged at the end.
size_t frag_part_floats(const Grid3& q_grid, int64_t heads);
// Work items of a call, those of its last, partial round, and how these are shared: `parts` parts of an item, `team` wavefronts a part.
struct LastRound { int total, items, team, parts; };
// The fragment order of K and V that launch_fwd_frag reads: for a call of few items that of 32x32x16 products, otherwise of 16x16x32.
bool frag_few(int64_t heads, int64_t Sq, int64_t Sk, const Grid3* q_grid);
// Whether the attention kernel makes the lists of a call itself; then the chunk means of k are in operand order.
bool frag_selects(int64_t heads, int64_t Sq, int64_t Sk, int bs_k, int idx_stride, const Grid3* halves_of, const Grid3* q_grid, bool one_length, int nbk, int width);
LastRound frag_last_round(int64_t heads, int64_t Sq, int64_t Sk, int bs_k, int idx_stride, const Grid3* halves_of, const Grid3* q_grid, bool one_length);
// halves_of (optional): idx and lens are HalfLists, idx_stride their row pitch (at most 4 096), of this grid of keys.
// gate_call (optional): idx and lens are still to be made.
size_t frag_fallback_ints(int64_t items);


// Backward of the blocked-order attention (bsa_bwd.hip), bf16 / fp16.  workspace: bwd_workspace_bytes() bytes, or at least
// those with `least` (then dS is not kept between the kernels and dQ is computed from scratch).
size_t bwd_workspace_bytes(int B, int Hn, int64_t Sq, int64_t Sk, int bs_q, int bs_k, int idx_stride, bool least = false);
int bwd_max_query_blocks();      // the dK / dV kernel stages a KV block's query blocks in LDS: Sq / bs_q may not exceed this
// With `thw` the caller's tensors are in token order: a pass in front brings q and dO into blocked order, k_s into transposed fragments
// (dS not kept: k_s and v into blocked order), with the row tables (token of every blocked-order slot of one (batch, head), -1 = padding) and the validity words, and the kernels store
// the gradient rows at their tokens.  Of launch_bwd's own tensors only idx, lens and tile_valid are then used.  Strides count
// elements.
struct BwdThw {
    Grid3 gq, gk;
    const void *q, *k, *v, *o, *dout;
    int64_t q_st[3], k_st[3], v_st[3], o_st[3], do_st[3];
    const float* lse;                 // [B * Hn][tokens]
    void *q_blocked, *v_blocked, *dout_blocked;      // B * Hn * Sq (v: Sk) rows of 128 elements; v where dS is not kept
    int32_t *q_rows, *k_rows;         // Sq and Sk entries
    uint64_t* valid;                  // Sk / 64 words
    void* dq; int64_t dq_st[3];
    void* dk; int64_t dk_st[3];
    void* dv; int64_t dv_st[3];
};
// unequal: the lists may differ much in length (for the schedule of dQ alone).  read_copies: a gradient is stored over k (with thw: or
// v) before the dK / dV kernel has read all of it, which then reads k_s and v in blocked order from the workspace; dS is not kept.
hipError_t launch_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout, const float* lse,
                      const int32_t* idx, const int32_t* lens, const uint64_t* tile_valid, void* dq, void* dk, void* dv,
                      int B, int Hn, int64_t Sq, int64_t Sk, int bs_q, int bs_k, int idx_stride, float sm_scale, int dtype,
                      void* workspace, size_t workspace_bytes, hipStream_t st, const BwdThw* thw = nullptr, bool unequal = false, bool read_copies = false);

}  // namespace bsa
