// The two projections of the attention module as one hand-written gfx950 GEMM:
//   out[M, N] = x[M, K] . w[N, K]^T (+ bias) (+ residual)            (plain epilogue)
//   q, k, v   = split(x . w^T + bias) per head, q and k normalised per head (RMSNorm over the 128
//               features of a head) and rotated (3-D RoPE), every head written as a contiguous
//               [tokens, 128] tensor                                    (QKV epilogue)
// bf16 operands, fp32 accumulation in v_mfma_f32_16x16x32_bf16.
//
// Shape of the computation.  Both operands have k as their fastest axis, which is the layout both MFMA
// operands want: lane l of a 16x16x32 product holds 8 consecutive k of row l % 16, starting at k = 8 (l / 16).
// The weight rows are the A operand and the token rows the B operand, so an accumulator register holds
// C^T: lane l has token l % 16 and, in its 4 registers, features 4 (l / 16) + r of the 16x16 block.  A lane
// therefore owns whole rotation pairs (features 2i, 2i + 1) and a quarter of the features of its tokens: the per-head
// sum of squares is an in-lane sum plus two exchanges.  16x16x32 and not 32x32x16: what bounds a large product is the
// board's power, and the small form moves half as many accumulators per multiplication.  Registers alone, random data, nothing but
// MFMAs: 2 070 TFLOP/s against 1 850; this kernel (then one tile a workgroup), 86 400 x 4 096 x 4 096: 2 149 us against 2 282, the
// clock under it 1.78 GHz against 1.65.
//
// A workgroup of eight wavefronts computes tiles of 256 tokens x 256 features, a wavefront 64 x 128 of a tile: for the
// QKV projection one head of 64 tokens.  Waves w and w + 4 share a SIMD and take turns: while group 0 (features 0 .. 127 of the
// tile) multiplies a k block of 64, 64 MFMAs, group 1 reads its operands of one from LDS and requests a slab of a later one, and
// the other way round, with a barrier at every change.  One wavefront a SIMD (128 x 128 of the tile) has a third fewer
// fragment reads but nothing to issue while it waits or requests: 2 500 us.  Per k block the workgroup brings 256 rows x 128 bytes of
// either operand (a half-slab of 32 KB, whole cache lines) from global memory straight into LDS
// (global_load_lds_dwordx4, no staging registers); five half-slab stages fill the 160 KB of LDS.  The LDS side of such a load is
// linear in the lane index, so the XOR swizzle that keeps the fragment reads (ds_read_b128, rows 128 bytes apart) free of bank
// conflicts is applied on the global side: the 16-byte slot p of row r receives k unit p ^ ((r >> 1) & 7).
//
// The stages, in phases (k block j is read by group 0 in phase 2j and by group 1 in phase 2j + 1): its two half-slabs are free from
// phase 2j + 2 on.  Group 0 requests the weights of block j + 1 in phase 2j, into the stage of block j - 1's tokens, and waits for them
// at the end of phase 2j + 1; group 1 requests the tokens of block j + 2 in phase 2j + 1, into the stage of block j - 1's
// weights, and waits for those of block j + 1 there.
//
// A workgroup stays and goes from tile to tile; the requests run on over the change, so that the first blocks of the next tile
// are there when it begins (one tile a workgroup: 2 135 us; 32 760 x 12 288 x 4 096 2 400 against 2 290).  The order of the tiles runs
// over blocks of 8 token tiles, and the workgroups of an XCD have a contiguous share of it, 8 x 4 tiles at a time: in step, they
// fetch a slab once for 4 or 8 of them.
//
// A LoRA side branch is more of the same sum: a tile's first k blocks are those of the rank axis (t . up^T, scaled where they end), for a pass
// that reads and writes the layer's output at 4 TB/s.  Its two blocks of 66 cost 3 % of the product (128 multiplications a lane included).
// A gated residual is added in the epilogue, for the same reason and by the rule of a residual: the library's product and gated_residual_kernel /
// this, us, 28 618 x 4 096 x 4 096 (rounds full) 734 / 734, 44 969 x 2 304 x 2 304 (0.88) 505 / 432, 25 128 x 1 280 (0.97) 112 / 81, 0.72
// full 5 795 x 3 968 168 / 172, K = 256 13.6 / 16.4 (506 rows, a launch less) to 26 / 21 (45 731).
// A token's gate is asked for before its sums (32 760 x 4 096 x 4 096 845 -> 840).  The residual's lines brought into the L2 three k blocks ahead of
// the epilogue (two loads a lane, whose wait falls into a phase) cost more than they save: 823 -> 842 with a residual.
//
// What bounds it: power, and the reading half of a phase.  Per k block and group 610 clocks to request 32 KB (the address unit of a
// CU takes 16 a load of 1 KB, and a wavefront issues in order) and 500 to read 96 KB of fragments, against 1 009 of MFMAs (an
// instrumented build).  By counters the MFMAs run 0.74 of the clocks at 1.72 GHz with a residual, 86 400 x 4 096 x 4 096, and 0.73 at 1.67 with the
// QKV epilogue, without a bank conflict.  Measured and not kept: the requests between the fragment reads (R 1 170 clocks)
// or between the MFMAs (both wait for the address unit: 0.66-0.70), MFMAs behind the barrier of a phase, with and without priority (0.75),
// an L2 prefetch three to eight blocks ahead (1-2 % slower), one barrier a k block with the groups half a block apart (0.54-0.74).
// hipBLASLt's kernel for the QKV shape runs 0.87 of its clocks at 1.53 GHz in the same runs.
#include "bsa_mfma.h"

#include <algorithm>

namespace bsa {
namespace {

using namespace mfma;

constexpr int kTileM = 256;              // tokens of a tile
constexpr int kTileN = 256;              // features of a tile
constexpr int kBK = 64;                  // k per pipeline step
constexpr int kPart = 256 * kBK * 2;     // bytes of one operand's slab
constexpr int kStages = 5;               // half-slabs resident in LDS: 160 KB
constexpr int kThreads = 512;
constexpr int kCus = 256;                // workgroups of a launch at most: one a CU
constexpr int kBlockM = 8;               // token tiles that the order of the tiles stays with

typedef bf16x8 V8;

constexpr int kMaxSlices = 8;

enum Epilogue { kPlain, kResidual, kGated, kQkv };

struct GemmArgs {
    const __bf16* x; int64_t ldx;
    const __bf16* w; int64_t ldw;
    const __bf16* bias;
    const __bf16* residual; int64_t ldr;
    __bf16* out; int64_t ldo;
    int M, N, K;
    int tiles_m, tiles_n;
    // QKV epilogue
    __bf16* dst[3];
    int64_t dB, dH, dS;
    const __bf16* norm_w[2];
    const float* tab;
    int Hn, S, Hg, Wg, t0, Ttab;
    float eps;
    const float* gate; int gate_rows;      // out = residual + gate * (...): a row of N for every gate_rows tokens
    // a LoRA side branch: t [M, slices * rank], up [per, rank] for every `per` features
    const __bf16* t; int64_t ldt;
    const __bf16* up[kMaxSlices];
    int per, rank;
    float scale;
};

// kSide: with a LoRA side branch.
template <int kEpi, bool kSide>
__global__ __launch_bounds__(kThreads, 2) void gemm_nt_kernel(const GemmArgs a) {
    constexpr bool QKV = kEpi == kQkv;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int group = wave >> 2, quarter = wave & 3;      // waves w and w + 4 share a SIMD

    // ---- tiles of this workgroup: every per_xcd-th of its XCD's (workgroup b runs on XCD b % 8)
    const int per_xcd = gridDim.x >> 3, xcd = blockIdx.x & 7;
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    const int t_end = (int)(tiles * (xcd + 1) >> 3), t_first = (int)(tiles * xcd >> 3) + (int)(blockIdx.x >> 3);
    if (t_first >= t_end) return;
    auto place = [&](int t, int& tile_m, int& tile_f) {
        const int block = t / (kBlockM * a.tiles_n), in = t - block * (kBlockM * a.tiles_n);
        const int rows = min(kBlockM, a.tiles_m - block * kBlockM);
        tile_f = in / rows;
        tile_m = block * kBlockM + in - tile_f * rows;
    };

    // ---- global -> LDS: group 0 brings weight rows (odd half-slabs), group 1 token rows (even ones), a wavefront 64 of them,
    // 8 rows (of 128 bytes: one cache line each) per load
    const char* from;
    uint32_t pitch;
    int last_row;
    int next_t = t_first, left = 0;                   // tile that is being brought, k blocks of it that are not yet
    const int side_blocks = kSide ? a.rank / kBK : 0, nblocks = side_blocks + a.K / kBK;
    bool side = kSide;                                // a tile's blocks are those of its side branch, then those of the layer
    const uint32_t lds0 = lds_address(smem);
    auto start_part = [&]() __attribute__((always_inline)) {
        int tm, tf;
        place(next_t, tm, tf);
        last_row = group ? a.M - 1 - tm * kTileM : a.N - 1 - tf * kTileN;
        if (kSide && side) {
            const int f = tf * kTileN, slice = f / a.per;                     // slices are whole tiles
            from = group ? reinterpret_cast<const char*>(a.t + (int64_t)tm * kTileM * a.ldt + slice * a.rank) : reinterpret_cast<const char*>(a.up[slice] + (int64_t)(f - slice * a.per) * a.rank);
            pitch = (uint32_t)(group ? a.ldt : a.rank) * 2u;
            left = side_blocks;
            return;
        }
        from = group ? reinterpret_cast<const char*>(a.x + (int64_t)tm * kTileM * a.ldx) : reinterpret_cast<const char*>(a.w + (int64_t)tf * kTileN * a.ldw);
        pitch = (uint32_t)(group ? a.ldx : a.ldw) * 2u;
        left = nblocks - side_blocks;
    };
    // half-slab h (even: token rows, odd: weight rows, of k block h / 2 of all of this workgroup's tiles) lives in stage h % kStages
    auto bring = [&](int stage) __attribute__((always_inline)) {
        const uint32_t to = lds0 + stage * kPart + quarter * 8192;
        int l = lane;
        asm volatile("" : "+v"(l));                   // eight offsets worked out anew cost less than registers for them
        const uint32_t unit = ((l & 7) ^ (l >> 4)) * 16;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int row = min(quarter * 64 + r * 8 + (l >> 3), last_row);       // edge tiles repeat their last row
            load_to_lds_16(from, __umul24(row, pitch) + (r & 1 ? unit ^ 64u : unit), to + r * 1024);
        }
        from += kBK * 2;
        if (--left == 0) {
            if (kSide && side) {
                side = false;
                start_part();
            } else {
                next_t += per_xcd;
                side = kSide;
                if (next_t < t_end) start_part();
            }
        }
    };

    // ---- LDS -> fragments
    const uint32_t lr = lane & 15, lg = lane >> 4;
    uint32_t unit_of[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) unit_of[ks] = ((4 * ks + lg) ^ ((lr >> 1) & 7)) * 16 + lr * 128;
    V8 af[2][8], bf[2][4];
    auto read_frags = [&](int stage_w, int stage_x) __attribute__((always_inline)) {
        const uint32_t sw = lds0 + stage_w * kPart + group * (128 * 128), sx = lds0 + stage_x * kPart + quarter * (64 * 128);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int i = 0; i < 8; ++i) af[ks][i] = lds_read_at<V8>(unit_of[ks] + sw + i * 2048);
#pragma unroll
            for (int j = 0; j < 4; ++j) bf[ks][j] = lds_read_at<V8>(unit_of[ks] + sx + j * 2048);
        }
    };
    f32x4_ acc[8][4];
    auto meet = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- pipeline
    start_part();
    if (group) {
        bring(0);
        if (left) {
            bring(2);
            asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        } else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
        bring(1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    meet();
    if (group) meet();
    int s_x = 0;                                     // stage of this block's token rows, (2 kb) % 5
    for (int t = t_first; t < t_end; t += per_xcd) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
        for (int kb = 0; kb < nblocks; ++kb) {
            const int s_w = s_x + 1 >= kStages ? s_x + 1 - kStages : s_x + 1;
            const int ahead = s_x + 3 + group, s_to = ahead >= kStages ? ahead - kStages : ahead;
            const bool more = left != 0;
            if (more) bring(s_to);
            __builtin_amdgcn_sched_barrier(0);
            read_frags(s_w, s_x);
            __builtin_amdgcn_sched_barrier(0);
            if (group && more) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else if (group) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            s_x = s_x + 2 >= kStages ? s_x + 2 - kStages : s_x + 2;
            meet();
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] = mfma16(af[ks][i], bf[ks][j], acc[i][j]);
            if constexpr (kSide) {
                if (kb + 1 == side_blocks && a.scale != 1.f) {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
#pragma unroll
                        for (int j = 0; j < 4; ++j)
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[i][j][r] *= a.scale;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (!group) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (!group || kb + 1 < nblocks || t + per_xcd < t_end) meet();
        }

        // ---- epilogue.  Feature of register r of block i: f0 + 16 i + 4 lg + r; token of block j: m0 + 16 j + lr.
        int tile_m, tile_f, el = lane;
        asm volatile("" : "+v"(el));
        const uint32_t lr = el & 15, lg = el >> 4;
        place(t, tile_m, tile_f);
        const int f0 = tile_f * kTileN + group * 128;         // first feature of this wavefront
        const int m0 = tile_m * kTileM + quarter * 64;        // first token
        if (f0 >= a.N) continue;
        int section = 0, head = 0;
        if constexpr (QKV) {
            const int per_section = a.Hn * 128;
            section = f0 / per_section;
            head = (f0 - section * per_section) >> 7;
            if (a.bias != nullptr) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint2 raw = *reinterpret_cast<const uint2*>(a.bias + f0 + 16 * i + 4 * lg);
                    const __bf16* bv = reinterpret_cast<const __bf16*>(&raw);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][j][e] += (float)bv[e];
                }
            }
            if (section < 2) {
#pragma clang fp contract(off)       // every product and sum below is rounded on its own, as in the eager expressions
                constexpr int D = 128;
                constexpr int nt = (D - 4 * (D / 6)) / 2, nh = D / 6, nw = D / 6;    // rotation pairs per axis: 22, 21, 21
                const __bf16* nwgt = a.norm_w[section];
                // the projection output is a bf16 tensor in the module this replaces: round before normalising
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float ss = 0.f;
#pragma unroll
                    for (int i = 0; i < 8; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float v = (float)(__bf16)acc[i][j][r];
                            acc[i][j][r] = v;
                            ss = fmaf(v, v, ss);
                        }
                    ss += __shfl_xor(ss, 16);
                    ss += __shfl_xor(ss, 32);
                    const float rs = __builtin_amdgcn_rsqf(ss * (1.0f / (float)D) + a.eps);    // as bsa_rope.h
                    // position of this lane's token of block j
                    const uint32_t tok = (uint32_t)min(m0 + 16 * j + (int)lr, a.M - 1);
                    const uint32_t s = tok % (uint32_t)a.S;
                    const uint32_t u = s / (uint32_t)a.Wg, v2 = u / (uint32_t)a.Hg;
                    const int wi = (int)(s - u * a.Wg), hi = (int)(u - v2 * a.Hg), ti = a.t0 + (int)v2;
                    const int cos_h = 2 * a.Ttab * nt, cos_w = cos_h + 2 * a.Hg * nh;
                    const int at_t = ti * nt, at_h = cos_h + hi * nh - nt, at_w = cos_w + wi * nw - nt - nh;     // + pair: cosines
                    const int to_sin_t = a.Ttab * nt, to_sin_h = a.Hg * nh, to_sin_w = a.Wg * nw;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint2 raw = *reinterpret_cast<const uint2*>(nwgt + 16 * i + 4 * lg);
                        const __bf16* wv = reinterpret_cast<const __bf16*>(&raw);
                        float f[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) f[e] = (float)(__bf16)((float)(__bf16)(acc[i][j][e] * rs) * (float)wv[e]);
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            const int pair = 8 * i + 2 * (int)lg + e;         // 8 i .. 8 i + 7: most blocks lie within one axis
                            const bool in_t = 8 * i + 7 < nt || (8 * i < nt && pair < nt), in_w = 8 * i >= nt + nh || (8 * i + 7 >= nt + nh && pair >= nt + nh);
                            const int at = (in_t ? at_t : in_w ? at_w : at_h) + pair;
                            const float c = a.tab[at], sn = a.tab[at + (in_t ? to_sin_t : in_w ? to_sin_w : to_sin_h)];
                            const float x0 = f[2 * e], x1 = f[2 * e + 1];
                            // two products, then one add, each rounded: the order of operations of the eager expression
                            acc[i][j][2 * e] = x0 * c + (-x1) * sn;
                            acc[i][j][2 * e + 1] = x1 * c + x0 * sn;
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);       // one block's table entries at a time: registers
                }
            }
        }
        // Two blocks of 16 features change places between the lanes so that a lane has eight features of its token in a row: 16
        // bytes of it, 64 of the four lanes that share it.
        const int piece = 16 * (lg & 1) + 8 * (lg >> 1);
        uint2 bias[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) bias[i] = make_uint2(0, 0);
        if (!QKV && a.bias != nullptr) {
#pragma unroll
            for (int i = 0; i < 8; ++i) bias[i] = *reinterpret_cast<const uint2*>(a.bias + f0 + 16 * i + 4 * lg);
        }
#pragma unroll
        for (int jj = 0; jj < 4; jj += 2) {
            uint4 res[2][4];
            if constexpr (kEpi == kResidual || kEpi == kGated) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const __bf16* row = a.residual + (int64_t)min(m0 + 16 * (jj + j) + (int)lr, a.M - 1) * a.ldr + f0 + piece;
#pragma unroll
                    for (int p = 0; p < 4; ++p) res[j][p] = *reinterpret_cast<const uint4*>(row + 32 * p);
                }
            }
#pragma unroll
            for (int j = jj; j < jj + 2; ++j) {
                const int tok = m0 + 16 * j + (int)lr;
                __bf16* to;
                if constexpr (QKV) {
                    const uint32_t bb = (uint32_t)tok / (uint32_t)a.S, s = (uint32_t)tok - bb * (uint32_t)a.S;
                    to = a.dst[section] + bb * a.dB + head * a.dH + s * a.dS;
                } else {
                    to = a.out + (int64_t)tok * a.ldo + f0;
                }
                f32x4_ gate[8];
                if constexpr (kEpi == kGated) {
                    const float* row = a.gate + (int64_t)((uint32_t)min(tok, a.M - 1) / (uint32_t)a.gate_rows) * a.N + f0 + 4 * lg;
#pragma unroll
                    for (int i = 0; i < 8; ++i) gate[i] = *reinterpret_cast<const f32x4_*>(row + 16 * i);
                }
                uint4 o[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    float v[2][4];
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            v[h][e] = QKV ? acc[2 * p + h][j][e] : acc[2 * p + h][j][e] + (float)reinterpret_cast<const __bf16*>(&bias[2 * p + h])[e];
                    if constexpr (kEpi == kResidual || kEpi == kGated) {
                        const uint4 r = res[j - jj][p];
                        const auto lo = __builtin_amdgcn_permlane16_swap(r.x, r.z, false, false);
                        const auto hi = __builtin_amdgcn_permlane16_swap(r.y, r.w, false, false);
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const uint32_t raw[2] = {lo[h], hi[h]};
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[h][e] = (float)reinterpret_cast<const __bf16*>(raw)[e] + (kEpi == kGated ? gate[2 * p + h][e] * v[h][e] : v[h][e]);
                        }
                    }
                    uint32_t w[2][2];
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            const __bf16 two[2] = {(__bf16)v[h][2 * e], (__bf16)v[h][2 * e + 1]};
                            w[h][e] = *reinterpret_cast<const uint32_t*>(two);
                        }
                    const auto lo = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
                    const auto hi = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
                    o[p] = make_uint4(lo[0], hi[0], lo[1], hi[1]);
                }
                if (tok < a.M) {
#pragma unroll
                    for (int p = 0; p < 4; ++p) *reinterpret_cast<uint4*>(to + 32 * p + piece) = o[p];
                }
            }
        }
    }
}


template <int kEpi, bool kSide = false>
int launch_gemm(GemmArgs& a, hipStream_t stream) {
    a.tiles_m = (a.M + kTileM - 1) / kTileM;
    a.tiles_n = (a.N + kTileN - 1) / kTileN;
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    const unsigned grid = (unsigned)std::min<int64_t>((tiles + 7) / 8 * 8, kCus);
    const size_t lds = (size_t)kStages * kPart;
    auto kernel = gemm_nt_kernel<kEpi, kSide>;
    // more than the 64 KB a kernel gets without asking; the attribute is per device, so it is set on every call
    const hipError_t ea = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (ea != hipSuccess) return set_error(BSA_ERR_HIP, "gemm: LDS size: %s", hipGetErrorString(ea));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), lds, stream, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? BSA_OK : set_error(BSA_ERR_HIP, "gemm launch: %s", hipGetErrorString(e));
}

int check_gemm_operands(const char* what, const void* x, int64_t ldx, const void* w, int64_t ldw, int64_t M, int N, int K) {
    if (!x || !w) return set_error(BSA_ERR_BAD_ARG, "%s: null pointer", what);
    if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffffLL) return set_error(BSA_ERR_BAD_ARG, "%s: M=%lld N=%d K=%d", what, (long long)M, N, K);
    if (K % kBK != 0) return set_error(BSA_ERR_UNSUPPORTED, "%s: K=%d must be a multiple of %d", what, K, kBK);
    if (N % 128 != 0) return set_error(BSA_ERR_UNSUPPORTED, "%s: N=%d must be a multiple of 128", what, N);
    if (ldx < K || ldw < K || ldx % 8 || ldw % 8) return set_error(BSA_ERR_BAD_ARG, "%s: row strides %lld, %lld (at least K, multiples of 8)", what, (long long)ldx, (long long)ldw);
    if (ldx >= (1 << 22) || ldw >= (1 << 22)) return set_error(BSA_ERR_UNSUPPORTED, "%s: row strides above 4M elements are not built", what);
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15u) return set_error(BSA_ERR_BAD_ARG, "%s: pointers must be 16-byte aligned", what);
    return BSA_OK;
}

}  // namespace

// Which linear layers (bsa_linear_bf16) this kernel serves: us of hipBLASLt (with a residual: an fp32 product and residual_add_kernel) /
// of this kernel.  With a residual where the tiles fill the rounds of 256 that they take to four fifths: 86 400 x 4 096 x 4 096 2 668 / 2 241, 4 096 rows
// 123 / 106, 2 048 (128 tiles) 72 / 82, 256 (16 tiles) 23 / 74, 8 192 x 2 048 x 2 048 80 / 58, 16 384 x 1 024 x 1 024 58 / 36; and where K is short, whatever
// the tiles: K = 256 16.9 / 10.7 for 16 rows, 60 / 33 for 86 400, 512 columns and K rows from 16 to 8 192 level.  Without one only there: K = 128 and
// 384 columns 14.2 / 9.9 (1 000 rows) to 37.6 / 27.2 (86 400), K = 256 and 768 13.9 / 12.1 to 67 / 53; the library's host time is 14.
// Rows must be those of whole 16-byte pieces, and out nowhere else than in a place of its own or the residual's: the
// library's route has read x before it writes a result, this kernel has not.
static bool gemm_takes(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* residual, const void* out, int64_t ldo,
                       int64_t M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffffLL || K % kBK || N % 128 || ldx % 8 || ldw % 8 || ldo % 8 || ldx < K || ldw < K || ldo < N || ldx >= (1 << 22) || ldw >= (1 << 22)) return false;
    const auto at = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
    if (((at(x) | at(w) | at(out) | at(residual)) & 15u) || (at(bias) & 7u)) return false;
    const auto rows = [](int64_t n, int64_t pitch, int64_t width) { return (uintptr_t)((n - 1) * pitch + width) * 2u; };
    const uintptr_t o = at(out), o_end = o + rows(M, ldo, N);
    const auto meets = [&](const void* p, uintptr_t bytes) { return p != nullptr && at(p) < o_end && o < at(p) + bytes; };
    return !(meets(x, rows(M, ldx, K)) || meets(w, rows(N, ldw, K)) || meets(bias, (uintptr_t)N * 2u) || (residual != out && meets(residual, o_end - o)));
}
static bool residual_serves(int64_t M, int N, int K) {
    const int64_t tiles = (M + kTileM - 1) / kTileM * ((N + kTileN - 1) / kTileN), round = (tiles + kCus - 1) / kCus * kCus;
    return K <= 256 || 5 * tiles >= 4 * round;
}
bool gemm_serves_linear(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* residual, const void* out, int64_t ldo,
                        int64_t M, int N, int K) {
    return (K <= 256 || residual != nullptr) && residual_serves(M, N, K) && gemm_takes(x, ldx, w, ldw, bias, residual, out, ldo, M, N, K);
}

// Which layers with a LoRA side branch run as one product, a rank of whole k blocks and slices of whole tiles: us, the library's product and
// lora_up_add_kernel / this kernel.  Rank 128, tiles that fill their rounds: 32 760 x 12 288 x 4 096 2 471 / 2 386 (the library alone 2 115), x 4 096 x 4 096
// 834 / 809, 86 400 x 4 096 x 4 096 2 276 / 2 192, 20 000 x 3 072 x 1 024 170 / 127.  Three quarters full 2 000 x 12 288 x 4 096 187 / 173, 0.73
// 12 000 x 2 048 x 2 048 105 / 94, two thirds 1 560 x 12 288 x 4 096 152 / 169, 0.56 9 000 x 2 048 x 2 048 89 / 90.  A short K has less to lose: K = 1 024
// 0.54 full 17 500 x 1 024 67 / 56, 3 000 x 3 072 45 / 29, a quarter full 4 000 x 1 024 24 / 27; K = 768 a third full 28 / 24, 0.07 12.9 / 22.5; K = 256
// 17.3 / 14.3 (506 x 256) to 33 / 17 (39 401).  With a gated residual as well, K = 256 19.4 / 19.1 to 41 / 23, 0.34 full 33 / 30, 0.84 27 580 x 2 048
// 287 / 235, 1.00 28 618 x 4 096 856 / 765.  Pointers and rows as above; out is memory of its own (check_own_memory).
static bool lora_serves(const void* x, const void* w, const void* bias, const void* t, int64_t ldt, const void* const* up, int n_sep, int rank,
                        const void* out, int64_t M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffffLL || n_sep <= 0 || n_sep > kMaxSlices || rank <= 0 || rank % kBK || rank > 128) return false;
    if (K % kBK || K >= (1 << 22) || N % n_sep || N / n_sep % kTileN || ldt < (int64_t)n_sep * rank || ldt % 8 || ldt >= (1 << 22)) return false;
    const auto at = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
    if (((at(x) | at(w) | at(t) | at(out)) & 15u) || (at(bias) & 7u)) return false;
    for (int i = 0; i < n_sep; ++i)
        if (!up[i] || (at(up[i]) & 15u)) return false;
    const int64_t tiles = (M + kTileM - 1) / kTileM * (N / kTileN), round = (tiles + kCus - 1) / kCus * kCus;
    return K <= 256 || (K <= 1024 ? 5 * tiles >= 2 * round : 4 * tiles >= 3 * round);
}

// What a layer with a side branch or behind a gate reads: neither route has read all of it before its first result is stored.
static int check_own_memory(const char* what, const void* x, const void* w, const void* bias, const void* t, int64_t ldt, const void* const* up, int n_sep, int rank,
                            const void* residual, const float* gate, int64_t groups, const void* out, int64_t M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return set_error(BSA_ERR_BAD_ARG, "%s: sizes must be positive", what);
    const auto at = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
    const uintptr_t o = at(out), o_end = o + (uintptr_t)M * N * 2u;
    const auto meets = [&](const void* p, uintptr_t bytes) { return p != nullptr && at(p) < o_end && o < at(p) + bytes; };
    bool over = meets(x, (uintptr_t)M * K * 2u) || meets(w, (uintptr_t)N * K * 2u) || meets(bias, (uintptr_t)N * 2u) || meets(residual, (uintptr_t)M * N * 2u) ||
                meets(gate, (uintptr_t)groups * N * sizeof(float));
    if (t != nullptr && n_sep > 0 && n_sep <= kMaxSlices && rank > 0 && ldt > 0) {      // refused otherwise
        over = over || meets(t, (uintptr_t)((M - 1) * ldt + (int64_t)n_sep * rank) * 2u);
        for (int i = 0; i < n_sep; ++i) over = over || meets(up[i], (uintptr_t)(N / n_sep) * rank * 2u);
    }
    return over ? set_error(BSA_ERR_BAD_ARG, "%s: out must be memory of its own", what) : BSA_OK;
}

static GemmArgs layer_args(const void* x, const void* w, const void* bias, void* out, int64_t M, int N, int K) {
    GemmArgs a = {};
    a.x = (const __bf16*)x; a.ldx = K; a.w = (const __bf16*)w; a.ldw = K; a.bias = (const __bf16*)bias;
    a.out = (__bf16*)out; a.ldo = N;
    a.M = (int)M; a.N = N; a.K = K;
    return a;
}
static void add_side(GemmArgs& a, const void* t, int64_t ldt, const void* const* up, int n_sep, int rank, float scale) {
    a.t = (const __bf16*)t; a.ldt = ldt; a.per = a.N / n_sep; a.rank = rank; a.scale = scale;
    for (int i = 0; i < n_sep; ++i) a.up[i] = (const __bf16*)up[i];
}

}  // namespace bsa

using namespace bsa;

extern "C" {

int bsa_gemm_bf16(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* residual,
                  int64_t ldr, void* out, int64_t ldo, int64_t M, int N, int K, void* stream) {
    const int rc = check_gemm_operands("gemm_bf16", x, ldx, w, ldw, M, N, K);
    if (rc != BSA_OK) return rc;
    if (!out) return set_error(BSA_ERR_BAD_ARG, "gemm_bf16: null pointer");
    if (ldo < N || ldo % 8 || (residual && (ldr < N || ldr % 8)))
        return set_error(BSA_ERR_BAD_ARG, "gemm_bf16: output / residual row strides (at least N, multiples of 8)");
    if ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(residual)) & 15u || reinterpret_cast<uintptr_t>(bias) & 7u)
        return set_error(BSA_ERR_BAD_ARG, "gemm_bf16: out and residual must be 16-byte aligned, bias 8-byte aligned");
    GemmArgs a = {};
    a.x = (const __bf16*)x; a.ldx = ldx; a.w = (const __bf16*)w; a.ldw = ldw; a.bias = (const __bf16*)bias;
    a.residual = (const __bf16*)residual; a.ldr = ldr; a.out = (__bf16*)out; a.ldo = ldo;
    a.M = (int)M; a.N = N; a.K = K;
    return residual ? launch_gemm<kResidual>(a, (hipStream_t)stream) : launch_gemm<kPlain>(a, (hipStream_t)stream);
}

int bsa_linear_lora_bf16(const void* x, const void* w, const void* bias, const void* t, int64_t ldt, const void* const* up, int n_sep, int rank,
                         float multiplier, float alpha_scale, void* out, int64_t M, int N, int K, void* workspace, size_t workspace_bytes, void* stream) {
    if (!x || !w || !t || !up || !out) return set_error(BSA_ERR_BAD_ARG, "linear_lora: null pointer");
    const int rc = check_own_memory("linear_lora", x, w, bias, t, ldt, up, n_sep, rank, nullptr, nullptr, 0, out, M, N, K);
    if (rc != BSA_OK) return rc;
    if (!lora_serves(x, w, bias, t, ldt, up, n_sep, rank, out, M, N, K)) {
        const int lrc = bsa_linear_bf16(x, w, bias, nullptr, out, M, N, K, workspace, workspace_bytes, stream);
        return lrc != BSA_OK ? lrc : bsa_lora_up_add(out, t, ldt, up, n_sep, rank, multiplier, alpha_scale, out, M, N, stream);
    }
    GemmArgs a = layer_args(x, w, bias, out, M, N, K);
    add_side(a, t, ldt, up, n_sep, rank, multiplier * alpha_scale);
    return launch_gemm<kPlain, true>(a, (hipStream_t)stream);
}

int bsa_linear_gated_bf16(const void* x, const void* w, const void* bias, const void* t, int64_t ldt, const void* const* up, int n_sep, int rank,
                          float multiplier, float alpha_scale, const void* residual, const float* gate, int rows_per_group, void* out,
                          int64_t M, int N, int K, void* workspace, size_t workspace_bytes, void* stream) {
    if (!x || !w || (t && !up) || !residual || !gate || !out) return set_error(BSA_ERR_BAD_ARG, "linear_gated: null pointer");
    if (M <= 0 || N <= 0 || K <= 0) return set_error(BSA_ERR_BAD_ARG, "linear_gated: sizes must be positive");
    if (rows_per_group <= 0 || M % rows_per_group != 0)
        return set_error(BSA_ERR_SHAPE, "linear_gated: %lld rows do not split into groups of %d", (long long)M, rows_per_group);
    const int own = check_own_memory("linear_gated", x, w, bias, t, ldt, up, n_sep, rank, residual, gate, M / rows_per_group, out, M, N, K);
    if (own != BSA_OK) return own;
    if (!(reinterpret_cast<uintptr_t>(gate) & 15u) && gemm_takes(x, K, w, K, bias, residual, out, N, M, N, K) &&
        (t ? lora_serves(x, w, bias, t, ldt, up, n_sep, rank, out, M, N, K) : residual_serves(M, N, K))) {
        GemmArgs a = layer_args(x, w, bias, out, M, N, K);
        a.residual = (const __bf16*)residual; a.ldr = N; a.gate = gate; a.gate_rows = rows_per_group;
        if (!t) return launch_gemm<kGated>(a, (hipStream_t)stream);
        add_side(a, t, ldt, up, n_sep, rank, multiplier * alpha_scale);
        return launch_gemm<kGated, true>(a, (hipStream_t)stream);
    }
    const int rc = t ? bsa_linear_lora_bf16(x, w, bias, t, ldt, up, n_sep, rank, multiplier, alpha_scale, out, M, N, K, workspace, workspace_bytes, stream)
                     : bsa_linear_bf16(x, w, bias, nullptr, out, M, N, K, workspace, workspace_bytes, stream);
    return rc != BSA_OK ? rc : bsa_gated_residual(residual, out, gate, out, M, rows_per_group, N, BSA_BF16, stream);
}

int bsa_qkv_projection(const void* x, int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* q_weight,
                       const void* k_weight, const float* rope_table, void* q, void* k, void* v,
                       const int64_t dst_strides[3], int B, int Hn, int T, int H, int W, int t_offset, int table_T,
                       int D, int K, float eps, void* stream) {
    if (D != 128) return set_error(BSA_ERR_UNSUPPORTED, "qkv_projection: head dim %d is not built (only 128)", D);
    if (B <= 0 || Hn <= 0 || T <= 0 || H <= 0 || W <= 0) return set_error(BSA_ERR_BAD_ARG, "qkv_projection: sizes must be positive");
    const int64_t S = (int64_t)T * H * W, M = (int64_t)B * S;
    if (S > 0x7fffffffLL || (int64_t)3 * Hn * D > 0x7fffffffLL) return set_error(BSA_ERR_UNSUPPORTED, "qkv_projection: too many tokens or features");
    const int rc = check_gemm_operands("qkv_projection", x, ldx, w, ldw, M, 3 * Hn * D, K);
    if (rc != BSA_OK) return rc;
    if (!q || !k || !v || !q_weight || !k_weight || !rope_table || !dst_strides)
        return set_error(BSA_ERR_BAD_ARG, "qkv_projection: null pointer");
    if (t_offset < 0 || table_T < t_offset + T)
        return set_error(BSA_ERR_SHAPE, "qkv_projection: frames %d..%d lie outside a table of %d frames", t_offset, t_offset + T, table_T);
    for (int i = 0; i < 3; ++i)
        if (dst_strides[i] < 0 || dst_strides[i] % 8) return set_error(BSA_ERR_BAD_ARG, "qkv_projection: strides must keep rows 16-byte aligned");
    if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15u ||
        (reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(q_weight) | reinterpret_cast<uintptr_t>(k_weight)) & 7u)
        return set_error(BSA_ERR_BAD_ARG, "qkv_projection: q, k, v must be 16-byte aligned, bias and norm weights 8-byte aligned");
    if (!(eps >= 0.f)) return set_error(BSA_ERR_BAD_ARG, "qkv_projection: eps must be non-negative");
    GemmArgs a = {};
    a.x = (const __bf16*)x; a.ldx = ldx; a.w = (const __bf16*)w; a.ldw = ldw; a.bias = (const __bf16*)bias;
    a.M = (int)M; a.N = 3 * Hn * D; a.K = K;
    a.dst[0] = (__bf16*)q; a.dst[1] = (__bf16*)k; a.dst[2] = (__bf16*)v;
    a.dB = dst_strides[0]; a.dH = dst_strides[1]; a.dS = dst_strides[2];
    a.norm_w[0] = (const __bf16*)q_weight; a.norm_w[1] = (const __bf16*)k_weight;
    a.tab = rope_table; a.Hn = Hn; a.S = (int)S; a.Hg = H; a.Wg = W; a.t0 = t_offset; a.Ttab = table_T; a.eps = eps;
    return launch_gemm<kQkv>(a, (hipStream_t)stream);
}

}  // extern "C"
