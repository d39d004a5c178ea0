// The operator on fp32 tensors: chunk means with the row tables (pool_f32_kernel) and the attention kernel
// (fwd_f32_kernel, v_mfma_f32_16x16x4), which reads q, k and v and writes o where they lie, through row tables.
//
// fp32 inputs are the plumbing configuration and a cross-check, so most calls are small: what counts is how many of
// the 1 024 SIMDs a call of a few dozen query rows reaches and how many launches it makes.  256 tokens x 4 heads took
// 93 us with a plain kernel behind four copies (62 us for 16 workgroups that walked their keys one by one, 20 us for
// the copies, 12 us for scores computed one column per lane).
#include "bsa_gate.h"
#include "bsa_mfma.h"

namespace bsa {
namespace {

using mfma::kD;
using mfma::kLazyTau;
using mfma::kLn2;
using mfma::kLog2e;
using mfma::kTile;

constexpr int64_t kF32SplitUnits = 4096;
// Units, and units times key blocks, up to which they select for themselves; the four units of a query block make its list four
// times.  With gate_kernel in front / like this, us: 64 units and 4 blocks 16.7 / 14.1, 512 and 128 44.5 / 40.9, 1 024 and 32 39.9 /
// 37.1, 1 024 and 64 50.8 / 48.1, 1 024 and 128 72.7 / 74.1, 2 048 and 64 83.6 / 87.2.
constexpr int64_t kF32GateUnits = 1024, kF32GateScores = 64 * 1024;

// ------------------------------------------------------------------ chunk means and row tables
// blockIdx.z 0: q, 1: k.  One workgroup per (chunk, batch * head): a thread sums 16-byte piece c of the rows rg, rg + 8,
// ... in ascending order, then the eight partial sums of a column are added in ascending rg (the order of
// permute_kernel, so the means carry the bits of the stand-alone entry points).
struct PoolF32 {
    const float* src;
    int64_t sB, sH, sS;
    Grid3 g;
    float* pooled;
    int32_t* rows;          // token row of every blocked-order slot, -1 for padding
};
__global__ __launch_bounds__(256) void pool_f32_kernel(PoolF32 a, PoolF32 b, int Hn) {
    __shared__ float red[8 * kD];
    const PoolF32 x = blockIdx.z == 0 ? a : b;
    const Grid3 g = x.g;
    const int blk = blockIdx.x, bh = blockIdx.y;
    if (blk >= g.blocks()) return;
    const int nw = blk % g.Nw, nh = (blk / g.Nw) % g.Nh, nt = blk / (g.Nw * g.Nh);
    const int bs = g.chunk();
    auto token = [&](int r) -> int {
        const int wi = r % g.w, hi = (r / g.w) % g.h, ti = r / (g.w * g.h);
        const int tt = nt * g.t + ti, hh = nh * g.h + hi, ww = nw * g.w + wi;
        return tt < g.T && hh < g.H && ww < g.W ? (tt * g.H + hh) * g.W + ww : -1;
    };
    if (bh == 0)
        for (int r = threadIdx.x; r < bs; r += 256) x.rows[(int64_t)blk * bs + r] = token(r);
    const int c = threadIdx.x & 31, rg = threadIdx.x >> 5;
    const float* base = x.src + (int64_t)(bh / Hn) * x.sB + (int64_t)(bh % Hn) * x.sH + 4 * c;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int r0 = rg; r0 < bs; r0 += 64) {          // bs is a multiple of 64: eight rows of a thread in flight
        int t[8];
        f32x4 val[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = token(r0 + 8 * j);
#pragma unroll
        for (int j = 0; j < 8; ++j) val[j] = *reinterpret_cast<const f32x4*>(base + (int64_t)max(t[j], 0) * x.sS);
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += t[j] >= 0 ? val[j][e] : 0.f;
    }
    *reinterpret_cast<f32x4*>(red + rg * kD + 4 * c) = acc;
    __syncthreads();
    if (threadIdx.x < kD) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) s += red[i * kD + threadIdx.x];
        x.pooled[((int64_t)bh * g.blocks() + blk) * kD + threadIdx.x] = s * (1.0f / bs);
    }
}

// ------------------------------------------------------------------ attention
// A wavefront owns 16 query rows.  S^T (16 keys x 16 queries) = K Q^T in 32 MFMAs over d, then O^T (128 d x 16 queries)
// += V^T P^T in 32: the accumulator of S^T (lane l: keys 4 (l / 16) + i of query l % 16) is the B operand of the second
// product when its step i contracts the keys 4 g + i, so P never moves.  Both products are free to take d in any order:
// step (j, e) of S^T contracts d = 16 j + 4 g + e, so a lane reads its key row in 16-byte pieces and four lanes share 64
// contiguous bytes; tile t of O^T holds d = 4 m + t (+ 60 from t = 4 on) in row m, so sixteen lanes read 256 contiguous
// bytes of a value row and a lane's results are contiguous.  No LDS in the loop: an fp32 MFMA takes 32 clocks for one
// register of each operand, so the 16 KB of a 16-key group against 2 048 clocks of MFMA ask for 32 B/clk of a CU's L1
// (64 B/clk), and half of that when the four wavefronts of a workgroup meet in it.
// kSplit 1: a workgroup is a 64-row query tile, a wavefront 16 of its rows.  kSplit 4: a workgroup is 16 query rows and
// its wavefronts take every fourth key group, merged through LDS at the end; chosen when a call has too few 16-row
// units to give every SIMD one (below).
struct F32Args {
    const float *q, *k, *v;
    float* o;
    float* lse;
    const int32_t *idx, *lens;
    const uint64_t* tile_valid;       // blocked order only; with a row table the token says it
    const int32_t *q_rows, *k_rows;   // null: blocked order
    int64_t q_st[3], k_st[3], v_st[3], o_st[3];
    int64_t Sq, Sk, lse_rows;
    int Hn, bs_q, bs_k, idx_stride;
    float qk_scale;
    const float *qc, *kc;             // kGate: chunk means
    int k_sel;
};

// kGate: the workgroup makes its block's list itself, as gate_kernel does (the same scores and choice, blocks ascending), instead
// of a launch in front that is longer than that.  Of the wavefronts' scores, 16 at a time, each
// is made once; the first wavefront selects.
constexpr int kF32GateBlocks = 128;
template <int kSplit, bool kGate>
__global__ __launch_bounds__(256) void fwd_f32_kernel(F32Args a) {
    constexpr int kPitch = kD + 4;
    __shared__ __attribute__((aligned(16))) float part_o[kSplit == 1 ? 1 : kSplit * 16 * kPitch];
    __shared__ float part_m[kSplit * 16], part_l[kSplit * 16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n16 = lane & 15, g = lane >> 4;
    const int64_t units = a.Sq / 16;                                  // 16-row units of one (batch, head)
    const int64_t unit_all = kSplit == 1 ? (int64_t)blockIdx.x * 4 + wave : (int64_t)blockIdx.x;
    const int64_t bh = unit_all / units;
    const int64_t slot0 = (unit_all - bh * units) * 16;
    const int64_t at = bh / a.Hn, hd = bh - at * a.Hn;
    const float* kb = a.k + at * a.k_st[0] + hd * a.k_st[1];
    const float* vb = a.v + at * a.v_st[0] + hd * a.v_st[1];
    const int nbq = (int)(a.Sq / a.bs_q), nbk = (int)(a.Sk / a.bs_k), per_block = a.bs_k / 16;
    const int64_t lrow = bh * nbq + slot0 / a.bs_q;
    __shared__ float gate_scores[kGate ? kF32GateBlocks : 1];
    __shared__ int32_t gate_list[kGate ? kF32GateBlocks : 1];
    const int32_t* list = kGate ? nullptr : a.idx + lrow * a.idx_stride;
    const int qtok = a.q_rows != nullptr ? a.q_rows[slot0 + n16] : (int)slot0 + n16;
    int ngroups = (kGate ? a.k_sel : __builtin_amdgcn_readfirstlane(min(max(a.lens[lrow], 0), a.idx_stride))) * per_block;
    if (!__any(qtok >= 0)) ngroups = 0;                               // query rows of padding only

    f32x4 qv[8], o[8];
    {
        const float* qp = a.q + at * a.q_st[0] + hd * a.q_st[1] + (int64_t)max(qtok, 0) * a.q_st[2] + 4 * g;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            qv[j] = *reinterpret_cast<const f32x4*>(qp + 16 * j);
            o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if constexpr (kGate) {
        f32x4 qm[8], km[8];
        score_row_f32(a.qc + lrow * kD + 4 * g, qm);                  // the block's mean as every row of the product
        for (int n0 = 16 * wave; n0 < nbk; n0 += 64) {
            score_row_f32(a.kc + (bh * nbk + min(n0 + n16, nbk - 1)) * kD + 4 * g, km);
            const f32x4 acc = score_tile_f32(qm, km);
            if (g == 0) gate_scores[n0 + n16] = acc[0];
        }
        __syncthreads();
        if (wave == 0) {
            uint32_t val[kF32GateBlocks / 64];
#pragma unroll
            for (int j = 0; j < kF32GateBlocks / 64; ++j) {
                const int i = j * 64 + lane;
                val[j] = i < nbk ? ord_of(__float_as_uint(gate_scores[min(i, nbk - 1)])) : 0u;
            }
            select_row<uint32_t, kF32GateBlocks / 64, false>(val, [&](int i) { return __float_as_uint(gate_scores[i]); }, lane, nbk, a.k_sel, nullptr,
                                                             gate_list, nullptr, nullptr);
        }
        __syncthreads();
    }
    // key group gi of the walk: its first blocked-order slot; tokens of its keys (-1: padding or masked)
    auto slot_of = [&](int gi) -> int64_t {
        const int blk = min(max(__builtin_amdgcn_readfirstlane(kGate ? gate_list[gi / per_block] : list[gi / per_block]), 0), nbk - 1);
        return (int64_t)blk * a.bs_k + (gi % per_block) * 16;
    };
    struct Rows { int k; int v[4]; };                                 // key n16 of the group; keys 4 g .. 4 g + 3
    auto rows_of = [&](int gi) -> Rows {
        Rows r;
        const int64_t s = slot_of(gi);
        if (a.k_rows != nullptr) {
            r.k = a.k_rows[s + n16];
            const int4 v4 = *reinterpret_cast<const int4*>(a.k_rows + s + 4 * g);
            r.v[0] = v4.x; r.v[1] = v4.y; r.v[2] = v4.z; r.v[3] = v4.w;
        } else {
            const uint32_t bits = a.tile_valid != nullptr ? (uint32_t)(a.tile_valid[s / kTile] >> (s % kTile)) : 0xffffu;
            r.k = (bits >> n16) & 1u ? (int)s + n16 : -1;
#pragma unroll
            for (int i = 0; i < 4; ++i) r.v[i] = (bits >> (4 * g + i)) & 1u ? (int)s + 4 * g + i : -1;
        }
        return r;
    };
    auto load_k = [&](const Rows& r, f32x4 (&x)[8]) {
        const float* p = kb + (int64_t)max(r.k, 0) * a.k_st[2] + 4 * g;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = *reinterpret_cast<const f32x4*>(p + 16 * j);
    };
    auto load_v = [&](const Rows& r, f32x4 (&x)[4][2]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float* p = vb + (int64_t)max(r.v[i], 0) * a.v_st[2] + 4 * n16;
            x[i][0] = *reinterpret_cast<const f32x4*>(p);
            x[i][1] = *reinterpret_cast<const f32x4*>(p + 64);
        }
    };
    float m = -INFINITY, l = 0.f;
    const int step = kSplit, first = kSplit == 1 ? 0 : wave;
    if (first < ngroups) {
        Rows now = rows_of(first), next = rows_of(min(first + step, ngroups - 1));
        f32x4 kx[8], vx[4][2];
        load_k(now, kx);
        load_v(now, vx);
        for (int gi = first; gi < ngroups; gi += step) {
            const Rows ahead = rows_of(min(gi + 2 * step, ngroups - 1));
            f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;                 // two chains: a dependent MFMA waits for its predecessor
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[j][0], qv[j][0], s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[j][1], qv[j][1], s1, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[j][2], qv[j][2], s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[j][3], qv[j][3], s1, 0, 0, 0);
            }
            load_k(next, kx);                                         // behind the last reader of this group's keys
            float p[4], mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[i] = now.v[i] >= 0 ? (s0[i] + s1[i]) * a.qk_scale : -INFINITY;
                mx = fmaxf(mx, p[i]);
            }
            // the running maximum is raised only when exceeded by 2^8 (every lane of a query then agrees on it)
            if (__any(mx > m + kLazyTau)) {
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                mx = fmaxf(mx, __shfl_xor(mx, 32));
                const float m_new = fmaxf(m, mx);
                const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
                m = m_new;
                l *= alpha;
#pragma unroll
                for (int t = 0; t < 8; ++t) o[t] *= alpha;
            }
            const float off = m == -INFINITY ? 0.f : m;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[i] = __builtin_amdgcn_exp2f(p[i] - off);
                l += p[i];
            }
            if (__any(min(min(now.v[0], now.v[1]), min(now.v[2], now.v[3])) < 0)) {      // 0 x inf of a stand-in row must not count
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (now.v[i] < 0) vx[i][0] = vx[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int t = 0; t < 8; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vx[i][t >> 2][t & 3], p[i], o[t], 0, 0, 0);
            load_v(next, vx);
            now = next;
            next = ahead;
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    float* op = a.o + at * a.o_st[0] + hd * a.o_st[1];
    if (kSplit == 1) {
        if (qtok < 0) return;
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        op += (int64_t)qtok * a.o_st[2] + 16 * g;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<f32x4*>(op + 64 * h + 4 * i) =
                    f32x4{o[4 * h][i], o[4 * h + 1][i], o[4 * h + 2][i], o[4 * h + 3][i]} * inv;
        if (a.lse != nullptr && g == 0) a.lse[bh * a.lse_rows + qtok] = l > 0.f ? (m + log2f(l)) * kLn2 : -INFINITY;
        return;
    }
    if (g == 0) { part_m[wave * 16 + n16] = m; part_l[wave * 16 + n16] = l; }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<f32x4*>(part_o + (wave * 16 + n16) * kPitch + 64 * h + 16 * g + 4 * i) =
                f32x4{o[4 * h][i], o[4 * h + 1][i], o[4 * h + 2][i], o[4 * h + 3][i]};
    __syncthreads();
    {
        const int row = threadIdx.x >> 4, d0 = (threadIdx.x & 15) * 8;
        const int tok = a.q_rows != nullptr ? a.q_rows[slot0 + row] : (int)slot0 + row;
        if (tok < 0) return;
        float M = -INFINITY, L = 0.f, scale[kSplit];
#pragma unroll
        for (int w = 0; w < kSplit; ++w) M = fmaxf(M, part_m[w * 16 + row]);
#pragma unroll
        for (int w = 0; w < kSplit; ++w) {
            const float mw = part_m[w * 16 + row];
            scale[w] = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
            L += part_l[w * 16 + row] * scale[w];
        }
        const float inv = L > 0.f ? 1.0f / L : 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < kSplit; ++w) sum += *reinterpret_cast<const f32x4*>(part_o + (w * 16 + row) * kPitch + d0 + 4 * h) * scale[w];
            *reinterpret_cast<f32x4*>(op + (int64_t)tok * a.o_st[2] + d0 + 4 * h) = sum * inv;
        }
        if (a.lse != nullptr && d0 == 0) a.lse[bh * a.lse_rows + tok] = L > 0.f ? (M + log2f(L)) * kLn2 : -INFINITY;
    }
}

}  // namespace

hipError_t launch_pool_f32(const void* q, const int64_t q_st[3], const Grid3& gq, float* q_pooled, int32_t* q_rows, const void* k,
                           const int64_t k_st[3], const Grid3& gk, float* k_pooled, int32_t* k_rows, int B, int Hn, hipStream_t st) {
    const PoolF32 a = {(const float*)q, q_st[0], q_st[1], q_st[2], gq, q_pooled, q_rows};
    const PoolF32 b = {(const float*)k, k_st[0], k_st[1], k_st[2], gk, k_pooled, k_rows};
    const int blocks = gq.blocks() > gk.blocks() ? gq.blocks() : gk.blocks();
    hipLaunchKernelGGL(pool_f32_kernel, dim3(blocks, B * Hn, 2), dim3(256), 0, st, a, b, Hn);
    return hipGetLastError();
}

hipError_t launch_fwd_f32(const void* q, const void* k, const void* v, const int32_t* idx, const int32_t* lens,
                          const uint64_t* tile_valid, void* o, float* lse, int B, int Hn, int64_t Sq, int64_t Sk, int bs_q, int bs_k,
                          int idx_stride, float sm_scale, hipStream_t st, const F32Layout* layout, const GateCall* gate_call) {
    F32Args a = {};
    a.q = (const float*)q; a.k = (const float*)k; a.v = (const float*)v; a.o = (float*)o;
    a.lse = lse; a.idx = idx; a.lens = lens; a.tile_valid = tile_valid;
    a.Sq = Sq; a.Sk = Sk; a.Hn = Hn; a.bs_q = bs_q; a.bs_k = bs_k; a.idx_stride = idx_stride;
    a.qk_scale = sm_scale * kLog2e;
    if (layout != nullptr) {
        a.q_rows = layout->q_rows; a.k_rows = layout->k_rows; a.lse_rows = layout->lse_rows;
        for (int i = 0; i < 3; ++i) {
            a.q_st[i] = layout->q_st[i]; a.k_st[i] = layout->k_st[i]; a.v_st[i] = layout->v_st[i]; a.o_st[i] = layout->o_st[i];
        }
    } else {
        a.lse_rows = Sq;
        a.q_st[0] = a.o_st[0] = (int64_t)Hn * Sq * kD;
        a.q_st[1] = a.o_st[1] = Sq * kD;
        a.k_st[0] = a.v_st[0] = (int64_t)Hn * Sk * kD;
        a.k_st[1] = a.v_st[1] = Sk * kD;
        a.q_st[2] = a.o_st[2] = a.k_st[2] = a.v_st[2] = kD;
    }
    // Up to 4 096 16-row units one workgroup each still is at most four wavefronts' worth per SIMD: the split walk is a
    // quarter as long.  Beyond, four units share a workgroup, and what they read of k and v.
    const int64_t units = (int64_t)B * Hn * (Sq / 16);
    if (gate_call != nullptr) {
        const GateCall& c = *gate_call;
        if (units <= kF32GateUnits && units * c.nbk <= kF32GateScores && c.nbk <= kF32GateBlocks && c.lists == nullptr && c.threshold == 0.f && c.width > 0) {
            a.qc = static_cast<const float*>(c.q_cmp);
            a.kc = static_cast<const float*>(c.k_cmp);
            a.k_sel = c.width;
            hipLaunchKernelGGL((fwd_f32_kernel<4, true>), dim3((unsigned)units), dim3(256), 0, st, a);
            return hipGetLastError();
        }
        const hipError_t e = c.make(c.ctx);
        if (e != hipSuccess) return e;
    }
    if (units <= kF32SplitUnits)
        hipLaunchKernelGGL((fwd_f32_kernel<4, false>), dim3((unsigned)units), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((fwd_f32_kernel<1, false>), dim3((unsigned)(units / 4)), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace bsa
