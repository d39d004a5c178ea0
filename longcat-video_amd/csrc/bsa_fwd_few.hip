// Block-sparse flash-attention forward for gfx950 (bf16 / fp16 MFMA) on fragment-order K and V, for calls of few work items
// (frag_few): every item has a wavefront, or a team of them, of its own at once, and SIMDs are left over.
//
// Why another kernel than that of bsa_fwd_frag.hip.  There the board's power is the bound, of which 16x16x32 products draw less.
// With SIMDs idle the clock is at its top and what bounds a wavefront is its own issue: a tile of 64 keys is 537 instructions
// there, with 128 products, and 450 here, with 64 products of 32x32x16, for 2 048 clocks of products either way.  Whole operator,
// 640 items of 80 tiles: 140.6 us there, 130.0 here (both sides by size at frag_few).  K and V come in the fragment order of the form:
//   K: [half kh][d step c = 0..7][lane l = 0..63][8 elements]
//        element j of lane l = K[key 32 kh + (l & 31)][d = 16 c + 8 (l >> 5) + j]
//      = the A operand of v_mfma_f32_32x32x16 for S^T (32 keys x 32 queries) += K . Q^T.
//   V: [half kh][key step s = 0..1][d tile t = 0..3][lane l][8 elements]
//        element j of lane l = V[key 32 kh + 16 s + 8 (j >> 2) + 4 (l >> 5) + (j & 3)][d = 32 t + (l & 31)]
//      = the A operand of O^T (32 d x 32 queries) += V^T . P^T, with the 16 keys of a step in the
//        order in which the accumulator registers of S^T hold them, so that P^T needs no shuffle.
// The rest is that kernel's: a wavefront's 64 query rows against its list, everything from global memory straight into registers,
// lazy running maximum, fp32 sums, one final rounding.
#include "bsa_frag.h"

namespace bsa {
namespace {

// Everything of one item and nothing of a next one.  kTeam: wavefronts of a workgroup, a SIMD of a compute unit each, that walk a share
// of the item's pairs (of a part's share, where the item is in parts as well) and put their sums together in LDS, in the order of the
// shares, wavefront w those of its 4 / kTeam tiles of d (choose_split).
template <typename T, int kWalk, int kTeam, bool kGate>
__global__ __launch_bounds__(64 * kTeam, 1) void fwd_few_kernel(
    const T* __restrict__ q, const char* __restrict__ kf, const char* __restrict__ vf,
    const int32_t* __restrict__ idx, const int32_t* __restrict__ lens, const uint64_t* __restrict__ tile_valid,
    T* __restrict__ o, float* __restrict__ lse, int64_t Sq, int64_t Sk, int bs_k, int idx_stride,
    float qk_scale, int items, int Hn, int64_t lse_S, FragLayout L, uint32_t kv_bytes, int32_t* __restrict__ lists_out,
    uint32_t* __restrict__ lens_out, Parts parts, FragGate G) {
    typedef typename Vec8<T>::type V8;
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    // log2 headroom before the running maximum is raised: probabilities reach 2^kTau, which the storage type of P
    // must hold (fp16 ends at 65 504) and the fp32 sums must hold times the number of keys
    constexpr float kTau = std::is_same<T, _Float16>::value ? 14.0f : 30.0f;
    touch_arguments<decltype(fwd_few_kernel<T, kWalk, kTeam, kGate>)>();
    // the item's list; then a team's sums; then 64 rows of the output of 256 B, 272 B apart
    constexpr int kOutPitch = kD + 8;
    constexpr int kOutBytes = kTile * kOutPitch * (int)sizeof(T);
    __shared__ __attribute__((aligned(16))) char ost_bytes[kTeam > 1 ? kTeamBytes<kTeam> : kOutBytes];
    T* const ost = reinterpret_cast<T*>(ost_bytes);
    constexpr int kWords = kWalk == kHalves ? 2 : 1;              // list words of a pair
    __shared__ int32_t out_rows[kTile];                          // token rows of the 64 query slots (row table given)
    uint32_t* const big = reinterpret_cast<uint32_t*>(ost);

    const int lane = threadIdx.x & 63;
    const int wave = kTeam > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
    const int lr = lane & 31, lh = lane >> 5;
    const int nqt = (int)(Sq / kTile);
    const int nsub = kWalk == kBlocks ? bs_k / kTile : 1, nsub_of_block = bs_k / kTile;
    const int tiles_bh = (int)(Sk / kTile), nbk = kWalk == kBlocks ? tiles_bh / L.by_sub : tiles_bh;     // kHalves does not ask for it
    const uint32_t lane_off = (uint32_t)lane * 16u;

    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kf), 0, (int)kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(vf), 0, (int)kv_bytes, 0x00020000);
    // at: byte offset of a 32-key half; c / f: fragment of the half
    auto k_frag = [&](uint32_t at, int c) -> V8 {
        return __builtin_bit_cast(V8, __builtin_amdgcn_raw_buffer_load_b128(krs, lane_off + (uint32_t)((c & 3) * 1024), at + (uint32_t)((c >> 2) * 4096), 0));
    };
    auto v_frag = [&](uint32_t at, int f) -> V8 {          // f = 4 * key step + d tile
        return __builtin_bit_cast(V8, __builtin_amdgcn_raw_buffer_load_b128(vrs, lane_off + (uint32_t)((f & 3) * 1024), at + (uint32_t)((f >> 2) * 4096), 0));
    };

    // ---- the item.  Workgroup b runs on XCD b % 8: every XCD takes a contiguous run of the items.
    const int n_all = parts.count * items, x = blockIdx.x & 7;
    if ((int)blockIdx.x >= n_all) return;
    const int local = x * (n_all >> 3) + min(x, n_all & 7) + (int)(blockIdx.x >> 3);
    const int part = parts.count > 1 ? local / parts.by_items : 0;
    auto uni = [](int v) -> int { return __builtin_amdgcn_readfirstlane(v); };
    const int item = uni(item_at(L, local - part * items, nqt));
    const int64_t list_row = item / L.by_block;
    const int bh = item / L.by_tiles;
    const int64_t qrow0 = (int64_t)(item - bh * nqt) * kTile;
    const int batch = bh / L.by_heads;
    const int64_t o_bh = (int64_t)batch * L.o_st[0] + (int64_t)(bh - batch * Hn) * L.o_st[1];
    const uint32_t half_base = (uint32_t)uni(bh * tiles_bh) * 2u;      // first half of the item's (batch, head)
    const int32_t* const list = idx + list_row * idx_stride;
    // what the first products wait for is asked for before any of it is waited for: the length of the list, its entries, as far as
    // one a thread goes (what lies behind its end is not used), the token rows
    const bool early = kTeam == 1 && !kGate && parts.count == 1;         // the walk starts at the list's first entry
    int n_listed = 0, my_entry = 0, first_rows[3] = {0, 0, 0}, first_ent[2] = {0, 0};
    if (!kGate) {
        n_listed = lens[list_row];
        if (idx_stride > 0) {
            my_entry = list[min((int)threadIdx.x, idx_stride - 1)];
            if (kTeam == 1) first_ent[0] = list[0];
            if (kTeam == 1 && kWalk == kHalves) first_ent[1] = list[1];
        }
    }
    if (L.q_rows != nullptr) {
        first_rows[0] = L.q_rows[qrow0 + lr];
        first_rows[1] = L.q_rows[qrow0 + 32 + lr];
        first_rows[2] = L.q_rows[qrow0 + lane];
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- registers
    V8 qreg[2][8];                                             // [32 queries][d step]
    // Register rings: K fragments of two steps, V fragments of two steps (each step: 4 fragments for its
    // first 16 keys, "A", and 4 for its last 16, "B").
    V8 kb[2][8], vb[2][8];
    f32x16 s[2][2];                                            // S^T of the current and of the next step
    V8 pb[2][2];                                               // P^T as B operand: [32 queries][A | B]
    f32x16 oacc[4][2];
    float m_i[2], l_i[2];
    // Softmax state per 32 queries: running maximum m_i (scaled, log2 units), its negative for the exponent
    // (0 while the maximum is -inf), and the unscaled logit above which the maximum has to be raised; the lower of these.
    float neg_m[2], raise_at[2], raise_low;
    const float inv_scale = 1.0f / qk_scale;
    // Raising the maximum has two parts.  Here: the new maximum, the exponent offset, the row sum (which already holds
    // every probability of the current step).  The output accumulators are rescaled one quarter of a step later
    // (rescale_out, behind slot 7 of the next step): the product of the current step's P_B, whose
    // probabilities were taken relative to the old maximum, is only issued in slots 0 .. 7 of that step.
    float alpha_p[2];
    bool rescale_pending = false;

    // ---- the walk: the pairs pair0 .. pair0 + npairs - 1 of the list
    int npairs = 0, pair0 = 0;
    int n_halves = 0;                // a team's walk over halves: those of this wavefront's share, from ents on
    const uint32_t* ents = big;      // the item's list in LDS
    // window of the walk: the entries of the halves 2 g + 1 .. 2 g + 5 of loop iteration g (one pair per iteration).  An entry is a half,
    // counted from half_base, | real keys << 20, as kHalves lists hold them; what is above 2^19 halves is lost in the shift to
    // bytes.  Positions behind the list: entry 0, no key.
    uint32_t w[5];
    auto offset_of = [&](uint32_t entry) -> uint32_t { return (entry << 13) + (half_base << 13); };
    static_assert(kHalfBytes == 1 << 13, "the shift");
    // Pair tp of the walk -> its entries.  The list is read from LDS (pair_raw, to be issued early) and made into entries later.
    struct Raw { uint32_t e[kWords]; };
    auto pair_raw = [&](int tp) -> Raw {
        const int tc = min(tp, npairs - 1) + pair0;
        Raw r;
        if constexpr (kWalk == kHalves && kTeam > 1) {
            r.e[0] = ents[2 * tc];
            r.e[1] = ents[min(2 * tc + 1, n_halves - 1)];
            if (2 * tc + 1 >= n_halves) r.e[1] &= kHalfId;      // an odd share: its last half once more, no key of it
        } else if constexpr (kWalk == kHalves) {
            const uint2 e = *reinterpret_cast<const uint2*>(ents + 2 * tc);               // the same address in every lane
            r.e[0] = e.x; r.e[1] = e.y;
        } else {
            r.e[0] = ents[kWalk == kTiles ? tc : tc / L.by_sub];
        }
        return r;
    };
    // first half of the pair's tile, counted from half_base (kTiles, kBlocks)
    auto tile_half = [&](int tp, const Raw& raw) -> uint32_t {
        if (tp >= npairs) return 0;
        const int blk = min(max(uni((int)raw.e[0]), 0), nbk - 1);                          // a malformed list: wrong numbers, never a fault
        const int tc = tp + pair0;
        return 2u * (uint32_t)(kWalk == kTiles ? blk : blk * nsub + tc - tc / L.by_sub * nsub);
    };
    // the validity word of a pair's tile (all keys valid without padding; kHalves: the entries say it), in two steps so that
    // a caller can ask for several words before it waits for the first
    auto pair_word = [&](uint32_t half) -> uint64_t { return kWalk == kHalves || tile_valid == nullptr ? ~0ull : tile_valid[half >> 1]; };
    auto pair_entries = [&](int tp, const Raw& raw, uint32_t half, uint64_t word, uint32_t (&e)[2]) {
        if (tp >= npairs) {
            e[0] = e[1] = 0;
        } else if (kWalk == kHalves) {
#pragma unroll
            for (int i = 0; i < kWords; ++i) e[i] = (uint32_t)uni((int)raw.e[i]);
        } else {
            const uint32_t lo = (uint32_t)uni((int)(uint32_t)word), hi = (uint32_t)uni((int)(uint32_t)(word >> 32));
            const int n = __builtin_popcountll((uint64_t)lo | ((uint64_t)hi << 32));
            e[0] = half | (uint32_t)min(n, 32) << kHalfCountShift;
            e[1] = (half + 1u) | (uint32_t)max(n - 32, 0) << kHalfCountShift;
        }
    };
    // accumulator i <-> key 8 (i / 4) + 4 lh + i % 4 of the step's 32 keys, query lr (+32)
    auto mask_pair = [&](f32x16 (&sv)[2], uint32_t entry) {
        if (__builtin_expect(entry < 32u << kHalfCountShift, 0)) {
            asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");       // the MFMAs into these accumulators have retired
            // the lane's part of the shift first: the tests below then use constants, not sixteen per-lane bit masks
            // that would have to be kept in registers (or spilled) all through the loop for this rare path
            uint32_t mine = ((1u << (entry >> kHalfCountShift)) - 1u) >> (4 * lh);
            asm volatile("" : "+v"(mine));
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (!((mine >> (8 * (i / 4) + (i % 4))) & 1u)) { sv[0][i] = -INFINITY; sv[1][i] = -INFINITY; }
        }
    };
    // the maximum over the two lanes that share a query
    auto over_lanes = [](float mx) -> float {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    };
    auto lane_max = [&](const f32x16 (&sv)[2], float (&mx)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            mx[qq] = fmaxf(sv[qq][0], sv[qq][1]);
#pragma unroll
            for (int i = 2; i < 16; i += 2) mx[qq] = fmaxf(fmaxf(mx[qq], sv[qq][i]), sv[qq][i + 1]);
        }
    };
    // mx: this lane's unscaled maxima over its 16 accumulators of the step that comes next.  The test needs no exchange
    // between the two key groups of a query: some lane exceeds the limit exactly when the combined maximum does.
    auto raise_max = [&](const float (&mx)[2]) __attribute__((always_inline)) {
        if (!__any(mx[0] > raise_at[0] || mx[1] > raise_at[1])) return;
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            const float m_new = fmaxf(m_i[qq], over_lanes(mx[qq]) * qk_scale);
            const float alpha = __builtin_amdgcn_exp2f(m_i[qq] - ((m_new == -INFINITY) ? 0.f : m_new));
            m_i[qq] = m_new;
            neg_m[qq] = (m_new == -INFINITY) ? 0.f : -m_new;
            raise_at[qq] = (m_new + kTau) * inv_scale;
            l_i[qq] *= alpha;
            alpha_p[qq] = alpha;
        }
        raise_low = fminf(raise_at[0], raise_at[1]);
        rescale_pending = true;
    };
    // The output accumulators live in AGPRs, which the VALU cannot multiply in place.  Written out register by
    // register through one temporary, so that this rare path does not make the compiler reserve VGPRs for a copy
    // of the accumulators.
    auto rescale_out = [&]() __attribute__((always_inline)) {
        asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMA into the accumulators has retired
        static_for<128>([&](auto n_c) {
            constexpr int n = decltype(n_c)::value, qq = n >> 6, t = (n >> 4) & 3, i = n & 15;
            float y = oacc[t][qq][i], tmp;
            asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\ts_nop 1\n\tv_accvgpr_write_b32 %0, %1"
                         : "+a"(y), "=&v"(tmp) : "v"(alpha_p[qq]));
            oacc[t][qq][i] = y;
        });
        asm volatile("s_nop 7" ::: "memory");                        // AGPR writes before the next MFMA reads them
        rescale_pending = false;
    };

    // Step u = 2 g + j (j static).  On entry S(u) is complete and the running maximum covers it; P_B(u-1) is
    // complete.  The 32 MFMAs of a step, in issue order ("slots"):
    //    0 ..  7   O^T += V_B(u-1)^T P_B(u-1)^T      the last 16 keys of the previous step
    //    8 .. 23   S(u+1)^T = K(u+1) Q^T
    //   24 .. 31   O^T += V_A(u)^T P_A(u)^T          the first 16 keys of this step
    // The VALU work on S(u) - per pair of accumulators two fma, two exp2, two additions for the row sum and one
    // rounding of the pair to the storage type, 16 pairs - is cut into pieces that go between the MFMAs so that
    // no gap holds more than an MFMA lasts: the first 14 pairs behind slots 0 .. 23 (the eight pairs of P_A
    // first: they are complete well before slot 24), the last two behind slots 24 .. 31 together with the row
    // maximum of S(u+1), which is complete by then.  Fragment registers are reloaded in bursts behind the last
    // MFMA that reads them: V_B(u+1) behind slot 7, K(u+3) behind slot 23, V_A(u+2) behind slot 31, so that every
    // fragment is requested two steps before it is used.  Within a burst the fragment that is used first is
    // requested last: loads return in order, so the wait in front of its first use covers the whole burst and
    // the fragments behind it need none of their own.  `between` puts scalar work of the walk behind the slots.
    auto step = [&](auto jj, auto between) __attribute__((always_inline)) {
        constexpr int j = decltype(jj)::value;
        constexpr int sc = j & 1, sn = sc ^ 1;                 // S(u) and S(u+1) alternate between two register sets
        constexpr int kslot = (j + 1) & 1;                     // ring slot of K(u+1), then of K(u+3)
        constexpr int vprev = (j + 1) & 1, vcur = j & 1;       // ring slots of V(u-1) / V(u+1) and of V(u) / V(u+2)
        // pair n: queries 32 (n & 1) .., accumulators 2 (n >> 1), + 1.  Its arithmetic comes in three pieces of about the
        // same cost - exponential of the first accumulator (h0), of the second (h1), and the use of both: row sum
        // and rounding (t) - in the order h0(0) h1(0) h0(1) t(0) h1(1) h0(2) t(1) h1(2) ...: the result of a
        // transcendental instruction cannot be consumed by the next instruction without a wait state.
        float pa[2][2];
        auto piece = [&](int p) {                               // p = 0 .. 47
            // p = 0: h0(0); p = 1: h1(0); p = 2 + 3 k: h0(k + 1); p = 3 + 3 k: t(k); p = 4 + 3 k: h1(k + 1); p = 47: t(15)
            const int k = p < 2 ? 0 : (p - 2) / 3, r = p < 2 ? 0 : (p - 2) % 3;
            const bool is_t = p == 47 || (p >= 2 && r == 1);
            const int n = p < 2 ? 0 : p == 47 ? 15 : (r == 1 ? k : k + 1);
            const int e = p < 2 ? p : (r == 0 ? 0 : 1);         // which accumulator of the pair (h0 / h1)
            const int qq = n & 1, i = 2 * (n >> 1);
            if (is_t) {
                l_i[qq] += pa[n & 1][0] + pa[n & 1][1];
                pb[qq][i >> 3][i & 7] = (T)pa[n & 1][0];
                pb[qq][i >> 3][(i + 1) & 7] = (T)pa[n & 1][1];
                asm volatile("" : "+v"(l_i[qq]), "+v"(pb[qq][i >> 3]));
            } else {
                pa[n & 1][e] = __builtin_amdgcn_exp2f(fmaf(s[sc][qq][i + e], qk_scale, neg_m[qq]));
                asm volatile("" : "+v"(pa[n & 1][e]));
            }
        };
        float highest = 0.f;                                    // of this lane's 32 accumulators of S(u+1)
        __builtin_amdgcn_sched_barrier(0);
        static_for<32>([&](auto slot_c) {
            constexpr int slot = decltype(slot_c)::value;
            // ---- the MFMA of this slot
            if constexpr (slot < 8) {
                constexpr int t = slot >> 1, qq = slot & 1;
                oacc[t][qq] = mfma32(vb[vprev][4 + t], pb[qq][1], oacc[t][qq]);
            } else if constexpr (slot < 24) {
                constexpr int c = (slot - 8) >> 1, qq = slot & 1;
                mfma_s<c == 0, qq == 1>(s[sn][qq], kb[kslot][c], qreg[qq][c]);
            } else {
                constexpr int t = (slot - 24) >> 1, qq = slot & 1;
                oacc[t][qq] = mfma32(vb[vcur][t], pb[qq][0], oacc[t][qq]);
            }
            // ---- reloads, in bursts behind the last MFMA that reads the fragments (single loads between the
            // arithmetic cost more issue time than they take): V_B(u+1), K(u+3), V_A(u+2)
            if constexpr (slot == 7) {
                const uint32_t at = offset_of(w[j]);
#pragma unroll
                for (int tt = 1; tt <= 4; ++tt) vb[vprev][4 + (tt & 3)] = v_frag(at, 4 + (tt & 3));
            }
            if constexpr (slot == 23) {
                const uint32_t at = offset_of(w[j + 2]);
#pragma unroll
                for (int cc = 1; cc <= 8; ++cc) kb[kslot][cc & 7] = k_frag(at, cc & 7);
            }
            if constexpr (slot == 31) {
                const uint32_t at = offset_of(w[j + 1]);
#pragma unroll
                for (int tt = 1; tt <= 4; ++tt) vb[vcur][tt & 3] = v_frag(at, tt & 3);
            }
            if constexpr (slot == 7) {
                if (__builtin_expect(rescale_pending, 0)) rescale_out();
            }
            // ---- VALU pieces: 42 of the 48 (14 pairs) behind slots 0 .. 23, one or two per slot; the other 6 behind
            // slots 24 .. 31 next to the row maximum of S(u+1).  S(u+1) is first read behind slot 25: its last MFMA
            // (slot 23) has retired by the time the MFMA of slot 25 has been issued, which the compiler cannot
            // check for the assembly MFMAs.
            if constexpr (slot < 24) {
                constexpr int lo = (slot * 42) / 24, hi = ((slot + 1) * 42) / 24;      // one or two pieces
                piece(lo);
                if constexpr (hi - lo > 1) piece(lo + 1);
            } else {
                constexpr int r = slot - 24;                    // 0 .. 7
                if constexpr (r == 0) { piece(42); piece(43); }
                if constexpr (r == 1) {
                    mfma_chain_end(s[sn][0]);
                    mfma_chain_end(s[sn][1]);
                    mask_pair(s[sn], w[j]);                    // the keys of step u + 1
                    highest = fmaxf(fmaxf(s[sn][0][0], s[sn][1][0]), s[sn][0][1]);
                    highest = fmaxf(fmaxf(highest, s[sn][1][1]), s[sn][0][2]);
                }
                if constexpr (r >= 2) {                         // the other 27, four or five a slot, value n: accumulator n / 2, queries 32 (n % 2) ..
                    constexpr int from = 5 + 27 * (r - 2) / 6, to = 5 + 27 * (r - 1) / 6;
#pragma unroll
                    for (int n = from; n < to; ++n) highest = fmaxf(highest, s[sn][n & 1][n >> 1]);
                }
                if constexpr (r == 2) piece(44);
                if constexpr (r == 4) piece(45);
                if constexpr (r == 6) piece(46);
                if constexpr (r == 7) piece(47);
            }
            between(slot_c);
            __builtin_amdgcn_sched_barrier(0);
        });
        // One test for all queries, of the highest value and the lowest limit, seldom met; then of each query's own.
        if (__builtin_expect(__any(highest > raise_low), 0)) {
            float mx[2];
            lane_max(s[sn], mx);
            raise_max(mx);
        }
    };

    auto first_fragments = [&](uint32_t at0, uint32_t at1) {
#pragma unroll
        for (int c = 0; c < 8; ++c) kb[0][c] = k_frag(at0, c);                      // K(0)
#pragma unroll
        for (int c = 0; c < 8; ++c) kb[1][c] = k_frag(at1, c);                      // K(1)
#pragma unroll
        for (int f = 0; f < 8; ++f) vb[0][f] = v_frag(at0, f);                      // V_A(0), V_B(0)
#pragma unroll
        for (int f = 0; f < 4; ++f) vb[1][f] = v_frag(at1, f);                      // V_A(1)
    };
    // list words in use
    auto list_length = [&](int n) -> int {
        n = min(max(uni(n), 0), idx_stride);
        return kWalk == kHalves ? (n + 1) & ~1 : min(n, kListEntries);
    };

    // Q as the B operand of S^T: lane holds rows lr and 32 + lr, d = 16 c + 8 lh .. + 8
    {
        const int64_t q_bh = (int64_t)batch * L.q_st[0] + (int64_t)(bh - batch * Hn) * L.q_st[1];
        V8 rows[2][8];
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            const int64_t row = L.q_rows != nullptr ? (int64_t)max(first_rows[qq], 0) : qrow0 + 32 * qq + lr;      // padded slots read token 0, never stored
            const T* qp = q + q_bh + row * L.q_st[2] + 8 * lh;
#pragma unroll
            for (int c = 0; c < 8; ++c) rows[qq][c] = *reinterpret_cast<const V8*>(qp + 16 * c);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (early && list_length(n_listed) > 0) {
            const uint32_t h0 = kWalk == kHalves ? (uint32_t)uni(first_ent[0]) & kHalfId : (uint32_t)(min(max(uni(first_ent[0]), 0), nbk - 1) * nsub) * 2u;
            first_fragments(offset_of(h0), offset_of(kWalk == kHalves ? (uint32_t)uni(first_ent[1]) & kHalfId : h0 + 1u));
        }
        __builtin_amdgcn_sched_barrier(0);
        if (L.q_rows != nullptr && wave == 0) out_rows[lane] = first_rows[2];
        if constexpr (kGate) {
            ents = make_list<T, kTeam, kWalk == kHalves>(G, ost_bytes, list_row, bh, nsub_of_block, tile_valid, lists_out, lens_out, lane, wave, n_listed);
        } else {
            const int n = list_length(n_listed);
            if ((int)threadIdx.x < n) big[threadIdx.x] = (uint32_t)my_entry;
            for (int e = threadIdx.x + 64 * kTeam; e < n; e += 64 * kTeam) big[e] = (uint32_t)list[e];
            __syncthreads();
        }
        // The queries 32 .. 63 are read by the assembly MFMAs from accumulation registers.  Their values pass through an
        // assembly statement that ties them to that register class.
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            asm volatile("" : "=v"(qreg[0][c]) : "0"(rows[0][c]));
            asm volatile("" : "=a"(qreg[1][c]) : "0"(rows[1][c]));
        }
    }
    const int nent = list_length(n_listed);
    if constexpr (kTeam > 1) {
        // This wavefront's share of the list, whole KV blocks of it, so that a walk over halves and one over tiles that masks
        // the empty halves cut at the same keys (and give the same bits).
        const int share = part * kTeam + wave, shares = parts.count * kTeam;
        if constexpr (kWalk == kHalves) {
            const int used = min(max(uni(n_listed), 0), idx_stride);      // without the repeat that makes the number even
            auto starts_block = [&](int base) -> uint64_t {       // of the list's entries base .. base + 63
                const uint32_t h = base + lane < used ? ents[base + lane] & kHalfId : 1u;
                return __ballot((h & 1u) == 0u && (int)(h >> 1) == (int)(h >> 1) / L.by_sub * (bs_k / kTile));
            };
            int n_blocks = 0;
            for (int base = 0; base < used; base += 64) n_blocks += __builtin_popcountll(starts_block(base));
            const int b0 = n_blocks * share / shares, b1 = n_blocks * (share + 1) / shares;      // 4 096 entries, 64 shares at most
            int p0 = 0, p1 = used, seen = 0;
            for (int base = 0; base < used; base += 64) {
                const uint64_t m = starts_block(base);
                const int rank = seen + __builtin_popcountll(m & (((uint64_t)1 << lane) - 1));
                const uint64_t at0 = __ballot(((m >> lane) & 1) != 0 && rank == b0), at1 = __ballot(((m >> lane) & 1) != 0 && rank == b1);
                if (at0 != 0) p0 = base + __builtin_ctzll(at0);
                if (at1 != 0) p1 = base + __builtin_ctzll(at1);
                seen += __builtin_popcountll(m);
            }
            ents += p0;
            n_halves = b1 > b0 ? p1 - p0 : 0;
            npairs = (n_halves + 1) >> 1;
        } else {
            const int b0 = nent * share / shares, b1 = nent * (share + 1) / shares;
            pair0 = b0 * nsub;
            npairs = (b1 - b0) * nsub;
        }
    } else {
        npairs = uni(kWalk == kHalves ? nent >> 1 : nent * nsub);
        if (parts.count > 1) {                                  // at most kMaxParts: the products fit 32 bits
            pair0 = npairs * part / parts.by_count;
            npairs = npairs * (part + 1) / parts.by_count - pair0;
        }
    }
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
        m_i[qq] = -INFINITY;
        l_i[qq] = 0.f;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) oacc[t][qq][i] = 0.f;
    }

    if (npairs > 0) {
        uint32_t first;                  // position 0 of the walk
        {
            // the three entries, then the three words, each kind in one sweep: one wait per kind instead of three
            Raw raw3[3];
            uint32_t h[3] = {0, 0, 0}, e[3][2];
            uint64_t word3[3];
#pragma unroll
            for (int r = 0; r < 3; ++r) raw3[r] = pair_raw(r);
            if (kWalk != kHalves) {
#pragma unroll
                for (int r = 0; r < 3; ++r) h[r] = tile_half(r, raw3[r]);
            }
#pragma unroll
            for (int r = 0; r < 3; ++r) word3[r] = pair_word(h[r]);
#pragma unroll
            for (int r = 0; r < 3; ++r) pair_entries(r, raw3[r], h[r], word3[r], e[r]);
            first = e[0][0];
            w[0] = e[0][1]; w[1] = e[1][0]; w[2] = e[1][1]; w[3] = e[2][0]; w[4] = e[2][1];
        }
        // ---- prologue.  In flight when the loop starts: K(1), K(2), V_A(0), V_B(0), V_A(1); the ring slot of
        // V_B(1) holds zeros, which the first step multiplies with P = 0 (there is no step -1).
        if (!early) first_fragments(offset_of(first), offset_of(w[0]));
#pragma unroll
        for (int f = 4; f < 8; ++f)
#pragma unroll
            for (int e = 0; e < 8; ++e) vb[1][f][e] = (T)0.f;
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
#pragma unroll
            for (int e = 0; e < 8; ++e) pb[qq][1][e] = (T)0.f;
            alpha_p[qq] = 1.f;
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (c == 0) { mfma_s<true, false>(s[0][0], kb[0][0], qreg[0][0]); mfma_s<true, true>(s[0][1], kb[0][0], qreg[1][0]); }
            else { mfma_s<false, false>(s[0][0], kb[0][c], qreg[0][c]); mfma_s<false, true>(s[0][1], kb[0][c], qreg[1][c]); }
        }
        const uint32_t third = offset_of(w[1]);
#pragma unroll
        for (int c = 0; c < 8; ++c) kb[0][c] = k_frag(third, c);                        // K(2), behind the last reader of K(0)
        asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");           // MFMA results before the VALU reads them
        mfma_chain_end(s[0][0]);
        mfma_chain_end(s[0][1]);
        mask_pair(s[0], first);
        // the first maximum: nothing is accumulated yet that it would rescale
        float mx[2];
        lane_max(s[0], mx);
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            m_i[qq] = over_lanes(mx[qq]) * qk_scale;
            neg_m[qq] = m_i[qq] == -INFINITY ? 0.f : -m_i[qq];
            raise_at[qq] = (m_i[qq] + kTau) * inv_scale;
        }
        raise_low = fminf(raise_at[0], raise_at[1]);

        // The entries that come into the window are made one iteration before they enter (a validity word may
        // be a load) and read from LDS one iteration before that, between the last MFMAs of an iteration.
        uint32_t in[2], in_next[2];
        auto make = [&](int tp, const Raw& raw, uint32_t (&e)[2]) {
            const uint32_t h = kWalk == kHalves ? 0u : tile_half(tp, raw);
            pair_entries(tp, raw, h, pair_word(h), e);
        };
        make(3, pair_raw(3), in);
        Raw raw = pair_raw(4);
        for (int g = 0; g < npairs; ++g) {
            step(std::integral_constant<int, 0>{}, [](auto) {});
            step(std::integral_constant<int, 1>{}, [&](auto slot_c) __attribute__((always_inline)) {
                constexpr int slot = decltype(slot_c)::value;
                if constexpr (slot == 27) make(g + 4, raw, in_next);
                if constexpr (slot == 29) raw = pair_raw(g + 5);
                if constexpr (slot >= 27 && slot < 31) asm volatile("" : "+s"(in_next[0]), "+s"(in_next[1]));
                if constexpr (slot == 31) {                     // behind the last reload that reads the window
                    w[0] = w[2]; w[1] = w[3]; w[2] = w[4]; w[3] = in[0]; w[4] = in[1];
                    in[0] = in_next[0]; in[1] = in_next[1];
#pragma unroll
                    for (int i = 0; i < 5; ++i) asm volatile("" : "+s"(w[i]));
                }
            });
        }
        if (kTeam <= 1) __syncthreads();          // the list in LDS has been read: the memory may become the staging tile (a team: below)
        // the last 16 keys of the last step (V_B of an odd step sits in ring slot 1)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int qq = 0; qq < 2; ++qq) oacc[t][qq] = mfma32(vb[1][4 + t], pb[qq][1], oacc[t][qq]);
        if (rescale_pending) rescale_out();
    }   // npairs > 0

    // accumulator i of d tile t <-> d = 32 t + 8 (i / 4) + 4 lh + i % 4, query 32 qq + lr.  A part is left in the register order that
    // merge_parts_kernel reads, that of the other kernel: its tile of 16 d, its 16 queries, its lane.
    auto part_place = [&](int t, int qq, int gq) -> int {
        return (((2 * t + (gq >> 1)) * 4 + 2 * qq + (lr >> 4)) * 64 + 16 * (2 * (gq & 1) + lh) + (lr & 15)) * 4;
    };
    if constexpr (kTeam > 1) {
        // ---- the wavefronts' sums together: sums[wave][register order], then maxima and row sums [wave][query].
        // 128 KB through LDS for a team of four, a microsecond; the rows leave from all wavefronts.
        float* const sums = reinterpret_cast<float*>(ost_bytes);
        float* const stats = sums + kTeam * kTile * kD;
        float inv[2], M[2], l_all[2];
        __syncthreads();                          // the list has been read
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            const float l = l_i[qq] + __shfl_xor(l_i[qq], 32);
            if (lh == 0) {
                stats[(2 * wave) * kTile + 32 * qq + lr] = m_i[qq];
                stats[(2 * wave + 1) * kTile + 32 * qq + lr] = l;
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int qq = 0; qq < 2; ++qq)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq)
                    *reinterpret_cast<float4*>(sums + wave * (kTile * kD) + (((t * 2 + qq) * 4 + gq) * 64 + lane) * 4) =
                        make_float4(oacc[t][qq][4 * gq], oacc[t][qq][4 * gq + 1], oacc[t][qq][4 * gq + 2], oacc[t][qq][4 * gq + 3]);
        __syncthreads();
        float factor[2][kTeam];
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            float m[kTeam];
#pragma unroll
            for (int v = 0; v < kTeam; ++v) m[v] = stats[(2 * v) * kTile + 32 * qq + lr];
            M[qq] = m[0];
#pragma unroll
            for (int v = 1; v < kTeam; ++v) M[qq] = fmaxf(M[qq], m[v]);
            l_all[qq] = 0.f;
#pragma unroll
            for (int v = 0; v < kTeam; ++v) {
                factor[qq][v] = m[v] > -INFINITY ? __builtin_amdgcn_exp2f(m[v] - M[qq]) : 0.f;      // a share without keys: no maximum, sums 0
                l_all[qq] += stats[(2 * v + 1) * kTile + 32 * qq + lr] * factor[qq][v];
            }
            inv[qq] = l_all[qq] > 0.f ? 1.0f / l_all[qq] : 0.f;
        }
        constexpr int kOwn = 4 / kTeam;           // tiles of d that a wavefront puts together
        float4 own[kOwn][2][4];
#pragma unroll
        for (int t = 0; t < kOwn; ++t)
#pragma unroll
            for (int qq = 0; qq < 2; ++qq)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                    for (int v = 0; v < kTeam; ++v) {
                        const float4 y = *reinterpret_cast<const float4*>(sums + v * (kTile * kD) + ((((wave * kOwn + t) * 2 + qq) * 4 + gq) * 64 + lane) * 4);
                        const float fw = factor[qq][v];
                        sum.x = fmaf(y.x, fw, sum.x); sum.y = fmaf(y.y, fw, sum.y); sum.z = fmaf(y.z, fw, sum.z); sum.w = fmaf(y.w, fw, sum.w);
                    }
                    own[t][qq][gq] = sum;
                }
        if (parts.count > 1) {
            float* const out = parts.buf + (int64_t)local * kPartFloats;
#pragma unroll
            for (int t = 0; t < kOwn; ++t)
#pragma unroll
                for (int qq = 0; qq < 2; ++qq)
#pragma unroll
                    for (int gq = 0; gq < 4; ++gq) *reinterpret_cast<float4*>(out + part_place(wave * kOwn + t, qq, gq)) = own[t][qq][gq];
            if (wave == 0 && lh == 0) {
#pragma unroll
                for (int qq = 0; qq < 2; ++qq) {
                    out[kTile * kD + 32 * qq + lr] = M[qq];
                    out[kTile * kD + kTile + 32 * qq + lr] = l_all[qq];
                }
            }
            return;
        }
        if (lse != nullptr && wave == 0 && lh == 0) {
#pragma unroll
            for (int qq = 0; qq < 2; ++qq) {
                const int64_t row = L.q_rows != nullptr ? out_rows[32 * qq + lr] : qrow0 + 32 * qq + lr;
                if (row >= 0) lse[(int64_t)bh * lse_S + row] = l_all[qq] > 0.f ? (M[qq] + __builtin_log2f(l_all[qq])) * kLn2 : -INFINITY;
            }
        }
        __syncthreads();                          // the sums have been read: the memory becomes the staging tile
#pragma unroll
        for (int qq = 0; qq < 2; ++qq)
#pragma unroll
            for (int t = 0; t < kOwn; ++t)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    const float4 y = own[t][qq][gq];
                    T out4[4] = {(T)(y.x * inv[qq]), (T)(y.y * inv[qq]), (T)(y.z * inv[qq]), (T)(y.w * inv[qq])};
                    *reinterpret_cast<uint2*>(ost + (32 * qq + lr) * kOutPitch + 32 * (wave * kOwn + t) + 8 * gq + 4 * lh) = *reinterpret_cast<uint2*>(out4);
                }
    } else {
        if (parts.count > 1) {
            float* const out = parts.buf + (int64_t)local * kPartFloats;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int qq = 0; qq < 2; ++qq)
#pragma unroll
                    for (int gq = 0; gq < 4; ++gq)
                        *reinterpret_cast<float4*>(out + part_place(t, qq, gq)) =
                            make_float4(oacc[t][qq][4 * gq], oacc[t][qq][4 * gq + 1], oacc[t][qq][4 * gq + 2], oacc[t][qq][4 * gq + 3]);
#pragma unroll
            for (int qq = 0; qq < 2; ++qq) {
                const float l = l_i[qq] + __shfl_xor(l_i[qq], 32);
                if (lh == 0) {
                    out[kTile * kD + 32 * qq + lr] = m_i[qq];
                    out[kTile * kD + kTile + 32 * qq + lr] = l;
                }
            }
            return;
        }
        // ---- combine the two key groups of every query, normalise
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            const float l = l_i[qq] + __shfl_xor(l_i[qq], 32), inv = l > 0.f ? 1.0f / l : 0.f;
            if (lse != nullptr && lh == 0) {
                const int64_t row = L.q_rows != nullptr ? out_rows[32 * qq + lr] : qrow0 + 32 * qq + lr;
                if (row >= 0) lse[(int64_t)bh * lse_S + row] = l > 0.f ? (m_i[qq] + __builtin_log2f(l)) * kLn2 : -INFINITY;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    T out4[4];
#pragma unroll
                    for (int jx = 0; jx < 4; ++jx) out4[jx] = (T)(oacc[t][qq][4 * gq + jx] * inv);
                    *reinterpret_cast<uint2*>(ost + (32 * qq + lr) * kOutPitch + 32 * t + 8 * gq + 4 * lh) = *reinterpret_cast<uint2*>(out4);
                }
        }
    }
    __syncthreads();
    // rows and pieces, then the stores: the LDS reads are all on their way before the first is waited for
    const int kc = threadIdx.x & 15, kr = threadIdx.x >> 4;
    constexpr int kRows = 4 * kTeam, kTurns = kTile / kRows;
    u32x4 pieces[kTurns];
    int32_t rows[kTurns];
#pragma unroll
    for (int i = 0; i < kTurns; ++i) {
        rows[i] = L.q_rows != nullptr ? out_rows[kr + kRows * i] : kr + kRows * i;
        pieces[i] = *reinterpret_cast<const u32x4*>(ost + (kr + kRows * i) * kOutPitch + kc * 8);
    }
#pragma unroll
    for (int i = 0; i < kTurns; ++i) asm volatile("" : "+v"(rows[i]), "+v"(pieces[i]));      // read here, not inside the branches below
#pragma unroll
    for (int i = 0; i < kTurns; ++i)
        if (rows[i] >= 0) *reinterpret_cast<u32x4*>(o + o_bh + ((L.q_rows != nullptr ? 0 : qrow0) + rows[i]) * L.o_st[2] + kc * 8) = pieces[i];
}

}  // namespace

hipError_t launch_fwd_few(const FragCall& c, const FragLayout& L, const Parts& parts, int items, int team, const FragGate* gate, int32_t* lists, uint32_t* list_lens,
                            uint32_t kv_bytes) {
    const dim3 grid((unsigned)(items * parts.count));
    const FragGate none = {};
#define BSA_FEW_W(T, WALK, TEAM, GATE)                                                                                                     \
    hipLaunchKernelGGL((fwd_few_kernel<T, WALK, TEAM, GATE>), grid, dim3(64 * TEAM), 0, c.st, (const T*)c.q, (const char*)c.kf, (const char*)c.vf, \
                       c.idx, c.lens, c.tile_valid, (T*)c.o, c.lse, c.Sq, c.Sk, c.bs_k, c.idx_stride, c.qk_scale, items, c.Hn, c.lse_rows, L, kv_bytes,  \
                       lists, list_lens, parts, gate != nullptr ? *gate : none)
#define BSA_FEW_G(T, TEAM, GATE)                                              \
    do {                                                                        \
        if (c.halves) BSA_FEW_W(T, kHalves, TEAM, GATE);                      \
        else if (c.bs_k == kTile) BSA_FEW_W(T, kTiles, TEAM, GATE);           \
        else BSA_FEW_W(T, kBlocks, TEAM, GATE);                               \
    } while (0)
#define BSA_FEW_T(T, TEAM)                                                    \
    do {                                                                        \
        if (gate != nullptr) BSA_FEW_G(T, TEAM, true);                        \
        else BSA_FEW_G(T, TEAM, false);                                       \
    } while (0)
#define BSA_FEW(TEAM)                                                         \
    do {                                                                        \
        if (c.dtype == BSA_BF16) BSA_FEW_T(__bf16, TEAM);                     \
        else BSA_FEW_T(_Float16, TEAM);                                       \
    } while (0)
    if (team == 4) BSA_FEW(4);
    else if (team == 2) BSA_FEW(2);
    else BSA_FEW(1);
#undef BSA_FEW
#undef BSA_FEW_T
#undef BSA_FEW_G
#undef BSA_FEW_W
    return hipGetLastError();
}

}  // namespace bsa
