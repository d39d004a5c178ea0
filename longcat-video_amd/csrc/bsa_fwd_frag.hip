// Block-sparse flash-attention forward for gfx950 (bf16 / fp16 MFMA) on K and V held in
// "fragment order".
//
// Why another layout.  The kernel of bsa_fwd.hip stages row-major K/V tiles in LDS, where every
// byte is written once and read twice (two wavefronts share each 32-key half): 96 KB of LDS
// traffic per 64 x 64 tile against 512 clocks of MFMA per SIMD, which makes LDS, not the matrix
// unit, its roofline.  Here a wavefront owns all 64 query rows of a work item, so every K and V
// fragment feeds four MFMAs (one per 16 query rows) and is needed by this wavefront alone: it is
// loaded from global memory straight into registers, in exactly the lane order the MFMA operand
// wants, and LDS carries nothing in the tile loop - no staging, no swizzle, no barrier.  That
// needs K and V in a layout whose every 1 KB is one operand fragment (below), written once per
// layer by prepare_kernel (bsa_prepare.hip) from the (T, H, W)-ordered tensors (a pass at HBM speed, which also
// replaces the zero-filled copies of the chunks at the padded high edge of the grid).
//
// Fragment order, per 64-key tile (16 KB for K, 16 KB for V; two 8 KB halves of 32 keys):
//   K: [half kh][d step c = 0..3][key block kb = 0..1][lane l = 0..63][8 elements]
//        element j of lane l = K[key 32 kh + 16 kb + (l & 15)][d = 32 c + 8 (l >> 4) + j]
//      = the A operand of v_mfma_f32_16x16x32 for S^T (16 keys x 16 queries) += K . Q^T.
//   V: [half kh][d tile t = 0..7][lane l][8 elements]
//        element j of lane l = V[key 32 kh + 16 (j >> 2) + 4 (l >> 4) + (j & 3)][d = 16 t + (l & 15)]
//      = the A operand of O^T (16 d x 16 queries) += V^T . P^T, with the 32 keys of a step in the
//        order in which the accumulator registers of S^T hold them, so that P^T needs no shuffle.
//
// 16x16x32 and not 32x32x16: the board's power is what bounds this kernel, and the small form moves half as many
// accumulators per multiplication (MFMAs alone on random data: 2 070 TFLOP/s against 1 850).  Calls that leave much of the chip
// idle are not bound by it and go to bsa_fwd_few.hip (frag_few).
//
// Work decomposition.  One wavefront (a workgroup of 64 threads, one per SIMD; two or four where
// they would be idle, see kTeam) = one work item =
// 64 query rows against its list of KV blocks, walked in steps of 32 keys (half a tile).  Per
// step: 32 MFMAs for S^T of the next step interleaved with the exp2 / row sum / rounding of the
// current one, then 32 MFMAs for O^T += V^T P^T interleaved with the row maximum of the next.
// K and V fragments of the following steps are in flight in register rings (two steps each).
// The output accumulators (128 registers) and the rings live in the 512-register file that a
// single wavefront per SIMD has to itself.
//
// Softmax: lazy running maximum as in bsa_fwd.hip, raised only when exceeded by 2^kTau, and for
// bf16 a form that takes no maxima where the norms bound the logits (kBounded); numerics
// follow flash_attn_bsa_varlen_mask.py:242-285: fp32 logits, scale * log2(e) applied after the
// dot, exp2, P rounded to the storage type for the P V product, fp32 row sum, one final rounding.
#include "bsa_frag.h"

namespace bsa {
namespace {

// ------------------------------------------------------------------ attention
// acc + x[2e]^2 + x[2e+1]^2 for a fragment of eight 16-bit values
__device__ __forceinline__ float dot2_self(bf16x8 x, int e, float acc) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 p = {x[2 * e], x[2 * e + 1]};
    return __builtin_amdgcn_fdot2_f32_bf16(p, p, acc, false);
}
__device__ __forceinline__ float dot2_self(f16x8 x, int e, float acc) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 p = {x[2 * e], x[2 * e + 1]};
    return __builtin_amdgcn_fdot2(p, p, acc, false);
}

// Lists of at most this many entries are staged in LDS for the next work item while the current one runs.
constexpr int kPipeList = 256;

// A workgroup (one wavefront) runs the work items b, b + round, b + 2 round, ... of its launch one after the other
// (or draws them from its XCD's queue).  What an item needs before its first MFMA - its list, its Q rows, its first K and
// V fragments - is requested while the item before it still runs, so that an item costs its tile walk and an
// epilogue, not a chain of three dependent memory round trips:
//   * lens and the first list entry of the item after next are scalar loads issued at the start of an item;
//   * the next item's list goes into registers at the start of an item and into its LDS buffer at the end;
//   * the next item's Q rows go from global memory straight into an LDS staging tile (LDS DMA) and from there into
//     the Q registers once the current item's last S^T product has been issued;
//   * the positions of the tile walk behind the end of the list name the next item's first tile, so the fragment
//     rings hold K(0), K(1), V(0) of the next item when the loop ends - what its prologue would load.
// K and V fragments are read through buffer resources (an SGPR base, a 32-bit scalar tile offset, the lane's
// 16 bytes): no 64-bit vector address arithmetic in the loop, and an offset outside the buffer reads zeros.
// kBounded: the kernel for items whose logits are bounded below the level at which the running maximum would move
// (see where the bound is tested): its steps take no row maxima.  An item that fails the test is not computed but
// appended to `fallback` (its count in fallback_count), and the other instantiation, which takes its items from that
// list, runs behind it.
// The schedule for lists of unequal length: a queue per XCD.  Section x holds the items [section_begin(x), section_begin(x + 1))
// of the call, a contiguous run of query tiles, and workgroup b draws from section b % 8, the XCD it runs on.
constexpr int kQueues = 8, kQueueChoice = kQueues, kQueueWords = kQueues + 1;      // a counter per section, the choice of schedule
static_assert(kQueueWords <= kFragQueueWords, "the caller's buffer holds the words");
__device__ __forceinline__ int section_begin(int n, int x) { return (int)(((int64_t)n * x) >> 3); }

// kTeam: 0, one wavefront a workgroup, which runs one item after another as above; otherwise a workgroup runs one item, with
// nothing prepared ahead and none of the code for it, as wavefronts that have a SIMD of a compute unit each.  1: a call of one
// round.  2, 4: a team.  Each of its wavefronts walks a share of the item's pairs (of a part's
// share, where the item is in parts as well) from the list that they stage together; then their sums are put together in LDS, in the
// order of the shares, wavefront w those of its 8 / kTeam tiles of d, and the rows leave from all of them.  For the items behind whole
// rounds, and calls that teams of two fill the chip with: see choose_split.
// kGate: the item's list does not exist yet (FragGate).  `fallback` and `fallback_count` are then where the lists ([BH][nbq][width]) and their
// lengths go, null: nowhere.  (As arguments of their own they would be 392 bytes, beyond what is asked for together, and two arguments that
// the kernel can do without in their place cost the layers 0.3 to 0.7 %, by where the loop then lies.)
// The first of a step's 96 pieces (six a pair, nine instructions' time) that stands behind MFMA g or a later one, in the kernel with maxima.
constexpr int first_piece(int g) {
    for (int p = 0; p < 96; ++p) {
        constexpr int before[6] = {0, 2, 3, 4, 6, 7};
        const int t = 9 * (p / 6) + before[p % 6];
        if ((t < 126 ? t * 48 / 126 : 48 + (t - 126) * 16 / 18) >= g) return p;
    }
    return 96;
}

template <typename T, int kWalk, bool kBounded, int kTeam, bool kGate>
// At a page: the queues' kernel, the same instructions, took 1 252 us of a call (16 heads of 20x30x52 by the CDF rule) at 0x500 of one and 1 245 at
// its start, where the linker had put it until other kernels left this file.  Level elsewhere.
__attribute__((aligned(4096))) __global__ __launch_bounds__(kTeam > 1 ? 64 * kTeam : 64, 1) void fwd_frag_kernel(
    const T* __restrict__ q, const char* __restrict__ kf, const char* __restrict__ vf,
    const int32_t* __restrict__ idx, const int32_t* __restrict__ lens, const uint64_t* __restrict__ tile_valid,
    T* __restrict__ o, float* __restrict__ lse, int64_t Sq, int64_t Sk, int bs_q, int bs_k, int idx_stride,
    float qk_scale, int item_begin, int item_end, int round, int Hn, int64_t lse_S, FragLayout L,
    const int32_t* __restrict__ order, uint32_t* __restrict__ queue, const uint32_t* __restrict__ gate, uint32_t gate_want,
    int bh_first, uint32_t kv_span_bytes, int q_offsets_32, const float* __restrict__ key_norm,
    int32_t* __restrict__ fallback, uint32_t* __restrict__ fallback_count, Parts parts, FragGate G) {
    typedef typename Vec8<T>::type V8;
    constexpr bool kOnce = kTeam > 0;
    static_assert(!kGate || kOnce, "a workgroup that selects has one item");
    // log2 headroom before the running maximum is raised: probabilities reach 2^kTau, which the storage type of P
    // must hold (fp16 ends at 65 504) and the fp32 sums must hold times the number of keys
    constexpr float kTau = std::is_same<T, _Float16>::value ? 14.0f : 30.0f;
    // How far the fixed reference of an item without row maxima may lie above the largest logit of its first keys (see
    // where the bound is tested): the largest probability of a row is then at least 2^-kSlack, which costs bf16 no bit (it
    // has fp32's exponents).  fp16 has none to spare - a probability below 2^-14 is subnormal - and always looks at the
    // maxima: RMS-normalised rows bound their logits at 16.3, beyond its headroom, so they would all fail a test without
    // slack and be computed behind the rounds, one list after another (16 heads of 13x30x53 in 4x4x8 chunks: 743 us
    // with the maxima, 822 with the test and no slack, 723 with a slack of 4, which left subnormal probabilities four bits
    // fewer).
    constexpr float kSlack = 60.0f;
    static_assert(!kBounded || std::is_same<T, __bf16>::value, "fp16 probabilities need the running maximum");
    static_assert(!kBounded || kTeam == 0, "a call of one round leaves nothing to another launch");
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    // six lines: 0.36 us for the first five where one by one they took 0.7 to 1.1; with the sixth a call of two prompts of 8 heads,
    // 7x15x26, takes 41.4 us for 41.9.  With what an item that nothing has prepared asks for at once (below) and the divisions
    // that went, the kernel of a single round is 1.3 us shorter: 15.1 -> 13.8 us for 5 heads of 9x27x12, 25.4 -> 24.2 for two
    // prompts of 8 heads of 7x15x26.
    touch_arguments<decltype(fwd_frag_kernel<T, kWalk, kBounded, kTeam, kGate>)>();
    if (gate != nullptr && *gate != gate_want) return;
    // output staging: 64 rows of 256 B, 272 B apart.  The same memory stages a list that is too long for the small
    // buffers (kListEntries words at most) during the tile loop of an item that was not prepared ahead of time.
    constexpr int kOutPitch = kD + 8;
    // A team has its list there, then the wavefronts' sums, then the rows of the output.
    constexpr int kOutBytes = kTile * kOutPitch * (int)sizeof(T);
    __shared__ __attribute__((aligned(16))) char ost_bytes[kTeam > 1 ? kTeamBytes<kTeam> : kOutBytes];
    T* const ost = reinterpret_cast<T*>(ost_bytes);
    constexpr int kWords = kWalk == kHalves ? 2 : 1;              // list words of a pair
    __shared__ __attribute__((aligned(8))) uint32_t lists[2][kOnce ? 2 : kPipeList * kWords];
    __shared__ int32_t out_rows[2][kTile];       // token rows of this and the next item's 64 query slots (row table given)
    __shared__ __attribute__((aligned(16))) char qstage[kOnce ? 16 : kTileBytes];      // Q of the next item, in register order
    __shared__ __attribute__((aligned(16))) char scale_room[kBounded ? 16 : kTeam > 1 ? 1024 * kTeam : 1024];
    uint32_t* const big = reinterpret_cast<uint32_t*>(ost);

    const int lane = threadIdx.x & 63;
    const int wave = kTeam > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
    const int lr = lane & 15, lg = lane >> 4;
    const int nqt = (int)(Sq / kTile);
    const int nsub = kWalk == kBlocks ? bs_k / kTile : 1, nsub_of_block = bs_k / kTile;
    const int tiles_bh = (int)(Sk / kTile), nbk = kWalk == kBlocks ? tiles_bh / L.by_sub : tiles_bh;     // kHalves does not ask for it
    const uint32_t lane_off = (uint32_t)lane * 16u;
    // the kernel that runs the fallback list takes as many items as the list holds
    const int n_launch = kBounded ? item_end - item_begin : parts.count > 1 ? parts.count * parts.items
                                  : (!kGate && fallback_count != nullptr ? __builtin_amdgcn_readfirstlane((int)min(*fallback_count, (uint32_t)(item_end - item_begin)))
                                                               : item_end - item_begin);

    const int64_t kv_bh_bytes = (int64_t)tiles_bh * kTileBytes;
    const __amdgpu_buffer_rsrc_t krs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kf) + bh_first * kv_bh_bytes, 0, (int)kv_span_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(vf) + bh_first * kv_bh_bytes, 0, (int)kv_span_bytes, 0x00020000);
    // at: byte offset of a 32-key half, counted from (batch, head) bh_first; c / f: fragment of the half
    auto k_frag = [&](uint32_t at, int c) -> V8 {
        return __builtin_bit_cast(V8, __builtin_amdgcn_raw_buffer_load_b128(krs, lane_off + (uint32_t)((c & 3) * 1024), at + (uint32_t)((c >> 2) * 4096), 0));
    };
    auto v_frag = [&](uint32_t at, int f) -> V8 {          // f: d tile
        return __builtin_bit_cast(V8, __builtin_amdgcn_raw_buffer_load_b128(vrs, lane_off + (uint32_t)((f & 3) * 1024), at + (uint32_t)((f >> 2) * 4096), 0));
    };

    // ---- which items this workgroup runs
    // The launch's items are taken in rounds of `round` (a multiple of 8).  Workgroup b runs on XCD b % 8: within
    // a round every XCD takes a contiguous run of the round's items.
    auto round_local = [&](int r) -> int {
        const int64_t r0 = (int64_t)r * round;
        if (r0 >= n_launch) return -1;
        const int n = min(round, n_launch - (int)r0), w = blockIdx.x, x = w & 7;
        if (w >= n) return -1;
        return (int)r0 + x * (n >> 3) + min(x, n & 7) + (w >> 3);
    };
    // From the queues (queue_plan_kernel): the section of this workgroup's XCD first, then what the others have left.
    int section_turn = 0;
    auto draw = [&]() -> int {
#pragma unroll 1
        for (; section_turn < kQueues; ++section_turn) {
            const int x = (blockIdx.x + section_turn) & (kQueues - 1);
            const int begin = section_begin(n_launch, x), n = section_begin(n_launch, x + 1) - begin;
            uint32_t drawn = 0;
            if (lane == 0) drawn = atomicAdd(queue + x, 1u);
            const uint32_t l = (uint32_t)__builtin_amdgcn_readfirstlane((int)drawn);
            if (l < (uint32_t)n) return begin + (int)l;
        }
        return -1;
    };
    int rounds_taken = 0;
    auto next_local = [&]() -> int { return !kOnce && queue != nullptr ? draw() : round_local(rounds_taken++); };
    // what is known of an item ahead of time: its number, the length of its list and its first entry (both as
    // they lie in memory; they are clamped where they are used)
    struct Desc { int item, nent, ent[2], local; float kn; };       // ent: the first list entry (kHalves: the first two)
    auto fetch = [&](int local) -> Desc {
        Desc d = {-1, 0, {0, 0}, local, INFINITY};
        if (local < 0) return d;
        if (!kBounded && kTeam != 1 && parts.count > 1) local -= local / parts.by_items * parts.items;
        d.item = order != nullptr ? item_begin + order[local] : item_at(L, item_begin + local, nqt);
        if (kGate) return d;
        const int64_t row = d.item / L.by_block;
        d.nent = lens[row];
        if (idx_stride > 0) {
            d.ent[0] = idx[row * idx_stride];
            if (kWalk == kHalves) d.ent[1] = idx[row * idx_stride + 1];
        }
        if (key_norm != nullptr) d.kn = key_norm[d.item / L.by_tiles];
        return d;
    };
    // The descriptor's loads are vector loads of one address (behind the stores of an earlier item the compiler
    // does not use the scalar cache): the values are the same in every lane and are made scalars where they are used,
    // not where they are loaded, so that the wait for them stands there.
    auto uni = [](int x) -> int { return __builtin_amdgcn_readfirstlane(x); };
    // list words in use
    auto list_length = [&](const Desc& d) -> int {
        if (d.item < 0) return 0;
        const int n = min(max(uni(d.nent), 0), idx_stride);
        return kWalk == kHalves ? (n + 1) & ~1 : min(n, kListEntries);
    };
    // the pair of halves that position 0 of d's walk names
    auto first_pair = [&](const Desc& d, uint32_t (&h)[2]) {
        const uint32_t base = (uint32_t)((d.item / L.by_tiles - bh_first) * tiles_bh) * 2u;
        if (kWalk == kHalves) {
            h[0] = base + ((uint32_t)uni(d.ent[0]) & kHalfId);
            h[1] = base + ((uint32_t)uni(d.ent[1]) & kHalfId);
        } else {
            h[0] = base + (uint32_t)(min(max(uni(d.ent[0]), 0), nbk - 1) * nsub) * 2u;
            h[1] = h[0] + 1u;
        }
    };

    // ---- registers that live across items
    V8 qreg[4][4];                                             // [16 queries][d step]
    // Register rings: K and V fragments of two steps.
    V8 kb[2][8], vb[2][8];
    f32x4_ s[2][2][4];                                         // S^T of the current and of the next step: [][key block][16 queries]
    V8 pb[4];                                                  // P^T as B operand, by 16 queries
    f32x4_ oacc[8][4];
    float m_i[4], l_i[4];
    // Softmax state per 16 queries: running maximum m_i (scaled, log2 units), its negative for the exponent
    // (0 while the maximum is -inf), and the unscaled logit above which the maximum has to be raised; the lowest of these.
    float neg_m[4], raise_at[4], raise_low;
    const float inv_scale = 1.0f / qk_scale;
    // Raising the
    // maximum has two parts.  Here: the new maximum, the exponent offset, the row sum (which already holds
    // every probability of the current step).  The output accumulators are rescaled one quarter of a step later
    // (rescale_out, behind slot 7 of the next step): the products of the current step's queries 32 .. 63, whose
    // probabilities were taken relative to the old maximum, are only issued in slots 0 .. 7 of that step.
    float alpha_p[4];
    bool rescale_pending = false;

    // Q fragments of 16 queries into their registers, and the lane's part of the rows' squared norms.  All of Q is
    // read by the assembly MFMAs from accumulation registers.  The values pass through an assembly statement that
    // ties them to that register class: a value that C++ code also reads (the squares) the compiler would keep in
    // ordinary registers and copy in front of every MFMA that names it, without the wait states such a copy needs.
    float q_sq[4] = {0.f, 0.f, 0.f, 0.f};
    auto take_q = [&](int qb, V8 (&rows)[4]) {
        float sq = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) sq = dot2_self(rows[c], e, sq);
        q_sq[qb] = sq;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            asm volatile("" : "=a"(qreg[qb][c]) : "0"(rows[c]));
        }
    };
    // a sum or a maximum over the four lanes that share a query
    auto over_lanes = [](float x, auto f) -> float {
        const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        const float y = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
        const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
        return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
    };
    const auto add = [](float a, float b) { return a + b; };

    // ---- per item
    int npairs = 0, pair0 = 0;       // the walk covers the pairs pair0 .. pair0 + npairs - 1 of the list
    int n_halves = 0;                // a team's walk over halves: those of this wavefront's share, from ents on
    uint32_t half_base = 0;          // first half of the item's (batch, head)
    uint32_t beyond[2] = {0, 0};     // the entries of the positions behind the end of the list
    const uint32_t* ents = big;      // the item's list in LDS
    // window of the walk: the entries of the halves 2 g + 1 .. 2 g + 5 of loop iteration g (one pair per iteration).  An entry is a half,
    // counted from half_base, | real keys << 20, as kHalves lists hold them; what is above 2^19 halves is lost in the shift to
    // bytes.
    uint32_t w[5];
    auto offset_of = [&](uint32_t entry) -> uint32_t { return (entry << 13) + (half_base << 13); };
    static_assert(kHalfBytes == 1 << 13, "the shift");

    // Pair tp of the walk -> its entries.  Positions behind the list name `beyond`, no key of theirs.  The list is read from LDS
    // (pair_raw, to be issued early) and made into entries later.
    struct Raw { uint32_t e[kWords]; };
    auto pair_raw = [&](int tp) -> Raw {
        const int tc = min(tp, npairs - 1) + pair0;
        Raw r;
        if constexpr (kWalk == kHalves && kTeam > 1) {
            r.e[0] = ents[2 * tc];
            r.e[1] = ents[min(2 * tc + 1, n_halves - 1)];
            if (2 * tc + 1 >= n_halves) r.e[1] &= kHalfId;      // an odd share: its last half once more, no key of it
        } else if constexpr (kWalk == kHalves) {
            const uint2 x = *reinterpret_cast<const uint2*>(ents + 2 * tc);               // the same address in every lane
            r.e[0] = x.x; r.e[1] = x.y;
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
            e[0] = beyond[0];
            e[1] = beyond[1];
        } else if (kWalk == kHalves) {
#pragma unroll
            for (int x = 0; x < kWords; ++x) e[x] = (uint32_t)uni((int)raw.e[x]);
        } else {
            // the same word in every lane; made a scalar by hand (behind the stores of an earlier item's output the
            // compiler reads it with a vector load)
            const uint32_t lo = (uint32_t)uni((int)(uint32_t)word), hi = (uint32_t)uni((int)(uint32_t)(word >> 32));
            const int n = __builtin_popcountll((uint64_t)lo | ((uint64_t)hi << 32));
            e[0] = half | (uint32_t)min(n, 32) << kHalfCountShift;
            e[1] = (half + 1u) | (uint32_t)max(n - 32, 0) << kHalfCountShift;
        }
    };
    // accumulator i of key block kk <-> key 16 kk + 4 lg + i of the step's 32 keys, query lr (+16, 32, 48)
    auto mask_pair = [&](f32x4_ (&sv)[2][4], uint32_t entry) {
        if (__builtin_expect(entry < 32u << kHalfCountShift, 0)) {
            asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");       // the MFMAs into these accumulators have retired
            // the lane's part of the shift first: the tests below then use constants, not eight per-lane bit masks
            // that would have to be kept in registers (or spilled) all through the loop for this rare path
            uint32_t mine = ((1u << (entry >> kHalfCountShift)) - 1u) >> (4 * lg);
            asm volatile("" : "+v"(mine));
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (!((mine >> (16 * kk + i)) & 1u)) {
#pragma unroll
                        for (int qb = 0; qb < 4; ++qb) sv[kk][qb][i] = -INFINITY;
                    }
        }
    };
    // mx: this lane's unscaled maxima over its 8 accumulators per query of the step that comes next.  The test
    // needs no exchange between the four key groups of a query: some lane exceeds the limit exactly when the
    // combined maximum does.
    auto raise_max = [&](const float (&mx)[4]) __attribute__((always_inline)) {
        if (!__any(mx[0] > raise_at[0] || mx[1] > raise_at[1] || mx[2] > raise_at[2] || mx[3] > raise_at[3])) return;
#pragma unroll
        for (int qb = 0; qb < 4; ++qb) {
            const float m_new = fmaxf(m_i[qb], over_lanes(mx[qb], [](float a, float b) { return fmaxf(a, b); }) * qk_scale);
            const float alpha = __builtin_amdgcn_exp2f(m_i[qb] - ((m_new == -INFINITY) ? 0.f : m_new));
            m_i[qb] = m_new;
            neg_m[qb] = (m_new == -INFINITY) ? 0.f : -m_new;
            raise_at[qb] = (m_new + kTau) * inv_scale;
            l_i[qb] *= alpha;
            alpha_p[qb] = alpha;
        }
        raise_low = fminf(fminf(raise_at[0], raise_at[1]), fminf(raise_at[2], raise_at[3]));
        rescale_pending = true;
    };
    auto lane_max = [&](const f32x4_ (&sv)[2][4], float (&mx)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int qb = 0; qb < 4; ++qb) {
            mx[qb] = fmaxf(sv[0][qb][0], sv[0][qb][1]);
            mx[qb] = fmaxf(fmaxf(mx[qb], sv[0][qb][2]), sv[0][qb][3]);
            mx[qb] = fmaxf(fmaxf(mx[qb], sv[1][qb][0]), sv[1][qb][1]);
            mx[qb] = fmaxf(fmaxf(mx[qb], sv[1][qb][2]), sv[1][qb][3]);
        }
    };
    // The output accumulators live in AGPRs, which the VALU cannot multiply in place.  Each goes through LDS and back into the
    // registers it came from, so that this rare path does not make the compiler reserve registers for copies of
    // them (element by element through moves it did, 220 to 340 of them, in scratch memory).
    auto rescale_out = [&]() __attribute__((always_inline)) {
        asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");   // the last MFMA into the accumulators has retired
        const uint32_t at = lds_address(scale_room) + threadIdx.x * 16u;
        static_for<32>([&](auto n_c) {
            constexpr int n = decltype(n_c)::value, qb = n & 3, t = n >> 2;
            f32x4_ y;
            asm volatile("ds_write_b128 %1, %2\n\ts_waitcnt lgkmcnt(0)\n\tds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(y) : "v"(at), "a"(oacc[t][qb]) : "memory");
            y *= alpha_p[qb];
            asm volatile("ds_write_b128 %1, %2\n\ts_waitcnt lgkmcnt(0)\n\tds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "+a"(oacc[t][qb]) : "v"(at), "v"(y) : "memory");
        });
        asm volatile("s_nop 7" ::: "memory");                        // AGPR writes before the next MFMA reads them
        rescale_pending = false;
    };

    // Step u = 2 g + j (j static).  On entry S(u) is complete and the running maximum covers it; the P of queries 32 .. 63 of
    // step u-1 are complete.  The 64 MFMAs of a step, in issue order (32 "slots" of two):
    //    0 ..  7   O^T += V(u-1)^T P(u-1)^T      queries 32 .. 63 of the previous step, a tile of d a slot
    //    8 .. 23   S(u+1)^T = K(u+1) Q^T         a fragment of K in two slots
    //   24 .. 31   O^T += V(u)^T P(u)^T          queries 0 .. 31 of this step
    // The VALU work on S(u) - per pair of accumulators two fma, two exp2, two additions for the row sum and one
    // rounding of the pair to the storage type, 16 pairs - is cut into pieces that go between the MFMAs so that
    // no gap holds more than two MFMAs last: the first 14 pairs behind slots 0 .. 23 (the eight pairs of queries 0 .. 31
    // first: they are complete well before slot 24), the last two behind slots 24 .. 31 together with the row
    // maximum of S(u+1), which is complete by then.  A fragment register is reloaded behind the last MFMA that reads it: V(u+1)
    // behind slots 0 .. 7, a step and a half before it is used, K(u+3) behind slots 9 .. 23, two steps.
    // `between` puts scalar work of the walk behind the slots.
    auto step = [&](auto jj, auto between) __attribute__((always_inline)) {
        constexpr int j = decltype(jj)::value;
        constexpr int sc = j & 1, sn = sc ^ 1;                 // S(u) and S(u+1) alternate between two register sets
        constexpr int kslot = (j + 1) & 1;                     // ring slot of K(u+1), then of K(u+3)
        constexpr int vprev = (j + 1) & 1, vcur = j & 1;       // ring slots of V(u-1), then V(u+1), and of V(u)
        // pair n: queries 16 qb .. with qb = 2 (n >> 3) + (n & 1), keys 2 ((n >> 1) & 3), + 1 of the lane's eight.  Its instructions go in
        // six: an exponential, an argument of the next pair, the sum of the pair before; the other exponential, the other argument, and
        // the pair before added to the row sum and rounded.  (The result of a transcendental instruction cannot be consumed by the
        // next instruction without a wait state.)
        float fx[2][2], pa[2][2], both;
        auto argument = [&](int m, int e) {
            const int qb = 2 * (m >> 3) + (m & 1), i = 2 * ((m >> 1) & 3);
            fx[m & 1][e] = fmaf(s[sc][i >> 2][qb][(i & 3) + e], qk_scale, neg_m[qb]);
            asm volatile("" : "+v"(fx[m & 1][e]));
        };
        auto piece = [&](int p) {                               // p = 0 .. 97
            const int n = p / 6, r = p % 6, m = n - 1;
            if ((r == 0 || r == 3) && n < 16) {
                pa[n & 1][r == 3] = __builtin_amdgcn_exp2f(fx[n & 1][r == 3]);
                asm volatile("" : "+v"(pa[n & 1][r == 3]));
            } else if ((r == 1 || r == 4) && n < 15) {
                argument(n + 1, r == 4);
            } else if (((r == 2 && n < 16) || p == 96) && m >= 0) {
                both = pa[m & 1][0] + pa[m & 1][1];
                asm volatile("" : "+v"(both));
            } else if (((r == 5 && n < 16) || p == 97) && m >= 0) {
                const int qb = 2 * (m >> 3) + (m & 1), i = 2 * ((m >> 1) & 3);
                l_i[qb] += both;
                pb[qb][i] = (T)pa[m & 1][0];
                pb[qb][i + 1] = (T)pa[m & 1][1];
                asm volatile("" : "+v"(l_i[qb]), "+v"(pb[qb]));
            }
        };
        // Behind MFMA g of 64.  An instruction takes four clocks of issue and an exponential eight; an MFMA sixteen in its pipe.
        // Without maxima a pair takes four gaps - of an exponential, two instructions, an exponential, three - and everything fits; with
        // them 14 pairs stand in the first 48 gaps, which leaves the last 16 room for the maxima of S(u+1).
        auto gap = [&](auto g_c) __attribute__((always_inline)) {
            constexpr int g = decltype(g_c)::value;
            if constexpr (g == 0) { argument(0, 0); argument(0, 1); }
            if constexpr (kBounded) {
                constexpr int p0 = 6 * (g >> 2), r = g & 3;
                if constexpr (r == 0) piece(p0);
                if constexpr (r == 1) { piece(p0 + 1); piece(p0 + 2); }
                if constexpr (r == 2) piece(p0 + 3);
                if constexpr (r == 3) { piece(p0 + 4); piece(p0 + 5); }
            } else {
                constexpr int from = first_piece(g), to = first_piece(g + 1);
                static_for<to - from>([&](auto p_c) { piece(from + decltype(p_c)::value); });
            }
            if constexpr (g == 63) { piece(96); piece(97); }
        };
        float highest = 0.f;                                    // of this lane's 32 accumulators of S(u+1), value n: key n / 4, queries n % 4
        auto next_s = [&](int n) { return s[sn][n >> 4][n & 3][(n >> 2) & 3]; };
        __builtin_amdgcn_sched_barrier(0);
        static_for<32>([&](auto slot_c) {
            constexpr int slot = decltype(slot_c)::value;
            // ---- the MFMAs of this slot
            if constexpr (slot == 0) asm volatile("s_nop 1");       // the last of pb[3] was written in front of this step
            if constexpr (slot < 8) {
                mfma_acc16(oacc[slot][2], vb[vprev][slot], pb[2]);
                __builtin_amdgcn_sched_barrier(0);
                gap(std::integral_constant<int, 2 * slot>{});
                __builtin_amdgcn_sched_barrier(0);
                mfma_acc16(oacc[slot][3], vb[vprev][slot], pb[3]);
            } else if constexpr (slot < 24) {
                constexpr int f = (slot - 8) >> 1, c = f >> 1, kk = f & 1, qb = 2 * (slot & 1);      // d step, key block
                mfma_s16<c == 0>(s[sn][kk][qb], kb[kslot][f], qreg[qb][c]);
                __builtin_amdgcn_sched_barrier(0);
                gap(std::integral_constant<int, 2 * slot>{});
                __builtin_amdgcn_sched_barrier(0);
                mfma_s16<c == 0>(s[sn][kk][qb + 1], kb[kslot][f], qreg[qb + 1][c]);
            } else {
                constexpr int t = slot - 24;
                mfma_acc16(oacc[t][0], vb[vcur][t], pb[0]);
                __builtin_amdgcn_sched_barrier(0);
                gap(std::integral_constant<int, 2 * slot>{});
                __builtin_amdgcn_sched_barrier(0);
                mfma_acc16(oacc[t][1], vb[vcur][t], pb[1]);
            }
            // ---- reloads, one by one behind the last MFMA that reads a fragment: V(u+1), K(u+3)
            if constexpr (slot < 8) vb[vprev][slot] = v_frag(offset_of(w[j]), slot);
            if constexpr (slot >= 8 && slot < 24 && slot % 2 == 1) kb[kslot][(slot - 9) / 2] = k_frag(offset_of(w[j + 2]), (slot - 9) / 2);
            if constexpr (slot == 7) {
                if (__builtin_expect(rescale_pending, 0)) rescale_out();
            }
            gap(std::integral_constant<int, 2 * slot + 1>{});
            if constexpr (slot >= 24) {
                constexpr int r = slot - 24;                    // 0 .. 7
                if constexpr (r == 1) {
#pragma unroll
                    for (int x = 0; x < 8; ++x) mfma_chain_end(s[sn][x >> 2][x & 3]);
                    mask_pair(s[sn], w[j]);                    // the keys of step u + 1
                    if constexpr (!kBounded) highest = fmaxf(fmaxf(next_s(0), next_s(1)), next_s(2));
                }
                if constexpr (!kBounded && r >= 2) {            // the other 29, five or four a slot
                    constexpr int from = 3 + (29 * (r - 2) + 5) / 6, to = 3 + (29 * (r - 1) + 5) / 6;
#pragma unroll
                    for (int n = from; n < (to < 32 ? to : 32); ++n) highest = fmaxf(highest, next_s(n));
                }
            }
            between(slot_c);
            __builtin_amdgcn_sched_barrier(0);
        });
        // One test for all queries, of the highest value and the lowest limit, seldom met; then of each query's own.
        if constexpr (!kBounded) {
            if (__builtin_expect(__any(highest > raise_low), 0)) {
                float mx[4];
                lane_max(s[sn], mx);
                raise_max(mx);
            }
        }
    };

    // ---- the workgroup's items
    Desc cur = {-1, 0, {0, 0}, -1, INFINITY}, nxt = cur;
#pragma unroll 1
    for (int i = 0; i < (kOnce ? 1 : 2); ++i) {        // one copy of the code: a launch's first item pays for every line of it, cold
        cur = nxt;
        nxt = fetch(next_local());
    }
    if (kOnce) cur = nxt;
    bool prepared = false;           // the current item's list, Q rows and first fragments were requested by the item before it
    int list_buf = 0;                // which of the small list buffers holds the current item's list, if prepared
    while (uni(cur.item) >= 0) {
        cur.item = uni(cur.item);
        const Desc nx2 = kOnce ? cur : fetch(next_local());      // in flight while this item runs
        const int bh = cur.item / L.by_tiles;
        const int qtile = cur.item - bh * nqt;
        const int64_t qrow0 = (int64_t)qtile * kTile;
        const int batch = bh / L.by_heads;
        const int64_t o_bh = (int64_t)batch * L.o_st[0] + (int64_t)(bh - batch * Hn) * L.o_st[1];
        // the token rows of an item that nothing has prepared: asked for beside its descriptor
        int32_t first_rows[5] = {0, 0, 0, 0, 0};
        if (!prepared && L.q_rows != nullptr) {
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) first_rows[qb] = L.q_rows[qrow0 + 16 * qb + lr];
            first_rows[4] = L.q_rows[qrow0 + lane];
        }
        // ... and so is a team's list, as far as one entry a thread goes (what lies behind its end is not used)
        int32_t team_entry = 0;
        if (kOnce && !kGate && idx_stride > 0) team_entry = idx[(int64_t)(cur.item / L.by_block) * idx_stride + min((int)threadIdx.x, idx_stride - 1)];
        __builtin_amdgcn_sched_barrier(0);
        int nent = list_length(cur);
        npairs = uni(kWalk == kHalves ? nent >> 1 : nent * nsub);
        if (!kOnce && !kBounded && parts.count > 1) {
            const int part = cur.local / parts.by_items;        // at most kMaxParts: the products fit 32 bits
            pair0 = npairs * part / parts.by_count;
            npairs = npairs * (part + 1) / parts.by_count - pair0;
        }
        half_base = (uint32_t)uni((bh - bh_first) * tiles_bh) * 2u;
        // the next item can be prepared while this one runs if this one has a loop to hide it behind, the next one
        // has a first tile to point the walk at, a list that fits a small buffer, and Q rows the LDS DMA can address
        const int next_nent = list_length(nxt);
        // (an item in parts has no first pair that is known ahead)
        const bool prepare_next = !kOnce && (kBounded || parts.count == 1) && nxt.item >= 0 && npairs > 0 && next_nent > 0 && next_nent <= kPipeList * kWords && q_offsets_32 != 0;
        beyond[0] = beyond[1] = 0;
        if (prepare_next) {
            first_pair(nxt, beyond);
#pragma unroll
            for (int x = 0; x < 2; ++x) beyond[x] = (uint32_t)uni((int)(beyond[x] - half_base)) & kHalfId;
        }
        const int nitem = prepare_next ? nxt.item : 0, nbh = nitem / L.by_tiles;
        const int64_t nqrow0 = (int64_t)(nitem - nbh * nqt) * kTile;
        const int32_t* nlist = idx + (int64_t)(nitem / L.by_block) * idx_stride;

        const bool early = (kTeam == 1 && !kGate) || (!kOnce && (kBounded || parts.count == 1));         // the walk starts at the list's first entry
        auto first_fragments = [&](uint32_t h0, uint32_t h1) {
#pragma unroll
            for (int c = 0; c < 8; ++c) kb[0][c] = k_frag(h0 << 13, c);                 // K(0)
#pragma unroll
            for (int c = 0; c < 8; ++c) kb[1][c] = k_frag(h1 << 13, c);                 // K(1)
#pragma unroll
            for (int f = 0; f < 8; ++f) vb[0][f] = v_frag(h0 << 13, f);                 // V(0)
        };
        if (!prepared) {
            // Nothing of this item is on its way yet.  Everything that its first product waits for is asked for before any of
            // it is waited for: the list, Q as the B operand of S^T (lane holds rows lr, 16 + lr, ..., d = 32 c + 8 lg .. +8) and,
            // where the walk starts at the list's first entry, which the descriptor holds, the first K and V fragments.
            int lane_now = lane;                                     // see the epilogue
            asm volatile("" : "+v"(lane_now));
            const int32_t* list = idx + (int64_t)(cur.item / L.by_block) * idx_stride;
            constexpr int kAhead = 4;
            int32_t entry[kAhead] = {0, 0, 0, 0};
            if (!kOnce && nent > 0) {
#pragma unroll
                for (int e = 0; e < kAhead; ++e) entry[e] = list[min(lane_now + 64 * e, nent - 1)];
            }
            const int64_t q_bh = (int64_t)batch * L.q_st[0] + (int64_t)(bh - batch * Hn) * L.q_st[1];
            V8 rows[4][4];
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) {
                const int64_t row = L.q_rows != nullptr ? (int64_t)max(first_rows[qb], 0) : qrow0 + 16 * qb + lr;      // padded slots read token 0, never stored
                const T* qp = q + q_bh + row * L.q_st[2] + 8 * lg;
#pragma unroll
                for (int c = 0; c < 4; ++c) rows[qb][c] = *reinterpret_cast<const V8*>(qp + 32 * c);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (early && npairs > 0) {
                uint32_t h[2];
                first_pair(cur, h);
                first_fragments((uint32_t)uni((int)h[0]), (uint32_t)uni((int)h[1]));
            }
            __builtin_amdgcn_sched_barrier(0);
            if (L.q_rows != nullptr && wave == 0) out_rows[list_buf][lane_now] = first_rows[4];
            if constexpr (!kOnce) {
#pragma unroll
                for (int e = 0; e < kAhead; ++e)
                    if (lane_now + 64 * e < nent) big[lane_now + 64 * e] = (uint32_t)entry[e];
                for (int e = lane_now + 64 * kAhead; e < nent; e += 64) big[e] = (uint32_t)list[e];
            } else if constexpr (kGate) {
                ents = make_list<T, kTeam, kWalk == kHalves>(G, ost_bytes, cur.item / L.by_block, bh, nsub_of_block, tile_valid, fallback, fallback_count, lane, wave, cur.nent);
                nent = list_length(cur);
                if (kTeam == 1) npairs = uni(kWalk == kHalves ? nent >> 1 : nent * nsub);
            } else {
                if ((int)threadIdx.x < nent) big[threadIdx.x] = (uint32_t)team_entry;
                for (int e = threadIdx.x + 64 * kTeam; e < nent; e += 64 * kTeam) big[e] = (uint32_t)list[e];
            }
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) take_q(qb, rows[qb]);
            if constexpr (!kGate) {
                ents = big;
                __syncthreads();
            }
            if constexpr (kTeam > 1) {
                // This wavefront's share of the list, whole KV blocks of it, so that a walk over halves and one over tiles that masks
                // the empty halves cut at the same keys (and give the same bits).
                const int share = (parts.count > 1 ? cur.local / parts.by_items : 0) * kTeam + wave, shares = parts.count * kTeam;
                if constexpr (kWalk == kHalves) {
                    const int used = min(max(uni(cur.nent), 0), idx_stride);      // without the repeat that makes the number even
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
            }
        } else {
            ents = lists[list_buf];
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) {
                V8 rows[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) rows[c] = *reinterpret_cast<const V8*>(qstage + (qb * 4 + c) * 1024 + lane_off);
                take_q(qb, rows);
            }
        }
#pragma unroll
        for (int qb = 0; qb < 4; ++qb) {
            m_i[qb] = -INFINITY;
            l_i[qb] = 0.f;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int qb = 0; qb < 4; ++qb)
#pragma unroll
                for (int i = 0; i < 4; ++i) oacc[t][qb][i] = 0.f;

        bool run = true;                     // this kernel computes the item (see the bound on q . k below)
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
            // ---- prologue.  In flight when the loop starts: K(1), K(2), V(0); the ring slot of
            // V(1) holds zeros, which the first step multiplies with P = 0 (there is no step -1).  A prepared item
            // finds all of them but K(2) requested already (K(0) sits where K(2) belongs until S(0) has been issued).
            if (!prepared && !early) first_fragments(half_base + (first & kHalfId), half_base + (w[0] & kHalfId));
#pragma unroll
            for (int f = 0; f < 8; ++f)
#pragma unroll
                for (int e = 0; e < 8; ++e) vb[1][f][e] = (T)0.f;
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) {
#pragma unroll
                for (int e = 0; e < 8; ++e) pb[qb][e] = (T)0.f;
                alpha_p[qb] = 1.f;
            }
            // the token rows of the next item's queries are looked up now; its list and its Q rows are asked for once
            // it is known that this item runs here
            int32_t next_rows[4] = {0, 0, 0, 0};
            if (prepare_next) {
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) {
                    const int64_t row = nqrow0 + 16 * qb + lr;
                    next_rows[qb] = L.q_rows != nullptr ? L.q_rows[row] : (int32_t)row;      // used (and clamped) behind S(0): no wait here
                }
            }
#pragma unroll
            for (int f = 0; f < 8; ++f)
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) {
                    if (f < 2) mfma_s16<true>(s[0][f & 1][qb], kb[0][f], qreg[qb][f >> 1]);
                    else mfma_s16<false>(s[0][f & 1][qb], kb[0][f], qreg[qb][f >> 1]);
                }
#pragma unroll
            for (int c = 0; c < 8; ++c) kb[0][c] = k_frag(offset_of(w[1]), c);              // K(2), behind the last reader of K(0)
            asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");           // MFMA results before the VALU reads them
#pragma unroll
            for (int x = 0; x < 8; ++x) mfma_chain_end(s[0][x >> 2][x & 3]);
            mask_pair(s[0], first);
            // the first maximum: nothing is accumulated yet that it would rescale
            float mx[4];
            lane_max(s[0], mx);
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) {
                m_i[qb] = over_lanes(mx[qb], [](float a, float b) { return fmaxf(a, b); }) * qk_scale;
                neg_m[qb] = m_i[qb] == -INFINITY ? 0.f : -m_i[qb];
                raise_at[qb] = (m_i[qb] + kTau) * inv_scale;
            }
            raise_low = fminf(fminf(raise_at[0], raise_at[1]), fminf(raise_at[2], raise_at[3]));
            rescale_pending = false;

            // Cauchy-Schwarz: no logit of this item exceeds |q| times the largest key norm of the head.  If that bound
            // lies below the level at which the running maximum would be raised, no later step can raise it, and the steps
            // of this kernel, which do not look at the row maxima (a fifth of the softmax instructions), give the same
            // result.  A bound above that level moves the reference up to where it holds, unless the probabilities would
            // then start too low (kSlack): such an item (a first half tile of padding, norms far above the logits) is left
            // to the kernel that does look: it is put on the fallback list, nothing of it is stored, and the item
            // after it starts from scratch.
            if constexpr (kBounded) {
                const float kn = __uint_as_float((uint32_t)uni((int)__float_as_uint(cur.kn)));
                bool fit = true;
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) {
                    const float bound = __builtin_sqrtf(over_lanes(q_sq[qb], add)) * 1.001f * kn * qk_scale;      // all of the row's d
                    const float lowest = m_i[qb] == -INFINITY ? -bound : m_i[qb];       // the row's largest logit is no smaller
                    const float ref = bound - kTau;
                    fit = fit && ref <= lowest + kSlack;                                // false for a NaN
                    if (ref > m_i[qb]) {
                        m_i[qb] = ref;
                        neg_m[qb] = -ref;
                    }
                }
                run = __all(fit);
                if (!run && lane == 0) fallback[atomicAdd(fallback_count, 1u)] = cur.item;
            }
            if (run) {
            if (prepare_next) {
                // What the next item needs and what takes long to arrive is asked for now.  Its list goes from global
                // memory straight into the list buffer that is not in use (LDS DMA, 64 entries per instruction; the
                // lanes behind the end of the list repeat its last entry); its Q rows go into the staging tile,
                // fragment (qb, c) as 1 KB in lane order.  These loads are invisible to the compiler's count of
                // outstanding loads, which can only make its waits for the fragment loads stricter than they need
                // be while the DMA is under way.
#pragma unroll
                for (int e = 0; e < kPipeList * kWords / 64; ++e)
                    if (64 * e < next_nent)
                        load_to_lds_4(nlist, (uint32_t)min(lane + 64 * e, next_nent - 1) * 4u, (uint32_t)uni((int)lds_address(&lists[list_buf ^ 1][64 * e])));
                // and the token rows of its 64 query slots, which its epilogue stores through
                if (L.q_rows != nullptr)
                    load_to_lds_4(L.q_rows + nqrow0, (uint32_t)lane * 4u, (uint32_t)uni((int)lds_address(&out_rows[list_buf ^ 1][0])));
                const int nbatch = nbh / L.by_heads;
                const int64_t nq_bh = (int64_t)nbatch * L.q_st[0] + (int64_t)(nbh - nbatch * Hn) * L.q_st[1];
                const char* qsrc = reinterpret_cast<const char*>(q + nq_bh);
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) {
                    const uint32_t voff = (uint32_t)max(next_rows[qb], 0) * (uint32_t)(L.q_st[2] * 2) + (uint32_t)(16 * lg);   // padded slots read token 0
#pragma unroll
                    for (int c = 0; c < 4; ++c) load_to_lds_16(qsrc + 64 * c, voff, lds_address(qstage + (qb * 4 + c) * 1024));
                }
            }
            // The entries that come into the window are made one iteration before they enter (a validity word may
            // be a load) and read from LDS one iteration before that.  All of it goes between the last MFMAs of an iteration: in a
            // row behind them, with masks worked out for every half, it was 55 instructions, and the matrix pipe had nothing
            // to do for 220 clocks of 2 048.
            uint32_t in[2];
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
                    if constexpr (slot == 26) w[0] = w[2];
                    if constexpr (slot == 27) { w[1] = w[3]; w[2] = w[4]; }
                    if constexpr (slot == 28) { w[3] = in[0]; w[4] = in[1]; }
                    if constexpr (slot == 29) make(g + 4, raw, in);
                    if constexpr (slot == 30) raw = pair_raw(g + 5);
                    if constexpr (slot >= 26) {
#pragma unroll
                        for (int x = 0; x < 5; ++x) asm volatile("" : "+s"(w[x]));
                        if constexpr (slot >= 29) asm volatile("" : "+s"(in[0]), "+s"(in[1]));
                    }
                });
            }
            if (kTeam <= 1) __syncthreads();          // the list in LDS has been read: the memory may become the staging tile (a team: below)
            if (prepare_next) {
                // The DMA of the next item's list and Q rows was issued in front of the loop and every iteration has
                // issued 32 loads since; loads complete in order, so all but the newest 24 done (the next item's first
                // fragments, which may still be on their way) means that the DMA has landed.  The wait stands here, in
                // front of the epilogue's stores, whose number depends on the data; Q moves into its registers when
                // the next item starts and the output accumulators are free.
                asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
            }
            // queries 32 .. 63 of the last step (V of an odd step sits in ring slot 1)
            asm volatile("s_nop 1");
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int qb = 2; qb < 4; ++qb) mfma_acc16(oacc[t][qb], vb[1][t], pb[qb]);
            asm volatile("s_nop 15" ::: "memory");           // the last of them has retired before the VALU reads it
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) mfma_acc_end(oacc[t][qb]);
            if (rescale_pending) rescale_out();
            }   // run
        }   // npairs > 0

        if constexpr (kTeam > 1) {
            // ---- the wavefronts' sums together: sums[wave][register order of a part], then maxima and row sums [wave][query].
            // 128 KB through LDS for a team of four, a microsecond; the rows leave from all wavefronts.
            float* const sums = reinterpret_cast<float*>(ost_bytes);
            float* const stats = sums + kTeam * kTile * kD;
            float inv[4], M[4], l_all[4];
            __syncthreads();                          // the list has been read
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) {
                const float l = over_lanes(l_i[qb], add);
                if (lg == 0) {
                    stats[(2 * wave) * kTile + 16 * qb + lr] = m_i[qb];
                    stats[(2 * wave + 1) * kTile + 16 * qb + lr] = l;
                }
            }
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) *reinterpret_cast<f32x4_*>(sums + wave * (kTile * kD) + ((t * 4 + qb) * 64 + lane) * 4) = oacc[t][qb];
            __syncthreads();
            float factor[4][kTeam];
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) {
                float m[kTeam];
#pragma unroll
                for (int w = 0; w < kTeam; ++w) m[w] = stats[(2 * w) * kTile + 16 * qb + lr];
                M[qb] = m[0];
#pragma unroll
                for (int w = 1; w < kTeam; ++w) M[qb] = fmaxf(M[qb], m[w]);
                l_all[qb] = 0.f;
#pragma unroll
                for (int w = 0; w < kTeam; ++w) {
                    factor[qb][w] = m[w] > -INFINITY ? __builtin_amdgcn_exp2f(m[w] - M[qb]) : 0.f;      // a share without keys: no maximum, sums 0
                    l_all[qb] += stats[(2 * w + 1) * kTile + 16 * qb + lr] * factor[qb][w];
                }
                inv[qb] = l_all[qb] > 0.f ? 1.0f / l_all[qb] : 0.f;
            }
            constexpr int kOwn = 8 / kTeam;           // tiles of d that a wavefront puts together
            float4 own[kOwn][4];
#pragma unroll
            for (int t = 0; t < kOwn; ++t)
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) {
                    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                    for (int w = 0; w < kTeam; ++w) {
                        const float4 x = *reinterpret_cast<const float4*>(sums + w * (kTile * kD) + (((wave * kOwn + t) * 4 + qb) * 64 + lane) * 4);
                        const float fw = factor[qb][w];
                        sum.x = fmaf(x.x, fw, sum.x); sum.y = fmaf(x.y, fw, sum.y); sum.z = fmaf(x.z, fw, sum.z); sum.w = fmaf(x.w, fw, sum.w);
                    }
                    own[t][qb] = sum;
                }
            if (parts.count > 1) {
                float* const out = parts.buf + (int64_t)cur.local * kPartFloats;
#pragma unroll
                for (int t = 0; t < kOwn; ++t)
#pragma unroll
                    for (int qb = 0; qb < 4; ++qb)
                        *reinterpret_cast<float4*>(out + (((wave * kOwn + t) * 4 + qb) * 64 + lane) * 4) = own[t][qb];
                if (wave == 0 && lg == 0) {
#pragma unroll
                    for (int qb = 0; qb < 4; ++qb) {
                        out[kTile * kD + 16 * qb + lr] = M[qb];
                        out[kTile * kD + kTile + 16 * qb + lr] = l_all[qb];
                    }
                }
                return;
            }
            if (lse != nullptr && wave == 0 && lg == 0) {
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) {
                    int64_t row = qrow0 + 16 * qb + lr;
                    if (L.q_rows != nullptr) row = out_rows[list_buf][16 * qb + lr];
                    if (row >= 0) lse[(int64_t)bh * lse_S + row] = l_all[qb] > 0.f ? (M[qb] + __builtin_log2f(l_all[qb])) * kLn2 : -INFINITY;
                }
            }
            __syncthreads();                          // the sums have been read: the memory becomes the staging tile
#pragma unroll
            for (int qb = 0; qb < 4; ++qb)
#pragma unroll
                for (int t = 0; t < kOwn; ++t) {
                    const float4 x = own[t][qb];
                    T out4[4] = {(T)(x.x * inv[qb]), (T)(x.y * inv[qb]), (T)(x.z * inv[qb]), (T)(x.w * inv[qb])};
                    *reinterpret_cast<uint2*>(ost + (16 * qb + lr) * kOutPitch + 16 * (wave * kOwn + t) + 4 * lg) = *reinterpret_cast<uint2*>(out4);
                }
            __syncthreads();
            const int kc = threadIdx.x & 15, kr = threadIdx.x >> 4;
            constexpr int kRows = 4 * kTeam, kTurns = kTile / kRows;
            u32x4 pieces[kTurns];
            int32_t rows[kTurns];
#pragma unroll
            for (int i = 0; i < kTurns; ++i) {
                rows[i] = L.q_rows != nullptr ? out_rows[list_buf][kr + kRows * i] : kr + kRows * i;
                pieces[i] = *reinterpret_cast<const u32x4*>(ost + (kr + kRows * i) * kOutPitch + kc * 8);
            }
#pragma unroll
            for (int i = 0; i < kTurns; ++i)
                if (rows[i] >= 0) *reinterpret_cast<u32x4*>(o + o_bh + ((L.q_rows != nullptr ? 0 : qrow0) + rows[i]) * L.o_st[2] + kc * 8) = pieces[i];
            return;
        }
        if (!kOnce && !kBounded && parts.count > 1) {
            float* const out = parts.buf + (int64_t)cur.local * kPartFloats;
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int qb = 0; qb < 4; ++qb) *reinterpret_cast<f32x4_*>(out + ((t * 4 + qb) * 64 + lane) * 4) = oacc[t][qb];
#pragma unroll
            for (int qb = 0; qb < 4; ++qb) {
                const float l = over_lanes(l_i[qb], add);
                if (lg == 0) {
                    out[kTile * kD + 16 * qb + lr] = m_i[qb];
                    out[kTile * kD + kTile + 16 * qb + lr] = l;
                }
            }
        } else if (run) {
        // ---- epilogue: combine the four key groups of every query, normalise, store through LDS ----
        float inv[4];
#pragma unroll
        for (int qb = 0; qb < 4; ++qb) {
            const float l = over_lanes(l_i[qb], add);
            inv[qb] = l > 0.f ? 1.0f / l : 0.f;
            if (lse != nullptr && lg == 0) {
                int64_t row = qrow0 + 16 * qb + lr;
                if (L.q_rows != nullptr) row = out_rows[list_buf][16 * qb + lr];
                if (row >= 0) lse[(int64_t)bh * lse_S + row] = l > 0.f ? ((kBounded ? -neg_m[qb] : m_i[qb]) + __builtin_log2f(l)) * kLn2 : -INFINITY;
            }
        }
        // accumulator i of d tile t <-> d = 16 t + 4 lg + i, query 16 qb + lr
#pragma unroll
        for (int qb = 0; qb < 4; ++qb) {
            T* orow = ost + (16 * qb + lr) * kOutPitch;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                T out4[4];
#pragma unroll
                for (int jx = 0; jx < 4; ++jx) out4[jx] = (T)(oacc[t][qb][jx] * inv[qb]);
                *reinterpret_cast<uint2*>(orow + 16 * t + 4 * lg) = *reinterpret_cast<uint2*>(out4);
            }
        }
        __syncthreads();                          // one wavefront: orders its LDS writes before the reads below
        {
            // The lane index goes through an opaque statement: what is derived from it here (sixteen row numbers and
            // their addresses) would otherwise be computed once in front of the item loop and held in registers, or
            // in scratch memory, all through the tile loop.
            int lane_now = lane;
            asm volatile("" : "+v"(lane_now));
            const int kc = lane_now & 15, kr = lane_now >> 4;
            // in three sweeps - the sixteen token rows, the sixteen pieces, the stores - so that the LDS reads are all
            // on their way before the first is waited for (row by row, every store sat behind two LDS round trips)
            int32_t rows[16];                         // relative to qrow0 without a row table
            u32x4 pieces[16];
            if (L.q_rows != nullptr) {
#pragma unroll
                for (int i = 0; i < 16; ++i) rows[i] = out_rows[list_buf][kr + 4 * i];
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) rows[i] = kr + 4 * i;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(rows[i]));
            const int64_t row_base = L.q_rows != nullptr ? 0 : qrow0;
#pragma unroll
            for (int i = 0; i < 16; ++i) pieces[i] = *reinterpret_cast<const u32x4*>(ost + (kr + 4 * i) * kOutPitch + kc * 8);
#pragma unroll
            for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(pieces[i]));      // read here, not inside the branches below
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (rows[i] >= 0) *reinterpret_cast<u32x4*>(o + o_bh + (row_base + rows[i]) * L.o_st[2] + kc * 8) = pieces[i];
        }
        }   // run
        if constexpr (kOnce) return;
        // ---- on to the next item
        prepared = prepare_next && run;
        if (prepared) list_buf ^= 1;
        __syncthreads();                          // the staging tile is free again
        cur = nxt;
        nxt = nx2;
    }   // work items
}

// Puts the parts of an item together: rescale to the largest of the running maxima, add, normalise, round, store.  One
// workgroup per item; bound by the parts' bytes (33 KB each).
template <typename T>
__global__ __launch_bounds__(256) void merge_parts_kernel(Parts parts, T* __restrict__ o, float* __restrict__ lse, int item_begin,
                                                          int nqt, int Hn, int64_t lse_S, FragLayout L) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4;
    const int item = item_at(L, item_begin + blockIdx.x, nqt), bh = item / L.by_tiles;
    const int64_t qrow0 = (int64_t)(item - bh * nqt) * kTile;
    const float* first = parts.buf + (int64_t)blockIdx.x * kPartFloats;
    const int64_t stride = (int64_t)parts.items * kPartFloats;
    float M[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY}, inv[4];
    int64_t row[4];
#pragma unroll
    for (int qb = 0; qb < 4; ++qb) {
        const int slot = 16 * qb + lr;
        row[qb] = L.q_rows != nullptr ? (int64_t)L.q_rows[qrow0 + slot] : qrow0 + slot;
        for (int p = 0; p < parts.count; ++p) M[qb] = fmaxf(M[qb], first[p * stride + kTile * kD + slot]);
        float l = 0.f;
        for (int p = 0; p < parts.count; ++p) {
            const float m = first[p * stride + kTile * kD + slot];
            if (m > -INFINITY) l += first[p * stride + kTile * kD + kTile + slot] * __builtin_amdgcn_exp2f(m - M[qb]);
        }
        inv[qb] = l > 0.f ? 1.0f / l : 0.f;
        if (lse != nullptr && wave == 0 && lg == 0 && row[qb] >= 0)
            lse[(int64_t)bh * lse_S + row[qb]] = l > 0.f ? (M[qb] + __builtin_log2f(l)) * kLn2 : -INFINITY;
    }
    T* const out = o + (int64_t)(bh / Hn) * L.o_st[0] + (int64_t)(bh % Hn) * L.o_st[1];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int chunk = wave * 8 + c, t = chunk >> 2, qb = c & 3;
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int p = 0; p < parts.count; ++p) {
            const float m = first[p * stride + kTile * kD + 16 * qb + lr];
            const float f = m > -INFINITY ? __builtin_amdgcn_exp2f(m - M[qb]) : 0.f;
            const float4 x = *reinterpret_cast<const float4*>(first + p * stride + (chunk * 64 + lane) * 4);
            sum.x = fmaf(x.x, f, sum.x); sum.y = fmaf(x.y, f, sum.y); sum.z = fmaf(x.z, f, sum.z); sum.w = fmaf(x.w, f, sum.w);
        }
        if (row[qb] < 0) continue;
        const float n = inv[qb];
        T x4[4] = {(T)(sum.x * n), (T)(sum.y * n), (T)(sum.z * n), (T)(sum.w * n)};
        *reinterpret_cast<uint2*>(out + row[qb] * L.o_st[2] + 16 * t + 4 * lg) = *reinterpret_cast<const uint2*>(x4);
    }
}

}  // namespace

// The price of a tile walked out of step, by which the queues' estimate is weighed against the rounds'.  Attention of 16 heads of
// 20x30x52 by the CDF threshold, queues / rounds, whole operator in us: smooth inputs 0.25 (lists of 32 to 49 blocks) 815 / 775,
// 0.5 (32 to 157) 1 200 / 1 485, 0.75 (54 to 313) 2 497 / 3 267, 32 heads of 24x45x80 at 0.5 (90 to 635) 8 592 / 10 396; random
// inputs (lists of one length, give or take three) 0.5 3 800 / 3 928, where rounds leave seven of eight wavefronts idle in
// the last; equal lists of 32 heads over whole rounds 1 840 / 1 848 smooth, 2 450 / 1 870 and 9 900 / 8 325 random.
constexpr double kQueuePrice = 1.4;
// Classes an octave of list length: 0 (query order alone) 1 441 us for the 0.5 case, 1 1 200, 2 1 229, 4 1 250; one counter over
// every head's tiles by exact length 1 834.
constexpr float kClassesPerOctave = 1.0f;

// The plan of the queue schedule, one launch.  Workgroup x < kQueues writes section x of `order`: its items in classes of
// similar list length, longest class first (so that the last items drawn are short), and within a class in the order of
// the query tiles.  Neighbouring tiles of a layer whose queries vary smoothly select largely the same blocks; drawn one after
// another by the workgroups of one XCD, with lists of about one length and so at about one pace, they find each other's
// tiles in its L2.  The last workgroup clears the counters and chooses between rounds and queues: a round lasts as long as
// its longest list, the queues keep every workgroup busy but walk out of step.
constexpr int kPlanThreads = 1024, kPlanClasses = 12, kPlanRounds = 8192;
__global__ __launch_bounds__(kPlanThreads) void queue_plan_kernel(const int32_t* __restrict__ lens, int nqt, FragLayout L,
                                                                  int total, int resident, int max_len, int32_t* __restrict__ order,
                                                                  uint32_t* __restrict__ queue) {
    __shared__ int sm[kPlanClasses * kPlanThreads];
    __shared__ int wave_sum[kPlanThreads / 64];
    __shared__ int longest_sm;
    __shared__ unsigned long long sum_sm;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    auto length_of = [&](int item) { return min(max(lens[item / L.by_block], 0), max_len); };
    auto wave_max = [](int x) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x = max(x, __shfl_xor(x, off));
        return x;
    };
    if (tid == 0) { longest_sm = 0; sum_sm = 0ull; }
    if (blockIdx.x == kQueues) {
        const int rounds = (total + resident - 1) / resident;
        if (tid < kQueues) queue[tid] = 0u;
        if (rounds > kPlanRounds) { if (tid == 0) queue[kQueueChoice] = 0u; return; }
        for (int r = tid; r < rounds; r += kPlanThreads) sm[r] = 0;
        __syncthreads();
        unsigned long long sum = 0ull;
        int longest = 0;
        for (int u0 = 64 * wave; u0 < total; u0 += kPlanThreads) {          // 64 consecutive items, mostly of one round
            const int u = min(u0 + lane, total - 1), l = length_of(item_at(L, u, nqt));
            sum += u0 + lane < total ? (unsigned long long)l : 0ull;
            longest = max(longest, l);
            const int most = wave_max(l), r = u0 / resident;
            if (r == min(u0 + 63, total - 1) / resident) { if (lane == 0) atomicMax(&sm[r], most); }
            else atomicMax(&sm[u / resident], l);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
        longest = wave_max(longest);
        if (lane == 0) {
            atomicAdd(&sum_sm, sum);
            atomicMax(&longest_sm, longest);
        }
        __syncthreads();
        if (tid == 0) {
            unsigned long long rounds_cost = 0ull;
            for (int r = 0; r < rounds; ++r) rounds_cost += (unsigned long long)sm[r];
            const double queue_cost = kQueuePrice * (double)sum_sm / (double)resident + (double)longest_sm;
            queue[kQueueChoice] = queue_cost < (double)rounds_cost ? 1u : 0u;
        }
        return;
    }
    const int begin = section_begin(total, blockIdx.x), end = section_begin(total, blockIdx.x + 1);
    const int per = (end - begin + kPlanThreads - 1) / kPlanThreads;
    const int first = min(begin + tid * per, end), last = min(first + per, end);      // this thread's items
    for (int c = 0; c < kPlanClasses; ++c) sm[c * kPlanThreads + tid] = 0;
    __syncthreads();
    int longest = 0;
    for (int u = first; u < last; ++u) longest = max(longest, length_of(item_at(L, u, nqt)));
    longest = wave_max(longest);
    if (lane == 0) atomicMax(&longest_sm, longest);
    __syncthreads();
    const float top = __builtin_log2f((float)max(longest_sm, 1));
    auto class_of = [&](int l) { return l <= 0 ? kPlanClasses - 1 : min((int)(kClassesPerOctave * (top - __builtin_log2f((float)l)) + 0.001f), kPlanClasses - 1); };
    for (int u = first; u < last; ++u) ++sm[class_of(length_of(item_at(L, u, nqt))) * kPlanThreads + tid];
    __syncthreads();
    // exclusive sums over (class, thread): twelve consecutive entries per thread, the threads' totals over the workgroup
    int own[kPlanClasses], run = 0;
#pragma unroll
    for (int c = 0; c < kPlanClasses; ++c) { own[c] = sm[tid * kPlanClasses + c]; run += own[c]; }
    int before = run;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int x = __shfl_up(before, off);
        if (lane >= off) before += x;
    }
    if (lane == 63) wave_sum[wave] = before;
    __syncthreads();
    before -= run;
    for (int w = 0; w < wave; ++w) before += wave_sum[w];
#pragma unroll
    for (int c = 0; c < kPlanClasses; ++c) { sm[tid * kPlanClasses + c] = before; before += own[c]; }
    __syncthreads();
    for (int u = first; u < last; ++u) {
        const int item = item_at(L, u, nqt);
        order[begin + sm[class_of(length_of(item)) * kPlanThreads + tid]++] = item;
    }
}

// Rounds per launch: five (four to six measure the same at 90 tiles per list and 1.5 % better than two, now that an
// item that was prepared by the one before it starts 7 us sooner than a launch's first; from eight on the items drift
// apart and the L2 hit rate falls); eight for short lists (six to ten measure the same, twenty lose 3 %).
constexpr int kRoundsPerLaunch = 5;
constexpr int kRoundsPerLaunchShort = 8;     // lists of at most kShortList tiles
constexpr int kShortList = 64;

// Tiles a wavefront walks in all of a call's rounds, up to which it runs the exact kernel alone (bounded / exact, us: 1 120 items
// of 4 tiles 55.0 / 52.8, of 16, the last round in teams, 83.3 / 81.4, of 32 116.9 / 115.6, of 64 183.5 / 184.0; 2 160 of 4 87.8 /
// 87.4, of 16 133.0 / 132.4, of 32 196.0 / 196.5; 2 700 of 11 132.6 / 133.8).
constexpr int kExactRoundTiles = 24;
constexpr int kOneRound = 1 << 30;           // more than a launch's items: each workgroup has one (kTeam > 0)

// Workgroups (of one wavefront) the device runs at once with this kernel: one per SIMD, at most kMostResident (256 compute
// units).
constexpr int kMostResident = 1024;
static int resident_wavefronts() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return kMostResident;
    if (cached[dev] == 0) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
        cached[dev] = 4 * cus < kMostResident ? 4 * cus : kMostResident;
    }
    return cached[dev];
}

// kf / vf: fragment-order K and V, [B * Hn][Sk / 64][16 KB].  q, o in blocked order (q_rows null) or in
// (T, H, W) order through the row table.  Scheduling: rounds of as many work items as the device runs at once,
// across (batch, head) boundaries, kRoundsPerLaunch rounds per launch, every workgroup running one item of each round;
// with `order` and `queue` also the schedule that draws items from the XCDs' queues, the choice between the two being
// made on the device.
__global__ void frag_zero_kernel(uint32_t* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// Into how many shares the items of the last, partial round are cut along their lists, so that the wavefronts it would leave
// idle help: a team of `team` wavefronts an item, or `parts` parts of such teams, whichever has the least estimated time.  A
// 64-key tile of a list takes 1.72 us of a wavefront when the chip is full, 1.15 us when it is half empty (its power then
// allows the full clock: with one price for both, rounds of 512 and 640 items were cut and a 480p layer took 1 838 us instead
// of 1 826, four heads of 720p 1 113 instead of 1 095); an item 6 us to start and end, 4.3 with a team of two, which stores
// side by side, 5.8 with one of four; the merge of parts a launch and their bytes (33 KB written and read).  Shares of fewer
// than 10 tiles are not worth a part.  Whole operator, one wavefront an item / two / four / two parts of teams of four, us: 16
// items of 2 tiles 20.3 / 17.4 / 18.5, 64 of 4 23.4 / 19.4 / 19.9, 64 of 8 29.3 / 23.0 / 22.2, 128 of 32 60.7 / 40.5 / 33.0 /
// 41.7, 128 of 128 184 / 108 / 71.5 / 64.3, 240 of 16 47.8 / 36.5 / 34.0 / 50.9, 384 of 32 72.4 / 52.9 / 62.9, 512 of 2 33.0 /
// 31.0 / 37.7, 512 of 64 120 / 87 / 95.
// Uncut, the items behind whole rounds (is_tail) were prepared by those before them and start at once; cut, they wait for
// another launch (4 us).  Items of one length behind one whole round, uncut / teams of two / of four: 56 of 8 64.3 / 63.9 / 64.0,
// of 16 88.9 / 84.6 / 82.7, of 64 225 / 197 / 183; 272 of 8 68.3 / 70.7, of 16 91.7 / 90.0, of 64 231 / 206; 416 of 16 94.2 / 93.0,
// of 64 232 / 214; behind two, 512 of 16 144.3 / 144.8, of 64 368 / 361.  As many shares as there are wavefronts are not made behind
// whole rounds: little is gained.
// Teams are made where all of them run at once.  Three rounds of teams of four were priced 8 % too low: three parts / teams, us, 544 items
// of 200 tiles 259 / 284, 640 of 200 282 / 292, of 280 368 / 383; a wavefront an item / teams, 640 of 100 177 / 173, 700 of 100 198 / 205,
// of 200 339 / 331, 768 of 64 131 / 138, of 200 327 / 320.  Where a list may be shorter than its width (the CDF rule, a caller's: one_length
// false) they lost more, behind kernels that select; teams / one round of wavefronts, at threshold 0.03, 0.0625, 0.25 and 1, us: 600
// items of 100 blocks 56.1 / 30.4, 63.0 / 35.2, 88.5 / 59.0, 171 / 153; 768 of 256 72.9 / 47.5, 87.4 / 56.2, 148.5 / 126.2, 404 / 410; 640
// of 320, which no wavefront scores by itself, 76.1 / 53.5, 88.0 / 65.7, 162 / 148, 444 / 454.
// The shares of a team of two are whole KV blocks of the list, which visits the sequence in order, while parts of single wavefronts
// are cut by halves.  On a grid whose last frames do not fill their chunks the second share is short: `heavier_half` is the first one's
// part of the halves over the mean, of blocks spread evenly.  Its wavefront walks that much longer on a chip that is as much emptier.
// Teams of two / parts, us, which were priced without it: 258 items of 13x26x43 in 4x4x8 chunks and 168 tiles 127 / 112, 342 of 9x36x57
// and 344 251 / 219, 336 of 5x46x53 in 4x4x4 and 168 137 / 129, 468 of 9x50x46 and 234 210 / 215.  Teams of four come out right without
// it: with it 80 items of 5x37x15 and 64 tiles would go to parts, 53 us for 41, 138 of 9x18x48 and 90 65 for 54.
static float heavier_half(const Grid3& k) {
    const int full = k.chunk() / 32, last = k.T % k.t == 0 ? full : (k.T % k.t * k.h * k.w + 31) / 32;      // halves of an inner chunk
    const float layers = (float)k.Nt, span = 0.5f * layers, inner = fminf(span, layers - 1.f);
    return 2.f * (inner * full + (span - inner) * last) / ((layers - 1.f) * full + last);
}
constexpr int kMaxParts = 16, kMaxPartRounds = 2, kMinPartTiles = 10;
struct Split { int team, parts; };
// halves_of: the grid of the keys where the lists are of halves, otherwise null
static Split choose_split(int items, int list_tiles, int resident, bool is_tail, bool one_length, const Grid3* halves_of) {
    Split best = {1, 1};
    float best_us = 0.f;
    for (int team = 1; team <= 4 && team <= list_tiles && (team == 1 || items * team + (is_tail ? 1 : 0) <= resident); team *= 2)
        for (int p = 1; p == 1 || (one_length && p <= kMaxParts && p * team * kMinPartTiles <= list_tiles && (int64_t)items * p * team <= kMaxPartRounds * resident); ++p) {
            const int groups = resident / team, rounds = (int)(((int64_t)items * p + groups - 1) / groups);
            const float start = team == 2 ? 4.3f : team == 4 ? 5.8f : is_tail && p == 1 ? 0.f : 6.f;
            const float weight = team == 2 && p == 1 && halves_of != nullptr ? heavier_half(*halves_of) : 1.f;
            const float full = (float)items * p / ((float)rounds * groups) / weight, tile_us = 1.15f + 1.14f * (full > 0.5f ? full - 0.5f : 0.f);
            const float us = rounds * (tile_us * list_tiles * weight / (p * team) + start) + (p > 1 ? 5.f + 0.0125f * items * p : 0.f) + (is_tail && p * team > 1 ? 4.f : 0.f);
            if ((team == 1 && p == 1) || us < best_us) { best = {team, p}; best_us = us; }
        }
    return best;
}
// Calls of so few items that SIMDs are left over run fwd_few_kernel, whose 32x32x16 products leave a wavefront more of its issue; where nearly
// all are busy the board's power is the bound again.  Whole operator in us, this file's kernel / that one, items x tiles: with a wavefront an item
// 640 x 20 53.7 / 50.3, x 80 140.6 / 130.0, 768 x 64 118.0 / 116.4, 800 x 20 56.9 / 56.9, x 80 145.5 / 145.2, 832 x 104 183.3 / 185.6, 896 x 64
// 126.2 / 128.9, 1 024 x 128 246.8 / 255.9; teams of two 384 x 64 70.6 / 69.0, 416 x 104 101.5 / 101.3, 448 x 112 111.4 / 113.0, 512 x 128
// 133.9 / 137.8; teams of four 128 x 64 43.6 / 39.6, 176 x 88 54.8 / 50.6, 208 x 104 61.0 / 60.0, 256 x 128 77.8 / 78.2.  So the line lies at
// 800 wavefronts, counted in full teams of two (of four it is level up to the most), and by the items alone, because K and V are prepared
// before the length of the lists, and with it the team, need be known (bsa_thw_prepare).
constexpr int kBusyWide = 800;
bool frag_few(int64_t heads, int64_t Sq, int64_t Sk, const Grid3* q_grid) {
    const int64_t items = heads * (q_grid != nullptr ? live_query_tiles(*q_grid) : Sq / kTile);
    return heads * (Sk / kTile) * (int64_t)kTileBytes < ((int64_t)1 << 32) && (items <= kBusyWide / 2 || (items > kMostResident / 2 && items <= kBusyWide));
}
struct Rounds {
    int heads_per_span;              // (batch, head)s that one buffer of K reaches
    bool one_span, few;
    int n_live, total, resident, list_tiles, tail;
    Split split;
};
static Rounds plan_rounds(int64_t heads, int64_t Sq, int64_t Sk, int bs_k, int idx_stride, const Grid3* halves_of, const Grid3* q_grid, bool one_length) {
    Rounds r;
    // The kernel addresses K and V through a buffer of less than 4 GB that starts at the first (batch, head) of a
    // launch: a launch covers as many heads as fit.  One head always does (fewer than 2^24 keys of 256 B).
    r.heads_per_span = (int)((((int64_t)1 << 32) - 1) / ((Sk / kTile) * (int64_t)kTileBytes));
    r.one_span = heads <= r.heads_per_span;
    // Query tiles without real rows drop out; they would walk their lists for nothing.  A 13x30x53 grid in 4x4x8 chunks has
    // 448 tiles, 371 of them with rows: 820 -> 727 us for 16 heads in fp16.  (Tiles with at most 32 rows, an eighth of a 30-row
    // grid's, stay whole: a walk with half of the MFMAs and the same loads took longer per tile, 206 against 179 us a round at
    // 720p, and a third longer overall where such tiles ran between full ones and put the items of an XCD out of step.)
    r.n_live = q_grid != nullptr && r.one_span ? live_query_tiles(*q_grid) : (int)(Sq / kTile);
    r.total = (int)(heads * r.n_live);
    r.resident = resident_wavefronts();
    r.list_tiles = halves_of != nullptr ? (idx_stride + 1) / 2 : idx_stride * (bs_k / kTile);
    // The items of the last, partial round are cut when its wavefronts would leave too much of the chip idle (and the exact
    // kernel reaches every head from one buffer); behind whole rounds and into parts only for lists of one length.
    r.tail = r.total % r.resident;
    r.split = {1, 1};
    // (frag_few goes by the whole chip: on a part of it such a call may have more than one round, which is not cut)
    r.few = frag_few(heads, Sq, Sk, q_grid);
    if (r.one_span && r.tail > 0 && (r.total < r.resident || (one_length && !r.few)))
        r.split = choose_split(r.tail, r.list_tiles, r.resident, r.total > r.resident, one_length, halves_of);
    return r;
}
// The lists of a call whose workgroups all run at once are made by those that walk them.  The kernels in front / like this, us, density
// 1/16: one wavefront an item, 768 items of 192 blocks 48.3 / 46.7, 672 of 224 49.0 / 47.3, 768 of 256 54.8 / 53.9, 1 024 of 256, the most
// that there are, 64.1 / 64.3 (at density 1/4 151.2 / 151.0); teams of four, 320 of 320 43.7 / 40.0, 512 of 512 66.6 / 62.5; one
// workgroup behind another pays for it twice (2 heads of 320 blocks, teams of four, density 1/4, 147 / 156).
bool frag_selects(int64_t heads, int64_t Sq, int64_t Sk, int bs_k, int idx_stride, const Grid3* halves_of, const Grid3* q_grid, bool one_length, int nbk, int width) {
    const Rounds r = plan_rounds(heads, Sq, Sk, bs_k, idx_stride, halves_of, q_grid, one_length);
    return r.one_span && r.split.parts == 1 && r.total * r.split.team <= r.resident && nbk <= (r.split.team == 1 ? kGateWaveBlocks : kGateMostBlocks) &&
           gate_here_bytes(nbk, width, bs_k / kTile, halves_of != nullptr) <= kTile * (kD + 8) * 2;
}
LastRound frag_last_round(int64_t heads, int64_t Sq, int64_t Sk, int bs_k, int idx_stride, const Grid3* halves_of, const Grid3* q_grid, bool one_length) {
    const Rounds r = plan_rounds(heads, Sq, Sk, bs_k, idx_stride, halves_of, q_grid, one_length);
    return {r.total, r.tail, r.split.team, r.split.parts};
}
// floats of the parts' buffer, whatever the length of the lists and whichever device runs the call (a caller asks for the size
// of a workspace once, for all of its devices): a partial round has no more items than the call, choose_split the limits
size_t frag_part_floats(const Grid3& g, int64_t heads) {
    const int64_t all = heads * live_query_tiles(g) * kMaxParts, most = (int64_t)kMaxPartRounds * kMostResident;
    return (size_t)(all < most ? all : most) * kPartFloats;
}

// int32 entries launch_fwd_frag's `fallback` argument must hold for `items` work items (64-row query tiles)
size_t frag_fallback_ints(int64_t items) { return 64 + (size_t)items; }

hipError_t launch_fwd_frag(const void* q, const void* kf, const void* vf, const int32_t* idx, const int32_t* lens,
                           const uint64_t* tile_valid, void* o, float* lse, int B, int Hn, int64_t Sq, int64_t Sk,
                           int bs_q, int bs_k, int idx_stride, float sm_scale, int dtype, hipStream_t st,
                           const int32_t* q_rows, const int64_t q_st[3], const int64_t o_st[3], int64_t lse_rows,
                           const Grid3* q_grid, int32_t* order, uint32_t* queue, const float* key_norm, int32_t* fallback, bool fallback_cleared,
                           const Grid3* halves_of, float* part_buf, const GateCall* gate_call) {
    const bool halves = halves_of != nullptr;
    // the C-ABI layer keeps lists within these limits (a list that is too long for the small buffers is staged in `ost`)
    if (idx_stride > (halves ? kHalfEntries : kListEntries)) return hipErrorInvalidValue;
    const float qk_scale = sm_scale * kLog2e;
    FragLayout L;
    L.q_rows = q_rows;
    for (int i = 0; i < 3; ++i) { L.q_st[i] = q_st[i]; L.o_st[i] = o_st[i]; }
    const int per_head = (int)(Sq / kTile);
    const int all_tiles = B * Hn * per_head;
    const uint32_t* gate = nullptr;
    const int64_t kv_bh_bytes = (Sk / kTile) * (int64_t)kTileBytes;
    if (kv_bh_bytes > ((int64_t)1 << 32) - 1) return hipErrorInvalidValue;
    // a buffer for parts comes with lists of one length
    const auto [heads_per_span, one_span, few, n_live, total, resident, list_tiles, tail, split] =
        plan_rounds((int64_t)B * Hn, Sq, Sk, bs_k, idx_stride, halves_of, q_grid, part_buf != nullptr);
    L.tiles = n_live < per_head ? q_rows + Sq : nullptr;
    L.n_live = n_live;
    L.by_live = divisor(n_live);
    L.by_tiles = divisor(per_head);
    L.by_block = divisor(bs_q / kTile);
    L.by_heads = divisor(Hn);
    L.by_sub = divisor(bs_k / kTile);
    const uint32_t whole_span = one_span ? (uint32_t)((int64_t)B * Hn * kv_bh_bytes) : 0u;
    // the LDS DMA that brings the next item's Q rows forms its addresses from 32-bit row offsets
    const int64_t q_rows_max = q_rows != nullptr ? lse_rows : Sq;
    const int q_offsets_32 = q_rows_max * q_st[2] * 2 + 512 < ((int64_t)1 << 32) ? 1 : 0;
    // The bf16 rounds run the kernel whose steps take no row maxima when the key norms are known, a place for the list of
    // the items it has to leave to the other kernel is given, and that kernel can reach every head from one buffer.
    // A short call runs the exact kernel alone: its steps are 3 % longer, but a last launch that finds nothing to do costs 4.7 us.
    Parts parts = {nullptr, 1, 0, divisor(1), divisor(1)};
    const bool bounded = !few && dtype == BSA_BF16 && key_norm != nullptr && fallback != nullptr && one_span && total > resident &&
                         (int64_t)total * list_tiles > (int64_t)kExactRoundTiles * resident;
    uint32_t* fb_count = bounded ? reinterpret_cast<uint32_t*>(fallback) : nullptr;
    int32_t* fb_list = bounded ? fallback + 64 : nullptr;
    FragGate here = {};
    int32_t* gate_lists = nullptr;      // with `here`: where the lists that the kernel makes go
    uint32_t* gate_lens = nullptr;
#define BSA_FRAG_LAUNCH_T(T, WALK, BD, TEAM, GATE, grid, begin, end, ord, que, want, bh0, span, fbl, fbc)                           \
    hipLaunchKernelGGL((fwd_frag_kernel<T, WALK, BD, TEAM, GATE>), grid, dim3(TEAM > 1 ? 64 * TEAM : 64), 0, st, (const T*)q, (const char*)kf, (const char*)vf, idx, \
                       lens, tile_valid, (T*)o, lse, Sq, Sk, bs_q, bs_k, idx_stride, qk_scale, begin, end, TEAM > 0 ? kOneRound : resident, Hn, lse_rows, \
                       L, ord, que, gate, want, bh0, span, q_offsets_32, key_norm, fbl, fbc, parts, here)
#define BSA_FRAG_LAUNCH_W(T, BD, TEAM, GATE, ...)                                                                      \
    do {                                                                                                               \
        if (halves) BSA_FRAG_LAUNCH_T(T, kHalves, BD, TEAM, GATE, __VA_ARGS__);                                        \
        else if (bs_k == kTile) BSA_FRAG_LAUNCH_T(T, kTiles, BD, TEAM, GATE, __VA_ARGS__);                             \
        else BSA_FRAG_LAUNCH_T(T, kBlocks, BD, TEAM, GATE, __VA_ARGS__);                                               \
    } while (0)
#define BSA_FRAG_LAUNCH(BD, ...)                                                                                       \
    do {                                                                                                               \
        if (dtype == BSA_BF16) BSA_FRAG_LAUNCH_W(__bf16, BD, 0, false, __VA_ARGS__);                                   \
        else BSA_FRAG_LAUNCH_W(_Float16, false, 0, false, __VA_ARGS__);                                                \
    } while (0)
#define BSA_FRAG_LAUNCH_LISTED(TEAM, ...)                                                                              \
    do {                                                                                                               \
        if (dtype == BSA_BF16) BSA_FRAG_LAUNCH_W(__bf16, false, TEAM, false, __VA_ARGS__);                             \
        else BSA_FRAG_LAUNCH_W(_Float16, false, TEAM, false, __VA_ARGS__);                                             \
    } while (0)
#define BSA_FRAG_LAUNCH_ONCE(TEAM, ...)                                                                                \
    do {                                                                                                               \
        if (here.qc != nullptr) {                                                                                      \
            if (dtype == BSA_BF16) BSA_FRAG_LAUNCH_W(__bf16, false, TEAM, true, __VA_ARGS__);                          \
            else BSA_FRAG_LAUNCH_W(_Float16, false, TEAM, true, __VA_ARGS__);                                          \
        } else {                                                                                                       \
            BSA_FRAG_LAUNCH_LISTED(TEAM, __VA_ARGS__);                                                                 \
        }                                                                                                              \
    } while (0)
    const bool once = few || (one_span && total <= resident && (split.team > 1 || split.parts == 1));
    if (gate_call != nullptr) {
        const GateCall& c = *gate_call;
        if (c.inside) {
            here = {static_cast<const uint16_t*>(c.q_cmp), static_cast<const uint16_t*>(c.k_cmp), c.nbk, c.width, c.threshold, c.scale, c.k_min,
                    pace_divisor(c.nbk, c.width)};
            gate_lists = c.lists;
            gate_lens = reinterpret_cast<uint32_t*>(c.lens);
            idx = lens = nullptr;
            if (halves) tile_valid = c.valid;
        } else {
            const hipError_t e = c.make(c.ctx);
            if (e != hipSuccess) return e;
        }
    }
    if (bounded && !fallback_cleared) hipLaunchKernelGGL(frag_zero_kernel, dim3(1), dim3(64), 0, st, fb_count, 1);
    // Lists of unequal length of one round need no plan: every item has a wavefront of its own from the start.
    if (queue != nullptr && one_span && total > resident && !few) {
        hipLaunchKernelGGL(queue_plan_kernel, dim3(kQueues + 1), dim3(kPlanThreads), 0, st, lens, per_head, L, total, resident, idx_stride,
                           order, queue);
        gate = queue + kQueueChoice;
        const dim3 grid((unsigned)(total < resident ? total : resident));
        if (bounded) BSA_FRAG_LAUNCH(true, grid, 0, total, order, queue, 1u, 0, whole_span, fb_list, fb_count);
        else BSA_FRAG_LAUNCH(false, grid, 0, total, order, queue, 1u, 0, whole_span, (int32_t*)nullptr, (uint32_t*)nullptr);
    }
    // kRoundsPerLaunch rounds per launch, every workgroup running one item of each: the items of a round start
    // together and keep in step (with many more rounds per launch they drift apart and the L2 hit rate falls).
    const int span = (list_tiles <= kShortList ? kRoundsPerLaunchShort : kRoundsPerLaunch) * resident;
    const int whole = once ? 0 : split.team * split.parts > 1 ? total - tail : total;
    for (int first = 0; first < whole;) {
        int end = first + span < whole ? first + span : whole;
        const int bh0 = one_span ? 0 : first / per_head;
        if (!one_span && (end - 1) / per_head - bh0 + 1 > heads_per_span) end = (bh0 + heads_per_span) * per_head;
        const int heads = one_span ? B * Hn : (end - 1) / per_head - bh0 + 1;
        const int n = end - first;
        const dim3 grid((unsigned)(n < resident ? n : resident));
        if (bounded)
            BSA_FRAG_LAUNCH(true, grid, first, end, (const int32_t*)nullptr, (uint32_t*)nullptr, 0u, bh0, (uint32_t)(heads * kv_bh_bytes), fb_list, fb_count);
        else
            BSA_FRAG_LAUNCH(false, grid, first, end, (const int32_t*)nullptr, (uint32_t*)nullptr, 0u, bh0, (uint32_t)(heads * kv_bh_bytes),
                            (int32_t*)nullptr, (uint32_t*)nullptr);
        first = end;
    }
    if (whole < total) {
        if (split.parts > 1) parts = {part_buf, split.parts, tail, divisor(split.parts), divisor(tail)};
        const int n = (total - whole) * split.parts;
        const dim3 grid((unsigned)(split.team == 1 && n > resident ? resident : n));
#define BSA_FRAG_TAIL grid, whole, total, (const int32_t*)nullptr, (uint32_t*)nullptr, 0u, 0, whole_span, gate_lists, gate_lens
        if (few) {
            const FragCall c = {q, kf, vf, idx, lens, tile_valid, o, lse, Sq, Sk, lse_rows, bs_k, idx_stride, Hn, dtype, qk_scale, halves, st};
            const hipError_t e = launch_fwd_few(c, L, parts, total, split.team, here.qc != nullptr ? &here : nullptr, gate_lists, gate_lens, whole_span);
            if (e != hipSuccess) return e;
        } else if (split.team == 4) BSA_FRAG_LAUNCH_LISTED(4, BSA_FRAG_TAIL);      // 4 x more than kBusyWide / 2 items are not one round: no selection inside
        else if (split.team == 2) BSA_FRAG_LAUNCH_ONCE(2, BSA_FRAG_TAIL);
        else if (once) BSA_FRAG_LAUNCH_ONCE(1, BSA_FRAG_TAIL);
        else BSA_FRAG_LAUNCH(false, BSA_FRAG_TAIL);
#undef BSA_FRAG_TAIL
    }
    if (split.parts > 1) {
        if (dtype == BSA_BF16)
            hipLaunchKernelGGL((merge_parts_kernel<__bf16>), dim3(tail), dim3(256), 0, st, parts, (__bf16*)o, lse, whole, per_head, Hn, lse_rows, L);
        else
            hipLaunchKernelGGL((merge_parts_kernel<_Float16>), dim3(tail), dim3(256), 0, st, parts, (_Float16*)o, lse, whole, per_head, Hn, lse_rows, L);
        parts = {nullptr, 1, 0, divisor(1), divisor(1)};
    }
    if (bounded) {
        // what the schedule that ran left over, be it the rounds or the queues: as many items as the list holds,
        // found out on the device.  Not behind the gate of either: only the one that ran has put items on the list.
        gate = nullptr;
        const dim3 grid((unsigned)(all_tiles < resident ? all_tiles : resident));
        BSA_FRAG_LAUNCH(false, grid, 0, all_tiles, (const int32_t*)fb_list, (uint32_t*)nullptr, 0u, 0, whole_span, (int32_t*)nullptr, fb_count);
    }
#undef BSA_FRAG_LAUNCH
#undef BSA_FRAG_LAUNCH_ONCE
#undef BSA_FRAG_LAUNCH_LISTED
#undef BSA_FRAG_LAUNCH_W
#undef BSA_FRAG_LAUNCH_T
    return hipGetLastError();
}

}  // namespace bsa
