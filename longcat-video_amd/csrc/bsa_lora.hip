// The up-projection of one LoRA side branch and its sum with the layer's output, in one pass (HBM-bound: the layer's output
// read and written once; the rank axis and the up weights stay in the caches).
//
//   out = T(org + s),  s = T(T(up * multiplier) * alpha),  up = T(lora_up(t)),  t = lora_down(x)
//
// with the eager expression's roundings.  lora_up is one matrix [N, rank], or n_sep of them for a fused layer, each with its
// own rank columns of t and its own N / n_sep output columns.
#include "bsa_mfma.h"

namespace bsa {
namespace {

using namespace mfma;

constexpr int kMaxSlices = 8, kMaxRank = 128;
constexpr int kCols = 256;           // output columns of a workgroup, 64 per wavefront
constexpr int kRows = 32;              // tokens of a turn
constexpr int kPitch = kCols + 8;    // elements between the staged rows
constexpr int kGroups = 768;         // workgroups of a launch, about: three a CU (1 536: 543 us, 6 144: 595, sizes below); never more than turns

struct UpSlices {
    const __bf16* w[kMaxSlices];     // [per, rank]
    int per;
};

// A workgroup keeps the up weights of its 256 columns in registers, in MFMA operand order, and walks over the tokens, 32 a
// turn: lane l of a product holds token l % 32 and four columns at a time, which go through LDS so that org is read and
// out is written in whole 512-byte runs.  t of the next turn is asked for as soon as its registers are free, org of a turn in
// front of its products.  kSteps: rank / 16.
//
// 32 760 tokens, rank 128, 12 288 columns in three slices and 4 096 in one: 537 us = 4.0 TB/s, for 943 us of up-projections
// (hipBLASLt, 364) and lora_add_kernel (579) before.  64 tokens a turn, two workgroups a CU 631; org a turn ahead 566 (its
// registers cost more than the wait).  It is taken wherever it is built and the engine's GEMM does not take the branch into its sum (lora_serves): one pass / separate ones, us, by tokens 1, 256, 4 096,
// 32 760: 4 096 columns, rank 16 4.3 / 20.8, 4.0 / 20.7, 12.0 / 32.6, 86 / 242, rank 128 4.5 / 20.6, 6.0 / 20.4, 22.8 / 29.3, 120 / 230;
// 12 288 in three, rank 16 4.0 / 41, 4.8 / 41, 33 / 85, 310 / 701, rank 128 4.5 / 41, 9.5 / 41, 50 / 80, 369 / 675; 512 columns, rank 128,
// 4.4 / 20.4, 5.7 / 20.2, 6.4 / 20.3, 23.7 / 31.4 (below 30 us the separate ones wait for the host).
template <int kSteps>
__global__ __launch_bounds__(256, 3) void lora_up_add_kernel(const __bf16* org, const __bf16* __restrict__ t, int64_t ldt, UpSlices up,
                                                             float multiplier, float alpha, __bf16* out, int64_t M, int N, int col_blocks,
                                                             int row_groups) {
    constexpr int kRank = 16 * kSteps;
    __shared__ __attribute__((aligned(16))) __bf16 stage[kRows * kPitch];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 31, lh = lane >> 5;
    const int col0 = (int)(blockIdx.x % col_blocks) * kCols, mine = col0 + 64 * wave;
    const bool active = mine < N;                                  // N is a multiple of 64
    const int slice = active ? mine / up.per : 0;
    bf16x8 a[2][kSteps];
    if (active) {
        const __bf16* w = up.w[slice] + (int64_t)(mine - slice * up.per + lr) * kRank + 8 * lh;
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int c = 0; c < kSteps; ++c) a[f][c] = *reinterpret_cast<const bf16x8*>(w + f * 32 * kRank + 16 * c);
    }
    const __bf16* tw = t + slice * kRank + 8 * lh;
    const int pc = threadIdx.x & 31, pr = threadIdx.x >> 5;        // 16-byte piece and row (of 8 at a time) of the copy
    const bool copies = col0 + 8 * pc < N;
    const __bf16* from = org + col0 + 8 * pc;
    __bf16* to = out + col0 + 8 * pc;
    const int64_t hop = (int64_t)row_groups * kRows;
    int64_t row0 = (int64_t)(blockIdx.x / col_blocks) * kRows;
    bf16x8 b[kSteps];
    auto load_t = [&](int64_t first) {
        const int64_t row = first + lr;
        const __bf16* tr = tw + (row < M ? row : M - 1) * ldt;
#pragma unroll
        for (int c = 0; c < kSteps; ++c) b[c] = *reinterpret_cast<const bf16x8*>(tr + 16 * c);
    };
    uint4 piece[kRows / 8];
    auto load_org = [&](int64_t first) {
#pragma unroll
        for (int i = 0; i < kRows / 8; ++i) {
            const int64_t row = first + pr + 8 * i;
            piece[i] = *reinterpret_cast<const uint4*>(from + (row < M ? row : M - 1) * N);
        }
    };
    if (active) load_t(row0);
    for (; row0 < M; row0 += hop) {
        if (copies) load_org(row0);
        if (active) {
            f32x16 acc[2];
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[f][i] = 0.f;
#pragma unroll
            for (int c = 0; c < kSteps; ++c)
#pragma unroll
                for (int f = 0; f < 2; ++f) acc[f] = mfma32(a[f][c], b[c], acc[f]);
            if (row0 + hop < M) load_t(row0 + hop);
            // accumulator i <-> column 32 f + 8 (i / 4) + 4 lh + i % 4 of token lr
            __bf16* srow = stage + lr * kPitch + 64 * wave + 4 * lh;
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    __bf16 x[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float u = (float)(__bf16)acc[f][4 * g + k];
                        x[k] = (__bf16)__fmul_rn((float)(__bf16)__fmul_rn(u, multiplier), alpha);
                    }
                    *reinterpret_cast<uint2*>(srow + 32 * f + 8 * g) = *reinterpret_cast<const uint2*>(x);
                }
        }
        __syncthreads();
        if (copies) {
#pragma unroll
            for (int i = 0; i < kRows / 8; ++i) {
                const int64_t row = row0 + pr + 8 * i;
                const uint4 sraw = *reinterpret_cast<const uint4*>(stage + (pr + 8 * i) * kPitch + 8 * pc);
                const __bf16* s = reinterpret_cast<const __bf16*>(&sraw);
                const __bf16* o = reinterpret_cast<const __bf16*>(&piece[i]);
                __bf16 res[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) res[k] = (__bf16)__fadd_rn((float)o[k], (float)s[k]);
                if (row < M) *reinterpret_cast<uint4*>(to + row * N) = *reinterpret_cast<const uint4*>(res);
            }
        }
        __syncthreads();
    }
}

}  // namespace
}  // namespace bsa

using namespace bsa;

extern "C" int bsa_lora_up_add(const void* org, const void* t, int64_t ldt, const void* const* up, int n_sep, int rank, float multiplier,
                               float alpha_scale, void* out, int64_t M, int N, void* stream) {
    if (!org || !t || !up || !out) return set_error(BSA_ERR_BAD_ARG, "lora_up_add: null pointer");
    if (M <= 0 || N <= 0 || n_sep <= 0 || rank <= 0) return set_error(BSA_ERR_BAD_ARG, "lora_up_add: sizes must be positive");
    if (n_sep > kMaxSlices || rank % 16 || rank > kMaxRank || N % n_sep || (N / n_sep) % 64)
        return set_error(BSA_ERR_UNSUPPORTED, "lora_up_add: rank a multiple of 16 up to 128, up to 8 slices of a multiple of 64 columns (rank %d, %d columns in %d)", rank, N, n_sep);
    if (ldt < (int64_t)n_sep * rank || ldt % 8) return set_error(BSA_ERR_BAD_ARG, "lora_up_add: rows of t lie %lld elements apart", (long long)ldt);
    UpSlices s{};
    s.per = N / n_sep;
    uintptr_t bits = reinterpret_cast<uintptr_t>(org) | reinterpret_cast<uintptr_t>(t) | reinterpret_cast<uintptr_t>(out);
    for (int i = 0; i < n_sep; ++i) {
        if (!up[i]) return set_error(BSA_ERR_BAD_ARG, "lora_up_add: null pointer");
        s.w[i] = static_cast<const __bf16*>(up[i]);
        bits |= reinterpret_cast<uintptr_t>(up[i]);
    }
    if (bits & 15u) return set_error(BSA_ERR_BAD_ARG, "lora_up_add: pointers must be 16-byte aligned");
    // a workgroup's turns lie `groups` turns apart, so that the workgroups of a moment share their tokens' rows
    const int col_blocks = (N + kCols - 1) / kCols;
    const int64_t turns = (M + kRows - 1) / kRows;
    int64_t groups = (kGroups + col_blocks - 1) / col_blocks;
    if (groups > turns) groups = turns;
    const dim3 grid((unsigned)(groups * col_blocks)), block(256);
#define BSA_LORA(S)                                                                                                                    \
    case S:                                                                                                                            \
        hipLaunchKernelGGL((lora_up_add_kernel<S>), grid, block, 0, (hipStream_t)stream, (const __bf16*)org, (const __bf16*)t, ldt, s, \
                           multiplier, alpha_scale, (__bf16*)out, M, N, col_blocks, (int)groups);                                      \
        break
    switch (rank / 16) {
        BSA_LORA(1); BSA_LORA(2); BSA_LORA(3); BSA_LORA(4); BSA_LORA(5); BSA_LORA(6); BSA_LORA(7); BSA_LORA(8);
    }
#undef BSA_LORA
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? BSA_OK : set_error(BSA_ERR_HIP, "lora_up_add launch: %s", hipGetErrorString(e));
}
