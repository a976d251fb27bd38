// Decode of Q4_0 rows of K = 9,216 to 16,384 in whole 1,024-weight blocks
// (G = 32 S groups, S = 9 .. 16 groups a range) — the down projections of
// the 7-8B models (Llama 3 8B and Mistral 7B: 4,096 x 14,336) — streamed
// through LDS.
//
// Why: a range here is S groups, so the reference's mapping (lane r of a
// half-wave owns range r, matmul.wgsl:207-243) has each lane load 16 bytes
// at a stride of 16 S bytes — 32 cache lines a load instruction — and the
// chunked kernel built on it (gemv.hip, gemv_chunked) reads 4,096 x 14,336
// at 1.5 TB/s. The mapping itself is what the order of addition fixes: a
// range's sum is one chain over its groups in order, so a range belongs to
// one lane and a row to 32 lanes. What changes is how the bytes arrive: a
// wave loads its step's two rows coalesced, eight lanes one range's half (its
// first or last ceil(S / 2) groups, up to 128 bytes in a row), and passes them to
// the ranges' lanes through its LDS stage, a half at a time.
//
// Why halves: the chains are serial, 32 S fmas with their decode, so a CU
// wants two waves a SIMD, and beside x (4 S KB) LDS holds eight stages of half
// a step but only four of a whole one. The whole step is in flight in
// registers all the same (64 of them; a half goes to the stage when the other
// has been taken), and the next step's loads go out before this one's decode.
// Four waves with whole stages, filled by global_load_lds, ran 4,096 x 14,336
// in two rounds of steps, neither hidden: 16.2 us; so 13.2 (4,096 x 9,216 11.0
// -> 9.8, gated 14,336 x 12,288 59.3 -> 48.5). The loads are plain ones: a
// range's halves share lines (non-temporal 14.6 us).
//
// Stage layout: a row's half of codes — 16-byte slot 8 r + (e xor r mod 8)
// holds the half's group e of range r — so that the lanes reading group e of
// their ranges fall in different banks; the row's 2 G bytes of scales in
// order. x is staged once a workgroup, range-interleaved as gemv_ranges
// stages it (float4 v of a range's group i at 256 i + 32 v + r).
// A row's 32 range sums meet in LDS and lane 0 or 1 adds them in order; the
// bits are every other kernel's.
#include <algorithm>

#include "decode.hpp"
#include "plan.hpp"
#include "product.hpp"
#include "stream.hpp"

namespace chm {

namespace {

constexpr uint32_t kWideWaves = 8;  // one workgroup a CU: x and eight half stages fill LDS
constexpr uint32_t kWideMinSpan = 9, kWideMaxSpan = 16;
constexpr uint32_t kWideSumPad = 36;  // a row's 32 range sums, 16-byte aligned
constexpr uint32_t kHalfSlots = 256;  // 16-byte slots of a row's half in the stage: 8 a range
constexpr uint32_t kScaleSlots = 2 * kWideMaxSpan * 2;  // and of a row's scales

// A wave's own LDS, written by some of its lanes and read by others: its LDS
// operations execute in order, so the compiler's view is all there is to order.
__device__ __forceinline__ void stage_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace

template <uint32_t S, bool FULL>
__global__ __launch_bounds__(64 * kWideWaves) void gemv_wide(Product a, uint32_t steps) {
    constexpr uint32_t G = 32 * S;
    constexpr uint32_t kHalf = (S + 1) / 2;  // groups of a range's first half; S - kHalf of its last
    static_assert(kHalf <= 8 && S / 8 <= 2, "a half is at most eight groups a range");
    __shared__ u32x4s_t x_stage[S * 256];
    __shared__ u32x4s_t codes_a[kWideWaves][2 * kHalfSlots];
    __shared__ u32x4s_t scales_a[kWideWaves][2 * kScaleSlots];
    __shared__ float sums_a[kWideWaves][2 * kWideSumPad];
    const float4* const xs = reinterpret_cast<const float4*>(x_stage);

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t h = lane >> 5, r = lane & 31u;
    const uint32_t token = a.last_token ? a.tokens - 1 : 0;
    u32x4s_t *const codes_s = codes_a[wave], *const scales_s = scales_a[wave];
    float* const sums_s = sums_a[wave];

    // Thread t stages range t % 32, float4 t / 32 % 8 of every second group,
    // clamped where the product is clipped; every load before any store, and
    // all of them before the first step's.
    constexpr uint32_t kPasses = (S + 1) / 2;
    const uint32_t sr = threadIdx.x & 31u, sv = (threadIdx.x >> 5) & 7u, si = threadIdx.x >> 8;
    float4 xv[kPasses];
    {
        const float4* src = reinterpret_cast<const float4*>(a.x + static_cast<uint64_t>(token) * G * 32);
#pragma unroll
        for (uint32_t k = 0; k < kPasses; ++k) xv[k] = src[(S * sr + min(2 * k + si, S - 1)) * 8 + sv];
    }

    // A step's loads. Instruction k of a row's half fills its slots 64 k ..
    // 64 k + 63, lane l slot 64 k + l = 8 rr + e', i.e. range rr's group (e' xor
    // rr mod 8) of the half; slots past the half's groups load its last again.
    // A row past the product loads the last row again.
    u32x4s_t half0[2][4], half1[2][4], scales[2];
    const uint32_t e = (lane & 7u) ^ ((lane >> 3) & 7u);
    const uint32_t from0 = S * (lane >> 3) + min(e, kHalf - 1);
    const uint32_t from1 = S * (lane >> 3) + min(kHalf + e, S - 1);
    auto load = [&](uint32_t step) {
#pragma unroll
        for (uint32_t hh = 0; hh < 2; ++hh) {
            const Piece w = piece_of(a, min(2 * step + hh, a.rows - 1));
            const u32x4s_t* codes = reinterpret_cast<const u32x4s_t*>(w.piece) + static_cast<uint64_t>(w.row) * G;
            const u32x4s_t* sc = reinterpret_cast<const u32x4s_t*>(w.piece + 16 * w.blocks + 2 * (static_cast<uint64_t>(w.row) * G));
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) half0[hh][k] = codes[8 * S * k + from0];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) half1[hh][k] = codes[8 * S * k + from1];
            scales[hh] = sc[min(lane, 4 * S - 1)];
        }
    };
    auto stage = [&](const u32x4s_t (&half)[2][4]) {
#pragma unroll
        for (uint32_t hh = 0; hh < 2; ++hh)
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) codes_s[kHalfSlots * hh + 64 * k + lane] = half[hh][k];
    };

    uint32_t step = blockIdx.x + gridDim.x * wave;
    const uint32_t waves = gridDim.x * kWideWaves;
    if (step < steps) load(step);
#pragma unroll
    for (uint32_t k = 0; k < kPasses; ++k) {
        const uint32_t i = 2 * k + si;
        const float4 q = clamp_input(a, xv[k]);
        if (i < S)
            x_stage[256 * i + 32 * sv + sr] = u32x4s_t{__float_as_uint(q.x), __float_as_uint(q.y),
                                                       __float_as_uint(q.z), __float_as_uint(q.w)};
    }
    __syncthreads();
    for (; step < steps; step += waves) {
        // The lane's range, both halves by way of the stage.
        u32x4s_t codes[S];
        uint32_t d[S];
        stage(half0);
#pragma unroll
        for (uint32_t hh = 0; hh < 2; ++hh) scales_s[kScaleSlots * hh + lane] = scales[hh];
        stage_sync();
        const u32x4s_t* const mine = codes_s + kHalfSlots * h + 8 * r;
        const uint16_t* const sc = reinterpret_cast<const uint16_t*>(scales_s + kScaleSlots * h) + S * r;
#pragma unroll
        for (uint32_t i = 0; i < kHalf; ++i) codes[i] = mine[i ^ (r & 7u)];
#pragma unroll
        for (uint32_t i = 0; i < S; ++i) d[i] = sc[i];
        stage_sync();
        stage(half1);
        stage_sync();
#pragma unroll
        for (uint32_t i = kHalf; i < S; ++i) codes[i] = mine[(i - kHalf) ^ (r & 7u)];
        if (step + waves < steps) load(step + waves);
        // The range's chain over its groups, its sum to LDS, then lanes 0 and 1
        // add rows 2 step and 2 step + 1's 32 sums in order (matmul.h:34-50).
        float s = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < S; ++i) {
            float xg[32];
#pragma unroll
            for (uint32_t v = 0; v < 8; ++v) {
                const float4 q = xs[256 * i + 32 * v + r];
                xg[4 * v] = q.x, xg[4 * v + 1] = q.y, xg[4 * v + 2] = q.z, xg[4 * v + 3] = q.w;
            }
            const uint32_t w[4] = {codes[i][0], codes[i][1], codes[i][2], codes[i][3]};
            s = chain_q4_0_wide(w, d[i], xg, s);
        }
        sums_s[kWideSumPad * h + r] = s;
        stage_sync();
        float total = 0.0f;
        if (lane < 2) total = ordered_total(sums_s + kWideSumPad * lane);
        float partner = 0.0f;
        if (FULL && a.epilogue == kGated) partner = __shfl_xor(total, 1);
        const uint32_t p = 2 * step + lane;
        if (lane < 2 && p < a.rows) emit<FULL>(a, p, 0, token, total, partner);
        stage_sync();
    }
}

// Whether this kernel takes the product: Q4_0, K a whole number of 1,024-
// weight blocks from 9,216 to 16,384 (every range S groups). Rows are copied
// one at a time, so members and gated products take any rows.
bool gemv_wide_takes(const Product& a, uint32_t format) {
    if (format != kQ4_0 || a.groups % 32 != 0) return false;
    const uint32_t span = a.groups / 32;
    return span >= kWideMinSpan && span <= kWideMaxSpan;
}

// A workgroup a CU, fewer where each then has four steps at least: the first
// steps go a workgroup each, so four waves of eight share a small product's x.
uint64_t gemv_wide_workgroups(uint32_t compute_units, uint64_t steps) {
    return std::min<uint64_t>(compute_units, (steps + 3) / 4);
}

template <uint32_t S>
static void go_wide(const Product& a, uint32_t compute_units, hipStream_t stream) {
    const uint32_t steps = (a.rows + 1) / 2;
    const uint32_t blocks = static_cast<uint32_t>(gemv_wide_workgroups(compute_units, steps));
    if (plain_epilogue(a))
        hipLaunchKernelGGL((gemv_wide<S, false>), dim3(blocks), dim3(64 * kWideWaves), 0, stream, a, steps);
    else
        hipLaunchKernelGGL((gemv_wide<S, true>), dim3(blocks), dim3(64 * kWideWaves), 0, stream, a, steps);
}

hipError_t launch_gemv_wide(const Product& a, uint32_t compute_units, hipStream_t stream) {
    switch (a.groups / 32) {
        case 9: go_wide<9>(a, compute_units, stream); break;
        case 10: go_wide<10>(a, compute_units, stream); break;
        case 11: go_wide<11>(a, compute_units, stream); break;
        case 12: go_wide<12>(a, compute_units, stream); break;
        case 13: go_wide<13>(a, compute_units, stream); break;
        case 14: go_wide<14>(a, compute_units, stream); break;
        case 15: go_wide<15>(a, compute_units, stream); break;
        case 16: go_wide<16>(a, compute_units, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace chm
