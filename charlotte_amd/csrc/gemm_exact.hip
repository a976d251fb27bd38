// Prefill on the matrix cores in the canonical order: bit-exact.
//
// gemm_exact — v_mfma_f32_32x32x2_f32 (K = 2, one 32 x 32 block) adds its two
// products one after the other, each as a fused multiply-add: d = fmaf(a1,
// b1, fmaf(a0, b0, c)) bit for bit (checked on the GPU by harness.hip's
// mfma_chain_check over random, cancelling, halfway, denormal, overflowing,
// infinite and NaN operands). So a range's chain s = fma(w_k, x_k, s), in k
// order from +0 (matmul.wgsl:121-126, 224-230), runs as a chain of these
// instructions, two ks at a time, for 1,024 outputs at once; a range's sums
// then add into the totals in order on the VALU (matmul.wgsl:134-137), as
// gemm_canonical adds them. Every output is gemm_canonical's bits, and
// decode's.
//
// What bounds it: the f32 matrix instructions and the VALU take turns on a
// SIMD — an instruction of the one adds its whole time to the other's (a
// probe of four independent products and n VALU instructions a wave, at one
// and two waves a SIMD: 72 cycles a product alone, + 4.4 a v_perm_b32 or
// v_fma_mix_f32, + 2.7 a v_add_f32 past the second) — so beside the products
// (64 cycles each, 98% of the FP32 peak where the K = 1 shape sustains 88%)
// the time is the VALU work a product, and the design is what keeps that
// small. The operands of ks 2m and 2m + 1 are one register whose lower
// half-wave holds k 2m and whose upper k 2m + 1: each lane decodes its own
// half of its row's weights (Half below: 32 instructions a Q4_0 group), and
// the inputs lie in LDS split into even and odd ks, so they are read as
// operands with no instruction between. A 32-row group and 64 tokens take 32
// products and about 40 VALU instructions, 32 more at a range's end.
//
// A workgroup takes 256 rows x TB x 32 tokens, eight waves of 32 rows each
// sharing its inputs: each group's are copied once, eight lanes a token's
// 128-byte line (a lane a token touches 64 lines a load, eight times over:
// with the loads spread among the products a line was fetched again for
// each), through registers into a ring of LDS stages, two groups between the
// workgroup's meetings (four: 144 against 142 us at 2,048 x 2,048 x 2,048,
// and a workgroup a CU less). Reading the inputs a slot ahead of their
// products, or spreading the decode among them by hand, measured no better:
// the SIMD's other waves cover the waits. Measured (Q4_0, two sides A/B):
// against the K = 1 form, 64 x 64 a wave with both operands in registers,
// 2,048 tokens through Llama 3.2 1B's layer 2,075 -> 1,968 us (120 -> 127
// TFLOP/s), 4,096 x 1,024 x 512 57 -> 46, 2 x 3,072 x 1,024 x 512 gated 100
// -> 81, 4,096 x 1,152 x 2,048 BF16 181 -> 158, 8,192 x 2,048 x 300 F32 276 ->
// 153 us.
//
// Result layout of the instruction (register v of 16, lane l): column l % 32,
// row 8 (v / 4) + 4 (l / 32) + v % 4 — rows p, p + 1 (p even) in one lane, so
// a gated product's gate and up totals (rows 2r, 2r + 1) meet there.
#include "decode.hpp"
#include "plan.hpp"
#include "product.hpp"
#include "stream.hpp"

namespace chm {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kWaveRows = 32;   // rows a wave
constexpr uint32_t kWaves = 8;       // waves a workgroup, each its own 32 rows

// The upper half-wave of `a` against the lower of `b`: afterwards a holds the
// two lower halves (a's, then b's), b the two upper ones.
__device__ __forceinline__ void swap32(float& a, float& b) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    const uint32_t s0 = s[0], s1 = s[1];
    a = __uint_as_float(s0), b = __uint_as_float(s1);
}

// A lane's share of one row's group for the K = 2 instruction: lane half h
// (lanes 0-31: 0) takes ks h, h + 2, ..., its sixteen weights w of weights_of.
// decode(r, h) works out what the whole group shares; four(j, w) gives ks
// 8j + h, 8j + 2 + h, 8j + 4 + h, 8j + 6 + h. Each lane makes its own half's
// weights alone, so the two lanes of a row do a group's decode between them.
template <uint32_t F>
struct Half;

// Q4_0: a code dword shifted by 8h holds its lane's codes in bytes 0 and 2;
// under 0x54 a half is 64 + m / 16 for its low byte m (chain_q4_0_wide), so
// a mask-and-or makes two of them: (64 + l / 16) 16d - 1032d = (l - 8) d and
// (64 + h) d - 72 d = (h - 8) d, exact. 1.75 instructions a weight.
template <>
struct Half<kQ4_0> {
    uint32_t w[4];
    float d, low, d16, high;
    __device__ __forceinline__ void decode(const Raw<kQ4_0>& r, uint32_t h) {
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = r.w[i] >> (8 * h);
        d = half_to_float(r.d);
        d16 = 16.0f * d, low = -1032.0f * d, high = -72.0f * d;
    }
    __device__ __forceinline__ void four(int j, float* o) const {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bool nib = j >= 2;
            const uint32_t c = w[2 * (j & 1) + i];
            const half2_t u = __builtin_bit_cast(
                half2_t, nib ? and_or(c, 0x00F000F0u, 0x54005400u) : and_or(c, 0x000F000Fu, 0x54005400u));
            o[2 * i] = __builtin_fmaf(static_cast<float>(u.x), nib ? d : d16, nib ? high : low);
            o[2 * i + 1] = __builtin_fmaf(static_cast<float>(u.y), nib ? d : d16, nib ? high : low);
        }
    }
};

// Q4_1: the codes as halves 1024 + q less 1024 (high nibbles 16 q, against
// d / 16: the same product), then fma(q, d, m) — weight()'s one rounding.
template <>
struct Half<kQ4_1> {
    uint32_t w[4];
    float d, m, d16;
    __device__ __forceinline__ void decode(const Raw<kQ4_1>& r, uint32_t h) {
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = r.w[i] >> (8 * h);
        d = half_to_float(r.dm & 0xFFFFu), m = half_to_float(r.dm >> 16);
        d16 = d * 0.0625f;
    }
    __device__ __forceinline__ void four(int j, float* o) const {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bool nib = j >= 2;
            const uint32_t c = w[2 * (j & 1) + i];
            const half2_t base = {1024.0f16, 1024.0f16};
            const half2_t u = __builtin_bit_cast(half2_t, nib ? and_or(c, 0x00F000F0u, 0x64006400u)
                                                              : and_or(c, 0x000F000Fu, 0x64006400u)) -
                              base;
            o[2 * i] = __builtin_fmaf(static_cast<float>(u.x), nib ? d16 : d, m);
            o[2 * i + 1] = __builtin_fmaf(static_cast<float>(u.y), nib ? d16 : d, m);
        }
    }
};

// Two code bytes of a dword, h and h + 2, lifted to binary16 1024 + b.
__device__ __forceinline__ uint32_t half_selector(uint32_t h) { return h ? 0x04030401u : 0x04020400u; }

template <>
struct Half<kQ8_0> {
    uint32_t w[8], selector;
    float d, offset;
    __device__ __forceinline__ void decode(const Raw<kQ8_0>& r, uint32_t h) {
        selector = half_selector(h);
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = r.w[i];
        d = half_to_float(r.d), offset = -1152.0f * d;
    }
    __device__ __forceinline__ void four(int j, float* o) const {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const half2_t u = lift(w[2 * j + i] ^ 0x80808080u, selector);
            o[2 * i] = __builtin_fmaf(static_cast<float>(u.x), d, offset);
            o[2 * i + 1] = __builtin_fmaf(static_cast<float>(u.y), d, offset);
        }
    }
};

// Q6_K: the 6-bit codes assembled as chain_q6_k assembles them.
template <>
struct Half<kQ6_K> {
    uint32_t lo[4], a[2], b[2], selector;
    float first, first_offset, second, second_offset;
    __device__ __forceinline__ void decode(const Raw<kQ6_K>& r, uint32_t h) {
        selector = half_selector(h);
#pragma unroll
        for (int i = 0; i < 4; ++i) lo[i] = r.lo[i];
#pragma unroll
        for (int i = 0; i < 2; ++i) a[i] = r.hi[i] & 0x33333333u, b[i] = (r.hi[i] >> 2) & 0x33333333u;
        const float d = half_to_float(r.d);
        first = d * static_cast<float>(static_cast<int8_t>(r.sc & 0xFFu));
        second = d * static_cast<float>(static_cast<int8_t>((r.sc >> 8) & 0xFFu));
        first_offset = -1056.0f * first, second_offset = -1056.0f * second;
    }
    __device__ __forceinline__ void four(int j, float* o) const {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t pairs = (j & 1) ? b[i] : a[i];  // weights 8j .. 8j + 7: pairs at bits 2j
            const uint32_t l = lo[2 * (j & 1) + i];
            const half2_t u = lift(j < 2 ? bitfield_insert(0x0F0F0F0Fu, l, pairs << 4)
                                         : bitfield_insert(0x0F0F0F0Fu, l >> 4, pairs),
                                   selector);
            const float scale = j < 2 ? first : second, offset = j < 2 ? first_offset : second_offset;
            o[2 * i] = __builtin_fmaf(static_cast<float>(u.x), scale, offset);
            o[2 * i + 1] = __builtin_fmaf(static_cast<float>(u.y), scale, offset);
        }
    }
};

// The plain formats: the lower half-wave loads ks 0 .. 15 of its row, the
// upper 16 .. 31; swapping two neighbours between the halves gives one
// register of ks 2m, 2m + 1 and one of ks 16 + 2m, 17 + 2m, as the halves
// take them.
template <uint32_t F>
struct HalfRaw : Raw<F> {
    __device__ __forceinline__ void load_half(const uint8_t* piece, uint64_t blocks, uint64_t gi, uint32_t) {
        this->load(piece, blocks, gi);
    }
};
template <uint32_t F>
struct PlainHalfRaw {
    static constexpr int kWords = F == kF32 ? 16 : 8;
    uint32_t w[kWords];
    __device__ __forceinline__ void load_half(const uint8_t* piece, uint64_t, uint64_t gi, uint32_t h) {
        const uint4* at = reinterpret_cast<const uint4*>(piece + 8 * kWords * gi + 4 * kWords * h);
#pragma unroll
        for (int v = 0; v < kWords / 4; ++v) {
            const uint4 q = at[v];
            w[4 * v] = q.x, w[4 * v + 1] = q.y, w[4 * v + 2] = q.z, w[4 * v + 3] = q.w;
        }
    }
};
template <>
struct HalfRaw<kF32> : PlainHalfRaw<kF32> {};
template <>
struct HalfRaw<kF16> : PlainHalfRaw<kF16> {};
template <>
struct HalfRaw<kBF16> : PlainHalfRaw<kBF16> {};

template <uint32_t F>
struct PlainHalf {
    float w[16];
    __device__ __forceinline__ void decode(const HalfRaw<F>& r, uint32_t) {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            float e, o;
            if constexpr (F == kF32) {
                e = __uint_as_float(r.w[2 * m]), o = __uint_as_float(r.w[2 * m + 1]);
            } else {
                e = F == kF16 ? half_to_float(r.w[m] & 0xFFFFu) : bf16_low(r.w[m]);
                o = F == kF16 ? half_to_float(r.w[m] >> 16) : bf16_high(r.w[m]);
            }
            swap32(e, o);
            w[m] = e, w[8 + m] = o;
        }
    }
    __device__ __forceinline__ void four(int j, float* o) const {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = w[4 * j + i];
    }
};
template <>
struct Half<kF32> : PlainHalf<kF32> {};
template <>
struct Half<kF16> : PlainHalf<kF16> {};
template <>
struct Half<kBF16> : PlainHalf<kBF16> {};

// A wave's range sums: 32 rows by TB token blocks of 32.
template <int TB>
struct Sums {
    f32x16 v[TB];
};

// SPLIT (the split along K, matmul.wgsl:592-695): `chunks` workgroups a tile,
// chunk c taking ranges [32c / chunks, 32(c + 1) / chunks) and writing each
// range's sum to range_sums ([32][tokens][rows], range first) instead of
// adding it to a total; combine_ranges (gemm.hip) then adds a row's sums in
// order. The range sums are the VALU split's bits, so the outputs are too.
// `quads`: rows a multiple of 4 and range_sums 16-byte aligned, so a lane's
// four registers of consecutive rows go out as one 16-byte store (C6's split
// 20.9 -> 18.3 us against a store a register).
template <int TB>
__device__ __forceinline__ void store_sums(const Product& a, const Sums<TB>& s, uint32_t range, uint32_t R, uint32_t T,
                                           float* range_sums, bool quads) {
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const uint32_t token = T + 32 * tb + (lane & 31u);
        if (token >= a.tokens) continue;
        float* const row = range_sums + (static_cast<uint64_t>(range) * a.tokens + token) * a.rows;
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
            const uint32_t p = R + 2 * v + 4 * (lane >> 5);
            const float q[4] = {s.v[tb][v], s.v[tb][v + 1], s.v[tb][v + 2], s.v[tb][v + 3]};
            if (quads) {
                if (p < a.rows) *reinterpret_cast<float4*>(row + p) = make_float4(q[0], q[1], q[2], q[3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (p + i < a.rows) row[p + i] = q[i];
            }
        }
    }
}

template <uint32_t F, int TB, bool FULL, bool CLIP, bool SPLIT = false>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_exact(Product a, uint32_t token_tiles, uint32_t row_tiles,
                                                             uint32_t chunks, float* range_sums, bool quads) {
    // A group's inputs a stage: [token][half][pair], 16-byte slots swizzled.
    constexpr uint32_t kStage = 256 * TB;  // float4s
    __shared__ float4 stages[4 * kStage];
    const uint32_t lane = threadIdx.x & 63u, half = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Uniform, and held so: what follows from them stays in scalar registers.
    const uint32_t tile_t = __builtin_amdgcn_readfirstlane(blockIdx.x % token_tiles);
    const uint32_t tile_r = __builtin_amdgcn_readfirstlane((blockIdx.x / token_tiles) % row_tiles);
    const uint32_t chunk = __builtin_amdgcn_readfirstlane(blockIdx.x / (token_tiles * row_tiles));
    const uint32_t T = tile_t * 32 * TB, R = (tile_r * kWaves + wave) * kWaveRows;
    const uint32_t G = a.groups;
    const auto lo_of = [&](uint32_t r) { return (r * G) >> 5; };  // range_lo; G is below 2^24
    const uint32_t chunk_r = __builtin_amdgcn_readfirstlane(32 * chunk / chunks);
    const uint32_t g_begin = lo_of(chunk_r);
    const uint32_t g_end = lo_of(__builtin_amdgcn_readfirstlane(32 * (chunk + 1) / chunks));
    if (g_begin >= g_end) return;  // a chunk of empty ranges (G < 32): nothing to write
    const uint32_t g_last = g_end - 1;

    // Rows and tokens past the product read its last row or token; their
    // outputs are never stored. A wave whose rows all lie past it still
    // copies its share of the inputs and meets the others.
    const Piece pc = piece_of(a, min(R + (lane & 31u), a.rows - 1));
    const uint64_t row0 = static_cast<uint64_t>(pc.row) * G;
    // Inputs: of a group's TB x 32 tokens x 8 chunks of 4 ks, thread t copies
    // chunk c = t % 8 of token t / 8 — eight lanes a token's 128-byte line — its
    // even ks and its odd ones to their halves of the token's slots. TB = 1
    // has half as many chunks as threads: the upper 256 take the next group's.
    const uint32_t ct = (threadIdx.x / 8) % (32 * TB), c = threadIdx.x % 8;
    constexpr uint32_t kGroupsACopy = TB == 1 ? 2 : 1;  // groups a copy covers
    const uint32_t copy_group = TB == 1 ? threadIdx.x >> 8 : 0;
    const float4* const x =
        reinterpret_cast<const float4*>(a.x) + min(T + ct, a.tokens - 1) * (G * uint64_t{8}) + c;
    float lo = 0.0f, hi = 0.0f;
    if constexpr (CLIP) lo = *a.clip[0], hi = *a.clip[1];
    // A token's eight 16-byte slots: half h's ks 8j + h .. 8j + 6 + h at slot
    // (4h + j) ^ (token % 8), so a read of one slot for 32 tokens spreads over the banks.
    float2* const store_at = reinterpret_cast<float2*>(stages + copy_group * kStage + 8 * ct);
    const uint32_t even_at = 2 * ((c / 2) ^ (ct & 7u)) + (c & 1u), odd_at = 2 * ((4 + c / 2) ^ (ct & 7u)) + (c & 1u);
    const float4* read_at[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) read_at[j] = stages + 8 * (lane & 31u) + ((4 * half + j) ^ (lane & 7u));

    constexpr int kCopies = 2 / kGroupsACopy;  // copies of a pair of groups
    struct Pair {
        float4 q[kCopies];
    };
    auto load_x = [&](Pair& p, uint32_t g) {
#pragma unroll
        for (int i = 0; i < kCopies; ++i) p.q[i] = x[8 * min(g + i + copy_group, g_last)];
    };
    auto store_x = [&](const Pair& p, uint32_t stage) {
#pragma unroll
        for (int i = 0; i < kCopies; ++i) {
            float4 q = p.q[i];
            if constexpr (CLIP) {
                q.x = clamp_to(q.x, lo, hi), q.y = clamp_to(q.y, lo, hi);
                q.z = clamp_to(q.z, lo, hi), q.w = clamp_to(q.w, lo, hi);
            }
            store_at[2 * kStage * (stage + i) + even_at] = make_float2(q.x, q.z);
            store_at[2 * kStage * (stage + i) + odd_at] = make_float2(q.y, q.w);
        }
    };
    // Every wave's stores of the next stages before any wave reads them, and
    // its reads of these before any stores over them.
    auto meet = [] {
        __asm__ __volatile__("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __asm__ __volatile__("" ::: "memory");
    };

    Sums<TB> s;
    float t[TB][16];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int v = 0; v < 16; ++v) t[tb][v] = 0.0f;
    // Range r, the one being summed, and the groups left in it. Below 32
    // groups a range that holds one holds it alone (group g's is range (32 g +
    // 31) / G); the empty ones hold zero and add nothing.
    uint32_t r = chunk_r;
    if (G < 32) r = __builtin_amdgcn_readfirstlane((32 * g_begin + 31) / G);
    uint32_t left = G < 32 ? 1u : lo_of(r + 1) - lo_of(r);
    bool fresh = true;  // the next product starts a range: its chain from +0

    auto group = [&](const HalfRaw<F>& raw, uint32_t stage, uint32_t g) {
        Half<F> ops;
        ops.decode(raw, half);
        const f32x16 zero = {};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float aw[4];
            ops.four(j, aw);
            float4 q[TB];
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) q[tb] = read_at[j][kStage * stage + 256 * tb];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float bx[TB];
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) bx[tb] = i == 0 ? q[tb].x : i == 1 ? q[tb].y : i == 2 ? q[tb].z : q[tb].w;
                if (j == 0 && i == 0) {
                    // a range's first product takes +0 as its accumulator, as
                    // fma(w, x, +0) does (the sums are never cleared)
                    if (fresh) {
#pragma unroll
                        for (int tb = 0; tb < TB; ++tb)
                            s.v[tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(aw[0], bx[tb], zero, 0, 0, 0);
                        continue;
                    }
                }
#pragma unroll
                for (int tb = 0; tb < TB; ++tb)
                    s.v[tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(aw[i], bx[tb], s.v[tb], 0, 0, 0);
            }
        }
        fresh = --left == 0;
        if (fresh) {  // range r ends
            if constexpr (SPLIT) {
                store_sums(a, s, r, R, T, range_sums, quads);
            } else {
#pragma unroll
                for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const float e = s.v[tb][v];
                        t[tb][v] = t[tb][v] + e;
                    }
            }
            if (G < 32) {
                if constexpr (SPLIT) r = __builtin_amdgcn_readfirstlane((32 * (g + 1) + 31) / G);
                left = 1;
            } else {
                ++r;
                left = lo_of(r + 1) - lo_of(r);
            }
        }
    };

    // Groups go in pairs: a group's codes are loaded one ahead, into one of
    // two buffers, a pair's inputs two pairs ahead, into registers, then LDS.
    // Every fetch is issued on every path (past the last group it reads the
    // last group again, unused), so the count of loads in flight at each wait
    // is the same on every path.
    HalfRaw<F> A, B;
    Pair px;
    auto fetch = [&](HalfRaw<F>& b, uint32_t g) { b.load_half(pc.piece, pc.blocks, row0 + min(g, g_last), half); };
    load_x(px, g_begin);
    fetch(A, g_begin);
    store_x(px, 0);
    load_x(px, g_begin + 2);
    meet();
    // A pair out of stages `stage`, stage + 1; false after the last group.
    auto pair = [&](uint32_t stage, uint32_t g) {
        fetch(B, g + 1);
        store_x(px, stage ^ 2);
        load_x(px, g + 4);
        group(A, stage, g);
        if (g + 1 >= g_end) return false;
        fetch(A, g + 2);
        group(B, stage + 1, g + 1);
        meet();
        return g + 2 < g_end;
    };
    for (uint32_t g = g_begin; pair(0, g) && pair(2, g + 2); g += 4) {
    }
    if constexpr (SPLIT) return;

#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const uint32_t token = T + 32 * tb + (lane & 31u);
        if (token < a.tokens) emit_block<FULL>(a, R, token, t[tb]);
    }
}


// A lane's share of one row's group for the K = 4 instruction: lane quarter q
// (lanes 16 q .. 16 q + 15) takes ks q, 4 + q, ..., 28 + q, its eight weights
// weight()'s values: eight(q, w) makes them from the group's bytes, byte q of
// each code dword, two dwords at a time.
template <uint32_t F>
struct Quarter;

// Byte q of `first` and of `second` as the low bytes of a dword's halves.
__device__ __forceinline__ uint32_t bytes_of(uint32_t first, uint32_t second, uint32_t q) {
    return __builtin_amdgcn_perm(second, first, 0x0C040C00u + 0x00010001u * q);
}

template <>
struct Quarter<kQ4_0> : Raw<kQ4_0> {
    __device__ __forceinline__ void eight(uint32_t q, float* o) const {
        const float s = half_to_float(d), s16 = 16.0f * s, low = -1032.0f * s, high = -72.0f * s;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t p = bytes_of(w[2 * i], w[2 * i + 1], q);
            // (64 + l / 16) 16 d - 1032 d and (64 + h) d - 72 d, as Half<kQ4_0>
            const half2_t l = __builtin_bit_cast(half2_t, and_or(p, 0x000F000Fu, 0x54005400u));
            const half2_t h = __builtin_bit_cast(half2_t, and_or(p, 0x00F000F0u, 0x54005400u));
            o[2 * i] = __builtin_fmaf(static_cast<float>(l.x), s16, low);
            o[2 * i + 1] = __builtin_fmaf(static_cast<float>(l.y), s16, low);
            o[4 + 2 * i] = __builtin_fmaf(static_cast<float>(h.x), s, high);
            o[5 + 2 * i] = __builtin_fmaf(static_cast<float>(h.y), s, high);
        }
    }
};

template <>
struct Quarter<kQ4_1> : Raw<kQ4_1> {
    __device__ __forceinline__ void eight(uint32_t q, float* o) const {
        const float s = half_to_float(dm & 0xFFFFu), m = half_to_float(dm >> 16), s16 = s * 0.0625f;
        const half2_t base = {1024.0f16, 1024.0f16};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t p = bytes_of(w[2 * i], w[2 * i + 1], q);
            const half2_t l = __builtin_bit_cast(half2_t, and_or(p, 0x000F000Fu, 0x64006400u)) - base;
            const half2_t h = __builtin_bit_cast(half2_t, and_or(p, 0x00F000F0u, 0x64006400u)) - base;
            o[2 * i] = __builtin_fmaf(static_cast<float>(l.x), s, m);
            o[2 * i + 1] = __builtin_fmaf(static_cast<float>(l.y), s, m);
            o[4 + 2 * i] = __builtin_fmaf(static_cast<float>(h.x), s16, m);
            o[5 + 2 * i] = __builtin_fmaf(static_cast<float>(h.y), s16, m);
        }
    }
};

template <>
struct Quarter<kQ8_0> : Raw<kQ8_0> {
    __device__ __forceinline__ void eight(uint32_t q, float* o) const {
        const float s = half_to_float(d), offset = -1152.0f * s;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // q + 128 (the sign bit flipped) under 0x64: 1152 + q
            const half2_t u = __builtin_bit_cast(half2_t, bytes_of(w[2 * i], w[2 * i + 1], q) ^ 0x64806480u);
            o[2 * i] = __builtin_fmaf(static_cast<float>(u.x), s, offset);
            o[2 * i + 1] = __builtin_fmaf(static_cast<float>(u.y), s, offset);
        }
    }
};

template <>
struct Quarter<kQ6_K> : Raw<kQ6_K> {
    __device__ __forceinline__ void eight(uint32_t q, float* o) const {
        const float s = half_to_float(d);
        const float first = s * static_cast<float>(static_cast<int8_t>(sc & 0xFFu));
        const float second = s * static_cast<float>(static_cast<int8_t>((sc >> 8) & 0xFFu));
        const float first_offset = -1056.0f * first, second_offset = -1056.0f * second;
        // the pairs' byte m = 4 (c % 2) + q holds dword c's: bits 0, 2 for the
        // low nibbles of dwords 0-1 and 2-3, bits 4, 6 for their high ones
        const uint32_t p01 = bytes_of(lo[0], lo[1], q), p23 = bytes_of(lo[2], lo[3], q), ph = bytes_of(hi[0], hi[1], q);
        constexpr uint32_t kNib = 0x000F000Fu;
        const uint32_t codes[4] = {bitfield_insert(kNib, p01, ph << 4), bitfield_insert(kNib, p23, ph << 2),
                                   bitfield_insert(kNib, p01 >> 4, ph), bitfield_insert(kNib, p23 >> 4, ph >> 2)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const half2_t u = __builtin_bit_cast(half2_t, and_or(codes[i], 0x003F003Fu, 0x64006400u));
            const float scale = i < 2 ? first : second, offset = i < 2 ? first_offset : second_offset;
            o[2 * i] = __builtin_fmaf(static_cast<float>(u.x), scale, offset);
            o[2 * i + 1] = __builtin_fmaf(static_cast<float>(u.y), scale, offset);
        }
    }
};

template <>
struct Quarter<kF32> {  // the quarter's own eight values
    uint32_t w[8];
    __device__ __forceinline__ void eight(uint32_t, float* o) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = __uint_as_float(w[j]);
    }
};

// BF16: value q of each four, half q % 2 of dword q / 2 of two.
template <>
struct Quarter<kBF16> : Raw<kBF16> {
    __device__ __forceinline__ void eight(uint32_t q, float* o) const {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            o[j] = __uint_as_float(__builtin_amdgcn_perm(w[2 * j + 1], w[2 * j], 0x01000C0Cu + 0x02020000u * q));
    }
};

template <>
struct Quarter<kF16> {  // the quarter's own eight halves, two a dword
    uint32_t w[4];
    __device__ __forceinline__ void eight(uint32_t, float* o) const {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o[2 * i] = half_to_float(w[i] & 0xFFFFu), o[2 * i + 1] = half_to_float(w[i] >> 16);
    }
};

// How sixteen rows' codes reach a wave, kBatch groups at a time: loaded by
// lanes that read a row's bytes side by side (the four lanes that decode a
// row's group would read the same bytes four times, sixteen lines a quarter
// of the wave), stored in the wave's LDS stage, and read back by each lane a
// group at a time. The quantized formats: four groups, lane l row l / 4's group
// l % 4; a record's 16-byte words at place 4 row + (group ^ (row / 2 % 4)),
// so that a read of one group for sixteen rows spreads over the banks.
template <uint32_t F>
struct Codes {
    static constexpr int kBatch = 4;
    static constexpr uint32_t kWide = F == kQ8_0 ? 2 : 1;                                 // 16-byte words a record
    static constexpr uint32_t kWords = 64 * (4 * kWide + (F == kQ6_K ? 2 : 0) + 1);  // LDS words
    Raw<F> raw;
    static __device__ __forceinline__ uint32_t load_row(uint32_t lane) { return lane >> 2; }
    __device__ __forceinline__ void load(const uint8_t* piece, uint64_t blocks, uint64_t row0, uint32_t g, uint32_t last,
                                         uint32_t lane) {
        raw.load(piece, blocks, row0 + min(g + (lane & 3u), last));
    }
    __device__ __forceinline__ void put(float* stage, uint32_t lane) const {
        uint4* const wide = reinterpret_cast<uint4*>(stage);
        const uint32_t row = lane >> 2, at = 4 * row + ((lane ^ (row >> 1)) & 3u);
        uint32_t tail;
        if constexpr (F == kQ6_K) {
            wide[at] = make_uint4(raw.lo[0], raw.lo[1], raw.lo[2], raw.lo[3]);
            reinterpret_cast<uint2*>(stage + 256)[lane] = make_uint2(raw.hi[0], raw.hi[1]);
            tail = raw.sc | (raw.d << 16);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < kWide; ++i)
                wide[64 * i + at] = make_uint4(raw.w[4 * i], raw.w[4 * i + 1], raw.w[4 * i + 2], raw.w[4 * i + 3]);
            if constexpr (F == kQ4_1)
                tail = raw.dm;
            else
                tail = raw.d;
        }
        reinterpret_cast<uint32_t*>(stage + kWords - 64)[lane] = tail;
    }
    static __device__ __forceinline__ void get(Quarter<F>& out, const float* stage, uint32_t j, uint32_t lane) {
        const uint4* const wide = reinterpret_cast<const uint4*>(stage);
        const uint32_t row = lane & 15u, at = 4 * row + (j ^ ((row >> 1) & 3u));
        const uint32_t tail = reinterpret_cast<const uint32_t*>(stage + kWords - 64)[4 * row + j];
        if constexpr (F == kQ6_K) {
            const uint4 l = wide[at];
            const uint2 h = reinterpret_cast<const uint2*>(stage + 256)[4 * row + j];
            out.lo[0] = l.x, out.lo[1] = l.y, out.lo[2] = l.z, out.lo[3] = l.w;
            out.hi[0] = h.x, out.hi[1] = h.y;
            out.sc = tail & 0xFFFFu, out.d = tail >> 16;
        } else {
#pragma unroll
            for (uint32_t i = 0; i < kWide; ++i) {
                const uint4 c = wide[64 * i + at];
                out.w[4 * i] = c.x, out.w[4 * i + 1] = c.y, out.w[4 * i + 2] = c.z, out.w[4 * i + 3] = c.w;
            }
            if constexpr (F == kQ4_1)
                out.dm = tail;
            else
                out.d = tail;
        }
    }
};

// F16 and BF16: a group, 64 bytes a row, lane l row l / 4's 16 bytes l % 4.
// BF16's are read back whole; F16's, whose values each cost a conversion past
// the pick, are stored [row][quarter][l % 4], a dword the quarter's two values
// of the eight (4 picks for 8, a lane reads its 16 bytes alone, and 126 registers
// in place of 136 let two 32 x 16 workgroups on a CU: 6,144 x 1,024 x 100
// 32.6 -> 32.3 us, 16,384 x 1,024 x 5 12.7 -> 10.8; BF16 so 1-2% slower).
template <uint32_t F>
struct HalfCodes {
    static constexpr int kBatch = 1;
    static constexpr uint32_t kWords = 256;
    uint32_t raw[4];
    static __device__ __forceinline__ uint32_t load_row(uint32_t lane) { return lane >> 2; }
    // 16-byte slot i of a row's four.
    static __device__ __forceinline__ uint32_t slot(uint32_t row, uint32_t i) { return 4 * row + (i ^ ((row >> 1) & 3u)); }
    __device__ __forceinline__ void load(const uint8_t* piece, uint64_t, uint64_t row0, uint32_t g, uint32_t last,
                                         uint32_t lane) {
        const uint4 c = reinterpret_cast<const uint4*>(piece + 64 * (row0 + min(g, last)))[lane & 3u];
        raw[0] = c.x, raw[1] = c.y, raw[2] = c.z, raw[3] = c.w;
    }
    __device__ __forceinline__ void put(float* stage, uint32_t lane) const {
        if constexpr (F == kF16) {
            uint32_t* const words = reinterpret_cast<uint32_t*>(stage);
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)  // half q % 2 of dword q / 2 of the first four values, and of the second
                words[4 * slot(lane >> 2, q) + (lane & 3u)] =
                    __builtin_amdgcn_perm(raw[2 + q / 2], raw[q / 2], q % 2 ? 0x07060302u : 0x05040100u);
        } else {
            reinterpret_cast<uint4*>(stage)[slot(lane >> 2, lane & 3u)] = make_uint4(raw[0], raw[1], raw[2], raw[3]);
        }
    }
    static __device__ __forceinline__ void get(Quarter<F>& out, const float* stage, uint32_t, uint32_t lane) {
        const uint4* const wide = reinterpret_cast<const uint4*>(stage);
        const uint32_t row = lane & 15u;
        constexpr uint32_t slots = F == kF16 ? 1 : 4;
#pragma unroll
        for (uint32_t i = 0; i < slots; ++i) {
            const uint4 c = wide[slot(row, F == kF16 ? lane >> 4 : i)];
            out.w[4 * i] = c.x, out.w[4 * i + 1] = c.y, out.w[4 * i + 2] = c.z, out.w[4 * i + 3] = c.w;
        }
    }
};
template <>
struct Codes<kF16> : HalfCodes<kF16> {};
template <>
struct Codes<kBF16> : HalfCodes<kBF16> {};

// Where element e of a 32-value line's chunk c (values 4c .. 4c + 3, e = k % 4)
// goes in operand order, and where a lane of quarter q reads values q, 4 + q,
// ..: [line][q][j], 16-byte slot 2q + j / 4 of a line's eight at (2q + j / 4) ^
// (line % 8), so that a read of one slot for 16 lines spreads over the banks.
__device__ __forceinline__ uint32_t operand_word(uint32_t line, uint32_t c, uint32_t e) {
    return 32 * line + 4 * ((2 * e + (c >> 2)) ^ (line & 7u)) + (c & 3u);
}
__device__ __forceinline__ uint32_t operand_slot(uint32_t line, uint32_t q, uint32_t i) {
    return 8 * line + ((2 * q + i) ^ (line & 7u));
}

// F32: a group, 128 bytes a row, in operand order as the inputs are.
template <>
struct Codes<kF32> {
    static constexpr int kBatch = 1;
    static constexpr uint32_t kWords = 512;
    float4 raw[2];
    static __device__ __forceinline__ uint32_t load_row(uint32_t lane) { return lane >> 3; }  // and 8 past it
    __device__ __forceinline__ void load(const uint8_t* const (&piece)[2], const uint64_t (&row0)[2], uint32_t g,
                                         uint32_t last, uint32_t lane) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            raw[i] = reinterpret_cast<const float4*>(piece[i] + 128 * (row0[i] + min(g, last)))[lane & 7u];
    }
    __device__ __forceinline__ void put(float* stage, uint32_t lane) const {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t line = 8 * i + (lane >> 3), c = lane & 7u;
            stage[operand_word(line, c, 0)] = raw[i].x;
            stage[operand_word(line, c, 1)] = raw[i].y;
            stage[operand_word(line, c, 2)] = raw[i].z;
            stage[operand_word(line, c, 3)] = raw[i].w;
        }
    }
    static __device__ __forceinline__ void get(Quarter<kF32>& out, const float* stage, uint32_t, uint32_t lane) {
        const uint4* const at = reinterpret_cast<const uint4*>(stage);
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
            const uint4 c = at[operand_slot(lane & 15u, lane >> 4, i)];
            out.w[4 * i] = c.x, out.w[4 * i + 1] = c.y, out.w[4 * i + 2] = c.z, out.w[4 * i + 3] = c.w;
        }
    }
};

// gemm_exact_short — a short step on the matrix cores: the canonical order
// with K split among a workgroup's waves, as gemm_short splits it on the
// VALU. A step of few tokens gives gemm_exact few waves, each walking all of
// K; here a workgroup takes RB x 16 rows by TB x 16 tokens and its eight
// waves four of the 32 ranges each. A range's chain runs on
// v_mfma_f32_16x16x4_f32 (K = 4, four fused multiply-adds an element in k
// order: harness.hip's mfma_chain_check): lane quarter q supplies ks 4j + q
// of row R + l % 16 as A (Quarter) and of token T + l % 16 as B, and register
// v of block (rb, tb) is row 4 (l / 16) + v, column l % 16.
//
// A wave copies what it multiplies itself — its rows' codes (Codes), and a
// group's inputs, eight lanes a token's 128-byte line — through its own LDS
// stage, where lanes find them in operand order; loads run four groups
// ahead. At a range's end its sums go to LDS ([range][block][lane], 16 bytes a
// lane), the wave's last range's (wave 0: its four ranges' total, added in
// order from zero) to its stage, no longer needed. After a barrier each
// thread adds two rows' sums in order, skipping empty ranges (G < 32) — rows
// p, p + 1 of one token, so a gated pair's totals meet in the thread:
// gemm_canonical's order, its bits.
//
// What bounds it: the f32 products and the VALU take turns on a SIMD
// (above): 8 products of 32 cycles a 16 x 16 block and group, beside 18 VALU
// instructions of Q4_0 decode a 16-row group and a few of addresses; then the
// L1's lines (a row's group read by the four lanes that decode it cost 26
// against 17 us at 16,384 x 2,048 x 5 tokens) and, at few groups a wave, the
// launch, the first loads' round trip and the combine. Measured against the
// K = 1 forms (a pair of ranges, or four, the blocks of one instruction, two
// groups' inputs staged by LDS copies), us: Q4_0 16,384 x 2,048 at 5 tokens
// 32.3 -> 15.6, 8,192 x 2,048 at 16 / 64 13.2 -> 9.7 / 33.2 -> 30.0, 2,048 x
// 8,192 at 5 / 32 18.7 -> 14.8 / 19.3 -> 15.2, 4,096 x 2,048 x 32 13.2 -> 9.7,
// 2,048 x 2,048 x 32 7.2 -> 6.3, 1,024 x 3,072 x 512 45.2 -> 40.1; Q6_K 1,152 x
// 6,912 x 203 54.6 -> 46.0; BF16 8,192 x 2,048 x 9 16.2 -> 10.2; F32 2,048 x 2,048
// x 32 11.0 -> 9.0; F16 3,072 x 1,024 x 64 (32 x 32) 11.3 -> 10.4.
// Sixteen waves for the 32 x 32 tile spill (33.5 against 32.2 us and far worse).
template <uint32_t F, int RB, int TB, uint32_t W, bool FULL, bool CLIP>
__global__ __launch_bounds__(64 * W, RB == 1 ? 4 : 2) void gemm_exact_short(Product a, uint32_t token_tiles) {
    constexpr int kSteps = 4;            // groups the inputs are loaded ahead
    constexpr uint32_t kEach = 32 / W;   // ranges a wave
    constexpr int kBatch = Codes<F>::kBatch;
    constexpr int kLoadRows = F == kF32 ? 2 : 1;
    constexpr uint32_t kBlock = 256 * RB * TB;  // floats of one range's sums
    constexpr uint32_t kCodeWords = RB * Codes<F>::kWords;
    constexpr uint32_t kStage = kCodeWords + TB * 512 > kBlock ? kCodeWords + TB * 512 : kBlock;
    __shared__ float4 sums4[(W - 1) * (kEach - 1) * kBlock / 4];  // the ranges but each wave's last, past wave 0's
    __shared__ float4 stage4[W * kStage / 4];
    float* const sums = reinterpret_cast<float*>(sums4);
    const uint32_t lane = threadIdx.x & 63u, q = lane >> 4, my = lane & 15u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t T = __builtin_amdgcn_readfirstlane(blockIdx.x % token_tiles) * (16 * TB);
    const uint32_t R = __builtin_amdgcn_readfirstlane(blockIdx.x / token_tiles) * (16 * RB);
    const uint32_t G = a.groups;
    const auto lo_of = [&](uint32_t r) { return (r * G) >> 5; };  // range_lo; G is below 2^24
    const uint32_t g_begin = lo_of(kEach * wave), g_end = lo_of(kEach * wave + kEach);
    float* const stage = reinterpret_cast<float*>(stage4) + wave * kStage;
    // The stage is this wave's own and its LDS operations run in order, so
    // ordering the compiler's view of them is all that is needed.
    auto order = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    f32x4 held[RB][TB];  // the last range's sums; wave 0: its ranges' total
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) held[rb][tb] = f32x4{};

    if (g_begin < g_end) {
        const uint32_t g_last = g_end - 1;
        // Rows and tokens past the product read its last row or token; their
        // outputs are never stored.
        const uint8_t* piece[RB][kLoadRows];
        uint64_t blocks[RB], row0[RB][kLoadRows];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int i = 0; i < kLoadRows; ++i) {
                const Piece pc = piece_of(a, min(R + 16 * rb + 8 * i + Codes<F>::load_row(lane), a.rows - 1));
                piece[rb][i] = pc.piece, blocks[rb] = pc.blocks, row0[rb][i] = static_cast<uint64_t>(pc.row) * G;
            }
        // copy i: token 8 i + lane / 8, its chunk lane % 8 (ks 4c .. 4c + 3)
        const float4* x[2 * TB];
        float* const inputs = stage + kCodeWords;
        uint32_t put_at[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) put_at[e] = operand_word(lane >> 3, lane & 7u, e);
#pragma unroll
        for (int i = 0; i < 2 * TB; ++i)
            x[i] = reinterpret_cast<const float4*>(a.x) + min(T + 8 * i + (lane >> 3), a.tokens - 1) * (G * uint64_t{8}) +
                   (lane & 7u);
        const float4* const get_low = reinterpret_cast<const float4*>(inputs) + operand_slot(my, q, 0);
        const float4* const get_high = reinterpret_cast<const float4*>(inputs) + operand_slot(my, q, 1);
        float lo = 0.0f, hi = 0.0f;
        if constexpr (CLIP) lo = *a.clip[0], hi = *a.clip[1];

        struct Inputs {
            float4 v[2 * TB];
        };
        auto fetch = [&](Inputs& b, uint32_t g) {
#pragma unroll
            for (int i = 0; i < 2 * TB; ++i) b.v[i] = x[i][8 * min(g, g_last)];
        };
        auto put = [&](const Inputs& b) {
#pragma unroll
            for (int i = 0; i < 2 * TB; ++i) {
                float4 v = b.v[i];
                if constexpr (CLIP) {
                    v.x = clamp_to(v.x, lo, hi), v.y = clamp_to(v.y, lo, hi);
                    v.z = clamp_to(v.z, lo, hi), v.w = clamp_to(v.w, lo, hi);
                }
                inputs[256 * i + put_at[0]] = v.x;
                inputs[256 * i + put_at[1]] = v.y;
                inputs[256 * i + put_at[2]] = v.z;
                inputs[256 * i + put_at[3]] = v.w;
            }
        };
        auto fetch_codes = [&](Codes<F> (&c)[RB], uint32_t g) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                if constexpr (F == kF32)
                    c[rb].load(piece[rb], row0[rb], g, g_last, lane);
                else
                    c[rb].load(piece[rb][0], blocks[rb], row0[rb][0], g, g_last, lane);
            }
        };
        // The range being summed and its groups left; below 32 groups the
        // ranges that hold one hold it alone (group g's is (32 g + 31) / G).
        uint32_t r = kEach * wave;
        if (G < 32) r = __builtin_amdgcn_readfirstlane((32 * g_begin + 31) / G);
        uint32_t left = G < 32 ? 1u : lo_of(r + 1) - lo_of(r);
        f32x4 s[RB][TB];  // +0 at a range's start: its first product is fma(w, x, +0)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) s[rb][tb] = f32x4{};
        Inputs buffers[kSteps];
        constexpr int kCodeBuffers = kSteps / kBatch;
        Codes<F> codes[kCodeBuffers][RB];
#pragma unroll
        for (int i = 0; i < kCodeBuffers; ++i) fetch_codes(codes[i], g_begin + kBatch * i);
#pragma unroll
        for (int i = 0; i < kSteps; ++i) fetch(buffers[i], g_begin + i);
        put(buffers[0]);
        // Group g, the i-th of four: its codes in the stage or on their way,
        // its inputs in the stage; `next` holds the next group's.
        auto step = [&](int i, Inputs& b, const Inputs& next, uint32_t g, bool more) {
            if (i % kBatch == 0) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) codes[i / kBatch][rb].put(stage + rb * Codes<F>::kWords, lane);
                if (more) fetch_codes(codes[i / kBatch], g + kSteps);
            }
            order();
            float4 bx[TB][2];
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) bx[tb][0] = get_low[128 * tb], bx[tb][1] = get_high[128 * tb];
            Quarter<F> quarter[RB];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) Codes<F>::get(quarter[rb], stage + rb * Codes<F>::kWords, i % kBatch, lane);
            order();
            put(next);
            if (more) fetch(b, g + kSteps);
            float w[RB][8];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) quarter[rb].eight(q, w[rb]);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) {
                    const float4 h = bx[tb][j / 4];
                    const float v = j % 4 == 0 ? h.x : j % 4 == 1 ? h.y : j % 4 == 2 ? h.z : h.w;
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb)
                        s[rb][tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[rb][j], v, s[rb][tb], 0, 0, 0);
                }
            }
            if (--left == 0) {
                const uint32_t at = ((kEach - 1) * (wave - 1) + r % kEach) * kBlock + 4 * lane;
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int tb = 0; tb < TB; ++tb) {
                        if (wave == 0) {
                            held[rb][tb] = held[rb][tb] + s[rb][tb];
                        } else if (r % kEach == kEach - 1) {
                            held[rb][tb] = s[rb][tb];
                        } else {
                            const float e0 = s[rb][tb][0], e1 = s[rb][tb][1], e2 = s[rb][tb][2], e3 = s[rb][tb][3];
                            *reinterpret_cast<float4*>(sums + at + 256 * (rb * TB + tb)) = make_float4(e0, e1, e2, e3);
                        }
                        s[rb][tb] = f32x4{};
                    }
                if (G < 32) {
                    r = __builtin_amdgcn_readfirstlane((32 * (g + 1) + 31) / G);
                    left = 1;
                } else {
                    ++r;
                    left = lo_of(r + 1) - lo_of(r);
                }
            }
        };
        // The last four groups load nothing more: their loads would be wasted
        // (a wave of a K = 2,048 product has four or eight groups in all),
        // and a load that may not be issued would make every wait one for all.
        uint32_t g = g_begin;
        for (; g + kSteps < g_end; g += kSteps) {
#pragma unroll
            for (int i = 0; i < kSteps; ++i) step(i, buffers[i], buffers[(i + 1) % kSteps], g + i, true);
        }
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
            if (g + i < g_end) step(i, buffers[i], buffers[(i + 1) % kSteps], g + i, false);
    }
    order();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) {
            const float e0 = held[rb][tb][0], e1 = held[rb][tb][1], e2 = held[rb][tb][2], e3 = held[rb][tb][3];
            *reinterpret_cast<float4*>(stage + 256 * (rb * TB + tb) + 4 * lane) = make_float4(e0, e1, e2, e3);
        }
    __syncthreads();

    // The ordered combine: thread t adds rows 2 h, 2 h + 1 of its lane's four.
    // With a read under each range's own test, an LDS round trip a range was a
    // tenth of a K = 1,024 tile: Q4_0 2,048 x 1,024 x 24 5.6 -> 4.9 us, 6,144 x
    // 1,024 x 100 29.9 -> 28.4, Q6_K gated 2 x 3,072 x 1,024 x 64 21.1 -> 20.3.
    const uint32_t block = threadIdx.x >> 7, l = threadIdx.x & 63u, h = (threadIdx.x >> 6) & 1u;
    if (block < RB * TB) {
        const uint32_t at = 256 * block + 4 * l + 2 * h;
        const float* const stages = reinterpret_cast<const float*>(stage4);
        float2 first = *reinterpret_cast<const float2*>(stages + at);
        float ta = first.x, tb = first.y;
        const auto sum_of = [&](uint32_t r) {
            return *reinterpret_cast<const float2*>(
                r % kEach == kEach - 1 ? stages + (r / kEach) * kStage + at
                                       : sums + ((kEach - 1) * (r / kEach - 1) + r % kEach) * kBlock + at);
        };
        if (G >= 32) {  // no range is empty: every read before the first add
            float2 v[32 - kEach];
#pragma unroll
            for (uint32_t r = kEach; r < 32; ++r) v[r - kEach] = sum_of(r);
#pragma unroll
            for (uint32_t r = kEach; r < 32; ++r) ta = ta + v[r - kEach].x, tb = tb + v[r - kEach].y;
        } else {
#pragma unroll
            for (uint32_t r = kEach; r < 32; ++r) {
                if (lo_of(r) < lo_of(r + 1)) {
                    const float2 v = sum_of(r);
                    ta = ta + v.x;
                    tb = tb + v.y;
                }
            }
        }
        const uint32_t token = T + 16 * (block % TB) + (l & 15u);
        const uint32_t p = R + 16 * (block / TB) + 4 * (l >> 4) + 2 * h;
        if (token < a.tokens) {
            if (p < a.rows) emit<FULL>(a, p, token, token, ta, tb);
            if (p + 1 < a.rows) emit<FULL>(a, p + 1, token, token, tb, 0.0f);
        }
    }
}

template <uint32_t F, int RB, int TB, uint32_t W>
void go_short(const Product& a, const Plan& plan, hipStream_t stream) {
    const dim3 grid(static_cast<uint32_t>(plan.workgroups)), block(64 * W);
    if (plain_epilogue(a))
        hipLaunchKernelGGL((gemm_exact_short<F, RB, TB, W, false, false>), grid, block, 0, stream, a, plan.token_tiles);
    else if (!clipped(a))
        hipLaunchKernelGGL((gemm_exact_short<F, RB, TB, W, true, false>), grid, block, 0, stream, a, plan.token_tiles);
    else
        hipLaunchKernelGGL((gemm_exact_short<F, RB, TB, W, true, true>), grid, block, 0, stream, a, plan.token_tiles);
}

template <uint32_t F>
void go_exact_short(const Product& a, const Plan& plan, hipStream_t stream) {
    if constexpr (F != kF32) {
        if (plan.tile_rows == 16 && plan.waves == 16) return go_short<F, 1, 1, 16>(a, plan, stream);
    }
    if (plan.tile_rows == 16) return go_short<F, 1, 1, 8>(a, plan, stream);
    if (plan.tile_tokens == 16) return go_short<F, 2, 1, 8>(a, plan, stream);
    go_short<F, 2, 2, 8>(a, plan, stream);
}

template <uint32_t F, int TB>
void go_exact_tile(const Product& a, const Plan& plan, float* range_sums, hipStream_t stream) {
    const dim3 grid(static_cast<uint32_t>(plan.workgroups)), block(64 * kWaves);
    const uint32_t tt = plan.token_tiles, rt = plan.row_tiles, ch = plan.chunks;
    if (range_sums) {  // a split product has no options and is not gated
        const bool quads = a.rows % 4 == 0 && reinterpret_cast<uintptr_t>(range_sums) % 16 == 0;
        hipLaunchKernelGGL((gemm_exact<F, TB, false, false, true>), grid, block, 0, stream, a, tt, rt, ch, range_sums,
                           quads);
    } else if (plain_epilogue(a)) {
        hipLaunchKernelGGL((gemm_exact<F, TB, false, false>), grid, block, 0, stream, a, tt, rt, 1u, nullptr, false);
    } else if (!clipped(a)) {
        hipLaunchKernelGGL((gemm_exact<F, TB, true, false>), grid, block, 0, stream, a, tt, rt, 1u, nullptr, false);
    } else {
        hipLaunchKernelGGL((gemm_exact<F, TB, true, true>), grid, block, 0, stream, a, tt, rt, 1u, nullptr, false);
    }
}

template <uint32_t F>
void go_exact(const Product& a, const Plan& plan, float* range_sums, hipStream_t stream) {
    if constexpr (F != kF32) {
        if (plan.tile_tokens == 64) return go_exact_tile<F, 2>(a, plan, range_sums, stream);
    }
    go_exact_tile<F, 1>(a, plan, range_sums, stream);
}

}  // namespace

// Tiles of 256 rows (eight waves of 32) by 64 or 32 tokens, token tile first,
// so the tiles reading one row tile's weights run together. A SIMD's waves
// share its matrix core, so a step takes as many rounds as its most loaded
// SIMD holds pairs of waves: 64 tokens where they give no more rounds than 32
// give half-length ones (a decoded weight then serves twice the products),
// else 32 — Llama 3.2 1B's QKV at 2,048 tokens: 1,536 pairs by 64 on 1,024
// SIMDs are two rounds, 3,072 by 32 one and a half. F32 always by 32.
void plan_gemm_exact(const Product& a, uint32_t format, uint32_t compute_units, bool split, Plan* plan) {
    *plan = Plan{};
    const uint64_t wave_rows = (a.rows + 63) / 64;
    const uint64_t simds = 4ull * compute_units;
    const uint64_t rounds64 = (wave_rows * ((a.tokens + 63) / 64) + simds - 1) / simds;
    const uint64_t rounds32 = (wave_rows * ((a.tokens + 31) / 32) + simds - 1) / simds;  // half-length rounds
    uint32_t tt = format != kF32 && rounds32 >= 2 * rounds64 ? 64 : 32;
    if (split) tt = format != kF32 && a.tokens > 32 ? 64 : 32;
    plan->kernel = split ? kGemmExactSplit : kGemmExact;
    plan->launches = split ? 2 : 1;
    plan->tile_tokens = tt;
    plan->tile_rows = kWaves * kWaveRows;
    plan->waves = kWaves;
    plan->token_tiles = (a.tokens + tt - 1) / tt;
    plan->row_tiles = (a.rows + plan->tile_rows - 1) / plan->tile_rows;
    plan->wave_rows = kWaveRows / 32;
    plan->wave_tokens = tt / 32;
    plan->tiles = static_cast<uint64_t>(plan->token_tiles) * plan->row_tiles;
    // Split: the ranges cut into as few chunks (a power of two, at most 32)
    // as still give every compute unit two workgroups where 32 can.
    uint32_t chunks = 1;
    if (split) {
        chunks = 2;
        while (chunks < 32 && plan->tiles * chunks < 2ull * compute_units) chunks *= 2;
    }
    plan->chunks = chunks;
    plan->workgroups = plan->tiles * chunks;
}

// The short-step form: workgroups of 32 rows x 32 or 16 tokens, or 16 x 16,
// token tile first.
void plan_gemm_exact_short(const Product& a, uint32_t format, uint32_t compute_units, Plan* plan) {
    *plan = Plan{};
    plan->kernel = kGemmExactShort;
    plan->launches = 1;
    // 16 x 16 tiles where they number at most two a compute unit, else 32 x
    // 32, a quarter as many (16 x 16 against 32 x 32 at three a compute unit:
    // 6,144 x 2,048 x 32 18.3 against 16.1 us, 6,144 x 4,096 x 32 23.5 against
    // 26.4); 32 x 16 for steps of at most 16 tokens, whose second 16 would be
    // padding. Sixteen waves (two ranges each) where the 16 x 16 tiles number
    // at most one a compute unit and a wave keeps two groups or more: 2,048 x
    // 8,192 x 32 16.4 against 18.2 us, 2,048 x 2,048 x 16 7.4 against 7.7, but
    // 1,024 x 1,024 x 64 5.9 against 5.7; F32 always eight (2,048 x 2,048 x 32
    // 9.7 against 12.1).
    const uint64_t quads = uint64_t{(a.tokens + 15) / 16} * ((a.rows + 15) / 16);
    const uint32_t tile = quads <= 2ull * compute_units ? 16 : 32;
    uint32_t tile_tokens = a.tokens <= 16 ? 16 : tile;
    // F16, and BF16 of K up to 2,048, past two rounds of 32 x 32 tiles: 32 x 16,
    // of which a CU holds two, one's first loads and combine beside the other's
    // products (us, 32 x 32 against 32 x 16: F16 6,144 x 1,024 x 100 32.3 and
    // 29.0, 6,144 x 4,096 x 200 160.6 and 131.9; BF16 gated 2 x 4,096 x 2,048 x
    // 100 62.9 and 54.1, but 6,144 x 4,096 x 128 78.4 and 81.4).
    const uint64_t squares = uint64_t{(a.tokens + 31) / 32} * ((a.rows + 31) / 32);
    if (tile == 32 && (format == kF16 || (format == kBF16 && a.groups <= 64)) && squares > 2ull * compute_units)
        tile_tokens = 16;
    plan->tile_tokens = tile_tokens;
    plan->tile_rows = tile;
    plan->waves = format != kF32 && quads <= compute_units && a.groups >= 64 ? 16 : 8;
    plan->token_tiles = (a.tokens + tile_tokens - 1) / tile_tokens;
    plan->row_tiles = (a.rows + tile - 1) / tile;
    plan->wave_rows = 1;
    plan->wave_tokens = 1;
    plan->tiles = static_cast<uint64_t>(plan->token_tiles) * plan->row_tiles;
    plan->workgroups = plan->tiles;
}

hipError_t launch_gemm_exact_short(const Product& a, uint32_t format, const Plan& plan, hipStream_t stream) {
    switch (format) {
        case kQ4_0: go_exact_short<kQ4_0>(a, plan, stream); break;
        case kQ4_1: go_exact_short<kQ4_1>(a, plan, stream); break;
        case kQ8_0: go_exact_short<kQ8_0>(a, plan, stream); break;
        case kQ6_K: go_exact_short<kQ6_K>(a, plan, stream); break;
        case kF32: go_exact_short<kF32>(a, plan, stream); break;
        case kF16: go_exact_short<kF16>(a, plan, stream); break;
        case kBF16: go_exact_short<kBF16>(a, plan, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// The tile; with `range_sums` (the split plan: room for 32 x tokens x rows
// floats), the split form and then combine_ranges.
hipError_t launch_gemm_exact(const Product& a, uint32_t format, const Plan& plan, float* range_sums,
                             hipStream_t stream) {
    switch (format) {
        case kQ4_0: go_exact<kQ4_0>(a, plan, range_sums, stream); break;
        case kQ4_1: go_exact<kQ4_1>(a, plan, range_sums, stream); break;
        case kQ8_0: go_exact<kQ8_0>(a, plan, range_sums, stream); break;
        case kQ6_K: go_exact<kQ6_K>(a, plan, range_sums, stream); break;
        case kF32: go_exact<kF32>(a, plan, range_sums, stream); break;
        case kF16: go_exact<kF16>(a, plan, range_sums, stream); break;
        case kBF16: go_exact<kBF16>(a, plan, range_sums, stream); break;
        default: return hipErrorInvalidValue;
    }
    if (range_sums) return launch_combine_ranges(a, range_sums, stream);
    return hipGetLastError();
}

}  // namespace chm
