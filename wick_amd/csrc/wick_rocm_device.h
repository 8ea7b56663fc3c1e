// Device-side helpers shared by the GEMV, GEMM and parity-hook kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wick_rocm {

// A device address as a kernel argument of its own.  The runtime looks up every argument that is a pointer among its allocations when
// the kernel is enqueued, 0.025 us each in a loop of one launch, more among others; numbers and structs it only copies.  Four pointers
// a launch / numbers: a prompt of 23 tokens behind 700 on the 350M shape, 121 launches, 655 / 623 us, of 100 tokens 709 / 700.
typedef uint64_t Address;
inline Address address(const void* p) { return reinterpret_cast<uint64_t>(p); }
template <typename T>
__device__ __forceinline__ T* in_global(Address a) {
    return (T*)(T __attribute__((address_space(1)))*)a;
}

// f16 bit pattern -> f32 (v_cvt_f32_f16; exact, subnormals kept).
__device__ __forceinline__ float f16_bits_to_f32(uint32_t bits) {
    uint16_t b = (uint16_t)bits;
    _Float16 h;
    __builtin_memcpy(&h, &b, 2);
    return (float)h;
}

// 4- and 16-byte vectors that only promise 4-byte alignment, so the compiler may
// still issue one wide global load for them.
struct __attribute__((packed, aligned(4))) u32x4_a4 {
    uint32_t v[4];
};
struct __attribute__((packed, aligned(4))) u32x2_a4 {
    uint32_t v[2];
};

// A "pair" is two consecutive weight blocks of one row: 36 B (Q4_0) or 68 B
// (Q8_0).  Rows hold an even number of blocks on the fast paths, so every pair
// starts 4-byte aligned and is read as whole dwords:
//   dword 0            = [ d0 (f16) | first two quant bytes of block 0 ]
//   dwords 1 .. NQ-1   = block 0 quants, shifted by two bytes
//   dword NQ           = [ last two quant bytes of block 0 | d1 (f16) ]
//   dwords NQ+1 .. 2NQ = block 1 quants, dword aligned
// NQ = quant dwords per block: 4 (Q4_0: 16 nibble bytes) or 8 (Q8_0: 32 int8).
template <int TYPE>
struct PairTraits;
template <>
struct PairTraits<2> {
    static constexpr int NQ = 4;
    static constexpr int DWORDS = 9;
    static constexpr int BYTES = 36;
};
template <>
struct PairTraits<8> {
    static constexpr int NQ = 8;
    static constexpr int DWORDS = 17;
    static constexpr int BYTES = 68;
};

// Native vectors with only 4-byte alignment promised, for the streaming builtin.
typedef uint32_t u32x4_native_a4 __attribute__((ext_vector_type(4), aligned(4)));

// STREAM = true marks the loads nontemporal: a GEMV reads every weight byte exactly
// once, and on MI355X streaming reads that do not allocate in the caches sustain
// about 10 % more HBM bandwidth than ordinary ones.  Tiles that are re-read by
// other workgroups (the GEMM) keep the default policy.
template <int DWORDS, bool STREAM = false>
__device__ __forceinline__ void load_pair(const uint8_t* __restrict__ p, uint32_t (&w)[DWORDS]) {
    static_assert(DWORDS % 4 == 1, "pair = 4*j + 1 dwords");
#pragma unroll
    for (int i = 0; i < DWORDS / 4; i++) {
        if constexpr (STREAM) {
            const u32x4_native_a4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4_native_a4*>(p + 16 * i));
            w[4 * i + 0] = t.x;
            w[4 * i + 1] = t.y;
            w[4 * i + 2] = t.z;
            w[4 * i + 3] = t.w;
        } else {
            u32x4_a4 t = *reinterpret_cast<const u32x4_a4*>(p + 16 * i);
            w[4 * i + 0] = t.v[0];
            w[4 * i + 1] = t.v[1];
            w[4 * i + 2] = t.v[2];
            w[4 * i + 3] = t.v[3];
        }
    }
    if constexpr (STREAM) {
        w[DWORDS - 1] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p + 4 * (DWORDS - 1)));
    } else {
        w[DWORDS - 1] = *reinterpret_cast<const uint32_t*>(p + 4 * (DWORDS - 1));
    }
}

// Splits a pair into the two f16 scale bit patterns and the two blocks' quant
// dwords (block 0 needs a two-byte funnel shift, v_alignbyte_b32).
template <int TYPE>
__device__ __forceinline__ void split_pair(const uint32_t (&w)[PairTraits<TYPE>::DWORDS], uint32_t& d0, uint32_t& d1,
                                           uint32_t (&q0)[PairTraits<TYPE>::NQ], uint32_t (&q1)[PairTraits<TYPE>::NQ]) {
    constexpr int NQ = PairTraits<TYPE>::NQ;
    d0 = w[0] & 0xffffu;
    d1 = w[NQ] >> 16;
#pragma unroll
    for (int j = 0; j < NQ; j++) {
        q0[j] = __builtin_amdgcn_alignbyte(w[j + 1], w[j], 2);
        q1[j] = w[NQ + 1 + j];
    }
}

// Exact i32 dot of one weight block with one Q8_0 activation block (8 dwords of
// int8: x[0..3] = elements 0..15, x[4..7] = elements 16..31).
//
// Q4_0 (wick/src/quant.rs:82-88): byte i of qs holds element i in its low nibble
// and element i+16 in its high nibble, value = nibble - 8.  The unsigned nibbles
// are dotted as they are and 8 * sum(x) is subtracted once; `xsum` is that
// block's sum of activation quants.
__device__ __forceinline__ int block_dot_q4_0(const uint32_t (&q)[4], const uint32_t (&x)[8], int xsum) {
    int s = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        uint32_t lo = q[j] & 0x0f0f0f0fu;
        uint32_t hi = (q[j] >> 4) & 0x0f0f0f0fu;
        s = __builtin_amdgcn_sdot4((int)lo, (int)x[j], s, false);
        s = __builtin_amdgcn_sdot4((int)hi, (int)x[4 + j], s, false);
    }
    return s - 8 * xsum;
}

__device__ __forceinline__ int block_dot_q8_0(const uint32_t (&q)[8], const uint32_t (&x)[8]) {
    int s = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) s = __builtin_amdgcn_sdot4((int)q[j], (int)x[j], s, false);
    return s;
}

__device__ __forceinline__ int block_xsum(const uint32_t (&x)[8]) {
    int s = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) s = __builtin_amdgcn_sdot4(0x01010101, (int)x[j], s, false);
    return s;
}

template <int TYPE>
__device__ __forceinline__ int block_dot(const uint32_t (&q)[PairTraits<TYPE>::NQ], const uint32_t (&x)[8], int xsum) {
    if constexpr (TYPE == 2) {
        return block_dot_q4_0(q, x, xsum);
    } else {
        (void)xsum;
        return block_dot_q8_0(q, x);
    }
}

// Q8_0 activation quantization arithmetic shared by the stand-alone quantizer and the
// fused GEMV (quantize_f32_to_q8_0_neon, wick/src/backend/simd.rs:255-323): d = amax/127,
// id = 1/d from the unrounded d, stored scale = f32(f16(d)),
// q = (i8)(i32) round-ties-even(x * id).  Every step is one correctly rounded
// binary32 operation.
__device__ __forceinline__ float q8_scale_and_inverse(float amax, float& id) {
    const float d = __fdiv_rn(amax, 127.0f);
    id = (d != 0.0f) ? __fdiv_rn(1.0f, d) : 0.0f;
    return (float)(_Float16)d;
}

__device__ __forceinline__ uint32_t q8_pack4(float v0, float v1, float v2, float v3, float id) {
    const int q0 = (int)__builtin_rintf(__fmul_rn(v0, id));
    const int q1 = (int)__builtin_rintf(__fmul_rn(v1, id));
    const int q2 = (int)__builtin_rintf(__fmul_rn(v2, id));
    const int q3 = (int)__builtin_rintf(__fmul_rn(v3, id));
    return (uint32_t)(q0 & 0xff) | ((uint32_t)(q1 & 0xff) << 8) | ((uint32_t)(q2 & 0xff) << 16) | ((uint32_t)(q3 & 0xff) << 24);
}

// Sum over groups of WIDTH consecutive lanes (WIDTH a power of two <= 64); every
// lane of a group ends with the group's total.  Within a row of 16 lanes the four
// butterfly steps are DPP operand modifiers on the add itself (no LDS crossbar, no
// wait): xor 1 and xor 2 as quad permutes, then the two mirror patterns, which
// complete the 8- and 16-lane sums because the smaller groups are already uniform.
// Only the 32- and 64-lane steps go through ds_bpermute.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false);
    return v + __builtin_bit_cast(float, moved);
}

// Maximum over groups of 8 consecutive lanes (the eight lanes that share one 32-element
// activation block in the quantizers), same three DPP steps, no LDS crossbar.
__device__ __forceinline__ float group_max8(float v) {
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, false)));
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, false)));
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, false)));
    return v;
}

// Sum over the same groups of 8 lanes.
__device__ __forceinline__ int group_sum8_i32(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false);
    return v;
}

template <int WIDTH>
__device__ __forceinline__ float group_sum(float v) {
    if constexpr (WIDTH >= 2) v = dpp_add<0xB1>(v);   // quad_perm [1,0,3,2]
    if constexpr (WIDTH >= 4) v = dpp_add<0x4E>(v);   // quad_perm [2,3,0,1]
    if constexpr (WIDTH >= 8) v = dpp_add<0x141>(v);  // row_half_mirror
    if constexpr (WIDTH >= 16) v = dpp_add<0x140>(v); // row_mirror
    if constexpr (WIDTH >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (WIDTH >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

// sums[e] += x of lane e of this lane's row of 16, times v[e].  A source of another lane is read two wait states after a vector instruction
// wrote it at the earliest, which the compiler does not see to in inline code.  Hence ONE piece of it, the wait and all that reads x: sixteen
// pieces of which the first waits may be put in another order (they write different sums), and x may be copied in front of any of them.
typedef float v16f __attribute__((ext_vector_type(16)));
__device__ __forceinline__ void fmac_row_lanes(v16f& sums, float x, const v16f& v) {
    float s[16];
#pragma unroll
    for (int e = 0; e < 16; e++) s[e] = sums[e];
#define WICK_FMAC_LANE(e) "v_fmac_f32_dpp %" #e ", %16, %[v" #e "] row_newbcast:" #e " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" WICK_FMAC_LANE(0) WICK_FMAC_LANE(1) WICK_FMAC_LANE(2) WICK_FMAC_LANE(3) WICK_FMAC_LANE(4) WICK_FMAC_LANE(5)
        WICK_FMAC_LANE(6) WICK_FMAC_LANE(7) WICK_FMAC_LANE(8) WICK_FMAC_LANE(9) WICK_FMAC_LANE(10) WICK_FMAC_LANE(11) WICK_FMAC_LANE(12)
        WICK_FMAC_LANE(13) WICK_FMAC_LANE(14) WICK_FMAC_LANE(15)
        : "+&v"(s[0]), "+&v"(s[1]), "+&v"(s[2]), "+&v"(s[3]), "+&v"(s[4]), "+&v"(s[5]), "+&v"(s[6]), "+&v"(s[7]), "+&v"(s[8]), "+&v"(s[9]),
          "+&v"(s[10]), "+&v"(s[11]), "+&v"(s[12]), "+&v"(s[13]), "+&v"(s[14]), "+&v"(s[15])
        : "v"(x), [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]), [v4] "v"(v[4]), [v5] "v"(v[5]), [v6] "v"(v[6]), [v7] "v"(v[7]),
          [v8] "v"(v[8]), [v9] "v"(v[9]), [v10] "v"(v[10]), [v11] "v"(v[11]), [v12] "v"(v[12]), [v13] "v"(v[13]), [v14] "v"(v[14]), [v15] "v"(v[15]));
#undef WICK_FMAC_LANE
#pragma unroll
    for (int e = 0; e < 16; e++) sums[e] = s[e];
}

// The same for a double over the whole wave, every lane gets the total: four DPP steps inside the rows of 16 lanes
// (each moves the two halves of the double), then the four row totals through scalar registers.  A butterfly of
// 64-bit shuffles costs twelve trips through the LDS crossbar, which is most of an RMSNorm prologue.
template <int CTRL>
__device__ __forceinline__ double dpp_add_f64(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum_f64(double v) {
    v = dpp_add_f64<0xB1>(v);   // quad_perm [1,0,3,2]
    v = dpp_add_f64<0x4E>(v);   // quad_perm [2,3,0,1]
    v = dpp_add_f64<0x141>(v);  // row_half_mirror
    v = dpp_add_f64<0x140>(v);  // row_mirror: every lane of a row holds the row's sum
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const double r0 = __hiloint2double(__builtin_amdgcn_readlane(hi, 0), __builtin_amdgcn_readlane(lo, 0));
    const double r1 = __hiloint2double(__builtin_amdgcn_readlane(hi, 16), __builtin_amdgcn_readlane(lo, 16));
    const double r2 = __hiloint2double(__builtin_amdgcn_readlane(hi, 32), __builtin_amdgcn_readlane(lo, 32));
    const double r3 = __hiloint2double(__builtin_amdgcn_readlane(hi, 48), __builtin_amdgcn_readlane(lo, 48));
    return (r0 + r1) + (r2 + r3);
}

// 1 / sqrt(total / k + eps) of an RMSNorm (rmsnorm, wick/src/backend/cpu.rs:577-594) in f64, rounded to f32 once.  The hardware's
// reciprocal root (22 bits and more) and one step of Halley's iteration for 1 / sqrt(s), y (1 + e / 2 + 3 e^2 / 8) with
// e = 1 - s y^2: the error is of order e^3, below f64's own rounding, in ten instructions where a division, a root and a
// division are a serial chain of some eighty in front of every projection of a decode step.
__device__ __forceinline__ float rms_inverse(double total, double inv_k, float eps) {
    const double s = __builtin_fma(total, inv_k, (double)eps);
    const double y = __builtin_amdgcn_rsq(s);
    const double e = __builtin_fma(-(s * y), y, 1.0);
    const double r = __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
    return (float)(__builtin_amdgcn_class(y, 0x100) ? r : y);  // positive normal; else 1 / sqrt of 0, inf or NaN as it stands
}

// f32 sum / maximum over the whole wave, every lane gets the result: DPP inside the rows, row results through scalar
// registers.
__device__ __forceinline__ float wave_sum_f32(float v) {
    v = group_sum<16>(v);
    const int b = __builtin_bit_cast(int, v);
    const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0)), r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32)), r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
    return (r0 + r1) + (r2 + r3);
}
template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) {
    return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_max_f32(float v) {
    v = dpp_max<0xB1>(v), v = dpp_max<0x4E>(v), v = dpp_max<0x141>(v), v = dpp_max<0x140>(v);
    const int b = __builtin_bit_cast(int, v);
    const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0)), r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32)), r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
    return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

// The greedy pick's ordering (cpu_argmax, wick/src/sampler.rs:7-19) as one unsigned key: NaN counts as -inf, values order
// by f32::total_cmp, and of equal values the larger index wins; 0 is below every real key.
__device__ __forceinline__ unsigned long long argmax_key(float f, uint32_t index) {
    if (f != f) f = -__builtin_inff();
    int32_t b = (int32_t)__float_as_uint(f);
    b ^= (int32_t)(((uint32_t)(b >> 31)) >> 1);                 // total_cmp's transform: signed order
    const uint32_t ordered = (uint32_t)b ^ 0x80000000u;          // ... as unsigned order
    return ((unsigned long long)ordered << 32) | index;          // equal values: the larger index wins
}

__device__ __forceinline__ float bits_f(uint32_t u) { return __uint_as_float(u); }

// ggml_expf (wick/src/backend/cpu.rs:604-652), operation for operation: bit-exact.
struct GgmlExp {
    float n, j, k;
    uint32_t e;
};
__device__ __forceinline__ GgmlExp ggml_expf_parts(float x) {
    const float R = bits_f(0x4B400000u), LOG2E = bits_f(0x3FB8AA3Bu);
    const float LN2_HI = bits_f(0x3F317200u), LN2_LO = bits_f(0x35BFBE8Eu);
    const float C1 = bits_f(0x3F7FFFF6u), C2 = bits_f(0x3EFFFEDBu), C3 = bits_f(0x3E2AAF33u);
    const float C4 = bits_f(0x3D2B9F17u), C5 = bits_f(0x3C072010u);
    const float z = __fadd_rn(R, __fmul_rn(x, LOG2E));
    const float n = __fsub_rn(z, R);
    const float b = __fsub_rn(__fsub_rn(x, __fmul_rn(n, LN2_HI)), __fmul_rn(n, LN2_LO));
    const uint32_t e = __float_as_uint(z) << 23;
    const float k = bits_f(e + 0x3F800000u);
    const float u = __fmul_rn(b, b);
    const float inner = __fadd_rn(__fadd_rn(C2, __fmul_rn(C3, b)), __fmul_rn(__fadd_rn(C4, __fmul_rn(C5, b)), u));
    const float j = __fadd_rn(__fmul_rn(C1, b), __fmul_rn(inner, u));
    return {n, j, k, e};
}
__device__ __forceinline__ float ggml_expf(float x) {
    const GgmlExp p = ggml_expf_parts(x);
    const float abs_n = fabsf(p.n);
    if (abs_n <= 126.0f) return __fadd_rn(p.k, __fmul_rn(p.j, p.k));
    if (abs_n > 192.0f) return p.n > 0.0f ? __builtin_inff() : 0.0f;
    const uint32_t d = p.n <= 0.0f ? 0x82000000u : 0u;
    const float s1 = bits_f(d + 0x7f000000u);
    const float s2 = bits_f(p.e - d);
    return __fmul_rn(__fadd_rn(s2, __fmul_rn(s2, p.j)), s1);
}
// silu_mul_inplace's element (wick/src/backend/cpu.rs:668-673): g / (1 + expf(-g)) * u, bit-exact.
__device__ __forceinline__ float silu_mul(float g, float u) { return __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, ggml_expf(-g))), u); }

// The same bits in some thirty instructions instead of forty, for 2^-60 <= |g| and |n| <= 60 (|g| < 41) alone: for code that takes many of
// them and asks once, by far and small over all of them (0 and 1 at first), whether they were.  There
//   n LN2_HI (6 + 15 bits) and j k (k a power of two) are exact, so that a fused operation rounds as the separate ones do, and
//   g / (1 + e^-g) needs neither scaling nor special cases: a Newton step on the hardware's reciprocal and two corrections by the exact
//   remainder, the last of which rounds correctly (Markstein 1990).
__device__ __forceinline__ float silu_mul_near(float g, float u, float& far, float& small) {
    const float x = -g, R = bits_f(0x4B400000u);
    const float z = __fadd_rn(R, __fmul_rn(x, bits_f(0x3FB8AA3Bu)));
    const float n = __fsub_rn(z, R);
    const float b = __fsub_rn(__builtin_fmaf(-n, bits_f(0x3F317200u), x), __fmul_rn(n, bits_f(0x35BFBE8Eu)));
    const float k = bits_f((__float_as_uint(z) << 23) + 0x3F800000u), b2 = __fmul_rn(b, b);
    const float lo = __fadd_rn(bits_f(0x3EFFFEDBu), __fmul_rn(bits_f(0x3E2AAF33u), b)), hi = __fadd_rn(bits_f(0x3D2B9F17u), __fmul_rn(bits_f(0x3C072010u), b));
    const float j = __fadd_rn(__fmul_rn(bits_f(0x3F7FFFF6u), b), __fmul_rn(__fadd_rn(lo, __fmul_rn(hi, b2)), b2));
    const float d = __fadd_rn(1.0f, __builtin_fmaf(j, k, k));
    const float y0 = __builtin_amdgcn_rcpf(d), y = __builtin_fmaf(__builtin_fmaf(-d, y0, 1.0f), y0, y0);
    const float q0 = __fmul_rn(g, y), q1 = __builtin_fmaf(__builtin_fmaf(-d, q0, g), y, q0);
    far = fmaxf(far, fabsf(n)), small = fminf(small, fabsf(g));
    return __fmul_rn(__builtin_fmaf(__builtin_fmaf(-d, q1, g), y, q1), u);
}
__device__ __forceinline__ bool silu_mul_was_near(float far, float small) { return far <= 60.0f && small >= 0x1p-60f; }

}  // namespace wick_rocm
