// hjm_mfma_ops.h -- matrix-core products and operand splits shared by the FP32 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hjm {

typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4_t mfma_bf16(u4_t a, u4_t b, f4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, a),
                                                   __builtin_bit_cast(bf8_t, b), c, 0, 0, 0);
}

// Exact three-way split of 8 FP32 values into packed bf16 parts (h + m + l = x): h keeps
// the top 8 significant bits, m the next 8, l the last 8 (each difference is exact).
struct Split8 {
    u4_t h, m, l;
};

__device__ __forceinline__ Split8 split8(const float* x)
{
#pragma clang fp contract(off)
    uint32_t hb[8], mb[8], lb[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t u = __builtin_bit_cast(uint32_t, x[i]);
        hb[i] = u & 0xffff0000u;
        const float r1 = x[i] - __builtin_bit_cast(float, hb[i]);
        mb[i] = __builtin_bit_cast(uint32_t, r1) & 0xffff0000u;
        const float r2 = r1 - __builtin_bit_cast(float, mb[i]);
        lb[i] = __builtin_bit_cast(uint32_t, r2);
    }
    Split8 s;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        // dword j = element 2j (low half) | element 2j+1 (high half)
        s.h[j] = __builtin_amdgcn_perm(hb[2 * j + 1], hb[2 * j], 0x07060302u);
        s.m[j] = __builtin_amdgcn_perm(mb[2 * j + 1], mb[2 * j], 0x07060302u);
        s.l[j] = __builtin_amdgcn_perm(lb[2 * j + 1], lb[2 * j], 0x07060302u);
    }
    return s;
}

__device__ __forceinline__ f4_t mfma_f16(u4_t a, u4_t b, f4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, a),
                                                  __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
}

// Two fp16 parts of 8 FP32 values, each rounded to nearest: h + l = x to 2^-22 |x| + 2^-25
// (the low part's subnormals end there).
struct SplitH8 {
    u4_t h, l;
};

// Three instructions per pair: v_cvt_pk_f16_f32, then the low parts by v_fma_mixlo/mixhi_f16
// (1.5 per value; the exact three-way bf16 split takes 5.5). The operands are opaque where the
// compiler would otherwise fold: a product feeding the conversions would be fused into one
// of them and not the other, and the low part would then belong to another high part; the
// pair is converted once; x - h stays an FMA with the opaque factor -1.
__device__ __forceinline__ SplitH8 split8h(const float* x)
{
    SplitH8 s;
    float neg1 = -1.f;
    asm("" : "+s"(neg1));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float a = x[2 * j], b = x[2 * j + 1];
        asm("" : "+v"(a), "+v"(b));
        h2_t h = {(_Float16)a, (_Float16)b};
        asm("" : "+v"(h));
        const h2_t l = {(_Float16)__builtin_fmaf((float)h[0], neg1, a),
                        (_Float16)__builtin_fmaf((float)h[1], neg1, b)};
        s.h[j] = __builtin_bit_cast(uint32_t, h);
        s.l[j] = __builtin_bit_cast(uint32_t, l);
    }
    return s;
}

}  // namespace hjm
