// The quantizers' arithmetic: (scale, zero) of a range and the codes of 8 values, on the device.
// Every code must be bit-exact with the float32 specification, so the arithmetic is spelled out
// one IEEE operation at a time, in the spec's order:
//   integer b bits, R = 2^b - 1: s = fp16((max - min) / R), z = fp16(min),
//       c = s == 0 ? 0 : clamp(rint((x - z) / s), 0, R)
//   fp8 e4m3fn, E = 448: z = fp16((max + min) * 0.5), s = fp16((max - min) / (2E)),
//       c = s == 0 ? 0x00 : e4m3fn_rne(clamp((x - z) / s, -E, E))
// rint rounds half to even; division is IEEE (correctly rounded, computed as in
// quotient()); no contraction.
// Each shortcut below equals the plain operations on the inputs its comment names: all of them are
// compared on the GPU by tests/gpu_checks/quant_math_check.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "kvq.h"

#pragma clang fp contract(off)

namespace kvq {

namespace {

constexpr float kFp8Max = 448.f;

typedef short s2q __attribute__((ext_vector_type(2)));
typedef uint32_t u2q __attribute__((ext_vector_type(2)));
typedef uint32_t u4q __attribute__((ext_vector_type(4)));
typedef _Float16 h8q __attribute__((ext_vector_type(8)));
typedef _Float16 h2q __attribute__((ext_vector_type(2)));

struct ScaleZero {
    uint32_t sz;  // (scale, zero) as stored: fp16 scale in the low half, zero in the high
    float r;      // RN(1 / s), 0 when s == 0
    __device__ __forceinline__ bool flat() const { return (sz & 0x7FFFu) == 0; }  // s == 0
};

// RN(d / R) for a constant R: q = RN(d RN(1/R)), one fma remainder and one fma correction
// (Markstein), d = +-inf passed through. The IEEE quotient for R = 15, 255 and 896 and every
// d = x - y of fp16 values with y not above x in the order of min / max, where -0 is below +0. (The
// one d this leaves out, -0 - +0, gives +0 where the division gives -0.) The empty asm keeps the
// correction and the conversion apart: fused into one v_fma_mixlo_f16 they would round once, where
// the spec rounds twice.
template <int R>
__device__ __forceinline__ float range_over(float d) {
    constexpr float ir = 1.f / R;
    const float q = d * ir;
    const float rem = __builtin_fmaf(-q, (float)R, d);
    float t = __builtin_fmaf(rem, ir, q);
    t = __builtin_fabsf(q) == INFINITY ? q : t;
    asm("" : "+v"(t));
    return t;
}

// RN(1 / s): v_rcp_f32 and one Newton step, the IEEE quotient for every positive finite fp16 s.
// s = inf gives NaN where the division gives 0: either way the quotients below are NaN.
__device__ __forceinline__ float reciprocal(float s) {
    const float r0 = __builtin_amdgcn_rcpf(s);
    const float e = __builtin_fmaf(-s, r0, 1.f);
    return __builtin_fmaf(e, r0, r0);
}

template <int FMT>
__device__ __forceinline__ ScaleZero make_params(float mn, float mx) {
    h2q sz;
    if (FMT == KVQ_KV_FP8_E4M3) {
        float mid = (mx + mn) * 0.5f;
        asm("" : "+v"(mid));  // not one v_fma_mixlo_f16, which loses the sign of a zero
        sz = h2q{(_Float16)range_over<2 * (int)kFp8Max>(mx - mn), (_Float16)mid};
    } else {
        sz = h2q{(_Float16)range_over<FMT == KVQ_KV_INT4 ? 15 : 255>(mx - mn), (_Float16)mn};
    }
    const float s = (float)sz[0];
    return ScaleZero{__builtin_bit_cast(uint32_t, sz), s == 0.f ? 0.f : reciprocal(s)};
}

// RN((x - z) / s) for fp16 x, z (d = fl(x - z) is 0 or |d| >= 2^-24) and a positive fp16 s,
// from the correctly rounded reciprocal r: q = RN(d r), the exact remainder d - s q by fma, and
// one fma correction (Markstein's theorem; its exceptions need a divisor significand of 24
// ones, and s has 11 significant bits). The codes it gives are compared for every such s, every
// finite or NaN x and 16 z each, the quotient itself on the CPU (tests/test_quotient_cpu.py). x, z
// and s are read in fp16 by v_fma_mix (x 1 - z; d - q s), half HI of x's dword: no conversions, and
// a channel's parameters take two registers. s = 0 gives r = 0 and a quotient of +-0 (NaN for a NaN
// x); d = -0, from x = -0 under z = +0, gives +0 (an FP8 code 0x00 where the spec's is 0x80, which
// stands for the same value).
template <int HI>
__device__ __forceinline__ float quotient(uint32_t x, const ScaleZero& p) {
    float d, rem;
    if constexpr (HI)
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(d) : "v"(x), "v"(p.sz));
    else
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[1,0,1]" : "=v"(d) : "v"(x), "v"(p.sz));
    const float q = d * p.r;
    asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel:[0,0,0] op_sel_hi:[0,1,0]" : "=v"(rem) : "v"(q), "v"(p.sz), "v"(d));
    return __builtin_fmaf(rem, p.r, q);
}

// Codes of 8 values of one row, packed as stored: INT4 one dword (low nibble = even value),
// INT8 / FP8 two. Element e uses q[CH * e] (CH = 1: per channel, 0: one pair for all).
//   INT8: v_cvt_pk_u8_f32 rounds half to even, clamps to [0, 255] (NaN: 0) and inserts the
//     byte - rint, both clamps, the conversion and the packing in one instruction, equal to
//     them on every fp32 value. INT4 the same after a clamp to 15 (v_med3; NaN: 0), the odd
//     values' bytes shifted into the high nibbles.
//   FP8: clamp to +-448 (NaN: -448), then v_cvt_scalef32_pk_fp8_f32 at scale 1, two codes
//     each: it equals the spec's software encode (mantissa rounded half to even at 2^(e-3),
//     subnormals at 2^-9) on every fp32 value of [-448, 448]
//     (tests/gpu_checks/fp8_encode_check.hip). `live` clears the codes of s = 0 (whose
//     quotient may be -0 or NaN); the integer formats give 0 there by themselves.
// 5 (INT8), 6 (INT4) and 5.5 (FP8) VALU instructions per value with the quotient.
template <int FMT>
struct Codes8 {
    static constexpr int N = FMT == KVQ_KV_INT4 ? 1 : 2;
    uint32_t w[N];
};

template <int FMT, int CH>
__device__ __forceinline__ Codes8<FMT> encode8(h8q v, const ScaleZero* q, const uint32_t* live) {
    const u4q x = __builtin_bit_cast(u4q, v);
    float t[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        t[2 * j] = quotient<0>(x[j], q[CH * 2 * j]);
        t[2 * j + 1] = quotient<1>(x[j], q[CH * (2 * j + 1)]);
    }
    Codes8<FMT> c;
    if constexpr (FMT == KVQ_KV_FP8_E4M3) {
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = __builtin_amdgcn_fmed3f(t[e], -kFp8Max, kFp8Max);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            s2q r = {0, 0};
            r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, t[4 * j], t[4 * j + 1], 1.0f, false);
            r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, t[4 * j + 2], t[4 * j + 3], 1.0f, true);
            c.w[j] = __builtin_bit_cast(uint32_t, r) & live[CH * j];
        }
    } else if constexpr (FMT == KVQ_KV_INT8) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) w = __builtin_amdgcn_cvt_pk_u8_f32(t[4 * j + e], e, w);
            c.w[j] = w;
        }
    } else {
        uint32_t even = 0, odd = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            even = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(t[2 * e], 0.f, 15.f), e, even);
            odd = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(t[2 * e + 1], 0.f, 15.f), e, odd);
        }
        c.w[0] = even | (odd << 4);
    }
    return c;
}

// encode8's `live` masks: all ones, or a zero byte for a value of scale 0 (FP8).
template <int FMT>
__device__ __forceinline__ void live_masks(const ScaleZero* q, uint32_t* live) {
    live[0] = live[1] = ~0u;
    if constexpr (FMT == KVQ_KV_FP8_E4M3) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (q[e].flat()) live[e / 4] &= ~(0xFFu << (8 * (e % 4)));
    }
}

}  // namespace

}  // namespace kvq
