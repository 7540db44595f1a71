// Exhaustive checks of the quantizers' arithmetic (kvq_decode_amd/csrc/quant_math.h, the code the
// kernels run) against the plain IEEE operations of the specification. Prints each check's number
// of cases and differences; exit status 0 = none. Test infrastructure, built by
// kvq_decode_amd.build, run by tests/test_quant_math_gpu.py.
//   params      (scale, zero, 1 / scale) of every pair of fp16 min and max, infinities included,
//               for each format: range_over, reciprocal and the roundings to fp16
//   reciprocal  every positive finite fp16
//   codes       every fp16 scale that is 0 or positive and finite, every x that is finite or NaN,
//               16 zeros for each: quotient, clamp, rounding and packing. FP8: x - z = -0, which
//               only x = -0 under z = +0 gives, must have the code +0 for the spec's -0
//   u8          v_cvt_pk_u8_f32 of every fp32 value: rounding half to even, clamps, NaN
//   minmax      packed-half min / max of every pair, NaN and both zeros included, against float's
#include <stdio.h>
#include <stdlib.h>

#include "quant_math.h"

using namespace kvq;

#define CK(x)                                                                            \
    do {                                                                                 \
        hipError_t e = (x);                                                              \
        if (e != hipSuccess) {                                                           \
            printf("HIP error %s at line %d\n", hipGetErrorString(e), __LINE__);         \
            exit(2);                                                                     \
        }                                                                                \
    } while (0)

typedef unsigned long long u64;

__device__ float half_of(uint32_t bits) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}
__device__ uint32_t bits_of(_Float16 h) { return __builtin_bit_cast(uint16_t, h); }
__device__ bool half_nan(uint32_t b) { return (b & 0x7FFFu) > 0x7C00u; }
// bits in the order of min / max: negative values descending below the positive ones
__device__ int order(uint32_t b) { return b & 0x8000u ? (int)(0xFFFFu - b) : (int)(b | 0x8000u); }
// a value the compiler cannot fuse into the next operation
__device__ float rounded(float x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ bool same_half(uint32_t a, uint32_t b) { return a == b || (half_nan(a) && half_nan(b)); }

// Adds a wave's cases and differences (each below 2^26 per lane) to the check's counters.
__device__ void add(u64* count, uint32_t cases, uint32_t bad) {
    for (int o = 32; o >= 1; o >>= 1) {
        cases += __shfl_xor(cases, o);
        bad += __shfl_xor(bad, o);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&count[0], (u64)cases);
        if (bad) atomicAdd(&count[1], (u64)bad);
    }
}

template <int FMT>
__global__ void params(u64* count) {
    uint32_t cases = 0, bad = 0;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < 1ull << 32; i += (u64)gridDim.x * blockDim.x) {
        const uint32_t lo = (uint32_t)i & 0xFFFFu, hi = (uint32_t)(i >> 16);
        if (half_nan(lo) || half_nan(hi) || order(lo) > order(hi)) continue;
        const float mn = half_of(lo), mx = half_of(hi);
        const float R = FMT == KVQ_KV_FP8_E4M3 ? 896.f : FMT == KVQ_KV_INT4 ? 15.f : 255.f;
        const _Float16 s = (_Float16)rounded(__fdiv_rn(rounded(mx - mn), R));
        const _Float16 z = FMT == KVQ_KV_FP8_E4M3
                               ? (_Float16)rounded(rounded(mx + mn) * 0.5f) : (_Float16)mn;
        const float r = (float)s == 0.f ? 0.f : __fdiv_rn(1.f, (float)s);
        const ScaleZero got = make_params<FMT>(mn, mx);
        const bool finite = (bits_of(s) & 0x7FFFu) < 0x7C00u;
        ++cases;
        bad += !same_half(got.sz & 0xFFFFu, bits_of(s)) || !same_half(got.sz >> 16, bits_of(z)) ||
               (finite && __float_as_uint(got.r) != __float_as_uint(r));
    }
    add(count, cases, bad);
}

__global__ void reciprocals(u64* count) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    const float s = half_of(b);  // b < 0x7C00
    add(count, b != 0, b != 0 && __float_as_uint(reciprocal(s)) != __float_as_uint(__fdiv_rn(1.f, s)));
}

// The spec's e4m3fn encode, restated in software (|t| <= 448).
__device__ uint32_t spec_e4m3fn(float t) {
    const uint32_t sign = (__float_as_uint(t) >> 31) << 7;
    const float a = fabsf(t);
    if (a < 0.015625f) return (uint32_t)__builtin_rintf(a * 512.f) | sign;
    int e = (int)((__float_as_uint(a) >> 23) & 0xFF) - 127;
    int m = (int)__builtin_rintf((a * __uint_as_float((uint32_t)(127 - e) << 23) - 1.f) * 8.f);
    if (m == 8) {
        m = 0;
        ++e;
    }
    return ((uint32_t)(e + 7) << 3) | (uint32_t)m | sign;
}

// The spec's code of x under scale s > 0 or 0 and zero z. A NaN counts as the lower clamp's value.
template <int FMT>
__device__ uint32_t spec_code(float x, float s, float z) {
    if (s == 0.f) return 0u;
    const float t = __fdiv_rn(rounded(x - z), s);
    if (FMT == KVQ_KV_FP8_E4M3) return spec_e4m3fn(fminf(fmaxf(t, -kFp8Max), kFp8Max));
    return (uint32_t)__builtin_rintf(fminf(fmaxf(t, 0.f), FMT == KVQ_KV_INT4 ? 15.f : 255.f));
}

// Block (scale, k of 16): zeros from a hash of both, the first 0; thread: runs of 8 values x.
template <int FMT>
__global__ void codes(u64* count) {
    const uint32_t sb = blockIdx.x;  // < 0x7C00
    uint32_t zb = (sb * 16 + blockIdx.y) * 2654435761u >> 16;
    if (blockIdx.y == 0) zb = 0;
    if ((zb & 0x7FFFu) >= 0x7C00u) zb &= 0x83FFu;  // not finite: the subnormal of its low bits
    const float s = half_of(sb), z = half_of(zb);
    const ScaleZero p = {sb | (zb << 16), s == 0.f ? 0.f : reciprocal(s)};
    const uint32_t live = p.flat() ? 0u : ~0u;
    uint32_t cases = 0, bad = 0;
    for (uint32_t x0 = 8 * threadIdx.x; x0 < 0x10000u; x0 += 8 * blockDim.x) {
        h8q v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = __builtin_bit_cast(_Float16, (uint16_t)(x0 + e));
        const Codes8<FMT> c = encode8<FMT, 0>(v, &p, &live);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (((x0 + e) & 0x7FFFu) == 0x7C00u) continue;  // an infinity widens its range to one
            const uint32_t got = FMT == KVQ_KV_INT4 ? c.w[0] >> (4 * e) & 15u
                                                    : c.w[e / 4 % Codes8<FMT>::N] >> (8 * (e % 4)) & 255u;
            ++cases;
            const bool minus_zero = FMT == KVQ_KV_FP8_E4M3 && x0 + e == 0x8000u && zb == 0;
            bad += got != (minus_zero ? 0u : spec_code<FMT>((float)v[e], s, z));
        }
    }
    add(count, cases, bad);
}

__global__ void u8(u64* count) {
    uint32_t cases = 0, bad = 0;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < 1ull << 32; i += (u64)gridDim.x * blockDim.x) {
        const float t = __uint_as_float((uint32_t)i);
        const uint32_t want = t != t ? 0u : (uint32_t)__builtin_rintf(fminf(fmaxf(t, 0.f), 255.f));
        ++cases;
        bad += __builtin_amdgcn_cvt_pk_u8_f32(t, 0, 0) != want;
    }
    add(count, cases, bad);
}

__global__ void minmax(u64* count) {
    uint32_t cases = 0, bad = 0;
    for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < 1ull << 32; i += (u64)gridDim.x * blockDim.x) {
        const uint32_t a = (uint32_t)i & 0xFFFFu, b = (uint32_t)(i >> 16);
        const h2q x = __builtin_bit_cast(h2q, a | (b << 16)), y = __builtin_bit_cast(h2q, b | (a << 16));
        const h2q mn = __builtin_elementwise_min(x, y), mx = __builtin_elementwise_max(x, y);
        const float fa = half_of(a), fb = half_of(b);
        const uint32_t n = bits_of((_Float16)fminf(fa, fb)), m = bits_of((_Float16)fmaxf(fa, fb));
        ++cases;
        bad += !same_half(bits_of(mn[0]), n) || !same_half(bits_of(mn[1]), n) ||
               !same_half(bits_of(mx[0]), m) || !same_half(bits_of(mx[1]), m);
    }
    add(count, cases, bad);
}

int failed = 0;

void check(const char* name, void (*kernel)(u64*), dim3 grid, int threads) {
    u64 *count, n[2] = {0, 0};
    CK(hipMalloc(&count, sizeof(n)));
    CK(hipMemcpy(count, n, sizeof(n), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, 0, count);
    CK(hipGetLastError());
    CK(hipDeviceSynchronize());
    CK(hipMemcpy(n, count, sizeof(n), hipMemcpyDeviceToHost));
    CK(hipFree(count));
    printf("%s: %llu cases, %llu differ\n", name, n[0], n[1]);
    fflush(stdout);
    failed |= n[1] != 0 || n[0] == 0;
}

int main() {
    const dim3 all(16384);
    check("params int8", params<KVQ_KV_INT8>, all, 256);
    check("params fp8", params<KVQ_KV_FP8_E4M3>, all, 256);
    check("params int4", params<KVQ_KV_INT4>, all, 256);
    check("reciprocal", reciprocals, dim3(0x7C00 / 256), 256);
    check("codes int8", codes<KVQ_KV_INT8>, dim3(0x7C00, 16), 256);
    check("codes fp8", codes<KVQ_KV_FP8_E4M3>, dim3(0x7C00, 16), 256);
    check("codes int4", codes<KVQ_KV_INT4>, dim3(0x7C00, 16), 256);
    check("u8", u8, all, 256);
    check("minmax", minmax, all, 256);
    return failed;
}
