// Shared device helpers and host-side status plumbing for the gfx950 MoE kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "moe_hip.h"

namespace moe {

constexpr int kWave = 64;        // CDNA wavefront width
constexpr int kMaxExperts = 64;  // one lane per expert in the routing kernels
constexpr int kMaxTopk = 8;
constexpr int kNumXcd = 8;       // MI355X: 8 XCDs, workgroups dispatched round-robin

// ---------------------------------------------------------------------------
// bf16 / fp16 conversion. bf16 is stored as uint16_t bit patterns.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float bf16_to_f32(uint16_t b) {
    return __uint_as_float(static_cast<uint32_t>(b) << 16);
}

// Round-to-nearest-even; NaN becomes the quiet NaN (bits >> 16) | 0x40. gfx950's
// v_cvt_pk_bf16_f32 implements exactly this mapping (checked against the
// integer formulation on all 2^32 inputs), so conversions use the instruction.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    const float2_t f = {lo, hi};
    const bf16x2_t h = __builtin_convertvector(f, bf16x2_t);
    uint32_t u;
    __builtin_memcpy(&u, &h, 4);
    return u;
}

__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
    const __bf16 h = static_cast<__bf16>(f);
    uint16_t u;
    __builtin_memcpy(&u, &h, 2);
    return u;
}

// Value of f rounded to bf16, as fp32.
__device__ __forceinline__ float round_bf16(float f) {
    return __uint_as_float(static_cast<uint32_t>(f32_to_bf16(f)) << 16);
}

__device__ __forceinline__ float f16_to_f32(uint16_t h) {
    _Float16 v;
    __builtin_memcpy(&v, &h, 2);
    return static_cast<float>(v);
}

__device__ __forceinline__ uint16_t f32_to_f16(float f) {
    _Float16 v = static_cast<_Float16>(f);
    uint16_t h;
    __builtin_memcpy(&h, &v, 2);
    return h;
}

// N elements at any element's address, moved as one vector (global loads and
// stores of up to 16 bytes need no wider alignment on gfx950).
template <typename T, int N>
struct __attribute__((packed, aligned(alignof(T)))) Unaligned {
    T v[N];
};

// Element access by storage dtype (MOE_DTYPE_*), used by the transport and
// activation kernels that support fp32 / fp16 / bf16.
template <int DT> struct Elem;
template <> struct Elem<MOE_DTYPE_F32> {
    using T = float;
    static __device__ __forceinline__ float load(T v) { return v; }
    static __device__ __forceinline__ T store(float f) { return f; }
    static __device__ __forceinline__ T store_product(float a, float b) { return a * b; }
};
template <> struct Elem<MOE_DTYPE_F16> {
    using T = uint16_t;
    static __device__ __forceinline__ float load(T v) { return f16_to_f32(v); }
    static __device__ __forceinline__ T store(float f) { return f32_to_f16(f); }
    // a * b rounded once (v_fma_mixlo_f16). Paired conversions (v_cvt_pk_f16_f32)
    // would round the fp32 product first; the empty asm keeps the compiler from pairing.
    static __device__ __forceinline__ T store_product(float a, float b) {
        T h = f32_to_f16(a * b);
        asm("" : "+v"(h));
        return h;
    }
};
template <> struct Elem<MOE_DTYPE_BF16> {
    using T = uint16_t;
    static __device__ __forceinline__ float load(T v) { return bf16_to_f32(v); }
    static __device__ __forceinline__ T store(float f) { return f32_to_bf16(f); }
    static __device__ __forceinline__ T store_product(float a, float b) { return f32_to_bf16(a * b); }
};

// ---------------------------------------------------------------------------
// SiLU, g / (1 + exp(-g)) with a correctly rounded fp32 division, in a fixed
// operation sequence that a CPU restatement with IEEE fp32 operations reproduces
// bit for bit. exp(x): Cody-Waite reduction x = n*ln2 + r (ln2 = 16-bit head +
// tail; n*ln2_hi is exact, so the fma rounds as a separate subtraction would),
// degree-7 Taylor polynomial of e^r in Horner form with separately rounded
// multiply and add, then ldexp; +inf above 88. Within 2 ulp of exp on [-80, 88].
// Below -80 any tiny exp leaves 1 + exp at 1, so one clamp stands for a test,
// and a NaN g is NaN through the division whatever exp is: about 40 VALU
// operations, which is what a bf16 or fp16 activation kernel is bound by.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float silu_f32(float g) {
#pragma clang fp contract(off)
    const float x = __builtin_amdgcn_fmed3f(-g, -80.0f, 1000.0f);
    const float n = rintf(x * __uint_as_float(0x3fb8aa3bu));  // log2(e)
    float r = __builtin_fmaf(-n, __uint_as_float(0x3f317200u), x);  // ln2 head
    r = r - n * __uint_as_float(0x35bfbe8eu);                  // ln2 tail
    float p = __uint_as_float(0x39500d01u);                    // 1/7!
    p = p * r + __uint_as_float(0x3ab60b61u);                  // 1/6!
    p = p * r + __uint_as_float(0x3c088889u);                  // 1/5!
    p = p * r + __uint_as_float(0x3d2aaaabu);                  // 1/4!
    p = p * r + __uint_as_float(0x3e2aaaabu);                  // 1/3!
    p = p * r + 0.5f;
    p = p * r + 1.0f;
    p = p * r + 1.0f;
    const float e = x > 88.0f ? __builtin_inff() : __builtin_amdgcn_ldexpf(p, static_cast<int>(n));
    return g / (1.0f + e);
}

inline int dtype_size(int dtype) {
    switch (dtype) {
        case MOE_DTYPE_F32: return 4;
        case MOE_DTYPE_F16: return 2;
        case MOE_DTYPE_BF16: return 2;
        default: return 0;
    }
}

// ---------------------------------------------------------------------------
// Host-side error reporting: a status code plus a thread-local message.
// ---------------------------------------------------------------------------
void set_error(const char* fmt, ...);
int fail(int status, const char* fmt, ...);
int check_launch(const char* what);

}  // namespace moe

#define MOE_REQUIRE(cond, status, ...)                \
    do {                                              \
        if (!(cond)) return ::moe::fail(status, __VA_ARGS__); \
    } while (0)
