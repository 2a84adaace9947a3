// Internal helpers shared by the libheterokv HIP sources (not part of the ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>
#include <atomic>

#include "../../include/heterokv.h"

namespace hkv {

// ---------------------------------------------------------------- errors
void set_error(const char* fmt, ...);
void clear_error();

#define HKV_REQUIRE(cond, code, ...)            \
    do {                                        \
        if (!(cond)) {                          \
            ::hkv::set_error(__VA_ARGS__);      \
            return (code);                      \
        }                                       \
    } while (0)

#define HKV_HIP_CHECK(expr)                                                        \
    do {                                                                           \
        hipError_t _e = (expr);                                                    \
        if (_e != hipSuccess) {                                                    \
            ::hkv::set_error("%s failed: %s", #expr, hipGetErrorString(_e));       \
            return HKV_ERR_HIP;                                                    \
        }                                                                          \
    } while (0)

// Launch-error check after a kernel launch.
#define HKV_LAUNCH_CHECK(name)                                                     \
    do {                                                                           \
        hipError_t _e = hipGetLastError();                                         \
        if (_e != hipSuccess) {                                                    \
            ::hkv::set_error("launch of %s failed: %s", name, hipGetErrorString(_e)); \
            return HKV_ERR_HIP;                                                    \
        }                                                                          \
    } while (0)

// Raises kernel fn's dynamic LDS limit to `bytes` on the current device, once per device
// (the attribute is held per device); `done` is the kernel's bitmask of devices already
// raised.  Safe to call from several host threads.
#define HKV_RAISE_LDS(fn, bytes, done)                                                        \
    do {                                                                                      \
        int _dev = 0;                                                                         \
        HKV_HIP_CHECK(hipGetDevice(&_dev));                                                   \
        const uint64_t _bit = 1ull << (_dev & 63);                                            \
        if (!((done).load(std::memory_order_acquire) & _bit)) {                               \
            HKV_HIP_CHECK(hipFuncSetAttribute((const void*)(fn),                              \
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (bytes))); \
            (done).fetch_or(_bit, std::memory_order_release);                                 \
        }                                                                                     \
    } while (0)

// The unpacked INT4 source of the fused entry points: present and aligned for the kernels'
// vector loads.
inline int check_fused_source(const HkvFusedArgs* f, const char* name) {
    if (f->num_tokens == 0) return HKV_OK;
    HKV_REQUIRE(f->k_codes && f->v_codes && f->k_scales && f->v_scales && f->k_zps && f->v_zps, HKV_ERR_ARG,
                "%s: null pointer", name);
    HKV_REQUIRE((((uintptr_t)f->k_codes | (uintptr_t)f->v_codes | (uintptr_t)f->k_scales | (uintptr_t)f->v_scales) & 15) == 0 &&
                    (((uintptr_t)f->k_zps | (uintptr_t)f->v_zps) & 3) == 0,
                HKV_ERR_ARG, "%s: codes and scales must be 16-byte aligned, zero points 4-byte", name);
    return HKV_OK;
}

constexpr int kHeadDim = 128;
constexpr int kBlockTokens = 16;
constexpr int kCodeRowBytes = kHeadDim / 2;          // 64 B of packed codes per token row
constexpr int kHeadCodeBytes = kBlockTokens * kCodeRowBytes;  // 1024 B per (block, head)

// Block record layout (bytes); see heterokv.h.  A record holds H head parts of
// kHeadPartBytes each; inside a part: K codes, V codes, K scales, V scales, K zero
// points, V zero points.
constexpr int kHeadPartBytes = 2208;
constexpr int kPartKc = 0, kPartVc = 1024, kPartKs = 2048, kPartVs = 2112, kPartKz = 2176, kPartVz = 2192;
struct RecordLayout {
    int64_t bytes;
    __host__ __device__ explicit RecordLayout(int H) : bytes((int64_t)H * kHeadPartBytes) {}
    __host__ __device__ static int64_t part(int h) { return (int64_t)h * kHeadPartBytes; }
    __host__ __device__ static int64_t kc(int h) { return part(h) + kPartKc; }
    __host__ __device__ static int64_t vc(int h) { return part(h) + kPartVc; }
    __host__ __device__ static int64_t ks(int h) { return part(h) + kPartKs; }
    __host__ __device__ static int64_t vs(int h) { return part(h) + kPartVs; }
    __host__ __device__ static int64_t kz(int h) { return part(h) + kPartKz; }
    __host__ __device__ static int64_t vz(int h) { return part(h) + kPartVz; }
};

// ---------------------------------------------------------------- kernel arguments
// A kernel's argument block is read with scalar loads, and a prologue whose loads depend
// on each other (a pointer tested, then a field on another 64-byte line read) misses
// the scalar cache one line at a time, a memory round trip each.  Touching every line of
// the block once, all loads issued together, at kernel entry makes the later argument
// loads hit the scalar cache: one round trip instead of a chain of them.
template <class P>
__device__ __forceinline__ void touch_kernel_args(const P& p) {
    constexpr int kWords = (int)(sizeof(P) / 4), kLines = (kWords + 15) / 16;
    const uint32_t* w = reinterpret_cast<const uint32_t*>(&p);
    uint32_t v[kLines];
#pragma unroll
    for (int i = 0; i < kLines; ++i) v[i] = w[16 * i < kWords ? 16 * i : kWords - 1];
    static_assert(kLines <= 8, "argument block of at most 8 lines");
    // one statement, so that every load is issued before the single wait
    asm volatile("" ::"s"(v[0]), "s"(v[1 < kLines ? 1 : 0]), "s"(v[2 < kLines ? 2 : 0]), "s"(v[3 < kLines ? 3 : 0]),
                 "s"(v[4 < kLines ? 4 : 0]), "s"(v[5 < kLines ? 5 : 0]), "s"(v[6 < kLines ? 6 : 0]),
                 "s"(v[7 < kLines ? 7 : 0]));
    __builtin_amdgcn_sched_barrier(0);   // nothing that reads an argument moves above the wait
}

// A wave-uniform read of a word the kernel does not write, through the scalar cache
// (a constant-address-space load): it completes on the scalar counter, so it does not
// queue behind the wave's vector loads, and no vector-to-scalar move waits for it.
// The scalar cache starts every kernel empty.
__device__ __forceinline__ int32_t load_uniform_i32(const int32_t* base, int64_t i) {
    typedef const __attribute__((address_space(4))) int32_t* const_i32_p;
    return *((const_i32_p)base + i);
}

// ---------------------------------------------------------------- numeric helpers
__device__ __forceinline__ float h2f(uint16_t b) {
    return __half2float(__ushort_as_half(b));
}
__device__ __forceinline__ uint16_t f2h_rn(float f) {
    return __half_as_ushort(__float2half_rn(f));
}
__device__ __forceinline__ float bf2f(uint16_t b) {
    return __uint_as_float(((uint32_t)b) << 16);
}
// float -> bfloat16, round to nearest even (NaN stays NaN), as c10::BFloat16.
__device__ __forceinline__ uint16_t f2bf_rn(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    uint32_t bias = 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)((u + bias) >> 16);
}

__device__ __forceinline__ float load_as_float(const void* p, int dtype, int64_t i) {
    if (dtype == HKV_DTYPE_F16) return h2f(((const uint16_t*)p)[i]);
    if (dtype == HKV_DTYPE_BF16) return bf2f(((const uint16_t*)p)[i]);
    return ((const float*)p)[i];
}

// Group quantization parameters, bit-exact with kv_compressor.py:76-84 (float32 math,
// IEEE division, clamp(min=1e-8) that keeps NaN, round half to even).
struct QParams {
    float scale;
    float zpf;
    float inv;     // RN(1 / scale)
    uint8_t zp;
};

__device__ __forceinline__ QParams qparams_from_minmax(float mn, float mx) {
    QParams q;
    float s = (mx - mn) / 15.0f;
    s = (s < 1e-8f) ? 1e-8f : s;          // torch.clamp(min=1e-8): NaN propagates
    float z = rintf(-mn / s);
    z = fminf(fmaxf(z, 0.0f), 15.0f);
    q.scale = s;
    q.zpf = z;
    q.inv = 1.0f / s;
    q.zp = (uint8_t)z;
    return q;
}

// x / scale rounded to nearest, without a division per element (Markstein): with
// y = RN(1/s), q = RN(x y) and the exact residual r = x - s q (one fma),
// RN(q + r y) is the correctly rounded quotient.  Only when the residual
// underflows (quotients below 2^-60 here) can it differ from x / s, and such a
// quotient leaves rint(quotient + zp) unchanged; checked for every fp16 value and
// 4096 random fp32 values against 20000 scales, all 16 zero points.  An infinite
// or NaN scale takes the plain division.
__device__ __forceinline__ float div_by_scale(float x, const QParams& q) {
    if (!(fabsf(q.scale) < INFINITY)) return x / q.scale;
    const float q0 = __fmul_rn(x, q.inv);
    const float r = __builtin_fmaf(-q0, q.scale, x);
    return __builtin_fmaf(r, q.inv, q0);
}

// kv_compressor.py:86-88: clamp(round(x / scale + zp), 0, 15)
__device__ __forceinline__ uint32_t quant_code(float x, const QParams& q) {
    float t = div_by_scale(x, q);
    t = t + q.zpf;
    t = rintf(t);
    t = fminf(fmaxf(t, 0.0f), 15.0f);
    return (uint32_t)t;
}

// quant_code before its rounding: x / scale + zp clamped to [0, 15].  Clamping first
// and rounding after gives the same code for integer bounds (a NaN clamps to 0);
// code_into() rounds to nearest even, as rintf does, with v_cvt_pk_u8_f32, which also
// writes the code into byte `sel` (0..3) of `word`.
__device__ __forceinline__ float quant_unrounded(float x, const QParams& q) {
    return fminf(fmaxf(div_by_scale(x, q) + q.zpf, 0.0f), 15.0f);
}
__device__ __forceinline__ uint32_t code_into(float t, uint32_t sel, uint32_t word) {
    return __builtin_amdgcn_cvt_pk_u8_f32(t, sel, word);
}

// Position of logical code k (0..7) inside a packed 32-bit word.
__host__ __device__ constexpr int nib_shift(int k) { return (k & 1) * 16 + (k >> 1) * 4; }

}  // namespace hkv
