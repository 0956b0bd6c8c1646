// Shared device helpers for the gfx950 quantized-linear kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

#include "../../include/gpu_api.h"

#define GPU_API extern "C" __attribute__((visibility("default")))

// Launch check in the reference's convention (csrc/common.cuh:128): a positive hipError_t on failure.
#define KCHECK()                                   \
    do {                                           \
        hipError_t e__ = hipGetLastError();        \
        if (e__ != hipSuccess) return (int)e__;    \
    } while (0)

// "Done once per device" flags for host-side set-up (a kernel's dynamic LDS limit, a memory pool attribute): one bit per
// device ordinal, set after the call has succeeded on that device.  Two threads that race both make the call, which is
// idempotent.  Devices past 63 are not remembered and make the call every time.
struct PerDeviceOnce {
    std::atomic<uint64_t> done{0};
    static int current() {
        int dev = 0;
        return hipGetDevice(&dev) == hipSuccess ? dev : -1;
    }
    bool is_done(int dev) const { return dev >= 0 && dev < 64 && ((done.load(std::memory_order_acquire) >> dev) & 1u); }
    void mark(int dev) { if (dev >= 0 && dev < 64) done.fetch_or((uint64_t)1 << dev, std::memory_order_release); }
};
// Raises a kernel's dynamic LDS limit on the current device, the first time it is asked for there.  0 or a hipError_t.
inline int allow_dynamic_lds(const void* kern, int bytes, PerDeviceOnce& once) {
    const int dev = PerDeviceOnce::current();
    if (once.is_done(dev)) return 0;
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return (int)e;
    once.mark(dev);
    return 0;
}

inline int device_cu_count() {
    static std::atomic<int> cached[64];   // compute units per device ordinal, 0 = not asked yet
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    const bool keep = dev >= 0 && dev < 64;
    if (keep && (n = cached[dev].load(std::memory_order_relaxed)) > 0) return n;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
    if (keep) cached[dev].store(n, std::memory_order_relaxed);
    return n;
}

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float u2f(uint32_t u) { return __builtin_bit_cast(float, u); }
__device__ __forceinline__ uint32_t f2u(float f) { return __builtin_bit_cast(uint32_t, f); }

// bf16 / f16 <-> f32; the narrowing conversions round to nearest even (v_cvt_pk_bf16_f32 / v_cvt_f16_f32).
__device__ __forceinline__ float bf16_to_f(uint16_t b) { return u2f((uint32_t)b << 16); }
__device__ __forceinline__ uint16_t f_to_bf16(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }
__device__ __forceinline__ float f16_to_f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
// The empty asm keeps the compiler from folding a preceding fp32 fma into v_fma_mixlo_f16, which rounds the exact
// fma result to f16 once; the reference rounds to fp32 first and converts afterwards, and ties differ between the two.
__device__ __forceinline__ uint16_t f_to_f16(float v) {
    asm("" : "+v"(v));
    return __builtin_bit_cast(uint16_t, (_Float16)v);
}

// Two floats -> packed bf16 pair (a in the low half), one v_cvt_pk_bf16_f32.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// A float rounded to bf16 and widened back, as one instruction: the pack conversion puts its second operand into the upper half,
// where the bits of a float are, and the bf16 of 0 below it.  (Converted into the lower half, the value takes a shift left, which
// like the conversion runs at half the rate of a plain add: 4.2 and 2.3 cycles of a SIMD per wave.)  The asm keeps the compiler
// from seeing a constant half, which it would convert by itself and put together with shifts again.
__device__ __forceinline__ float rnd_bf16(float v) {
    float zero;
    asm("v_mov_b32 %0, 0" : "=v"(zero));
    return u2f(pack_bf16x2(zero, v));
}

// Round a float to the precision of the dtype code and widen back (rnd<T>, csrc/common.cuh:25-28).
template <int DT> __device__ __forceinline__ float rnd_dt(float v) {
    if (DT == DT_BF16) return rnd_bf16(v);
    if (DT == DT_F16) return f16_to_f(f_to_f16(v));
    return v;
}
template <int DT> __device__ __forceinline__ float ld_dt(const void* p, int64_t i) {
    if (DT == DT_BF16) return bf16_to_f(((const uint16_t*)p)[i]);
    if (DT == DT_F16) return f16_to_f(((const uint16_t*)p)[i]);
    return ((const float*)p)[i];
}
template <int DT> __device__ __forceinline__ void st_dt(void* p, int64_t i, float v) {
    if (DT == DT_BF16) ((uint16_t*)p)[i] = f_to_bf16(v);
    else if (DT == DT_F16) ((uint16_t*)p)[i] = f_to_f16(v);
    else ((float*)p)[i] = v;
}
template <int DT> struct dt_size { static constexpr int value = DT == DT_F32 ? 4 : 2; };

// Two floats -> packed f16 pair as one v_cvt_pk_f16_f32, and back.  The empty asm for the reason given at f_to_f16.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
    asm("" : "+v"(a), "+v"(b));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
}
__device__ __forceinline__ void unpack_f16x2(uint32_t u, float& a, float& b) {
    const f16x2 h = __builtin_bit_cast(f16x2, u);
    a = (float)h[0];
    b = (float)h[1];
}

// Reductions over the 64 lanes of a wave, result in every lane: data-parallel-primitive moves inside rows of 16 lanes,
// then the two row-swap instructions.  (A shuffle goes through the LDS and costs its latency six times.)
template <int CTRL> __device__ __forceinline__ int dpp_int(int x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, false); }
__device__ __forceinline__ float wave_max_f32(float v) {
    const auto mv = [](float x, auto ctrl) { return __builtin_bit_cast(float, dpp_int<decltype(ctrl)::value>(__builtin_bit_cast(int, x))); };
    v = fmaxf(v, mv(v, std::integral_constant<int, 0xB1>{}));    // quad_perm [1,0,3,2]
    v = fmaxf(v, mv(v, std::integral_constant<int, 0x4E>{}));    // quad_perm [2,3,0,1]
    v = fmaxf(v, mv(v, std::integral_constant<int, 0x141>{}));   // row_half_mirror
    v = fmaxf(v, mv(v, std::integral_constant<int, 0x140>{}));   // row_mirror
    auto s = __builtin_amdgcn_permlane16_swap(f2u(v), f2u(v), false, false);
    v = fmaxf(u2f(s[0]), u2f(s[1]));
    s = __builtin_amdgcn_permlane32_swap(f2u(v), f2u(v), false, false);
    return fmaxf(u2f(s[0]), u2f(s[1]));
}
__device__ __forceinline__ double wave_sum_f64(double v) {
    const auto mv = [](double x, auto ctrl) {
        const int64_t b = __builtin_bit_cast(int64_t, x);
        constexpr int C = decltype(ctrl)::value;
        return __builtin_bit_cast(double, ((int64_t)dpp_int<C>((int)(b >> 32)) << 32) | (uint32_t)dpp_int<C>((int)b));
    };
    v += mv(v, std::integral_constant<int, 0xB1>{});
    v += mv(v, std::integral_constant<int, 0x4E>{});
    v += mv(v, std::integral_constant<int, 0x141>{});
    v += mv(v, std::integral_constant<int, 0x140>{});
    const auto join = [](uint32_t hi, uint32_t lo) { return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo); };
    uint64_t b = __builtin_bit_cast(uint64_t, v);
    auto l = __builtin_amdgcn_permlane16_swap((uint32_t)b, (uint32_t)b, false, false);
    auto h = __builtin_amdgcn_permlane16_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    v = join(h[0], l[0]) + join(h[1], l[1]);
    b = __builtin_bit_cast(uint64_t, v);
    l = __builtin_amdgcn_permlane32_swap((uint32_t)b, (uint32_t)b, false, false);
    h = __builtin_amdgcn_permlane32_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    return join(h[0], l[0]) + join(h[1], l[1]);
}

// 1/sqrt(a) in fp64, rounded to fp32: two Newton steps on the hardware's fp32 estimate (23 bits, then 45, then the rounding
// of fp64), a tenth of the instructions of the fp64 square root and division, which serve the ends of the range.
__device__ __forceinline__ float rsqrt_cr(float a) {
    if (!(a > 1e-30f && a < 1e30f)) return (float)(1.0 / sqrt((double)a));
    const double d = (double)a;
    double y = (double)__builtin_amdgcn_rsqf(a);
#pragma unroll
    for (int i = 0; i < 2; ++i) y = __builtin_fma(0.5 * y, __builtin_fma(-d * y, y, 1.0), y);
    return (float)y;
}

// Workgroup -> tile.  Workgroups are dealt round-robin to the 8 XCDs (each with its own L2), so first renumber them
// XCD-contiguously, then walk tiles in panels of 4 tile rows so that the 32 workgroups an XCD runs at once cover a
// 4 x 8 patch of tiles and share A rows / W rows in that XCD's L2.
// A persistent kernel calls this three times per tile (two operand streams and the epilogue), and two integer divisions
// are about a hundred dependent scalar instructions each time, so the divisions are multiplications: `magic` =
// panel_magic(tiles_m, tiles_n) from the host turns lin / (4 * tiles_n) into a multiply-high, and the rows of a panel
// are 4, or 1..3 in the last one.  magic == 0 (shapes beyond the multiply's exact range) divides.
__host__ __device__ inline uint32_t panel_magic(int tiles_m, int tiles_n) {
    // floor(n / d) == (n * ceil(2^32 / d)) >> 32 for n, d <= 65536
    const int64_t per_panel = 4 * (int64_t)tiles_n, ntiles = (int64_t)tiles_m * tiles_n;
    if (per_panel > 65536 || ntiles > 65536) return 0;
    return (uint32_t)(((1ull << 32) + (uint64_t)per_panel - 1) / (uint64_t)per_panel);
}
__device__ __forceinline__ void tile_of_block(int b, int nblocks, int tiles_m, int tiles_n, int& tm, int& tn, uint32_t magic = 0) {
    const int base = nblocks >> 3, rem = nblocks & 7;
    const int xcd = b & 7, idx = b >> 3;
    const int lin = xcd * base + (xcd < rem ? xcd : rem) + idx;
    constexpr int GM = 4;
    const int per_panel = GM * tiles_n;
    const int panel = magic ? (int)__umulhi((uint32_t)lin, magic) : lin / per_panel;
    const int first_m = panel * GM;
    const int rows = tiles_m - first_m < GM ? tiles_m - first_m : GM;
    const int in_panel = lin - panel * per_panel;
    int q;   // in_panel / rows
    if (rows == 4) q = in_panel >> 2;
    else if (rows == 2) q = in_panel >> 1;
    else if (rows == 1) q = in_panel;
    else if (magic) q = (int)__umulhi((uint32_t)in_panel, 0x55555556u);   // rows == 3, in_panel < 65536
    else q = in_panel / rows;
    tm = first_m + in_panel - q * rows;
    tn = q;
}


// Integer sums of a matrix instruction as floats without v_cvt_f32_i32: the accumulator starts at the bits of 1.5 * 2^23, where floats
// have a step of 1 and room for +-2^22, so that its bits are a float all the way, and an exact subtraction takes the start off again.
// Two waves of a SIMD issue fp32 additions, multiplications and fma on registers side by side, 1.05 ns each (2.2 cycles), also beside
// another wave's slower instruction; conversions, maxima, packing, left shifts and anything with a scalar operand take 1.85 ns, one at a time.
// A kernel that starts its sums there holds their largest magnitude below kSumRoom by a static_assert.
constexpr int kSumOne = 0x4B400000, kSumRoom = 1 << 22;
__device__ __forceinline__ float sum_value(int bits) { return __builtin_bit_cast(float, bits) - 12582912.f; }

// Four consecutive elements of a dtype-coded array <-> four floats (8- or 16-byte vector access).
template <int OUT_DT> __device__ __forceinline__ void load4(const void* p, int64_t i, float* v) {
    if (OUT_DT == DT_F32) {
        const float4 f = *reinterpret_cast<const float4*>((const float*)p + i);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    } else {
        const uint2 u = *reinterpret_cast<const uint2*>((const uint16_t*)p + i);
        if (OUT_DT == DT_BF16) {
            v[0] = u2f(u.x << 16); v[1] = u2f(u.x & 0xffff0000u); v[2] = u2f(u.y << 16); v[3] = u2f(u.y & 0xffff0000u);
        } else {
            v[0] = f16_to_f((uint16_t)(u.x & 0xffffu)); v[1] = f16_to_f((uint16_t)(u.x >> 16));
            v[2] = f16_to_f((uint16_t)(u.y & 0xffffu)); v[3] = f16_to_f((uint16_t)(u.y >> 16));
        }
    }
}
template <int OUT_DT> __device__ __forceinline__ void store4(void* p, int64_t i, const float* v) {
    if (OUT_DT == DT_F32) {
        *reinterpret_cast<float4*>((float*)p + i) = make_float4(v[0], v[1], v[2], v[3]);
    } else if (OUT_DT == DT_BF16) {
        uint2 u;
        u.x = pack_bf16x2(v[0], v[1]);
        u.y = pack_bf16x2(v[2], v[3]);
        *reinterpret_cast<uint2*>((uint16_t*)p + i) = u;
    } else {
        uint2 u;
        u.x = pack_f16x2(v[0], v[1]);
        u.y = pack_f16x2(v[2], v[3]);
        *reinterpret_cast<uint2*>((uint16_t*)p + i) = u;
    }
}

