// W6 requantizer for the reference's two-plane format: a bf16 weight in its original basis -> ConvRot256 -> 6-bit codes
// (nibble plane, then 2-bit plane), one fp8-e4m3 relative scale per 32 columns, one fp32 scale per row.  Replaces
// gpu_w6_requant, csrc/vendor/w6a8_requant.cu: same float expressions (cited by line), bit for bit.
//
// A load-time / LoRA-bake kernel: 2 B read + 0.78 B written per weight, bound by its vector instructions (about 4000 cycles
// of them per 1024 values).  A wave owns chunks of 1024 values, 16 consecutive ones per lane, and keeps them in registers from
// the load to the packed stores: a scale group is two neighbouring lanes, a rotation group sixteen.  A workgroup takes as many
// rows as fill its waves best and cuts them into chunks as if they were one, so only its last wave can have idle lanes; the rows'
// maxima meet in LDS.  5376 x 5376, whole rows to a workgroup, the sixth
// wave a quarter full: 69.4 us; three rows on 16 waves: 55.  (One thread per group over a row in LDS, as the reference has it,
// leaves a third of the lanes idle and reads LDS at a stride of 32 words: 170 us; the copy rate of the part allows 16 us.)
#include "common.hpp"
#include "convrot.hpp"

namespace {

constexpr int kG = 32;   // columns per relative scale
constexpr int kMaxRows = 16;   // rows of a workgroup

// float -> fp8 e4m3 bits, round to nearest even, saturating at 448 (finite inputs)
__device__ __forceinline__ uint32_t f_to_e4m3(float x) {
    const uint32_t sgn = (f2u(x) >> 31) << 7;
    const float a = fabsf(x);
    if (a != a) return sgn | 0x7f;
    if (a > 448.f) return sgn | 0x7e;
    if (a < 0.015625f) return sgn | (uint32_t)nearbyintf(a * 512.f);
    const uint32_t u = f2u(a);
    int e = (int)(u >> 23) - 127;
    const float frac = u2f((u & 0x007fffffu) | 0x3f800000u);                     // in [1, 2)
    int m = (int)nearbyintf((frac - 1.f) * 8.f);
    if (m == 8) { m = 0; ++e; }
    const uint32_t code = ((uint32_t)(e + 7) << 3) | (uint32_t)m;
    return sgn | (code > 0x7e ? 0x7e : code);
}
__device__ __forceinline__ float e4m3_to_f(uint32_t v) {
    const uint32_t e = (v >> 3) & 0xf, m = v & 7;
    const float f = e == 0 ? (float)m * 0.001953125f : (e == 15 && m == 7) ? __builtin_nanf("") : u2f(((e + 120) << 23) | (m << 20));
    return (v & 0x80) ? -f : f;
}
// Level i of a group's grid, i counted from the middle (f = i - 31, a whole number in a float), :59-61.
__device__ __forceinline__ float level(float f, float s) { return __builtin_amdgcn_fmed3f(__builtin_rintf(f * s), -127.0f, 127.0f); }
// The other lane of an even/odd pair.
__device__ __forceinline__ float pair_lane(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, false));
}

// Four values of a group -> their code bytes (level index + 1), :63-80,126-148.  Wanted is the pair of neighbouring levels
// with level(l) < t <= level(l + 1), l in -31..30 (ends beyond t count as bracketing it).  Any f in -30..30 next to the
// pair settles it by one look: l is f when level(f) is below t, else f - 1.
//   plain (every lane's step in [1, 4], every |t| < 127): f = rint(t / s).  f s is within s/2 of t and a level within 1/2
//     of its product, so level(f - 1) < t <= level(f + 1) for s >= 1, whichever way t / s falls at a tie; no level
//     reaches the clamp at +-127; and f s is a 6-bit times a 4-bit number, so adding 1.5 * 2^23 rounds it as rint does.  The
//     sign of level(f) - t stands for the compare: a level of zero is +0 here.  (Below, it can be -0, and -0 - (+0) has the sign
//     of a smaller level: steps below 1/62 around a zero value, i.e. zero blocks in a row that is not zero.)
//   else: levels are whole numbers, so the first level at or above t is the first that reaches ceil(t), i.e. whose product
//     reaches ceil(t) - 1/2 (or passes it, where that tie rounds down to an even number).  With z that quotient, rint(z) is
//     that position or the one before it: a whole z needs the tie looked at, any other is farther from a whole number
//     than the last bit of the division reaches.  Outside [-127, 127] every level is on one side of t: an end of the grid.
//     NaN: a value's is the middle of the grid (the reference's conversion of the estimate to an integer gives 0) and above
//     no threshold; a step's (an infinite row scale) makes every level -127, the clamp's lower end.
// `x0` is the hash input of value 0 without its low four bits' share, kc[j] that share (see the caller).
template <bool PLAIN>
__device__ __forceinline__ uint32_t codes4(const float* v, float inv_sc, float s, float inv_s, uint32_t x0, const uint32_t* kc) {
    constexpr float M = 12582912.f;
    uint32_t out = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float t = v[j] * inv_sc;
        float f, lf, lg;
        if (PLAIN) f = __builtin_fmaf(t, inv_s, M) - M;
        else f = t > (s != s ? -127.f : 127.f) ? 30.f : t <= -127.f ? -30.f : __builtin_rintf((__builtin_ceilf(t) - 0.5f) * inv_s);
        f = PLAIN || t == t ? __builtin_amdgcn_fmed3f(f, -30.f, 30.f) : 0.f;
        lf = PLAIN ? __builtin_fmaf(f, s, M) - M : level(f, s);
        const float g = PLAIN ? f - __builtin_copysignf(1.f, lf - t) : lf < t ? f + 1.f : f - 1.f;   // the pair's other end
        lg = PLAIN ? __builtin_fmaf(g, s, M) - M : level(g, s);
        const uint32_t h = x0 + kc[j];                                            // x * 747796405 + 2891336453, :21-25
        const uint32_t w = ((h >> ((h >> 28u) + 4u)) ^ h) * 277803737u;
        const float u = (float)(((w >> 22u) ^ w) & 0xffffff00u) * 0x1.0p-32f;     // :27-31, the 24 bits left where they are
        const float thr = __builtin_fmaf(u, fabsf(lg - lf), fminf(lf, lg));
        const float half = PLAIN ? __builtin_copysignf(0.5f, thr - t) : t > thr ? -0.5f : 0.5f;   // negative where t is above the threshold
        out = __builtin_amdgcn_cvt_pk_u8_f32(fminf(f, g) - half + 32.25f, j, out);
    }
    return out;
}

// The maximum over the 16 lanes of a rotation group, in all of them.
__device__ __forceinline__ float group_max(float x) {
    const auto step = [&](auto ctrl) {
        x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false)));
    };
    step(std::integral_constant<int, 0xB1>{});    // lane ^ 1
    step(std::integral_constant<int, 0x4E>{});    // lane ^ 2
    step(std::integral_constant<int, 0x141>{});   // the other half of eight
    step(std::integral_constant<int, 0x140>{});   // the other half of sixteen
    return x;
}

// rpb rows per workgroup, `groups` = K / 256 rotation groups each; wave w takes the chunks w, w + waves, ... of all of them.
// group / `groups` is (group * inv_groups) >> 16.
template <int C>
__global__ void __launch_bounds__(1024) w6_requant_kernel(const uint16_t* w, uint8_t* packed, uint8_t* s_rel, float* s_channel, int N, int K,
                                                         uint64_t seed, int groups, uint32_t inv_groups, int rpb) {
    extern __shared__ __attribute__((aligned(16))) float tiles[];   // a rotation tile per wave
    __shared__ uint32_t row_max[kMaxRows];                          // the bits of a maximum that is never negative
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int64_t n0 = (int64_t)blockIdx.x * rpb;
    const int ngroups = (N - n0 < rpb ? (int)(N - n0) : rpb) * groups;
    float v[C][16], gs[C], gmax[C];
    if (threadIdx.x < kMaxRows) row_max[threadIdx.x] = 0u;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int chunk = wave + c * nw, group = chunk * 4 + (lane >> 4);
        const bool act = group < ngroups;               // a lane's 16 values are all in or all out
        if (act) {
            const uint4* src = reinterpret_cast<const uint4*>(w + n0 * K + chunk * convrot::kChunk + lane * 16);
            const uint4 a = src[0], b = src[1];
            const uint32_t ww[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[c][2 * i] = u2f(ww[i] << 16);
                v[c][2 * i + 1] = u2f(ww[i] & 0xffff0000u);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) v[c][i] = 0.f;
        }
        // ConvRot256 (:174-206) as the row quantizer does it; the rotated row is kept in the weight dtype (:209-217)
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) m = fmaxf(fmaxf(m, fabsf(v[c][i])), fabsf(v[c][i + 1]));
        if (__builtin_amdgcn_ballot_w64(m >= convrot::kOnceLimit) == 0) convrot::rotate_chunk<256, true>(v[c], tiles + wave * convrot::kLdsPerWave, lane);
        else convrot::rotate_chunk<256>(v[c], tiles + wave * convrot::kLdsPerWave, lane);
        m = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            v[c][i] = rnd_bf16(v[c][i]);
            v[c][i + 1] = rnd_bf16(v[c][i + 1]);
            m = fmaxf(fmaxf(m, fabsf(v[c][i])), fabsf(v[c][i + 1]));
        }
        // the group's step by two alternating-least-squares rounds, :94-117.  num adds its 32 terms in index order: the odd
        // lane of the pair goes on where the even one ends.  den sums whole numbers below 2^15: exact in any order.
        m = fmaxf(m, pair_lane(m));
        float step = fmaxf(m / 31.0f, 1e-8f), inv = 1.0f / step;
        bool nan = false;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            float q[16], num = 0.f, den = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                q[i] = __builtin_rintf(v[c][i] * inv);
                if (it > 0) q[i] = __builtin_amdgcn_fmed3f(q[i], -31.0f, 31.0f);   // the first step is the largest value's 31st part
                num = __builtin_fmaf(v[c][i], q[i], num);
                den = __builtin_fmaf(q[i], q[i], den);
            }
            den += pair_lane(den);
            const float head = pair_lane(num);
            num = lane & 1 ? head : 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) num = __builtin_fmaf(v[c][i], q[i], num);
            const float other = pair_lane(num);
            num = lane & 1 ? num : other;
            nan = num != num;
            step = fmaxf(num / fmaxf(den, 1e-8f), 1e-8f);
            inv = 1.0f / step;
        }
        // the group's largest decoded magnitude, :118-119: products and roundings are monotonic, so it is the largest
        // value's (a NaN takes -31 in the reference's clamp)
        const float amax = group_max(fmaxf(0.f, (nan ? 31.0f : fminf(31.0f, __builtin_rintf(m * inv))) * step));   // 0 * inf counts for nothing
        if (act && (lane & 15) == 0) atomicMax(row_max + (group * inv_groups >> 16), f2u(amax));
        gs[c] = step;
        gmax[c] = nan ? __builtin_inff() : m;   // a group with a NaN is not for the plain form of codes4
    }
    __syncthreads();

    // The hash multiplies index ^ seed; a lane's first index is a multiple of 16, so the product splits into one for the
    // upper 28 bits and one for the four low bits, which is the same in all lanes.
    const uint32_t s32 = (uint32_t)seed ^ (uint32_t)(seed >> 32);
    uint32_t kc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) kc[i] = ((s32 ^ (uint32_t)i) & 15u) * 747796405u + 2891336453u;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int group = (wave + c * nw) * 4 + (lane >> 4);
        if (group >= ngroups) continue;
        const int row = (int)(group * inv_groups >> 16), e0 = (group - row * groups) * 256 + (lane & 15) * 16;
        const int64_t n = n0 + row;
        const float sc = fmaxf(u2f(row_max[row]) / 127.0f, 1e-8f), inv_sc = 1.0f / sc;   // :121
        if (e0 == 0) s_channel[n] = sc;
        const uint32_t bits = f_to_e4m3(gs[c] / sc);                                // :126-151
        if (!(lane & 1)) s_rel[n * (K / kG) + e0 / kG] = (uint8_t)bits;
        const float sr = e4m3_to_f(bits), inv_sr = 1.0f / fmaxf(sr, 1e-30f);
        const uint32_t x0 = ((uint32_t)(n * K + e0) ^ (s32 & ~15u)) * 747796405u;
        uint32_t cw[4] = {0u, 0u, 0u, 0u};
        if (__builtin_amdgcn_ballot_w64(!(gmax[c] * inv_sc < 127.f && sr >= 1.f && sr <= 4.f)) == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) cw[i] = codes4<true>(v[c] + 4 * i, inv_sc, sr, inv_sr, x0, kc + 4 * i);
        } else {
#pragma unroll 1
            for (int i = 0; i < 4; ++i) {
                // the loop stays rolled: this is the rare form
                float x[4];
                uint32_t k4[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    x[j] = i == 0 ? v[c][j] : i == 1 ? v[c][4 + j] : i == 2 ? v[c][8 + j] : v[c][12 + j];
                    k4[j] = i == 0 ? kc[j] : i == 1 ? kc[4 + j] : i == 2 ? kc[8 + j] : kc[12 + j];
                }
                const uint32_t o = codes4<false>(x, inv_sc, sr, inv_sr, x0, k4);
                cw[0] = i == 0 ? o : cw[0];
                cw[1] = i == 1 ? o : cw[1];
                cw[2] = i == 2 ? o : cw[2];
                cw[3] = i == 3 ? o : cw[3];
            }
        }
        // nibbles of codes 2j, 2j + 1 share a byte; the top bits of four codes share one (the product lines them up in
        // its upper byte, and nothing below carries into it)
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t nib = cw[i] & 0x0f0f0f0fu;
            lo[i] = nib | (nib >> 4);                   // bytes 0 and 2
            hi[i] = ((cw[i] >> 4) & 0x03030303u) * 0x01041040u;   // byte 3
        }
        uint8_t* lo_plane = packed + n * (int64_t)(K / 4 * 3);
        *reinterpret_cast<uint2*>(lo_plane + e0 / 2) =
            make_uint2(__builtin_amdgcn_perm(lo[1], lo[0], 0x06040200u), __builtin_amdgcn_perm(lo[3], lo[2], 0x06040200u));
        *reinterpret_cast<uint32_t*>(lo_plane + K / 2 + e0 / 4) =
            __builtin_amdgcn_perm(hi[1], hi[0], 0x0c0c0703u) | (__builtin_amdgcn_perm(hi[3], hi[2], 0x0c0c0703u) << 16);
    }
}

// Rows of a workgroup: one, or as many more as give the CUs clearly fewer waves to run: all of a workgroup's, however few lanes its
// last has, times the workgroups of the busiest CU.  us, one row and the rows chosen: 5376 x 5376 66.6 and 56.4 (three), 4096 x 1280
// 20.3 and 15.9 (four), 8192 x 256 19.4 and 10.9 (four), 4096 x 1536 19.1 and 16.5 (two); within 6 % the larger workgroups
// lose by their barriers (4096 x 7680 59.7 and, two rows in 15 waves, 64.3).  With up to three workgroups per CU a SIMD waits for its
// own waves: a workgroup's go to the four SIMDs from the first on, so that two workgroups of two waves meet on the same two SIMDs and
// one of four does not (448 x 2048 8.1 and 6.9, 453 x 5120 10.9 and 9.9; 1400 shapes: 19 more than 4 % slower than with fixed rows, with this 5).
int rows_per_group(int64_t N, int groups) {
    const uint32_t cus = (uint32_t)device_cu_count(), rows = (uint32_t)N;
    struct Choice { int r; uint32_t wgs; double waves; uint32_t on_simd; };   // wgs: of the busiest CU
    const auto choice = [&](int r) {
        const uint32_t wgs = ((rows + r - 1) / r + cus - 1) / cus;
        return Choice{r, wgs, (double)wgs * ((r * groups + 3) / 4), wgs * ((r * groups + 15) / 16)};
    };
    const int most = 64 / groups < kMaxRows ? 64 / groups : kMaxRows;
    Choice best = choice(1);
    for (int r = 2; r <= most; ++r) {
        const Choice c = choice(r);
        if (c.waves < 0.92 * best.waves) best = c;
    }
    for (int r = 2; r <= most && best.wgs <= 3; ++r) {
        const Choice c = choice(r);
        if (c.waves <= best.waves && c.on_simd < best.on_simd) best = c;
    }
    return best.r;
}

template <int C>
int launch_requant(const void* w, void* packed, void* s_rel, void* s_channel, int N, int K, uint64_t seed, int rpb, hipStream_t st) {
    const int groups = K / 256, chunks = (rpb * groups + 3) / 4, nw = (chunks + C - 1) / C;
    const int smem = nw * convrot::kLdsPerWave * (int)sizeof(float);
    static PerDeviceOnce once;
    if (smem > 64 * 1024)
        if (const int e = allow_dynamic_lds((const void*)w6_requant_kernel<C>, 16 * convrot::kLdsPerWave * (int)sizeof(float), once)) return e;
    hipLaunchKernelGGL(w6_requant_kernel<C>, dim3((unsigned)((N + rpb - 1) / rpb)), dim3(nw * 64), smem, st, (const uint16_t*)w,
                       (uint8_t*)packed, (uint8_t*)s_rel, (float*)s_channel, N, K, seed, groups, (65536u + groups - 1) / groups, rpb);
    KCHECK();
    return 0;
}

}  // namespace

// weight bf16 [N, K] -> packed [N, 3K/4], s_rel e4m3 [N, K/32], s_channel f32 [N].  Rounding is always stochastic, keyed by
// element index and seed, as in the reference's launcher (csrc/vendor/w6a8_requant.cu:242-251).
GPU_API int gpu_w6_requant(const void* weight, void* packed, void* s_rel, void* s_channel, int64_t N, int K, uint64_t seed,
                           void* stream) {
    if (K <= 0 || K % 256) return -1;
    if (K > 39680 || N > 0x7fffffff) return -2;
    if (N <= 0) return 0;
    // a chunk per wave up to 16 waves per row; longer rows give a wave two or three
    const int groups = K / 256, chunks = (groups + 3) / 4;
    hipStream_t st = (hipStream_t)stream;
    if (chunks > 32) return launch_requant<3>(weight, packed, s_rel, s_channel, (int)N, K, seed, 1, st);
    if (chunks > 16) return launch_requant<2>(weight, packed, s_rel, s_channel, (int)N, K, seed, 1, st);
    return launch_requant<1>(weight, packed, s_rel, s_channel, (int)N, K, seed, rows_per_group(N, groups), st);
}

// Test hook: rows of a workgroup of gpu_w6_requant.
GPU_API int gpu_internal_w6_requant_rows(int64_t N, int K) {
    if (N <= 0 || N > 0x7fffffff || K <= 0 || (K % 256) != 0 || K > 39680) return -1;
    return K > 16 * convrot::kChunk ? 1 : rows_per_group(N, K / 256);
}
