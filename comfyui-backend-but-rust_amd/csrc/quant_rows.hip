// Per-row absmax int8 quantization with the optional ConvRot group rotation, for gfx950 (wave64).
//
// Arithmetic follows the reference's quantizers exactly (csrc/kernels.cu:184-258 for bf16/f32 rows,
// csrc/sd.cu:578-598 for fp16 rows, csrc/common.cuh:99-126 for the staged radix-4 Hadamard butterflies): same
// float operation order, same rounding points.  The structure does not: a row is cut into chunks of 1024 values, one
// wave per chunk, each lane holding 16 consecutive values in registers.  Radix-4 stages with strides 1 and 4 run inside
// a lane; for the wider strides the chunk makes one trip through a wave-private LDS tile so that those butterflies are
// again lane-local, then returns to row order for the 16-byte code stores.
#include "common.hpp"
#include "convrot.hpp"
#include "rowmath.hpp"
#include "act_tables.hpp"

namespace {
using namespace convrot;

enum { MODE_BF16 = 0, MODE_F32 = 1, MODE_SD_F16 = 2, MODE_ROT_F32 = 3 };

struct QuantArgs {
    const void* x;
    int64_t x_stride;  // elements between rows
    int8_t* q;         // [M, K]
    float* scales;     // [M]
    float* out_f;      // MODE_ROT_F32: rotated rows [M, K]
    int M, K;
    int wpr;           // waves per row
    int rpb;           // rows per block
    uint64_t seed;     // nonzero: stochastic rounding keyed by element index + seed (gpu_convrot_requant)
    // row prologue (csrc/kernels.cu:21-37), PRO kernels only
    int pro;
    const void* g;          // GATE: logits [M, g_stride]
    int64_t g_stride;
    int64_t up_offset;      // SWIGLU, SITU: column of the second half inside the x row
    const float* norm_w;    // RMS, LAYERNORM, LN_AFFINE
    const float* norm_b;    // LN_AFFINE
    float eps;
    const void* mod_scale;  // [K] in the row dtype
    const void* mod_shift;
    int d, dp;              // PRO_SD_UNPAD: heads of d values, each stored dp wide
    int per;                // PRO_SD_GN: channels per group; g holds the (mean, rstd) pairs, g_stride the pixels per image
    ActTables tab;          // activation tables for 16-bit rows (null members: evaluate per element)
};

// Sources of the SD UNet's fused quantizers (csrc/sd.cu:611-663), fp16 rows only.  Its LayerNorm source is PRO_LN_AFFINE.
enum { PRO_SD_GEGLU = 101, PRO_SD_UNPAD = 102, PRO_SD_GN = 103 };

// csrc/kernels.cu:1355-1359
constexpr uint32_t kPcgMul = 747796405u, kPcgAdd = 2891336453u;
// The hash's upper 24 bits in place, as a float: 2^32 times the noise in [0, 1).  In place they take one three-operand bit operation
// where a shift down to whole numbers takes a second instruction, and the power of two rides in the addition that follows
// (12288 x 3072 bf16 39.7 -> 37.4 us).
__device__ __forceinline__ float pcg_noise_state(uint32_t state) {   // state: x * kPcgMul + kPcgAdd
    const uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
    return (float)(((word >> 22u) ^ word) & 0xffffff00u);
}
template <int MODE> __device__ __forceinline__ void load16(const void* x, int64_t off, float* v) {
    if (MODE == MODE_BF16) {
        const uint4* p = reinterpret_cast<const uint4*>((const uint16_t*)x + off);
        const uint4 a = p[0], b = p[1];
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[2 * i] = u2f(w[i] << 16);
            v[2 * i + 1] = u2f(w[i] & 0xffff0000u);
        }
    } else if (MODE == MODE_SD_F16) {
        const uint4* p = reinterpret_cast<const uint4*>((const uint16_t*)x + off);
        const uint4 a = p[0], b = p[1];
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[2 * i] = f16_to_f((uint16_t)(w[i] & 0xffffu));
            v[2 * i + 1] = f16_to_f((uint16_t)(w[i] >> 16));
        }
    } else {
        const float4* p = reinterpret_cast<const float4*>((const float*)x + off);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 f = p[i];
            v[4 * i] = f.x; v[4 * i + 1] = f.y; v[4 * i + 2] = f.z; v[4 * i + 3] = f.w;
        }
    }
}

// Sum over the waves of one row in fp64, rounded to fp32 once (every wave of the block calls it).
__device__ __forceinline__ float row_sum_f64(double v, double* red, int wave, int lane, int wpr, int rloc) {
    v = wave_sum_f64(v);
    if (wpr == 1) return (float)v;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < wpr; ++i) t += red[rloc * wpr + i];
    return (float)t;
}

// The rotation of a row's chunks and the maximum of their magnitudes over the lane's values.  `exact`: the values are bf16
// or f16 numbers (rotate_chunk's condition for scaling once; bf16 ones are also checked against the overflow limit).
template <int MODE, int G, int C>
__device__ __forceinline__ float rotate_and_max(const QuantArgs& p, float (&v)[C][16], int64_t m, bool row_ok, int wr, int lane, float* wl, bool exact) {
    float amax = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int e0 = (wr + c * p.wpr) * kChunk + lane * 16;
        const bool act = row_ok && e0 < p.K;
        if constexpr (G != 0) {
            // scaled once where that is exact (rotate_chunk): f16 rows always, bf16 values below the overflow limit
            bool once = G != 128 && MODE == MODE_SD_F16 && exact;
            if (G != 128 && MODE == MODE_BF16 && exact) {
                float big = 0.f;
#pragma unroll
                for (int i = 0; i < 16; i += 2) big = fmaxf(fmaxf(big, fabsf(v[c][i])), fabsf(v[c][i + 1]));
                once = __builtin_amdgcn_ballot_w64(big >= kOnceLimit) == 0;
            }
            if (once) rotate_chunk<G, true>(v[c], wl, lane);
            else rotate_chunk<G>(v[c], wl, lane);
        }
        if (MODE == MODE_ROT_F32) {
            if (act) {
                float4* o = reinterpret_cast<float4*>(p.out_f + m * (int64_t)p.K + e0);
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = make_float4(v[c][4 * i], v[c][4 * i + 1], v[c][4 * i + 2], v[c][4 * i + 3]);
            }
        } else if (MODE == MODE_SD_F16) {
            // the maximum is taken over the half-rounded row (csrc/sd.cu:587), which is also what is divided below
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                unpack_f16x2(pack_f16x2(v[c][i], v[c][i + 1]), v[c][i], v[c][i + 1]);
                amax = fmaxf(fmaxf(amax, fabsf(v[c][i])), fabsf(v[c][i + 1]));
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; i += 2) amax = fmaxf(fmaxf(amax, fabsf(v[c][i])), fabsf(v[c][i + 1]));
        }
    }
    return amax;
}

// Scale and codes of a row whose maximum is `amax`; a lane's values start at column first + c * step of it.
template <int MODE, int C, bool SR>
__device__ __forceinline__ void store_codes(const QuantArgs& p, float (&v)[C][16], int64_t m, bool row_ok, int first, int step, float amax) {
    float scale, st, rinv = 0.f;
    bool by_rcp = true;   // f16 rows: st is a finite half
    if (MODE == MODE_SD_F16) {
        scale = fmaxf(amax, 1e-30f) / 127.f;                       // csrc/sd.cu:589
        const float sh = rnd_dt<DT_F16>(scale);
        st = sh > 0.f ? sh : scale;                                // :593
        by_rcp = __builtin_amdgcn_ballot_w64(!(sh > 0.f && sh < __builtin_inff())) == 0;
        rinv = __builtin_amdgcn_rcpf(st);
    } else if (MODE == MODE_BF16) {
        scale = fmaxf(fminf(amax, 3.38953139e38f) * (1.f / 127.f), 1.0e-30f);  // csrc/kernels.cu:241
        st = rnd_dt<DT_BF16>(scale);
        rinv = __builtin_amdgcn_rcpf(st);
    } else {
        scale = fmaxf(fminf(amax, 3.402823466e+38f) * (1.f / 127.f), 1.0e-30f);
        st = scale;
    }
    if (row_ok && first == 0) p.scales[m] = scale;

    // Stochastic rounding: the hash of element index + seed, its halves folded, starts with a product.  Where a row's keys stay
    // below 2^32 the fold changes nothing and a lane's 16 products differ by constants.  With that, the fp32 addition above
    // (fp64 and 64-bit integers before) and the clamp in the pack conversion 12288 x 3072 bf16 took 42 us instead of 53 (45
    // where the keys pass 2^32), now 37, bound by vector instructions: the same rows rounded to nearest take 26.
    const uint64_t key0 = (uint64_t)(m * (int64_t)p.K) + p.seed;
    const auto store = [&](auto fast_tag) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int e0 = first + c * step;
            if (!(row_ok && e0 < p.K)) continue;
            uint32_t w[4];
            const uint32_t state0 = ((uint32_t)key0 + (uint32_t)e0) * kPcgMul + kPcgAdd;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (MODE == MODE_SD_F16) {
                    // t = half(x / st).  Both operands carry 11 significant bits: their quotient never equals a midpoint of two
                    // halves and is 2^-23 (relative) away at least, more than the error left after one correction of x * rcp.
                    // clamp(rint(t), -128, 127): a half around 1536 has a step of 1, so t + 1536 is 0x6600 + rint(t) and its
                    // low byte the code; the maximum turns a NaN into the -128 that fminf(127, fmaxf(-128, NaN)) gives.
                    float qt[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float x = v[c][4 * i + j];
                        if constexpr (decltype(fast_tag)::value) {
                            const float q0 = x * rinv;
                            qt[j] = __builtin_fmaf(__builtin_fmaf(-q0, st, x), rinv, q0);
                        } else {
                            qt[j] = x / st;
                        }
                    }
                    uint32_t h[2];
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        f16x2 t = __builtin_bit_cast(f16x2, pack_f16x2(qt[2 * j], qt[2 * j + 1]));
                        t = __builtin_elementwise_min(__builtin_elementwise_max(t, f16x2{-128, -128}), f16x2{127, 127});
                        h[j] = __builtin_bit_cast(uint32_t, t + f16x2{1536, 1536});
                    }
                    w[i] = __builtin_amdgcn_perm(h[1], h[0], 0x06040200u);
                    continue;
                }
                uint32_t acc = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float x = v[c][4 * i + j];
                    float t;
                    if (MODE == MODE_BF16) {
                        // Both operands carry 8 significant bits, so their exact quotient is never closer than 2^-17
                        // (relative) to a bf16 rounding boundary: a 1-ulp reciprocal times the numerator rounds to the
                        // same bf16 value as the IEEE quotient does.
                        t = rnd_dt<DT_BF16>(rnd_dt<DT_BF16>(x) * rinv);
                    } else {
                        t = x / st;
                    }
                    if (SR && (MODE == MODE_BF16 || MODE == MODE_F32)) {   // csrc/kernels.cu:1385-1388
                        uint32_t state;
                        if constexpr (decltype(fast_tag)::value) {
                            state = state0 + (uint32_t)(4 * i + j) * kPcgMul;
                        } else {
                            const uint64_t key = key0 + e0 + 4 * i + j;
                            state = ((uint32_t)key ^ (uint32_t)(key >> 32)) * kPcgMul + kPcgAdd;
                        }
                        // bf16: t plus the rounded noise, rounded once to bf16 as __hadd's instruction does (csrc/kernels.cu:1341-1343).
                        // The fp32 sum rounds first and changes nothing: it is inexact only where the smaller operand is below
                        // 2^-15 of the larger, which leaves the sum 2^-10 (relative) or more away from every midpoint of two bf16 values.
                        const float noise = pcg_noise_state(state);
                        const float r = floorf(MODE == MODE_F32 ? __builtin_fmaf(noise, 0x1.0p-32f, t)
                                                                : rnd_dt<DT_BF16>(__builtin_fmaf(rnd_dt<DT_BF16>(noise), 0x1.0p-32f, t)));
                        acc = __builtin_amdgcn_cvt_pk_u8_f32(r + 128.f, j, acc);   // the clamp as below; r is a whole number
                    } else if (MODE == MODE_F32) {
                        const int qi = (int)fminf(127.f, fmaxf(-128.f, nearbyintf(t)));
                        acc |= ((uint32_t)qi & 0xffu) << (8 * j);
                    } else {
                        // clamp(rint(t), -128, 127) + 128 as one instruction: t is a 16-bit float, so t + 128 is exact
                        // wherever t has a bit at 2^-16 or above set, and below that both t and t + 128 round to the
                        // same integer; v_cvt_pk_u8_f32 rounds to nearest even, saturates to 0..255 (NaN to 0, which is
                        // the -128 that fminf(127, fmaxf(-128, NaN)) gives) and drops the byte into place.
                        acc = __builtin_amdgcn_cvt_pk_u8_f32(t + 128.f, j, acc);
                    }
                }
                w[i] = (SR || MODE != MODE_F32) ? acc ^ 0x80808080u : acc;
            }
            *reinterpret_cast<uint4*>(p.q + m * (int64_t)p.K + e0) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    };
    if constexpr (MODE == MODE_SD_F16) {
        if (by_rcp) store(std::true_type{});
        else store(std::false_type{});
    } else if constexpr (SR) {
        if (key0 < ((uint64_t)1 << 32) - (uint64_t)p.K) store(std::true_type{});
        else store(std::false_type{});
    } else {
        store(std::true_type{});
    }
}

// CLS: the class of the row prologue (csrc/kernels.cu:88-182), which runs on the values as they are loaded, with the
// reference's rounding points; p.pro selects the prologue within its class at run time.  Row sums are fp64, rounded once;
// the activation functions are correctly rounded.  The classes keep what is cheap in registers apart from what calls
// the fp64 routines: in one kernel for all, SwiGLU and the norms had the 123 registers of those calls, four waves per SIMD
// (GEGLU 8192 x 2560 53.3 us, LayerNorm 8192 x 640 14.9 us; by class 48.8 and 13.3).
// SR: stochastic rounding keyed by element index + p.seed (gpu_convrot_requant); a kernel variant of its own, so that the
// plain quantizer carries neither the hash nor a branch per element.
enum {
    CLS_PLAIN,
    CLS_NORM,    // RMS, LAYERNORM, ADALN, LN_MOD, LN_AFFINE
    CLS_GATED,   // bf16 rows: GATE, SWIGLU, SILU; f16 rows: GEGLU through its table
    CLS_REST     // everything that may evaluate an fp64 routine, and the SD gathers
};
template <int MODE, int G, int C, int CLS, bool SR = false>
__global__ void __launch_bounds__(512, C > 3 ? 2 : 4) quant_rows_kernel(QuantArgs p) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ float red[8];
    __shared__ double dred[8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rloc = wave / p.wpr, wr = wave - rloc * p.wpr;
    const int64_t m = (int64_t)blockIdx.x * p.rpb + rloc;
    const bool row_ok = m < p.M;
    float* wl = lds + wave * kLdsPerWave;
    // the row dtype T of the prologue's roundings, and how a T vector is loaded
    constexpr int TD = MODE == MODE_BF16 ? DT_BF16 : MODE == MODE_SD_F16 ? DT_F16 : DT_F32;
    constexpr int TMODE = MODE == MODE_BF16 ? MODE_BF16 : MODE == MODE_SD_F16 ? MODE_SD_F16 : MODE_F32;
    auto R = [](float x) { return rnd_dt<TD>(x); };
    // dst[i] = rnd(f(src[i])) for the 16 values of a lane: through a table of all 65536 bf16 inputs when it is there (one
    // test for the 16 lookups, which then issue as a batch), else evaluated
    auto map16 = [](const uint16_t* tab, const float* src, float* dst, auto f) {
        if (MODE == MODE_BF16 && tab) {
#pragma unroll
            for (int i = 0; i < 16; ++i) dst[i] = bf16_to_f(tab[f2u(src[i]) >> 16]);
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) dst[i] = rnd_dt<TD>(f(src[i]));
        }
    };

    float v[C][16];
    constexpr bool NORM = CLS == CLS_NORM, GATED = CLS == CLS_GATED, REST = CLS == CLS_REST;
    const int pro = CLS == CLS_PLAIN ? PRO_PLAIN : p.pro;
    const bool ln = NORM && (pro == PRO_LAYERNORM || pro == PRO_LN_MOD || pro == PRO_LN_AFFINE);
    double part = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int e0 = (wr + c * p.wpr) * kChunk + lane * 16;
        const bool act = row_ok && e0 < p.K;
        if (REST && MODE == MODE_SD_F16 && pro == PRO_SD_UNPAD) {                     // csrc/sd.cu:650-652
            const uint16_t* r = (const uint16_t*)p.x + m * p.x_stride;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int k = e0 + i;
                v[c][i] = act ? f16_to_f(r[(k / p.d) * p.dp + k % p.d]) : 0.f;
            }
        } else if (act) {
            load16<MODE>(p.x, m * p.x_stride + e0, v[c]);
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) v[c][i] = 0.f;
        }
        if (NORM && act) {
            if (ln) {
#pragma unroll
                for (int i = 0; i < 16; ++i) part += (double)v[c][i];
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) part += (double)v[c][i] * (double)v[c][i];
            }
        }
        if (GATED && act) {
            float u[16];
            if (MODE == MODE_SD_F16) {                                               // GEGLU, csrc/sd.cu:642-649, row = [value | gate]
                load16<TMODE>(p.x, m * p.x_stride + p.up_offset + e0, u);
#pragma unroll
                for (int i = 0; i < 16; ++i) u[i] = f16_to_f(p.tab.gelu_f16[f_to_f16(u[i])]);
#pragma unroll
                for (int i = 0; i < 16; ++i) v[c][i] = R(v[c][i] * u[i]);
            } else if (pro == PRO_GATE) {                                            // csrc/kernels.cu:95-100
                load16<TMODE>(p.g, m * p.g_stride + e0, u);
#pragma unroll
                for (int i = 0; i < 16; ++i) v[c][i] = R(v[c][i] * R(sigmoid_of_bf16(u[i])));
            } else {                                                                 // :101-106
                const bool two = pro == PRO_SWIGLU;
                if (two) load16<TMODE>(p.x, m * p.x_stride + p.up_offset + e0, u);
#pragma unroll
                for (int i = 0; i < 16; ++i) v[c][i] = R(silu_of_bf16(v[c][i]));
                if (two) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[c][i] = R(v[c][i] * u[i]);
                }
            }
        }
        if (REST && act) {
            if (MODE == MODE_SD_F16) {
                if (pro == PRO_SD_GEGLU) {
                    float gg[16];
                    load16<TMODE>(p.x, m * p.x_stride + p.up_offset + e0, gg);
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[c][i] = R(v[c][i] * R(gelu_f(gg[i])));
                } else if (pro == PRO_SD_GN) {                                       // csrc/sd.cu:653-662
                    const float2* stats = (const float2*)p.g + (m / p.g_stride) * (int64_t)(p.K / p.per) * 2;
                    float nw[16], nb[16];
                    load16<MODE_F32>(p.norm_w, e0, nw);
                    load16<MODE_F32>(p.norm_b, e0, nb);
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const float2 st = stats[((e0 + i) / p.per) * 2];
                        v[c][i] = R(__builtin_fmaf((v[c][i] - st.x) * st.y, nw[i], nb[i]));
                    }
                }
            } else if (pro == PRO_GATE) {                                            // f32 rows from here: csrc/kernels.cu:95-112
                float gg[16];
                load16<TMODE>(p.g, m * p.g_stride + e0, gg);
#pragma unroll
                for (int i = 0; i < 16; ++i) v[c][i] = R(v[c][i] * R(sigmoid_f(gg[i])));
            } else if (pro == PRO_SWIGLU || pro == PRO_SITU || pro == PRO_SITU_FAST) {
                float u[16];
                load16<TMODE>(p.x, m * p.x_stride + p.up_offset + e0, u);
                if (pro == PRO_SWIGLU) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[c][i] = R(R(silu_f(v[c][i])) * u[i]);
                } else if (MODE == MODE_BF16 && p.tab.situ_gate_bf16) {
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        v[c][i] = p.tab.situ_gate_bf16[f2u(u[i]) >> 16] * p.tab.situ_hidden_bf16[f2u(v[c][i]) >> 16];
                } else {   // one float expression, not rounded to T; the lossy id runs the same accurate form
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[c][i] = situ_f(v[c][i], u[i]);
                }
            } else if (pro == PRO_SILU) {
#pragma unroll
                for (int i = 0; i < 16; ++i) v[c][i] = R(silu_f(v[c][i]));
            } else if (pro == PRO_GELU) {
                map16(p.tab.gelu_bf16, v[c], v[c], [](float x) { return gelu_f(x); });
            } else if (pro == PRO_GELU_TANH) {
                map16(p.tab.gelu_tanh_bf16, v[c], v[c], [](float x) { return gelu_tanh_f(x); });
            }
        }
    }
    if constexpr (NORM) {
        if (ln) {        // :133-145
            const float mean = row_sum_f64(part, dred, wave, lane, p.wpr, rloc) / (float)p.K;
            part = 0.0;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int e0 = (wr + c * p.wpr) * kChunk + lane * 16;
                if (!(row_ok && e0 < p.K)) continue;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    v[c][i] -= mean;
                    part += (double)v[c][i] * (double)v[c][i];
                }
            }
        }
        const float ss = row_sum_f64(part, dred, wave, lane, p.wpr, rloc);
        const float rstd = rsqrt_cr(ss / (float)p.K + p.eps);                        // :148
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int e0 = (wr + c * p.wpr) * kChunk + lane * 16;
            if (!(row_ok && e0 < p.K)) continue;
            const bool mod = p.mod_scale != nullptr;
            // the form is chosen once per 16 values, and each loads only what it takes
            float a[16], b[16];
            const auto load_mod = [&]() {
                if (mod) {
                    load16<TMODE>(p.mod_scale, e0, a);
                    load16<TMODE>(p.mod_shift, e0, b);
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i) a[i] = b[i] = 0.f;
                }
            };
            if (pro == PRO_ADALN) {                                                  // :163-166, one rounding
                load_mod();
#pragma unroll
                for (int i = 0; i < 16; ++i) v[c][i] = R(__builtin_fmaf(v[c][i] * rstd, 1.f + a[i], b[i]));
            } else if (pro == PRO_LN_MOD) {                                          // ln_finish, :40-46
                load_mod();
#pragma unroll
                for (int i = 0; i < 16; ++i) v[c][i] = R(__builtin_fmaf(R(v[c][i] * rstd), R(1.f + a[i]), b[i]));
            } else if (pro == PRO_LN_AFFINE) {
                load16<MODE_F32>(p.norm_w, e0, a);
                load16<MODE_F32>(p.norm_b, e0, b);
#pragma unroll
                for (int i = 0; i < 16; ++i) v[c][i] = R(__builtin_fmaf(v[c][i] * rstd, a[i], b[i]));
            } else {                                                                 // RMS, LAYERNORM: :171-179
                if (p.norm_w) {
                    load16<MODE_F32>(p.norm_w, e0, a);
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[c][i] = R(v[c][i] * rstd * a[i]);
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[c][i] = R(v[c][i] * rstd);
                }
                if (mod) {
                    load_mod();
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[c][i] = R(R(R(1.f + a[i]) * v[c][i]) + b[i]);
                }
            }
        }
    }
    const bool exact = !REST || (pro != PRO_SITU && pro != PRO_SITU_FAST);   // those hand on unrounded fp32 values
    float amax = rotate_and_max<MODE, G, C>(p, v, m, row_ok, wr, lane, wl, exact);
    if constexpr (MODE != MODE_ROT_F32) {
        amax = wave_max_f32(amax);
        if (p.wpr > 1) {  // uniform over the block
            if (lane == 0) red[wave] = amax;
            __syncthreads();
            amax = 0.f;
            for (int i = 0; i < p.wpr; ++i) amax = fmaxf(amax, red[rloc * p.wpr + i]);
        }
        store_codes<MODE, C, SR>(p, v, m, row_ok, wr * kChunk + lane * 16, p.wpr * kChunk, amax);
    }
}

// GEGLU of f16 rows ahead of the quantizer (csrc/sd.cu:642-649, row = [value | gate]), one workgroup of 16 waves per CU that
// walks the rows with the table of gelu in its LDS.  Read per lane from the 128 KB table in global memory the activation costs
// the CU's address path a cycle per lane (8192 x 2560: 48.8 us on a GEMM's output); from the LDS the 64 lanes of a read
// spread over the 64 banks.  71 KB of magnitudes serve both signs (act_tables.hpp).
// C == 1: a wave per chunk, the next row's loads issued before this row's arithmetic, one barrier per row (33 us).  C == 2, 3:
// a wave per row, no barrier, the waves' loads and arithmetic drift apart by themselves (28 us), for rows of that many
// chunks where the rows divide well over the waves.  About 1500 cycles of vector instructions per chunk make 16 us of
// that; the traffic alone is 20.
// Two gates (packed f16) and their table entries -> rnd(gelu) of both, packed: max(x, 0) + g, the first as half of x + |x| so
// that a NaN and -inf (gelu: NaN) stay what they are.
__device__ __forceinline__ uint32_t gelu_index_x2(uint32_t gw) {   // the entries' indices, packed
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, gw & 0x7fff7fffu), u16x2{kGeluEnd, kGeluEnd}));
}
__device__ __forceinline__ uint32_t gelu_f16x2(uint32_t gw, float t0, float t1) {
    float g0, g1;
    unpack_f16x2(gw, g0, g1);
    return pack_f16x2(__builtin_fmaf(g0 + fabsf(g0), 0.5f, t0), __builtin_fmaf(g1 + fabsf(g1), 0.5f, t1));
}

constexpr int kGegluWaves = 16;
constexpr int kGegluTable = (kGeluEnd + 4) / 4 * 4;   // floats
template <int G, int C>
__global__ void __launch_bounds__(kGegluWaves * 64) geglu_rows_kernel(QuantArgs p) {
    constexpr bool PF = C == 1;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ float red[2][kGegluWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rloc = wave / p.wpr, wr = wave - rloc * p.wpr;
    const int row0 = (rloc < p.rpb ? rloc : 0) * p.wpr;   // the row's first wave; waves past the last row read along
    float* wl = lds + kGegluTable + wave * kLdsPerWave;
    for (int i = threadIdx.x * 4; i <= kGeluEnd; i += kGegluWaves * 64 * 4)   // the table is padded to whole vectors
        *reinterpret_cast<float4*>(lds + i) = *reinterpret_cast<const float4*>(p.tab.gelu_f16_g + i);
    uint4 x[C][2], g[C][2];
    const auto load = [&](int64_t m) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int e0 = (wr + c * p.wpr) * kChunk + lane * 16;
            if (rloc < p.rpb && m < p.M && e0 < p.K) {
                const uint4* s = reinterpret_cast<const uint4*>((const uint16_t*)p.x + m * p.x_stride + e0);
                const uint4* t = reinterpret_cast<const uint4*>((const uint16_t*)p.x + m * p.x_stride + p.up_offset + e0);
                x[c][0] = s[0]; x[c][1] = s[1];
                g[c][0] = t[0]; g[c][1] = t[1];
            } else {
                x[c][0] = x[c][1] = g[c][0] = g[c][1] = make_uint4(0u, 0u, 0u, 0u);
            }
        }
    };
    int64_t m = (int64_t)blockIdx.x * p.rpb + rloc;
    if (PF) load(m);
    __syncthreads();
    const int64_t step = (int64_t)gridDim.x * p.rpb, first = m;
    for (int it = 0; (int64_t)blockIdx.x * p.rpb + it * step < p.M; ++it) {   // the same count in every wave
        m = first + it * step;
        const bool row_ok = rloc < p.rpb && m < p.M;
        if (!PF) load(m);
        float v[C][16];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const uint32_t gw[8] = {g[c][0].x, g[c][0].y, g[c][0].z, g[c][0].w, g[c][1].x, g[c][1].y, g[c][1].z, g[c][1].w};
            const uint32_t xw[8] = {x[c][0].x, x[c][0].y, x[c][0].z, x[c][0].w, x[c][1].x, x[c][1].y, x[c][1].z, x[c][1].w};
            float t[16];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t a = gelu_index_x2(gw[i]);
                t[2 * i] = lds[a & 0xffffu];
                t[2 * i + 1] = lds[a >> 16];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t act = gelu_f16x2(gw[i], t[2 * i], t[2 * i + 1]);
                // the product of two halves is exact in fp32, so the packed f16 product is its one rounding
                const f16x2 pr = __builtin_bit_cast(f16x2, xw[i]) * __builtin_bit_cast(f16x2, act);
                v[c][2 * i] = (float)pr[0];
                v[c][2 * i + 1] = (float)pr[1];
            }
        }
        if (PF) load(m + step);
        float amax = wave_max_f32(rotate_and_max<MODE_SD_F16, G, C>(p, v, m, row_ok, wr, lane, wl, true));
        if (p.wpr > 1) {   // uniform over the workgroup; the slots alternate, so one barrier per row is enough
            float* r = red[it & 1];
            if (lane == 0) r[wave] = amax;
            __syncthreads();
            amax = 0.f;
            for (int i = 0; i < p.wpr; ++i) amax = fmaxf(amax, r[row0 + i]);
        }
        store_codes<MODE_SD_F16, C, false>(p, v, m, row_ok, wr * kChunk + lane * 16, p.wpr * kChunk, amax);
    }
}

template <int G, int C>
int launch_geglu(QuantArgs a, int wpr, int cus, hipStream_t st) {
    constexpr int lds = (kGegluTable + (G ? kGegluWaves * kLdsPerWave : 0)) * (int)sizeof(float);
    static PerDeviceOnce once;
    if (const int e = allow_dynamic_lds(reinterpret_cast<const void*>(geglu_rows_kernel<G, C>), lds, once)) return e;
    a.wpr = wpr;
    a.rpb = kGegluWaves / wpr;
    const int groups = (a.M + a.rpb - 1) / a.rpb;
    hipLaunchKernelGGL((geglu_rows_kernel<G, C>), dim3(groups < cus ? groups : cus), dim3(kGegluWaves * 64), lds, st, a);
    KCHECK();
    return 0;
}

// GEGLU with the table in LDS: chunks per wave and waves per row.  Filling the table takes a workgroup 2.5 us: it pays from about
// 5000 chunks on (1024 x 5120: 13.0 us either way; 2048 x 5120 18.4 against 21.4, 512 x 2560 7.4 against 5.9).  A round of the
// wave-per-row form takes about 3.3 us per chunk of its rows and 4 us of the launch's start more than the other form, whose rounds
// take 4.1 us.
struct GegluForm { int chunks, wpr; };   // no chunks: the table stays in global memory
GegluForm geglu_form(int M, int K, int cus) {
    const int nchunks = (K + kChunk - 1) / kChunk;
    if ((int64_t)M * nchunks < 5120) return {0, 0};
    if (nchunks > kGegluWaves) return {2, (nchunks + 1) / 2};
    const auto rounds = [&](int rpb) { return (M + (int64_t)rpb * cus - 1) / ((int64_t)rpb * cus); };
    if (nchunks <= 3 && 3.3 * nchunks * rounds(kGegluWaves) + 4. < 4.1 * rounds(kGegluWaves / nchunks)) return {nchunks, 1};
    return {1, nchunks};
}

// LayerNorm of f16 rows ahead of the quantizer (csrc/sd.cu:633-640) for widths that leave a wave per row many idle lanes: a workgroup takes as
// many rows as fill its waves and cuts them into chunks as if they were one.  A rotation group of 64 is four lanes of one row;
// their sums and maxima meet in LDS, and every lane adds those of its row.  Bound by vector instructions (about 700 per wave: the fp64
// sums, the rotation, the divisions), of which idle lanes take as many as busy ones.
// us, a wave per row and this: 8192 x 640 11.7 and 9.5, 8192 x 320 10.9 and 6.3, 16384 x 768 20.1 and 17.0, 2048 x 512 4.8 and 4.35, 256 x 320
// 4.0 and 3.7.  Beyond 768 columns the longer sums and barriers cost what the lanes give (8192 x 832 12.3 and 12.7, 8192 x 1280 18.5 and
// 20.3), as more than four waves do (8192 x 448 in seven 7.6, in four 7.4; 1024 x 448 4.9 and 4.2); below 1024 rows only
// whole rows of one wave pay (256 x 448, nine rows on four waves, 4.1; a wave per row 4.0).
constexpr int kLnWaves = 4;
struct LnForm { int rows, waves; };   // of a workgroup; no rows: a wave per chunk of a row
LnForm ln_form(int M, int K) {
    LnForm best{0, 0};
    if (K % 64 != 0 || K > 768) return best;
    double busy = 1.2 * K / kChunk;   // share of the lanes with values
    for (int waves = 1; waves <= (M < 1024 ? 1 : kLnWaves); ++waves) {
        const int rows = waves * kChunk / K < 16 ? waves * kChunk / K : 16;
        const double b = (double)rows * K / (waves * kChunk);
        if (b > (best.rows ? 1.06 : 1.) * busy) {
            best = {rows, waves};
            busy = b;
        }
    }
    return best;
}
template <int G, int NQ>   // NQ: a quarter of a row's groups at least
__global__ void __launch_bounds__(kLnWaves * 64) ln_rows_f16_kernel(QuantArgs p, int gpr, uint32_t inv_gpr) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ double sums[2][kLnWaves * 16];
    __shared__ float maxima[kLnWaves * 16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int group = wave * 16 + (lane >> 2);   // of 64 columns; row = group / gpr
    const int rloc = (int)(group * inv_gpr >> 16), e0 = (int)threadIdx.x * 16 - rloc * p.K;
    const int64_t m = (int64_t)blockIdx.x * p.rpb + rloc;
    const bool act = rloc < p.rpb && m < p.M;
    int at[NQ];   // a group past the row's (or of no row) is read from its first, and not counted
#pragma unroll
    for (int i = 0; i < NQ; ++i) at[i] = act ? rloc * gpr + (i * 4 + (lane & 3) < gpr ? i * 4 + (lane & 3) : 0) : 0;
    const auto row_sum = [&](double part, double* meet) {
        const auto mv = [](double x, auto ctrl) {
            const int64_t b = __builtin_bit_cast(int64_t, x);
            constexpr int C = decltype(ctrl)::value;
            return __builtin_bit_cast(double, ((int64_t)dpp_int<C>((int)(b >> 32)) << 32) | (uint32_t)dpp_int<C>((int)b));
        };
        const auto quad = [&](double x) {
            x += mv(x, std::integral_constant<int, 0xB1>{});
            return x + mv(x, std::integral_constant<int, 0x4E>{});
        };
        part = quad(part);
        if ((lane & 3) == 0) meet[group] = part;
        __syncthreads();
        double t = 0.0;   // every fourth of the row's, the other three from the neighbours
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const double x = meet[at[i]];
            t += i * 4 + (lane & 3) < gpr ? x : 0.0;
        }
        return (float)quad(t);
    };
    float v[1][16], a[16], b[16];
    if (act) {
        load16<MODE_SD_F16>(p.x, m * p.x_stride + e0, v[0]);
        load16<MODE_F32>(p.norm_w, e0, a);
        load16<MODE_F32>(p.norm_b, e0, b);
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[0][i] = a[i] = b[i] = 0.f;
    }
    double part = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) part += (double)v[0][i];
    const float mean = row_sum(part, sums[0]) / (float)p.K;
    part = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        v[0][i] -= mean;
        part += (double)v[0][i] * (double)v[0][i];
    }
    const float rstd = rsqrt_cr(row_sum(part, sums[1]) / (float)p.K + p.eps);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[0][i] = act ? rnd_dt<DT_F16>(__builtin_fmaf(v[0][i] * rstd, a[i], b[i])) : 0.f;
    float amax = rotate_and_max<MODE_SD_F16, G, 1>(p, v, m, act, 0, lane, lds + wave * kLdsPerWave, true);
    const auto quad_max = [](float x) {
        x = fmaxf(x, __builtin_bit_cast(float, dpp_int<0xB1>(__builtin_bit_cast(int, x))));
        return fmaxf(x, __builtin_bit_cast(float, dpp_int<0x4E>(__builtin_bit_cast(int, x))));
    };
    amax = quad_max(amax);
    if ((lane & 3) == 0) maxima[group] = amax;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NQ; ++i) amax = fmaxf(amax, maxima[at[i]]);
    amax = quad_max(amax);
    store_codes<MODE_SD_F16, 1, false>(p, v, m, act, e0, 0, amax);
}

template <auto KERN>
int launch_kernel(const QuantArgs& a, int nw, int lds_per_wave, hipStream_t st) {
    hipLaunchKernelGGL(KERN, dim3((a.M + a.rpb - 1) / a.rpb), dim3(nw * 64), nw * lds_per_wave, st, a);   // 8 waves: 35 KB
    KCHECK();
    return 0;
}

template <int MODE, int G, int C>
int launch(const QuantArgs& a, int nw, hipStream_t st) {
    constexpr int lds = G ? kLdsPerWave * (int)sizeof(float) : 0;
    constexpr bool CAN_SR = (MODE == MODE_BF16 || MODE == MODE_F32) && G == 256;
    if (a.pro == PRO_PLAIN) {
        if (CAN_SR && a.seed != 0) return launch_kernel<quant_rows_kernel<MODE, G, C, CLS_PLAIN, CAN_SR>>(a, nw, lds, st);
        return launch_kernel<quant_rows_kernel<MODE, G, C, CLS_PLAIN>>(a, nw, lds, st);
    }
    if constexpr (MODE == MODE_SD_F16) {
        if (const LnForm f = ln_form(a.M, a.K); a.pro == PRO_LN_AFFINE && f.rows) {
            QuantArgs r = a;
            r.rpb = f.rows;
            const int gpr = a.K / 64;
            const auto kern = gpr <= 8 ? ln_rows_f16_kernel<G, 2> : ln_rows_f16_kernel<G, 3>;
            hipLaunchKernelGGL(kern, dim3((a.M + f.rows - 1) / f.rows), dim3(f.waves * 64), f.waves * lds, st, r, gpr, (65536u + gpr - 1) / gpr);
            KCHECK();
            return 0;
        }
    }
    if (a.pro == PRO_RMS || a.pro == PRO_LAYERNORM || a.pro == PRO_ADALN || a.pro == PRO_LN_MOD || a.pro == PRO_LN_AFFINE)
        return launch_kernel<quant_rows_kernel<MODE, G, C, CLS_NORM>>(a, nw, lds, st);
    if constexpr (MODE == MODE_BF16 || MODE == MODE_SD_F16) {
        const bool gated = MODE == MODE_BF16 ? a.pro == PRO_GATE || a.pro == PRO_SWIGLU || a.pro == PRO_SILU
                                             : a.pro == PRO_SD_GEGLU && a.tab.gelu_f16;
        if constexpr (MODE == MODE_SD_F16) {
            if (gated) {
                const int cus = device_cu_count();
                const GegluForm f = geglu_form(a.M, a.K, cus);
                if (f.chunks == 1) return launch_geglu<G, 1>(a, f.wpr, cus, st);
                if (f.chunks == 2) return launch_geglu<G, 2>(a, f.wpr, cus, st);
                if (f.chunks == 3) return launch_geglu<G, 3>(a, f.wpr, cus, st);
            }
        }
        if (gated) return launch_kernel<quant_rows_kernel<MODE, G, C, CLS_GATED>>(a, nw, lds, st);
    }
    return launch_kernel<quant_rows_kernel<MODE, G, C, CLS_REST>>(a, nw, lds, st);
}

template <int MODE, int G>
int launch_c(const QuantArgs& a, int nw, int C, hipStream_t st) {
    return C == 1 ? launch<MODE, G, 1>(a, nw, st) : C == 2 ? launch<MODE, G, 2>(a, nw, st) : C == 3 ? launch<MODE, G, 3>(a, nw, st) : launch<MODE, G, 4>(a, nw, st);
}

// g: rotation group width (0, 64, 128, 256).  A row goes to 1, 2, 4 or 8 waves, up to three chunks of 1024 values each (four beyond
// 24 chunks, and in the f32 requantizer), and to more of them where the launch would have fewer than `enough` waves: short
// waves overlap their loads with each other's arithmetic, but a row's waves wait for its slowest, and a norm's for each other
// twice more.  us per call, a wave per chunk (two beyond 8 chunks, on 8 waves) against this: bf16 rotate 128 4608 x 3072 14.2 either way,
// 18601 x 5376 76 and 62; f32 7440 x 5376 40.7 and 36.4, with LayerNorm 90 and 52, bf16 66 and 42; f32 requantizer 54 and 46 there.
//   * Without a rotation (and in the f16 gathers) there is less to wait for: always the most waves.
//   * Six and seven chunks go to eight waves, not to as many: idle ones cost less than uneven SIMDs (bf16 2232 x 5376 8.4, 8.8).
//   * Nine and ten stay on four waves: on eight, a third of the slots would be empty (bf16 rotate 128 1302 x 9216 12.5, 13.6).
//   * Three chunks on two waves and five on four are the worst of both (bf16 13020 x 3072: 1 wave 28.8, 2 29.1, 3 26.4; f16 4882 x
//     5120: 4 waves 23.0, 5 20.3), so those go straight to a wave per chunk.
template <int MODE>
int run_quant(QuantArgs a, int g, hipStream_t st) {
    if (a.M <= 0) return 0;
    const int nchunks = (a.K + kChunk - 1) / kChunk;
    if (nchunks > 32) return -2;
    const bool norm = a.pro == PRO_RMS || a.pro == PRO_LAYERNORM || a.pro == PRO_ADALN || a.pro == PRO_LN_MOD || a.pro == PRO_LN_AFFINE;
    const bool light = g == 0 || a.pro == PRO_SD_UNPAD || a.pro == PRO_SD_GN;
    const int64_t enough = norm ? 2048 : MODE == MODE_F32 && a.pro == PRO_PLAIN ? 6144 : light ? INT64_MAX : 12288;
    int wpr = 1;
    while (wpr < 8 && (nchunks + wpr - 1) / wpr > (MODE == MODE_F32 && a.seed ? 4 : 3)) wpr *= 2;
    while (wpr < 8 && wpr < nchunks && a.M * (int64_t)wpr < (wpr == 4 && nchunks < 11 && nchunks > 8 ? 2048 : enough))
        wpr = nchunks == 3 || nchunks == 5 ? nchunks : 2 * wpr;
    const int C = (nchunks + wpr - 1) / wpr;
    const int nw = wpr < 2 ? 2 : wpr;   // two rows per workgroup at least
    a.wpr = wpr;
    a.rpb = nw / wpr;
    switch (g) {
        case 0: return launch_c<MODE, 0>(a, nw, C, st);
        case 64: return launch_c<MODE, 64>(a, nw, C, st);
        case 128: if (MODE == MODE_SD_F16 || MODE == MODE_ROT_F32) return -1; return launch_c<MODE == MODE_F32 || MODE == MODE_BF16 ? MODE : MODE_BF16, 128>(a, nw, C, st);
        default: return launch_c<MODE, 256>(a, nw, C, st);
    }
}

// The activation tables, for the prologues that evaluate erf / tanh on a 16-bit row.
void attach_tables(QuantArgs& a, hipStream_t st) {
    const int p = a.pro;
    if (p == PRO_SITU || p == PRO_SITU_FAST || p == PRO_GELU || p == PRO_GELU_TANH || p == PRO_SD_GEGLU)
        if (const ActTables* t = act_tables(st)) a.tab = *t;
}

int rotate_group(int rotate) { return rotate == 0 ? 0 : (rotate == 64 || rotate == 128) ? rotate : 256; }

bool known_prologue(int p) { return p >= PRO_PLAIN && p <= PRO_SITU_FAST && p != PRO_LN_AFFINE_SILU; }

// One linear of a few rows in a launch: every workgroup quantizes the rows for itself (a wave per row, the code of the
// quantizer above, so the codes are its codes) while its weights are on their way from HBM straight into the registers
// that the matrix instruction reads, then multiplies them with 64 columns, 16 per wave.  Bound by latency: one trip to memory beside
// the quantizer's chain of LDS round trips.  M=3, K=256 -> N=18432, us per linear replayed from a graph: 4.5, as a quantizer and
// a GEMM 7.0; a call from Python 4.9 where it is native code, 8.1 without, host work.
constexpr int kLinRows = 8, kLinK = 1024, kLinCols = 64;
struct LinArgs {
    const int8_t* W;
    const float* ws;
    const void* bias;
    void* D;
    int N;
    bool vec_ok;   // four consecutive outputs, biases and scales are aligned vectors
};
template <int MODE, int G, int OUT_DT>
__global__ void __launch_bounds__(256) linear_rows_kernel(QuantArgs p, LinArgs a) {
    __shared__ __attribute__((aligned(16))) int8_t codes[kLinRows * kLinK];
    __shared__ float xs[kLinRows];
    __shared__ __attribute__((aligned(16))) float tiles[G ? 4 * kLdsPerWave : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane & 15, quarter = lane >> 4;
    const int nb = (int)blockIdx.x * kLinCols + wave * 16;
    const int wrow = nb + row < a.N ? nb + row : a.N - 1;   // a row past the end is read as the last one and not stored
    const v4i* src = reinterpret_cast<const v4i*>(a.W + (int64_t)wrow * p.K + quarter * 16);
    v4i w[kLinK / 64];
#pragma unroll
    for (int k = 0; k < kLinK / 64; ++k)
        if (k * 64 < p.K) w[k] = src[k * 4];
    QuantArgs r = p;
    r.q = codes;
    r.scales = xs;
    r.wpr = 1;
    for (int m = wave; m < p.M; m += 4) {
        float v[1][16];
        if (lane * 16 < p.K) {
            load16<MODE>(p.x, m * p.x_stride + lane * 16, v[0]);
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) v[0][i] = 0.f;
        }
        const float amax = wave_max_f32(rotate_and_max<MODE, G, 1>(r, v, m, true, 0, lane, tiles + (G ? wave * kLdsPerWave : 0), true));
        store_codes<MODE, 1, false>(r, v, m, true, lane * 16, 0, amax);
    }
    __syncthreads();
    v4i acc{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < kLinK / 64; ++k) {
        if (k * 64 >= p.K) break;
        v4i c{0, 0, 0, 0};
        if (row < p.M) c = *reinterpret_cast<const v4i*>(codes + row * p.K + k * 64 + quarter * 16);
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[k], c, acc, 0, 0, 0);
    }
    // a lane holds row lane % 16 and the columns 4 * (lane / 16) + j
    const int n = nb + 4 * quarter;
    if (row >= p.M || n >= a.N) return;
    const int64_t o = (int64_t)row * a.N + n;
    float ws[4], b[4] = {0.f, 0.f, 0.f, 0.f}, out[4];
    if (a.vec_ok) {
        load4<DT_F32>(a.ws, n, ws);
        if (a.bias) load4<OUT_DT>(a.bias, n, b);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            ws[j] = n + j < a.N ? a.ws[n + j] : 0.f;
            if (a.bias && n + j < a.N) b[j] = ld_dt<OUT_DT>(a.bias, n + j);
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = __builtin_fmaf((float)acc[j] * xs[row], ws[j], b[j]);
    if (a.vec_ok) {
        store4<OUT_DT>(a.D, o, out);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) if (n + j < a.N) st_dt<OUT_DT>(a.D, o + j, out[j]);
    }
}

template <int MODE, int G>
int launch_linear_rows(const QuantArgs& q, const LinArgs& a, int out_dt, hipStream_t st) {
    const dim3 grid((unsigned)((a.N + kLinCols - 1) / kLinCols));
    if (out_dt == DT_F32) hipLaunchKernelGGL((linear_rows_kernel<MODE, G, DT_F32>), grid, dim3(256), 0, st, q, a);
    else if (out_dt == DT_F16) hipLaunchKernelGGL((linear_rows_kernel<MODE, G, DT_F16>), grid, dim3(256), 0, st, q, a);
    else hipLaunchKernelGGL((linear_rows_kernel<MODE, G, DT_BF16>), grid, dim3(256), 0, st, q, a);
    KCHECK();
    return 0;
}
template <int MODE>
int run_linear_rows(const QuantArgs& q, const LinArgs& a, int g, int out_dt, hipStream_t st) {
    return g == 0 ? launch_linear_rows<MODE, 0>(q, a, out_dt, st) : g == 64 ? launch_linear_rows<MODE, 64>(q, a, out_dt, st)
         : g == 128 ? launch_linear_rows<MODE, 128>(q, a, out_dt, st) : launch_linear_rows<MODE, 256>(q, a, out_dt, st);
}

// Rows of at most one wave's chunk, few enough of them that quantizing them in every workgroup costs less than a launch: at
// N=18432, one kernel against two, 8 rows 5.9 and 7.2 us (K=256), 9.7 and 10.9 (K=1024), 16 rows 8.9 and 7.3, 13.3 and 11.0.
bool linear_in_one(const void* W, int dtype, int64_t M, int64_t N, int64_t K, int grp, int out_dt) {
    return M > 0 && M <= kLinRows && K > 0 && K <= kLinK && K % (grp ? grp : 64) == 0 && N > 0 && N <= 0x7fffffff - kLinCols &&
           (dtype == DT_BF16 || dtype == DT_F32) && out_dt >= DT_F32 && out_dt <= DT_BF16 && ((uintptr_t)W & 15) == 0;
}

}  // namespace

GPU_API int gpu_quant_rows(int dtype, int prologue, const void* x, int64_t x_stride, const void* g, int64_t g_stride,
                           int64_t up_offset, const float* norm_w, float eps, const void* mod_scale,
                           const void* mod_shift, int8_t* q, float* scales, int M, int K, int rotate, void* stream) {
    const int grp = rotate_group(rotate);
    const int need = grp == 0 ? 64 : grp;
    if (K <= 0 || (K % need) != 0) return -1;
    if (dtype != DT_BF16 && dtype != DT_F32) return -4;
    if (!known_prologue(prologue)) return -3;   // the id list of csrc/kernels.cu:280-292
    if (K > 32768) return -2;
    QuantArgs a{x, x_stride, q, scales, nullptr, M, K, 1, 1, 0, prologue, g, g_stride, up_offset, norm_w, nullptr, eps, mod_scale,
                mod_shift};
    if (dtype == DT_BF16 && M > 0) attach_tables(a, (hipStream_t)stream);
    return dtype == DT_BF16 ? run_quant<MODE_BF16>(a, grp, (hipStream_t)stream) : run_quant<MODE_F32>(a, grp, (hipStream_t)stream);
}

GPU_API int gpu_linear_w8a8(int dtype, const void* x, int64_t x_stride, const int8_t* W, const float* ws, const void* bias, void* D,
                            void* scratch, int64_t M, int64_t N, int64_t K, int rotate, int out_dt, void* stream) {
    const int grp = rotate_group(rotate);
    hipStream_t st = (hipStream_t)stream;
    if (linear_in_one(W, dtype, M, N, K, grp, out_dt)) {
        const QuantArgs q{x, x_stride, nullptr, nullptr, nullptr, (int)M, (int)K, 1, 1, 0, PRO_PLAIN};
        const uintptr_t size = out_dt == DT_F32 ? 4 : 2;
        const LinArgs a{W, ws, bias, D, (int)N,
                        N % 4 == 0 && (((uintptr_t)D | (uintptr_t)bias) & (4 * size - 1)) == 0 && ((uintptr_t)ws & 15) == 0};
        return dtype == DT_BF16 ? run_linear_rows<MODE_BF16>(q, a, grp, out_dt, st) : run_linear_rows<MODE_F32>(q, a, grp, out_dt, st);
    }
    if (M < 0 || M > 0x7fffffff || K < 0 || K > 0x7fffffff) return -200;
    const bool refuse = M > 0 && (!scratch || ((uintptr_t)scratch & 15));   // after what the quantizer refuses, of no rows
    int8_t* codes = (int8_t*)scratch;
    float* xs = (float*)(codes + M * K);   // K % 64 == 0: aligned as scratch is
    if (const int rc = gpu_quant_rows(dtype, PRO_PLAIN, x, x_stride, nullptr, 0, 0, nullptr, 0.f, nullptr, nullptr, codes, xs,
                                      refuse ? 0 : (int)M, (int)K, rotate, stream)) return rc;
    if (refuse) return -1;
    return gpu_int8_gemm(codes, W, xs, ws, bias, D, M, N, K, out_dt, stream);
}

GPU_API int gpu_quant_rows_b(int dtype, int prologue, const void* x, int64_t x_stride, const float* norm_w,
                             const float* norm_b, float eps, const void* mod_scale, const void* mod_shift, int8_t* q,
                             float* scales, int M, int K, int rotate, void* stream) {
    if ((K % 256) != 0) return -1;
    if (dtype != DT_BF16) return -4;
    if (prologue != PRO_LN_MOD && prologue != PRO_LN_AFFINE) return -3;
    if (K <= 0) return -1;
    if (K > 32768) return -2;
    QuantArgs a{x, x_stride, q, scales, nullptr, M, K, 1, 1, 0, prologue, nullptr, 0, 0, norm_w, norm_b, eps, mod_scale, mod_shift};
    return run_quant<MODE_BF16>(a, rotate_group(rotate), (hipStream_t)stream);
}

GPU_API int gpu_rotate_rows_f32(int prologue, const float* x, int64_t x_stride, int64_t up_offset, const float* norm_w,
                                float eps, float* out, int M, int K, void* stream) {
    if (K <= 0 || (K % 256) != 0) return -1;
    if (prologue != PRO_PLAIN && prologue != PRO_RMS && prologue != PRO_SWIGLU) return -3;
    if (K > 32768) return -2;
    QuantArgs a{x, x_stride, nullptr, nullptr, out, M, K, 1, 1, 0, prologue, nullptr, 0, up_offset, norm_w, nullptr, eps, nullptr,
                nullptr};
    return run_quant<MODE_ROT_F32>(a, 256, (hipStream_t)stream);
}

GPU_API int gpu_sd_quant_rows(const void* x, int64_t x_stride, int8_t* q, float* scales, int M, int K, int rotate,
                              void* stream) {
    if ((rotate != 0 && rotate != 64 && rotate != 256) || (rotate && K % rotate)) return -1;
    if (K <= 0 || (K % 16) != 0) return -1;   // 16 values per lane
    if (K > 32768) return -2;
    QuantArgs a{x, x_stride, q, scales, nullptr, M, K, 1, 1};
    return run_quant<MODE_SD_F16>(a, rotate, (hipStream_t)stream);
}

// The SD UNet's fused quantizers (csrc/sd.cu:608-724): the half row of LayerNorm / GEGLU / head un-padding / GroupNorm,
// computed on the values as the fp16 quantizer loads them; it is rounded to half there as in the reference.
extern "C" int gpu_internal_sd_group_stats(const void* x, void* stats, int n_images, int64_t P, int C, int G, float eps,
                                           void* stream);
namespace {
int sd_fused(QuantArgs a, int rotate, hipStream_t st) {
    if ((rotate != 0 && rotate != 64 && rotate != 256) || (rotate && a.K % rotate)) return -1;   // csrc/sd.cu:682
    if (a.K <= 0 || (a.K % 16) != 0) return -1;
    if (a.K > 32768) return -2;
    if (a.M <= 0) return 0;
    attach_tables(a, st);
    return run_quant<MODE_SD_F16>(a, rotate, st);
}
}  // namespace

GPU_API int gpu_sd_ln_quant_rows(const void* x, int64_t x_stride, const float* w, const float* b, float eps, int8_t* q,
                                 float* scales, int M, int K, int rotate, void* stream) {
    QuantArgs a{x, x_stride, q, scales, nullptr, M, K, 1, 1, 0, PRO_LN_AFFINE, nullptr, 0, 0, w, b, eps, nullptr, nullptr};
    return sd_fused(a, rotate, (hipStream_t)stream);
}
GPU_API int gpu_sd_geglu_quant_rows(const void* in, int8_t* q, float* scales, int M, int I, int rotate, void* stream) {
    QuantArgs a{in, 2 * (int64_t)I, q, scales, nullptr, M, I, 1, 1, 0, PRO_SD_GEGLU, nullptr, 0, I, nullptr, nullptr, 0.f, nullptr,
                nullptr};
    return sd_fused(a, rotate, (hipStream_t)stream);
}
GPU_API int gpu_sd_unpad_quant_rows(const void* src, int8_t* q, float* scales, int M, int H, int d, int dp, int rotate,
                                    void* stream) {
    if (H <= 0 || d <= 0 || dp < d) return -1;
    QuantArgs a{src, (int64_t)H * dp, q, scales, nullptr, M, H * d, 1, 1, 0, PRO_SD_UNPAD, nullptr, 0, 0, nullptr, nullptr, 0.f,
                nullptr, nullptr, d, dp};
    return sd_fused(a, rotate, (hipStream_t)stream);
}
GPU_API int gpu_sd_group_norm_quant_rows(const void* x, const float* w, const float* b, void* sums, int N, int64_t P, int C, int G,
                                         float eps, int8_t* q, float* scales, int rotate, void* stream) {
    if (G <= 0 || C % G) return -1;                                                             // csrc/sd.cu:713
    if ((rotate != 0 && rotate != 64 && rotate != 256) || (rotate && C % rotate) || C <= 0 || C % 16) return -1;
    if (N <= 0 || P <= 0) return 0;
    const int rc = gpu_internal_sd_group_stats(x, sums, N, P, C, G, eps, stream);
    if (rc) return rc;
    QuantArgs a{x, C, q, scales, nullptr, (int)(N * P), C, 1, 1, 0, PRO_SD_GN, sums, P, 0, w, b, eps, nullptr, nullptr, 0, 0, C / G};
    return sd_fused(a, rotate, (hipStream_t)stream);
}

// x [N, K] in its original basis -> rotated int8 rows + row scales: the 256-wide quantizer with rounding to nearest
// (seed 0) or stochastic rounding keyed by element index + seed.  Replaces gpu_convrot_requant, csrc/kernels.cu:1361-1420;
// as there, any dtype other than DT_F32 is read as bf16.
GPU_API int gpu_convrot_requant(int dtype, const void* x, void* q, void* s, int64_t N, int K, uint64_t seed, void* stream) {
    if (K <= 0 || (K % 256) != 0) return -1;
    if (K > 32768 || N > 0x7fffffff) return -2;
    QuantArgs a{x, K, (int8_t*)q, (float*)s, nullptr, (int)N, K, 1, 1, seed};
    return dtype == DT_F32 ? run_quant<MODE_F32>(a, 256, (hipStream_t)stream) : run_quant<MODE_BF16>(a, 256, (hipStream_t)stream);
}

// Test hook: the form of the GEGLU quantizer that a shape takes, 100 * chunks per wave + waves per row; 0: the one for few chunks.
GPU_API int gpu_internal_geglu_form(int M, int K) {
    const GegluForm f = geglu_form(M, K, device_cu_count());
    return 100 * f.chunks + f.wpr;
}

// Test hook: out[i] = bf16 bits of sigmoid (which 0) or silu (1) of the bf16 bits in[i], or f16 bits of gelu (2) of the f16
// bits in[i], as the prologues evaluate them.
namespace {
__global__ void __launch_bounds__(256) act_probe_kernel(int which, const uint16_t* in, uint16_t* out, int n, const float* gelu) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    if (which == 2) {
        const uint32_t a = gelu_index_x2(in[i]);
        out[i] = (uint16_t)gelu_f16x2(in[i], gelu[a & 0xffffu], 0.f);
        return;
    }
    const float x = bf16_to_f(in[i]);
    out[i] = f_to_bf16(which == 0 ? sigmoid_of_bf16(x) : silu_of_bf16(x));
}
}  // namespace
GPU_API int gpu_internal_act_probe(int which, const void* in, void* out, int n, void* stream) {
    if (which < 0 || which > 2 || !in || !out || n <= 0) return -1;
    const ActTables* t = which == 2 ? act_tables((hipStream_t)stream) : nullptr;
    if (which == 2 && !t) return -1;
    hipLaunchKernelGGL(act_probe_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, which, (const uint16_t*)in,
                       (uint16_t*)out, n, t ? t->gelu_f16_g : nullptr);
    KCHECK();
    return 0;
}
