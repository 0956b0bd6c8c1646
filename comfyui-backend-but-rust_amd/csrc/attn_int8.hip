// INT8 attention for head dim 128 on gfx950: Q and K rotated and quantized per scale group, V per channel, integer
// scores and integer P.V partials on v_mfma_i32_32x32x32_i8, softmax state in fp32.
//
// Semantics follow the reference's Sage-style path (csrc/attn_int8.cu:118-160 chains the stages;
// csrc/vendor/sage/quant_qk_int8.cu:72-157 rotation, :296-413 Q groups, :422-575 K groups, :591-756 K anchor;
// csrc/vendor/sage/quant_v_int8.cu:94-190 V; csrc/vendor/sage/qk_int_sv_i8_cuda.cuh + attn_utils.cuh:700-800 the tile
// update with u8 probabilities).  The design is for CDNA4:
//   * keys ride in src0 and queries in src1 of the score MFMA, so a lane ends up with one query row and 16 keys per
//     32-key block: row maxima and sums are in-lane plus one exchange with lane ^ 32;
//   * those 16 scores are, in order, exactly the 16 K-bytes that lane must supply as src1 of the P.V MFMA when V^T is
//     stored with the matching key order, so probabilities never cross lanes;
//   * the matrix cores multiply signed bytes only: probabilities 0..255 are fed as p - 128 and the accumulator starts
//     at 128 * (column sums of the V tile), which the V quantizer leaves in the workspace.  The integers are exact.
// The workspace layout is private to this file.
#include <climits>
#include <cstdio>
#include <type_traits>

#include "common.hpp"

namespace {

constexpr float kU8Offset = 7.9943534f;
// Head dims 64, 128 and 256 (csrc/attn_int8.cu:42-45).  A row's channels lie on D/16 consecutive lanes, sixteen channels
// each; the Q quantizer's row block is 32 rows, 16 at head dim 256.
constexpr int lanes_per_row(int D) { return D / 16; }
constexpr int q_block_rows(int D) { return D == 256 ? 16 : 32; }

struct AttnArgs {
    const void *q, *k, *v;
    void* o;
    int8_t *qi, *ki, *vt;
    float *qs, *ks, *vs;
    int* anchors;
    float* vmax;   // [kv head][v_chunks][D]: largest |v| of each chunk of keys
    int* vsum;
    int b, lq, lk, h, hk, rep, qg, kb, ck, nblk;
    int64_t q_bs, q_rs, q_hs, k_bs, k_rs, k_hs, v_bs, v_rs, v_hs, o_bs, o_rs, o_hs;
    float sm, sink;
    int vec_ok, in_vec, v_vec, nr_vec, use_anchor;   // nr_vec: qw, kw and rope are 16-byte aligned
    int rot4;   // lk <= 256: the rotation is only the H4 on runs of four channels, without the sign diagonal
    // per-head RMSNorm (+ weight) and RoPE ahead of the quantizers (csrc/kernels.cu:482-540 through
    // csrc/vendor/sage/quant_qk_int8.cu:160-291): q_norm / k_norm say which of Q and K take it
    const float *qw, *kw, *rope;   // [128] or null (ones); rope [L][64] x (cos, sin) or null
    float eps;
    int q_norm, k_norm, rope_mode;
    const float* bias;    // per-key logit bias of the caller, f32 [lk], or null
    float* kbias;         // prepared: bias * log2e per key of every tile (-inf: not kept / padding), then one value per tile
    int whole, parts;     // row blocks with one workgroup each; workgroups that share the keys of every other row block
    float* part;          // their results, and per row block how many of them are there
    uint32_t* done;
    float* tbias;         // per tile: the bias all its keys share (times log2e), NaN when they differ, -inf when none is kept
};

// fmaxf as the reference's device code uses it: a NaN operand is dropped.
__device__ __forceinline__ float fmax_nn(float a, float b) { return __builtin_fmaxf(a, b); }

// Cross-lane moves inside a row's lanes, as data-parallel-primitive modifiers (no LDS traffic).  A row's 16-channel blocks lie
// on its lanes so that each move of a block bit is one such modifier: blocks 4..7 of eight run backwards, which makes
// block ^ 4 the mirror of the eight lanes.
template <int CTRL> __device__ __forceinline__ float dpp_mov(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <int D> __device__ __forceinline__ int block_of_lane(int lane) { return D == 64 || !(lane & 4) ? lane : lane ^ 3; }   // within the row
__device__ __forceinline__ float block_xor1(float x) { return dpp_mov<0xB1>(x); }    // quad_perm [1,0,3,2]
__device__ __forceinline__ float block_xor2(float x) { return dpp_mov<0x4E>(x); }    // quad_perm [2,3,0,1]
__device__ __forceinline__ float block_xor4(float x) { return dpp_mov<0x141>(x); }   // half-row mirror
__device__ __forceinline__ float block_xor8(float x) { return dpp_mov<0x128>(x); }   // row_ror:8 within a row of 16 lanes

// Normalized Walsh-Hadamard over the 16 << LB channels of one row held by 1 << LB consecutive lanes, sixteen adjacent
// channels per lane (ol = the lane's block), after the sign diagonal when SIGN (head dim 128 only).  Same operation
// order as the oracle: H4 on runs of four channels, radix-2 butterflies over the higher channel bits in ascending order
// (two in the lane, LB across lanes), one scaling.  LB = 3: H128 (the reference's convrot128 / convrot128_plain), LB = 2:
// H64 (convrot64).
template <int LB, bool SIGN> __device__ __forceinline__ void rot_wh(float (&v)[16], int ol) {
    if (SIGN) {
        const uint32_t word = (ol >> 1) == 0 ? 0x1035997bu : (ol >> 1) == 1 ? 0x8087f5eeu : (ol >> 1) == 2 ? 0xee2e4e1au : 0x71132418u;
        const uint32_t keep = word >> ((ol & 1) * 16);
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = u2f(f2u(v[e]) ^ ((((keep >> e) & 1u) ^ 1u) << 31));
    }
#pragma unroll
    for (int g = 0; g < 16; g += 4) {
        const float a0 = v[g] + v[g + 1], a1 = v[g] - v[g + 1], a2 = v[g + 2] + v[g + 3], a3 = v[g + 2] - v[g + 3];
        v[g] = (a0 + a2) * 0.5f;
        v[g + 1] = (a1 + a3) * 0.5f;
        v[g + 2] = (a0 - a2) * 0.5f;
        v[g + 3] = (a1 - a3) * 0.5f;
    }
#pragma unroll
    for (int bit = 4; bit < 16; bit <<= 1)
#pragma unroll
        for (int e = 0; e < 16; ++e)
            if (!(e & bit)) {
                const float lo = v[e], hi = v[e | bit];
                v[e] = lo + hi;
                v[e | bit] = lo - hi;
            }
    // other - v in the upper block of a pair, v + other in the lower: one fma on an exact product by -1 or 1
    const float s1 = ol & 1 ? -1.f : 1.f, s2 = ol & 2 ? -1.f : 1.f, s4 = ol & 4 ? -1.f : 1.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = __builtin_fmaf(v[e], s1, block_xor1(v[e]));
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = __builtin_fmaf(v[e], s2, block_xor2(v[e]));
    if (LB == 3) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = __builtin_fmaf(v[e], s4, block_xor4(v[e]));
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] *= LB == 3 ? 0.1767766952966369f : 0.25f;
}

// The rotation of sequences of at most 256 keys (csrc/vendor/sage/quant_qk_int8.cu:1160-1166, ROTATION 4): the
// normalized H4 on each run of four adjacent channels and nothing else.
__device__ __forceinline__ void rot4(float (&v)[16]) {
#pragma unroll
    for (int g = 0; g < 16; g += 4) {
        const float a0 = v[g] + v[g + 1], a1 = v[g] - v[g + 1], a2 = v[g + 2] + v[g + 3], a3 = v[g + 2] - v[g + 3];
        v[g] = (a0 + a2) * 0.5f;
        v[g + 1] = (a1 + a3) * 0.5f;
        v[g + 2] = (a0 - a2) * 0.5f;
        v[g + 3] = (a1 - a3) * 0.5f;
    }
}

// The rotation the quantizers apply to a row of head dim D (csrc/vendor/sage/quant_qk_int8.cu:1150-1195): the H4 blocks
// alone up to 256 keys, beyond that H64 at head dim 64, sign diagonal + H128 at 128, the plain H128 on each half at 256.
template <int D> __device__ __forceinline__ void rotate_row(float (&v)[16], int ol, bool h4_only) {
    if (h4_only) rot4(v);
    else if (D == 64) rot_wh<2, false>(v, ol);
    else if (D == 128) rot_wh<3, true>(v, ol);
    else rot_wh<3, false>(v, ol & 7);
}

// Maximum over the lanes of a row.
template <int D> __device__ __forceinline__ float max_row(float m) {
    m = fmax_nn(m, block_xor1(m));
    m = fmax_nn(m, block_xor2(m));
    if (D >= 128) m = fmax_nn(m, block_xor4(m));
    if (D == 256) m = fmax_nn(m, block_xor8(m));
    return m;
}

// Sum of squares of one 128-channel row in the order of the reference's warp of 32 lanes (csrc/kernels.cu:497-513,
// csrc/common.cuh:30-34): lane L accumulates its four channels by fma in index order, then the lanes add pairwise at
// distances 16, 8, 4, 2, 1.  Lane L owns channels 4L..4L+3, or, with split = rope_mode 2 (with or without a table),
// channels 2L, 2L+1, 64+2L, 65+2L.  Here eight lanes hold sixteen adjacent channels each (o8 = the lane's block),
// so a lane carries four (eight, split) of the reference's lanes; all eight lanes get the sum.
__device__ __forceinline__ float sumsq128(const float (&v)[16], int o8, bool split) {
    if (!split) {
        float s[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s[i] = v[4 * i] * v[4 * i];
            s[i] = __builtin_fmaf(v[4 * i + 1], v[4 * i + 1], s[i]);
            s[i] = __builtin_fmaf(v[4 * i + 2], v[4 * i + 2], s[i]);
            s[i] = __builtin_fmaf(v[4 * i + 3], v[4 * i + 3], s[i]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] += block_xor4(s[i]);   // distance 16
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] += block_xor2(s[i]);   // 8
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] += block_xor1(s[i]);   // 4
        return (s[0] + s[2]) + (s[1] + s[3]);                   // 2, then 1
    }
    // split: the lanes of the low half start each chain (channels 2L, 2L+1), the lanes of the high half finish it
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float p = __builtin_fmaf(v[2 * i + 1], v[2 * i + 1], v[2 * i] * v[2 * i]);
        const float q = block_xor4(p);
        s[i] = __builtin_fmaf(v[2 * i + 1], v[2 * i + 1], __builtin_fmaf(v[2 * i], v[2 * i], q));   // meaningful where o8 >= 4
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] += block_xor2(s[i]);       // distance 16
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] += block_xor1(s[i]);       // 8
    const float t = ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));   // 4, 2, 1
    const float u = block_xor4(t);
    return o8 >= 4 ? t : u;
}

// The same sum by one thread over a row in memory.
__device__ inline float sumsq128_serial(const float* x, bool split) {
    float s[32];
    for (int l = 0; l < 32; ++l) {
        const int i0 = split ? 2 * l : 4 * l, i2 = split ? 64 + 2 * l : 4 * l + 2;
        float t = x[i0] * x[i0];
        t = __builtin_fmaf(x[i0 + 1], x[i0 + 1], t);
        t = __builtin_fmaf(x[i2], x[i2], t);
        s[l] = __builtin_fmaf(x[i2 + 1], x[i2 + 1], t);
    }
    for (int o = 16; o > 0; o >>= 1)
        for (int l = 0; l < o; ++l) s[l] += s[l + o];
    return s[0];
}

__device__ __forceinline__ void round_bf16x2(float& x, float& y) {
    x = rnd_bf16(x);
    y = rnd_bf16(y);
}

// Per-head RMSNorm, weight and RoPE of one 128-channel row held by eight lanes (sixteen adjacent channels each), as the
// reference applies them to q and k ahead of the quantizer (csrc/kernels.cu:482-540, csrc/vendor/sage/quant_qk_int8.cu:
// 211-278): v = T((v * rstd) * w), rstd = 1/sqrt(mean(v^2) + eps) with the sum in the reference's order (sumsq128);
// rope mode 1 turns the pairs (2p, 2p+1), mode 2 the pairs (j, j + 64), with (cos, sin) = rope_row[2p], rope_row[2p+1];
// the result is rounded to bf16 again.  This build's definition of the two parts the reference leaves to its machine:
// 1/sqrt is correctly rounded (the reference's rsqrtf is an approximation of up to two units in the last place), and
// c*a - s*b, s*a + c*b contract to one fma each on their first product.  w == nullptr means ones; rope_row == nullptr
// means no rotation.  All eight lanes must call it.
// The caller has loaded the lane's weights (ones for a null w) and, unless rope_mode is 0, its pairs of (cos, sin): rope_mode 1
// those of its own channel pairs, 2 those of channels (block & 3) * 16 .. + 15, thirty-two floats.
__device__ __forceinline__ void norm_row(float (&v)[16], int o8, const float (&w)[16], float eps, bool split) {
    const float rstd = rsqrt_cr(sumsq128(v, o8, split) / 128.f + eps);
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        v[e] = v[e] * rstd * w[e];
        v[e + 1] = v[e + 1] * rstd * w[e + 1];
        round_bf16x2(v[e], v[e + 1]);
    }
}
__device__ __forceinline__ void rope_pairs(float (&v)[16], const float (&cs)[16]) {
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        const float a = v[e], b = v[e + 1];
        v[e] = __builtin_fmaf(cs[e], a, -(cs[e + 1] * b));
        v[e + 1] = __builtin_fmaf(cs[e + 1], a, cs[e] * b);
        round_bf16x2(v[e], v[e + 1]);
    }
}
__device__ __forceinline__ void rope_halves(float (&v)[16], int o8, const float* r) {
    const float sgn = o8 < 4 ? -1.f : 1.f;
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        v[e] = __builtin_fmaf(v[e], r[2 * e], sgn * (block_xor4(v[e]) * r[2 * e + 1]));
        v[e + 1] = __builtin_fmaf(v[e + 1], r[2 * e + 2], sgn * (block_xor4(v[e + 1]) * r[2 * e + 3]));
        round_bf16x2(v[e], v[e + 1]);
    }
}
__device__ __forceinline__ void load16_f32(const float* p, float (&v)[16]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const float4 f = reinterpret_cast<const float4*>(p)[g];
        v[4 * g] = f.x; v[4 * g + 1] = f.y; v[4 * g + 2] = f.z; v[4 * g + 3] = f.w;
    }
}
// What the quantizer kernels are instantiated for: no norm; norm with 16-byte aligned tables and rope by pairs or none; any
// other.  The first two do without the registers of what follows them.
enum { NORM_NONE, NORM_PAIRS, NORM_ANY };
// N rows at once, so that their tables are all in flight before the first is used: row_of(j) is row j's position.
template <int NM, int N, class RowOf>
__device__ __forceinline__ void norm_rope_rows(float (&v)[N][16], int o8, const float* w, const float* rope, float eps, int mode, RowOf row_of) {
    float wv[16];
    if (NM == NORM_PAIRS && w) {
        load16_f32(w + o8 * 16, wv);
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) wv[e] = NM == NORM_ANY && w ? w[o8 * 16 + e] : 1.f;
    }
    if constexpr (NM == NORM_PAIRS) {
        float cs[N][16];
        if (rope) {
#pragma unroll
            for (int j = 0; j < N; ++j) load16_f32(rope + (int64_t)row_of(j) * 128 + o8 * 16, cs[j]);
        }
#pragma unroll
        for (int j = 0; j < N; ++j) {
            norm_row(v[j], o8, wv, eps, false);
            if (rope) rope_pairs(v[j], cs[j]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            norm_row(v[j], o8, wv, eps, mode == 2);
            if (!rope) continue;
            const float* r = rope + (int64_t)row_of(j) * 128;
            if (mode == 1) {
                float cs[16];
#pragma unroll
                for (int e = 0; e < 16; ++e) cs[e] = r[o8 * 16 + e];
                rope_pairs(v[j], cs);
            } else {
                rope_halves(v[j], o8, r + (o8 & 3) * 32);
            }
        }
    }
}

// Sixteen codes rn(v * inv), for |v * inv| below 2^22: around 1.5 * 2^23 a float has a step of 1, so adding that leaves the
// rounded number in the low bits, two's complement.  No clamp: inv is the reciprocal of (largest |v|) / 127 + 1e-7.  A NaN
// gives 0 (its payload's low byte), as the reference's conversion does.
__device__ __forceinline__ uint32_t pack_low_bytes(float a, float b, float c, float d) {
    return __builtin_amdgcn_perm(__builtin_amdgcn_perm(f2u(d), f2u(c), 0x0c0c0400u), __builtin_amdgcn_perm(f2u(b), f2u(a), 0x0c0c0400u), 0x05040100u);
}
__device__ __forceinline__ uint4 codes16(const float (&v)[16], float inv) {
    constexpr float M = 12582912.f;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = pack_low_bytes(v[4 * e] * inv + M, v[4 * e + 1] * inv + M, v[4 * e + 2] * inv + M, v[4 * e + 3] * inv + M);
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// Four consecutive elements: one 8-byte load when the caller's strides and base allow it.
template <int DT> __device__ __forceinline__ void ld4_dt(const void* p, int64_t i, bool vec, float (&v)[4]) {
    if (vec) {
        load4<DT>(p, i, v);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = ld_dt<DT>(p, i + c);
    }
}

template <int DT> __device__ __forceinline__ void ld16_dt(const void* p, int64_t i, bool vec, float (&v)[16]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        float x[4];
        ld4_dt<DT>(p, i + g * 4, vec, x);
#pragma unroll
        for (int c = 0; c < 4; ++c) v[g * 4 + c] = x[c];
    }
}

// N rows' sixteen channels, all loads issued before the first is used.
template <int DT, int N, class RowOf>
__device__ __forceinline__ void load_rows(const void* p, int64_t base, int64_t rs, int vec, float (&v)[N][16], RowOf row_of) {
    if (vec == 2) {
        uint4 w[N][2];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint4* q = reinterpret_cast<const uint4*>((const uint16_t*)p + base + (int64_t)row_of(j) * rs);
            w[j][0] = q[0];
            w[j][1] = q[1];
        }
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint32_t u[8] = {w[j][0].x, w[j][0].y, w[j][0].z, w[j][0].w, w[j][1].x, w[j][1].y, w[j][1].z, w[j][1].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (DT == DT_BF16) {
                    v[j][2 * e] = u2f(u[e] << 16);
                    v[j][2 * e + 1] = u2f(u[e] & 0xffff0000u);
                } else {
                    unpack_f16x2(u[e], v[j][2 * e], v[j][2 * e + 1]);
                }
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) ld16_dt<DT>(p, base + (int64_t)row_of(j) * rs, vec, v[j]);
    }
}

// The K anchor of one (kv head, batch).  The nine sampled keys go to LDS (a thread per channel); the sums then follow the
// reference's block of 128 threads in four warps: thread t walks channels t and t + 128 with one set of accumulators
// (head dim 256), threads past the head dim hold zeros (64), warps add by a shuffle-down tree and the four warps in
// order (csrc/vendor/sage/quant_qk_int8.cu:640-756).  A chain of LDS trips by few threads, which short calls wait for: rows and parts of
// sums lie so that their readers meet in different banks, maxima go over lanes instead of 128 reads of one thread, and every thread picks the
// candidate itself.  us a call, with rows 128 floats apart, one thread's maxima and the candidate through LDS, and this: with norm and rope
// 300 x 24 x 128 27.2 and 26.1, 1024 x 24 x 128 44.9 and 43.9; 256 x 10 x 64 16.6 and 16.3, 2 x 1600 x 7 x 64 33.6 and 33.3; 4608 x 24 x 128 and
// 2 x 4096 x 10 x 64 the same.  (cos and sin asked for beside the keys: 26.8 and 45.3, registers of the whole launch.)
template <int DT, int D>
__device__ __forceinline__ void anchor_body(const AttnArgs& a, const int hi, const int bi) {
    __shared__ __align__(16) float s[9][D + 4];
    constexpr int PART = 36;   // floats from one 32-thread part of a sum to the next: the parts' readers meet in other banks
    __shared__ __align__(16) float dist[10][4 * PART], best_energy[4 * PART];   // nine candidates, then the energy
    __shared__ float amax[2], bmax[2];
    const int tid = threadIdx.x, c = tid & (D - 1), slot = (tid >> 5) * PART + (tid & 31);
    const int64_t base = bi * a.k_bs + hi * a.k_hs;
    bool normed = false;
    if constexpr (D == 128) {
        if (a.k_norm) {
            normed = true;
            // the nine sampled keys as the K quantizer will see them: norm_rope_row's arithmetic with a thread per channel
            __shared__ float rstd9[9];
            __shared__ float nrm[9][D];
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const int row = (int)((int64_t)i * (a.lk - 1) / 8);
                s[i][c] = ld_dt<DT>(a.k, base + (int64_t)row * a.k_rs + c);
            }
            __syncthreads();
            if (tid < 9) rstd9[tid] = (float)(1.0 / sqrt((double)(sumsq128_serial(s[tid], a.rope_mode == 2) / 128.f + a.eps)));
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 9; ++i) nrm[i][c] = rnd_dt<DT_BF16>(s[i][c] * rstd9[i] * (a.kw ? a.kw[c] : 1.f));
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                float x = nrm[i][c];
                if (a.rope) {
                    const int row = (int)((int64_t)i * (a.lk - 1) / 8);
                    const float* r = a.rope + (int64_t)row * D;
                    if (a.rope_mode == 1) {
                        const float cs = r[c & ~1], sn = r[c | 1], other = nrm[i][c ^ 1];
                        x = rnd_dt<DT_BF16>((c & 1) ? __builtin_fmaf(sn, other, cs * x) : __builtin_fmaf(cs, x, -(sn * other)));
                    } else {
                        const int j = c & 63;
                        const float cs = r[2 * j], sn = r[2 * j + 1], other = nrm[i][c ^ 64];
                        x = rnd_dt<DT_BF16>(c < 64 ? __builtin_fmaf(x, cs, -(other * sn)) : __builtin_fmaf(x, cs, other * sn));
                    }
                }
                s[i][c] = x;
            }
        }
    }
    if (!normed && tid < D) {
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int row = (int)((int64_t)i * (a.lk - 1) / 8);
            s[i][c] = ld_dt<DT>(a.k, base + (int64_t)row * a.k_rs + c);
        }
    }
    __syncthreads();
    if (tid < 128) {
        float e = 0.f, m = 0.f, d9[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) d9[i] = 0.f;
        for (int ch = tid; ch < D; ch += 128) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const float x = s[i][ch];
                e = fmaf(x, x, e);
                m = fmax_nn(m, fabsf(x));
                sum += x;
            }
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const float d = fmaf(9.f, s[i][ch], -sum);
                d9[i] = fmaf(d, d, d9[i]);
            }
        }
        dist[9][slot] = e;
        m = wave_max_f32(m);
        if ((tid & 63) == 0) amax[tid >> 6] = m;
#pragma unroll
        for (int i = 0; i < 9; ++i) dist[i][slot] = d9[i];
    }
    __syncthreads();
    auto tree = [](const float* x) {
        float t[32];
        for (int i = 0; i < 32; ++i) t[i] = x[i];
        for (int off = 16; off > 0; off >>= 1)
            for (int i = 0; i < off; ++i) t[i] += t[i + off];
        return t[0];
    };
    __shared__ float warp_sum[11][4];   // nine candidate distances, then the two energies
    if (tid < 40) warp_sum[tid / 4][tid % 4] = tree(&dist[tid / 4][(tid % 4) * PART]);
    __syncthreads();
    int best = 0;   // every thread for itself: broadcasts cost less than a barrier
    float best_d = 3.402823466e+38F;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        float d = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) d += warp_sum[i][w];
        if (d < best_d) { best = i; best_d = d; }
    }
    if (tid < 128) {
        float be = 0.f, bm = 0.f;
        for (int ch = tid; ch < D; ch += 128) {
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                const float r = s[i][ch] - s[best][ch];
                be = fmaf(r, r, be);
                bm = fmax_nn(bm, fabsf(r));
            }
        }
        best_energy[slot] = be;
        bm = wave_max_f32(bm);
        if ((tid & 63) == 0) bmax[tid >> 6] = bm;
    }
    __syncthreads();
    if (tid < 4) warp_sum[10][tid] = tree(&best_energy[tid * PART]);
    __syncthreads();
    if (tid == 0) {
        float e0 = 0.f, e1 = 0.f;
        for (int w = 0; w < 4; ++w) {
            e0 += warp_sum[9][w];
            e1 += warp_sum[10][w];
        }
        const float m0 = fmax_nn(amax[0], amax[1]), m1 = fmax_nn(bmax[0], bmax[1]);
        a.anchors[bi * a.hk + hi] = (a.use_anchor && e1 < e0 && m1 <= m0 * 1.125f) ? (int)((int64_t)best * (a.lk - 1) / 8) : -1;
    }
}

// Q: a scale group is the rows g, g+8, .. of a block of 32 rows (16 at head dim 256), a row D/16 lanes of 16 channels each.
// Two runs of lanes share a group's rows at head dims 64 and 128 (one run has them all at 256), so that a lane holds two
// rows and the registers leave room for every workgroup of a usual call to be resident at once (four rows per lane, with
// norm and rope: 158 registers, 37 us at 4608 x 24; two: 100 registers, 22 us).
constexpr int q_runs(int D) { return D == 256 ? 1 : 2; }
constexpr int q_groups_per_wave(int D) { return 64 / lanes_per_row(D) / q_runs(D); }
template <int DT, int D, int NM>
__device__ __forceinline__ void quant_q_body(const AttnArgs& a, const int hi, const int ty, const int bi) {
    constexpr int LPR = lanes_per_row(D), NRUN = q_runs(D), GPW = q_groups_per_wave(D), WQ = q_block_rows(D), NR = WQ / 8 / NRUN;
    const int lane = threadIdx.x & 63, ol = block_of_lane<D>(lane & (LPR - 1)), part = (lane / LPR) % NRUN;
    const int gid = (ty * 4 + (threadIdx.x >> 6)) * GPW + lane / (LPR * NRUN);   // scale group of the head: block * 8 + g
    if (gid >= a.qg * 8) return;
    const int t = gid >> 3, g = gid & 7;
    const int64_t bh = (int64_t)bi * a.h + hi, base = bi * a.q_bs + hi * a.q_hs + ol * 16;
    float v[NR][16];
    const auto true_row = [&](int j) { return t * WQ + g + 8 * (part * NR + j); };
    const auto row_of = [&](int j) { return true_row(j) < a.lq ? true_row(j) : a.lq - 1; };
    load_rows<DT, NR>(a.q, base, a.q_rs, a.in_vec, v, row_of);
    if constexpr (NM != NORM_NONE) {
        if (a.q_norm) norm_rope_rows<NM, NR>(v, ol, a.qw, a.rope, a.eps, a.rope_mode, row_of);
    }
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        rotate_row<D>(v[j], ol, a.rot4);
        if (true_row(j) < a.lq) {
#pragma unroll
            for (int e = 0; e < 16; ++e) mx = fmax_nn(mx, fabsf(v[j][e]));
        }
    }
    mx = max_row<D>(mx);
    if (D == 128) mx = fmax_nn(mx, block_xor8(mx));
    if (D == 64) mx = fmax_nn(mx, block_xor4(mx));   // a lane of the other run: all of them hold its maximum
    const float sc = mx / 127.f + 1e-7f, inv = 1.f / sc;
    if (ol == 0 && part == 0) a.qs[bh * a.qg * 8 + gid] = sc;
#pragma unroll
    for (int j = 0; j < NR; ++j)
        if (true_row(j) < a.lq) *reinterpret_cast<uint4*>(a.qi + (bh * a.lq + true_row(j)) * D + ol * 16) = codes16(v[j], inv);
}

// K: one workgroup of NT threads per tile of CK keys.  A scale group is the keys with (key % 8) / 2 == g; its CK/4 rows
// are shared out over the runs of D/16 lanes that serve the group, whose maxima meet in LDS.  The tile is assembled in
// LDS in fragment order, [32-key block][channel step of 32][half of 16 channels][key][16 bytes] (the 64 lanes of the
// attention kernel read one contiguous KB per load), and leaves as 16-byte stores over its contiguous CK * D bytes;
// keys past lk are zeros.
constexpr int stage2_threads(int CK) { return CK == 128 ? 512 : 256; }
template <int DT, int CK, int D, int NM>
__device__ __forceinline__ void quant_k_body(const AttnArgs& a, const int hi, const int t, const int bi, uint8_t* stage) {
    constexpr int NT = stage2_threads(CK), LPR = lanes_per_row(D), RUNS = NT / LPR, NSUB = RUNS / 4;
    constexpr int R = (CK / 4) / NSUB;   // rows per run
    static_assert(R >= 1 && R * NSUB * 4 == CK, "rows of a group divide over its runs");
    __shared__ float omax[RUNS];
    __shared__ __align__(16) float shift[D];
    const int ol = block_of_lane<D>(threadIdx.x & (LPR - 1)), run = threadIdx.x / LPR, g = run & 3, sub = run >> 2;
    const int64_t bh = (int64_t)bi * a.hk + hi, base = bi * a.k_bs + hi * a.k_hs + ol * 16;
    const int anchor = a.anchors[bh];
    float v[R][16];
    const auto tile_row = [&](int j) { const int i = sub * R + j; return (i / 2) * 8 + g * 2 + (i % 2); };   // i: index within the group
    const auto row_of = [&](int j) {
        const int row = t * CK + tile_row(j);
        return row < a.lk ? row : a.lk - 1;
    };
    load_rows<DT, R>(a.k, base, a.k_rs, a.in_vec, v, row_of);
    // the anchor as the keys are seen: one run of lanes takes it through the norm, the others read it from LDS
    if (anchor >= 0 && run == 0) {
        float x[1][16];
        const auto anchor_row = [&](int) { return anchor; };
        load_rows<DT, 1>(a.k, base, a.k_rs, a.in_vec, x, anchor_row);
        if constexpr (NM != NORM_NONE) {
            if (a.k_norm) norm_rope_rows<NM, 1>(x, ol, a.kw, a.rope, a.eps, a.rope_mode, anchor_row);
        }
#pragma unroll
        for (int e = 0; e < 16; e += 4) *reinterpret_cast<float4*>(shift + ol * 16 + e) = make_float4(x[0][e], x[0][e + 1], x[0][e + 2], x[0][e + 3]);
    }
    if constexpr (NM != NORM_NONE) {
        if (a.k_norm) norm_rope_rows<NM, R>(v, ol, a.kw, a.rope, a.eps, a.rope_mode, row_of);
    }
    __syncthreads();
    float bias[16];
    if (anchor >= 0) {
        load16_f32(shift + ol * 16, bias);
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) bias[e] = 0.f;
    }
    int rt[R];
#pragma unroll
    for (int j = 0; j < R; ++j) rt[j] = tile_row(j);
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[j][e] -= bias[e];
        rotate_row<D>(v[j], ol, a.rot4);
        if (t * CK + rt[j] < a.lk) {
#pragma unroll
            for (int e = 0; e < 16; ++e) mx = fmax_nn(mx, fabsf(v[j][e]));
        }
    }
    mx = max_row<D>(mx);
    if (ol == 0) omax[run] = mx;
    __syncthreads();
    mx = 0.f;
#pragma unroll
    for (int x = 0; x < NSUB; ++x) mx = fmax_nn(mx, omax[x * 4 + g]);
    const float sc = mx / 127.f + 1e-7f, inv = 1.f / sc;
    if (sub == 0 && ol == 0) a.ks[(bh * a.kb + t) * 4 + g] = sc;
#pragma unroll
    for (int j = 0; j < R; ++j) {
        uint4 w = make_uint4(0u, 0u, 0u, 0u);
        if (t * CK + rt[j] < a.lk) w = codes16(v[j], inv);
        *reinterpret_cast<uint4*>(stage + (rt[j] / 32) * (32 * D) + (ol >> 1) * 1024 + (ol & 1) * 512 + (rt[j] % 32) * 16) = w;
    }
    __syncthreads();
    uint4* out = reinterpret_cast<uint4*>(a.ki + (bh * a.nblk + (int64_t)t * (CK / 32)) * (32 * D));
#pragma unroll
    for (int i = 0; i < CK * D / 16 / NT; ++i)
        out[i * NT + threadIdx.x] = *reinterpret_cast<const uint4*>(stage + (i * NT + threadIdx.x) * 16);
}

// V abs-max per channel over a chunk of the keys of one (kv head, batch), eight channels per thread.  The chunks' maxima are
// stored side by side and folded by every workgroup that needs them: 32 chunks at most, which a fold reads in one trip.  (Four channels per
// thread, loads of eight bytes: the launch at 4608 x 24 x 128 with norm and rope 27.9 us, this way 24.6.)
__host__ __device__ constexpr int v_chunks(int lk) { return lk >= 32 * 128 ? 32 : (lk + 127) / 128; }
template <int DT, int D>
__device__ __forceinline__ void v_absmax_body(const AttnArgs& a, const int hi, const int chunk, const int bi) {
    constexpr int TPR = D / 8, RL = 256 / TPR;   // threads per row, rows per pass
    __shared__ float red[RL][D];
    const int c8 = threadIdx.x % TPR, rl = threadIdx.x / TPR, chunks = v_chunks(a.lk);
    const int64_t base = bi * a.v_bs + hi * a.v_hs + c8 * 8;
    float mx[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const int rows = (a.lk + chunks - 1) / chunks, r0 = chunk * rows, r1 = r0 + rows < a.lk ? r0 + rows : a.lk;
    if (a.v_vec == 2) {
        for (int r = r0 + rl; r < r1; r += 4 * RL) {
            uint4 u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)   // rows past the chunk's last are read as that
                u[i] = *reinterpret_cast<const uint4*>((const uint16_t*)a.v + base + (int64_t)(r + i * RL < r1 ? r + i * RL : r1 - 1) * a.v_rs);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t w[4] = {u[i].x, u[i].y, u[i].z, u[i].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float x, y;
                    if (DT == DT_BF16) {
                        x = u2f(w[e] << 16);
                        y = u2f(w[e] & 0xffff0000u);
                    } else {
                        unpack_f16x2(w[e], x, y);
                    }
                    mx[2 * e] = fmax_nn(mx[2 * e], fabsf(x));
                    mx[2 * e + 1] = fmax_nn(mx[2 * e + 1], fabsf(y));
                }
            }
        }
    } else {
        for (int r = r0 + rl; r < r1; r += RL)
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                float x[4];
                ld4_dt<DT>(a.v, base + (int64_t)r * a.v_rs + e, a.v_vec, x);
#pragma unroll
                for (int c = 0; c < 4; ++c) mx[e + c] = fmax_nn(mx[e + c], fabsf(x[c]));
            }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) red[rl][c8 * 8 + c] = mx[c];
    __syncthreads();
    if (threadIdx.x < D) {
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < RL; ++i) m = fmax_nn(m, red[i][threadIdx.x]);
        a.vmax[(((int64_t)bi * a.hk + hi) * chunks + chunk) * D + threadIdx.x] = m;
    }
}

// V codes: a workgroup per key tile (two tiles of 64 keys at head dim 64).  A thread takes eight channels of four keys, so that four codes
// of a channel are a dword of the order vt[(kv head, block of 32 keys)][d][32], where position h*16 + j of a row holds key
// (j/4)*8 + h*4 + j%4 of the block: the order a lane of the attention kernel holds its 16 scores in.  The tile is assembled in LDS
// (eight channels 272 bytes apart: writes of a wave meet in pairs instead of sixteens) and leaves as 16-byte stores.  Keys past lk
// are zeros.  128 x the column sums of a tile go to vsum[(kv head, key tile)][d].  Bound by the chain of loads: the rows are asked for
// ahead of the channels' maxima.  A workgroup per 32 keys with 16 byte reads and two atomics per output row, rows loaded behind the
// maxima, as a launch of its own: 4608 x 24 x 128 13.0 us, this, as a launch of its own, 7.4; 2 x 4096 x 10 x 64 7.8 and 5.5.
constexpr int v_tiles(int CK, int D) { return stage2_threads(CK) * 32 / D > CK ? 2 : 1; }
constexpr int v_stage_bytes(int CK, int D) { return v_tiles(CK, D) * CK / 32 * (D / 8) * 272; }
template <int DT, int CK, int D>
__device__ __forceinline__ void quant_v_body(const AttnArgs& a, const int hi, const int unit, const int bi, uint8_t* stage) {
    constexpr int NT = stage2_threads(CK), CPR = D / 8, GROUP = 272, BLOCK = CPR * GROUP;   // bytes of eight channels, of 32 keys
    constexpr int TILES = v_tiles(CK, D), KEYS = TILES * CK, KPP = NT / CPR * 4, PASSES = KEYS / KPP, PARTS = NT / D;
    static_assert(PASSES * KPP == KEYS && PARTS >= 1 && PARTS * D == NT, "threads divide over keys and channels");
    __shared__ float part_max[PARTS][D];
    __shared__ __align__(16) float inv_s[D];
    __shared__ int sums[TILES][D];
    const int64_t bh = (int64_t)bi * a.hk + hi;
    const int c8 = threadIdx.x % CPR, kg = threadIdx.x / CPR, key0 = unit * KEYS + kg * 4;
    const int64_t base = bi * a.v_bs + hi * a.v_hs + c8 * 8;
    float v[PASSES][4][8];
    const auto row_at = [&](int p, int j) {   // rows past the end read the last one
        const int key = key0 + p * KPP + j;
        return base + (int64_t)(key < a.lk ? key : a.lk - 1) * a.v_rs;
    };
    if (a.v_vec == 2) {
        uint4 u[PASSES][4];
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
#pragma unroll
            for (int j = 0; j < 4; ++j) u[p][j] = *reinterpret_cast<const uint4*>((const uint16_t*)a.v + row_at(p, j));
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t w[4] = {u[p][j].x, u[p][j].y, u[p][j].z, u[p][j].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (DT == DT_BF16) {
                        v[p][j][2 * e] = u2f(w[e] << 16);
                        v[p][j][2 * e + 1] = u2f(w[e] & 0xffff0000u);
                    } else {
                        unpack_f16x2(w[e], v[p][j][2 * e], v[p][j][2 * e + 1]);
                    }
                }
            }
    } else {
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 8; e += 4) {
                    float x[4];
                    ld4_dt<DT>(a.v, row_at(p, j) + e, a.v_vec, x);
#pragma unroll
                    for (int c = 0; c < 4; ++c) v[p][j][e + c] = x[c];
                }
    }
    {
        const int d = threadIdx.x % D, part = threadIdx.x / D, chunks = v_chunks(a.lk);
        const float* src = a.vmax + bh * chunks * D + d;
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < 32 / PARTS; ++i) {   // a chunk twice changes nothing
            const int c = i * PARTS + part;
            m = fmax_nn(m, src[(c < chunks ? c : chunks - 1) * D]);
        }
        part_max[part][d] = m;
        __syncthreads();
        if (threadIdx.x < D) {
            m = 0.f;
#pragma unroll
            for (int i = 0; i < PARTS; ++i) m = fmax_nn(m, part_max[i][d]);
            const float sc = fmax_nn(m * (1.f / 127.f), 1e-12f);
            if (unit == 0) a.vs[bh * D + d] = sc;
            inv_s[d] = 1.f / sc;
#pragma unroll
            for (int i = 0; i < TILES; ++i) sums[i][d] = 0;
        }
    }
    __syncthreads();
    float inv[8];
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
        const float4 f = *reinterpret_cast<const float4*>(inv_s + c8 * 8 + e);
        inv[e] = f.x; inv[e + 1] = f.y; inv[e + 2] = f.z; inv[e + 3] = f.w;
    }
    // Codes as codes16 makes them: |v| <= 127 scales.  Bytes of keys past lk are cleared.
    constexpr float M = 12582912.f;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const int left = a.lk - (key0 + p * KPP), k4 = kg + p * (KPP / 4);
        const uint32_t keep = left >= 4 ? 0xffffffffu : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
        uint8_t* dst = stage + (k4 >> 3) * BLOCK + c8 * GROUP + (k4 & 1) * 16 + ((k4 & 7) >> 1) * 4;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            *reinterpret_cast<uint32_t*>(dst + e * 32) =
                pack_low_bytes(v[p][0][e] * inv[e] + M, v[p][1][e] * inv[e] + M, v[p][2][e] * inv[e] + M, v[p][3][e] * inv[e] + M) & keep;
    }
    __syncthreads();
    uint4* out = reinterpret_cast<uint4*>(a.vt + (bh * a.nblk + (int64_t)unit * (KEYS / 32)) * (32 * D));
#pragma unroll
    for (int i = 0; i < 2 * PASSES; ++i) {
        const int id = i * NT + threadIdx.x, blk = id / (2 * D), d = id / 2 % D;
        const uint4 w = *reinterpret_cast<const uint4*>(stage + blk * BLOCK + (d / 8) * GROUP + (d % 8) * 32 + (id & 1) * 16);
        if (TILES == 1 || unit * TILES + blk / (CK / 32) < a.kb) out[id] = w;
        int sum = 0;
        for (const uint32_t x : {w.x, w.y, w.z, w.w}) sum = __builtin_amdgcn_sdot4((int)x, 0x01010101, sum, false);
        sum += dpp_int<0xB1>(sum);   // the row's other half
        if (!(id & 1)) atomicAdd(&sums[blk / (CK / 32)][d], sum);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < TILES * D; i += NT) {
        const int t = unit * TILES + i / D;
        if (t < a.kb) a.vsum[(bh * a.kb + t) * D + i % D] = 128 * sums[i / D][i % D];
    }
}

// Two launches carry the four bodies above: work that does not depend on each other shares a launch, heads fastest so
// that neighbouring workgroups read neighbouring memory.  Stage 1: anchors, the V maxima and Q.  Stage 2: K (needs the anchors) and V
// (needs the maxima).  Three launches, the maxima beside K and combined by atomics on memory that stage 1 cleared: 4608 x 24 x 128
// with norm and rope 245.3 us a call, this way 236.3; 2 x 4096 x 10 x 64 112.8 and 108.7.
template <int DT, int D, int NM>
__global__ __launch_bounds__(256) void attn_stage1_kernel(AttnArgs a) {
    if (a.parts > 1)   // finished parts, counted by the attention kernel
        for (int i = blockIdx.x * 256 + threadIdx.x; i < (a.lq + 127) / 128 * a.h * a.b - a.whole; i += gridDim.x * 256) a.done[i] = 0u;
    int id = blockIdx.x;
    const int n_anchor = a.hk * a.b;
    if (id < n_anchor) {
        anchor_body<DT, D>(a, id % a.hk, id / a.hk);
        return;
    }
    id -= n_anchor;
    const int chunks = v_chunks(a.lk), n_v = a.hk * chunks * a.b;
    if (id < n_v) {
        v_absmax_body<DT, D>(a, id % a.hk, (id / a.hk) % chunks, id / (a.hk * chunks));
        return;
    }
    id -= n_v;
    constexpr int GPB = 4 * q_groups_per_wave(D);   // scale groups per workgroup
    const int ny = (a.qg * 8 + GPB - 1) / GPB;
    quant_q_body<DT, D, NM>(a, id % a.h, (id / a.h) % ny, id / (a.h * ny));
}

template <int DT, int CK, int D, int NM>
__global__ __launch_bounds__(stage2_threads(CK)) void attn_stage2_kernel(AttnArgs a) {
    __shared__ __align__(16) uint8_t stage[v_stage_bytes(CK, D) > CK * D ? v_stage_bytes(CK, D) : CK * D];
    int id = blockIdx.x;
    const int n_k = a.hk * a.kb * a.b;
    if (id < n_k) {
        quant_k_body<DT, CK, D, NM>(a, id % a.hk, (id / a.hk) % a.kb, id / (a.hk * a.kb), stage);
        return;
    }
    id -= n_k;
    const int units = (a.kb + v_tiles(CK, D) - 1) / v_tiles(CK, D);
    quant_v_body<DT, CK, D>(a, id % a.hk, (id / a.hk) % units, id / (a.hk * units), stage);
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* glb_ptr_t;

// The attention: a workgroup of four waves owns 128 query rows, a wave 32 of them.  The K tile, the V tile and the
// tile's 128 x column sums are contiguous in the workspace, in the order the fragment reads want them, so the four waves
// copy them global -> LDS with DMA loads (no registers) into one of two stages, a tile ahead; one barrier per tile.
// FD (no mask, 64-key tiles): the reference's unfused probability path in every tile, which its build takes for f16
// outputs and at most 512 keys (csrc/vendor/sage/sage_attn_launcher.cu:187-191, qk_int_sv_i8_cuda.cuh:132-139,637-700):
// every tile's maximum starts at a raw score of -50000 and the denominator sums the unrounded probabilities in
// per-thread partials (attn_utils.cuh:922-940).  Without FD only the last tile takes that form.
template <int OUT_DT, int CK, bool MASK = false, bool FD = false, int D = 128>
__global__ __launch_bounds__(256, D == 256 ? 1 : 2) void attn_int8_kernel(AttnArgs a) {
    constexpr int NB = CK / 32, NS = D / 32, KV = CK * D, STAGE = 2 * KV + D * 4, WQ = q_block_rows(D);
    static_assert(!MASK || D == 128, "the key-bias form exists for head dim 128 only");
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, hh = lane >> 5;
    const int hi = blockIdx.y, bi = blockIdx.z;
    const int row0 = blockIdx.x * 128 + wave * 32;
    const int64_t bh = (int64_t)bi * a.h + hi, kvh = (int64_t)bi * a.hk + hi / a.rep;
    // rows past lq are computed on a clamped row and never stored: every wave takes part in the copies and barriers
    const int r = row0 + l32, rc = r < a.lq ? r : a.lq - 1;

    auto fetch = [&](int t) {
        uint8_t* st = smem + (t & 1) * STAGE;
        const int64_t tile = (kvh * a.nblk + (int64_t)t * NB) * (32 * D) + lane * 16;
#pragma unroll
        for (int j = 0; j < KV / 4096; ++j) {
            const int c = wave + 4 * j;
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(a.ki + tile + c * 1024), (lds_ptr_t)(st + c * 1024), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(a.vt + tile + c * 1024), (lds_ptr_t)(st + KV + c * 1024), 16, 0, 0);
        }
        if (wave == 0 && lane < D / 4)
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(a.vsum + (kvh * a.kb + t) * D + lane * 4), (lds_ptr_t)(st + 2 * KV), 16, 0, 0);
    };
    fetch(0);

    v4i qf[NS];
    {
        const int8_t* qrow = a.qi + (bh * a.lq + rc) * D + hh * 16;
#pragma unroll
        for (int s = 0; s < NS; ++s) qf[s] = *reinterpret_cast<const v4i*>(qrow + s * 32);
    }
    const float q_scale = a.qs[(bh * a.qg + r / WQ) * 8 + (r & 7)];

    float ro[NS][16];
#pragma unroll
    for (int x = 0; x < NS; ++x)
#pragma unroll
        for (int i = 0; i < 16; ++i) ro[x][i] = 0.f;
    float m = -50000.f, dsum = 1.f;
    float dsum2 = 0.f;   // the unfused and per-key mask routes keep the reference's four partial denominators per row: two per lane
    bool kept = false;   // that route: some key of this lane was kept
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    // One key tile.  The last tile (the only one that can hold keys past lk) is a separate instantiation, so that the
    // validity compares exist only there.
    auto tile = [&](const int t, auto last_tag) {
        constexpr bool last = decltype(last_tag)::value;
        const uint8_t* st = smem + (t & 1) * STAGE;
        const int key0 = t * CK;
        // Channel steps outside, key blocks inside: consecutive MFMAs write different accumulators, so none waits for
        // the one before it.
        v16i S[NB];
#pragma unroll
        for (int blk = 0; blk < NB; ++blk) S[blk] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int blk = 0; blk < NB; ++blk) {
                const v4i kf = *reinterpret_cast<const v4i*>(st + blk * (32 * D) + s * 1024 + lane * 16);
                S[blk] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[s], S[blk], 0, 0, 0);
            }
        if constexpr (!last) fetch(t + 1);   // the other stage: every wave left it at the barrier that ended the last tile
        const float* ksc = a.ks + (kvh * a.kb + t) * 4 + hh * 2;
        const float gs0 = a.sm * (q_scale * ksc[0]), gs1 = a.sm * (q_scale * ksc[1]);

        // Probabilities: v_cvt_pk_u8_f32 rounds to nearest even, saturates to 0..255 (NaN to 0) and writes one byte of a
        // dword, which is the reference's cvt.rni.sat.u8 plus the packing.  p - 128 as a signed byte is p ^ 0x80.
        v4i pf[NB];
        uint32_t psum = 0;
        float tile_m, o_scale, t_scale;
        auto rescale = [&]() {
            tile_m = fmax_nn(tile_m, __shfl_xor(tile_m, 32));
            const float smaller = __builtin_amdgcn_exp2f(-fabsf(m - tile_m));
            o_scale = m < tile_m ? smaller : 1.f;
            t_scale = tile_m < m ? smaller : 1.f;
            m = fmax_nn(m, tile_m);
        };
        // integer route: exp2(fma(score, group scale, negm)), the unmasked path and a tile with one bias for all its keys
        auto probabilities = [&](auto masked, const float negm) {
#pragma unroll
            for (int blk = 0; blk < NB; ++blk) {
                uint32_t w[4];
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    uint32_t packed = 0u;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        float e = __builtin_amdgcn_exp2f(fmaf((float)S[blk][g4 * 4 + c], c < 2 ? gs0 : gs1, negm));
                        if constexpr (decltype(masked)::value) {
                            const int key = key0 + blk * 32 + g4 * 8 + hh * 4 + c;
                            e = key < a.lk ? e : 0.f;
                        }
                        packed = __builtin_amdgcn_cvt_pk_u8_f32(e, c, packed);
                    }
                    psum = __builtin_amdgcn_sad_u8(packed, 0u, psum);
                    w[g4] = packed ^ 0x80808080u;
                }
                pf[blk] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
                __builtin_amdgcn_sched_barrier(0);   // one block at a time: the converted scores die here
            }
        };
        auto int_maxima = [&](int& i0, int& i1) {
            i0 = i1 = INT_MIN;
#pragma unroll
            for (int blk = 0; blk < NB; ++blk)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    if ((i % 4) < 2) i0 = max(i0, S[blk][i]);
                    else i1 = max(i1, S[blk][i]);
                }
        };
        // float route of the masked forms: scores already carry scale and bias; exp2(score - tile_m)
        float fsc[MASK ? NB : 1][16];
        auto float_probabilities = [&](auto sum_floats) {
#pragma unroll
            for (int blk = 0; blk < NB; ++blk) {
                uint32_t w[4];
                float e[4][4];
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    uint32_t packed = 0u;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        e[g4][c] = __builtin_amdgcn_exp2f(fsc[MASK ? blk : 0][g4 * 4 + c] + (-tile_m));
                        packed = __builtin_amdgcn_cvt_pk_u8_f32(e[g4][c], c, packed);
                    }
                    psum = __builtin_amdgcn_sad_u8(packed, 0u, psum);
                    w[g4] = packed ^ 0x80808080u;
                }
                if constexpr (decltype(sum_floats)::value) {
                    // the reference's thread l of a row owns keys 2l, 2l+1, 8+2l, 9+2l of each 16: this lane carries
                    // threads 2hh (c = 0, 1) and 2hh + 1 (c = 2, 3); a 16-key group is two g4 steps
#pragma unroll
                    for (int fk = 0; fk < 2; ++fk) {
                        dsum += ((e[2 * fk][0] + e[2 * fk][1]) + (e[2 * fk + 1][0] + e[2 * fk + 1][1])) * t_scale;
                        dsum2 += ((e[2 * fk][2] + e[2 * fk][3]) + (e[2 * fk + 1][2] + e[2 * fk + 1][3])) * t_scale;
                    }
                }
                pf[blk] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
                __builtin_amdgcn_sched_barrier(0);
            }
        };

        if constexpr (!MASK && (FD || last)) {
            // The unfused form: every tile with FD, and the last tile always (the reference's last iteration has no fused
            // variant, qk_int_sv_i8_cuda.cuh:956-1000).  Maxima start at a raw score of -50000, keys past lk drop out
            // (-1e30 raw), and the denominator takes the unrounded probabilities, in the two per-thread partials of the
            // reference that this lane carries (threads 2hh: c = 0, 1 and 2hh + 1: c = 2, 3 of each 16 keys).
            int i0 = -50000, i1 = -50000;
#pragma unroll
            for (int blk = 0; blk < NB; ++blk)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    int sv = S[blk][i];
                    if constexpr (last) {
                        const int key = key0 + blk * 32 + (i / 4) * 8 + hh * 4 + (i % 4);
                        sv = key < a.lk ? sv : INT_MIN;
                    }
                    if ((i % 4) < 2) i0 = max(i0, sv);
                    else i1 = max(i1, sv);
                }
            tile_m = fmax_nn(fmaf((float)i0, gs0, -kU8Offset), fmaf((float)i1, gs1, -kU8Offset));
            rescale();
            dsum *= o_scale;
            dsum2 *= o_scale;
#pragma unroll
            for (int blk = 0; blk < NB; ++blk) {
                uint32_t w[4];
                float e[4][4];
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    uint32_t packed = 0u;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        e[g4][c] = __builtin_amdgcn_exp2f(fmaf((float)S[blk][g4 * 4 + c], c < 2 ? gs0 : gs1, -tile_m));
                        if constexpr (last) {
                            const int key = key0 + blk * 32 + g4 * 8 + hh * 4 + c;
                            e[g4][c] = key < a.lk ? e[g4][c] : 0.f;
                        }
                        packed = __builtin_amdgcn_cvt_pk_u8_f32(e[g4][c], c, packed);
                    }
                    w[g4] = packed ^ 0x80808080u;
                }
#pragma unroll
                for (int fk = 0; fk < 2; ++fk) {
                    dsum += ((e[2 * fk][0] + e[2 * fk][1]) + (e[2 * fk + 1][0] + e[2 * fk + 1][1])) * t_scale;
                    dsum2 += ((e[2 * fk][2] + e[2 * fk][3]) + (e[2 * fk + 1][2] + e[2 * fk + 1][3])) * t_scale;
                }
                pf[blk] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
                __builtin_amdgcn_sched_barrier(0);
            }
        } else if constexpr (!MASK) {
            // Group maxima on the integers (exact in fp32: |score| < 2^24).
            int i0, i1;
            int_maxima(i0, i1);
            tile_m = fmax_nn(fmaf((float)i0, gs0, -kU8Offset), fmaf((float)i1, gs1, -kU8Offset));
            rescale();
            dsum *= o_scale;
            probabilities(std::false_type{}, -tile_m);
            dsum += (float)psum * t_scale;
        } else {
            // this lane's prepared biases: four consecutive keys per (blk, g4)
            auto load_bias = [&](float (&bj)[NB][16]) {
#pragma unroll
                for (int blk = 0; blk < NB; ++blk)
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) {
                        const float4 b4 = *reinterpret_cast<const float4*>(a.kbias + key0 + blk * 32 + g4 * 8 + hh * 4);
                        bj[blk][g4 * 4] = b4.x; bj[blk][g4 * 4 + 1] = b4.y; bj[blk][g4 * 4 + 2] = b4.z; bj[blk][g4 * 4 + 3] = b4.w;
                    }
            };
            if constexpr (CK == 64) {
                // per-key mask: scaled score, plus the bias where the key is kept, -50000 elsewhere; the denominator sums
                // the unrounded probabilities in the reference's per-thread partials
                float bj[NB][16];
                load_bias(bj);
                float mx = -50000.f;
#pragma unroll
                for (int blk = 0; blk < NB; ++blk)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const bool keep = bj[blk][i] != -__builtin_inff();   // padding past lk is prepared as -inf too
                        kept = kept || keep;
                        const float rs = (float)S[blk][i] * ((i % 4) < 2 ? gs0 : gs1);
                        fsc[MASK ? blk : 0][i] = keep ? rs + bj[blk][i] : -50000.f;
                        mx = fmax_nn(mx, fsc[MASK ? blk : 0][i]);
                    }
                tile_m = mx - kU8Offset;
                rescale();
                dsum *= o_scale;
                dsum2 *= o_scale;
                float_probabilities(std::true_type{});
            } else {
                const float tb = a.tbias[t];   // uniform: a scalar branch
                if (!last && __builtin_isfinite(tb)) {
                    int i0, i1;
                    int_maxima(i0, i1);
                    tile_m = fmax_nn(fmaf((float)i0, gs0, -kU8Offset) + tb, fmaf((float)i1, gs1, -kU8Offset) + tb);
                    rescale();
                    probabilities(std::false_type{}, tb - tile_m);
                } else {
                    float bj[NB][16];
                    load_bias(bj);
                    float mx = -50000.f;
#pragma unroll
                    for (int blk = 0; blk < NB; ++blk)
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            fsc[MASK ? blk : 0][i] = fmaf((float)S[blk][i], (i % 4) < 2 ? gs0 : gs1, bj[blk][i]);
                            mx = fmax_nn(mx, fsc[MASK ? blk : 0][i]);
                        }
                    tile_m = mx - kU8Offset;
                    rescale();
                    float_probabilities(std::false_type{});
                }
                dsum *= o_scale;
                dsum += (float)psum * t_scale;
            }
        }

        // P.V: the 32-channel blocks of the output keep their own accumulators (the scores are dead by now), key blocks
        // outside, so that consecutive MFMAs are independent here too; four output blocks at a time.
#pragma unroll
        for (int x0 = 0; x0 < NS; x0 += 4) {
            constexpr int NX = NS < 4 ? NS : 4;
            v16i acc[NX];
#pragma unroll
            for (int x = 0; x < NX; ++x) {
                const int* vsp = reinterpret_cast<const int*>(st + 2 * KV) + (x0 + x) * 32 + hh * 4;
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const v4i c4 = *reinterpret_cast<const v4i*>(vsp + g4 * 8);
                    acc[x][g4 * 4 + 0] = c4[0];
                    acc[x][g4 * 4 + 1] = c4[1];
                    acc[x][g4 * 4 + 2] = c4[2];
                    acc[x][g4 * 4 + 3] = c4[3];
                }
            }
#pragma unroll
            for (int blk = 0; blk < NB; ++blk)
#pragma unroll
                for (int x = 0; x < NX; ++x) {
                    const v4i vf = *reinterpret_cast<const v4i*>(st + KV + ((blk * D + (x0 + x) * 32 + l32) * 32 + hh * 16));
                    acc[x] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, pf[blk], acc[x], 0, 0, 0);
                }
#pragma unroll
            for (int x = 0; x < NX; ++x)
#pragma unroll
                for (int i = 0; i < 16; ++i) ro[x0 + x][i] = fmaf((float)acc[x][i], t_scale, ro[x0 + x][i] * o_scale);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's share of the next tile has landed
        __syncthreads();
    };
    for (int t = 0; t + 1 < a.kb; ++t) tile(t, std::false_type{});
    tile(a.kb - 1, std::true_type{});

    dsum += dsum2;   // (d0 + d1) and (d2 + d3) of the reference's four threads
    float dtot = dsum + __shfl_xor(dsum, 32);
    bool row_kept = true;
    if constexpr (MASK && CK == 64) row_kept = (__shfl_xor((int)kept, 32) | (int)kept) != 0;   // a row with no kept key gives zeros
    // `sink` more keys of score zero and value zero: each adds exp2(0 - m) to the denominator, nothing to the output
    if (a.sink != 0.f) dtot = fmaf(a.sink, __builtin_amdgcn_exp2f(-m), dtot);
    const float rcp = 1.f / dtot;
    if (r < a.lq) {
        const int64_t ob = bi * a.o_bs + (int64_t)r * a.o_rs + hi * a.o_hs;
#pragma unroll
        for (int x = 0; x < NS; ++x)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d0 = x * 32 + g4 * 8 + hh * 4;
                const float4 s4 = *reinterpret_cast<const float4*>(a.vs + kvh * D + d0);
                float out[4] = {ro[x][g4 * 4] * rcp * s4.x, ro[x][g4 * 4 + 1] * rcp * s4.y, ro[x][g4 * 4 + 2] * rcp * s4.z,
                                ro[x][g4 * 4 + 3] * rcp * s4.w};
                if constexpr (MASK && CK == 64) {
                    if (!row_kept) out[0] = out[1] = out[2] = out[3] = 0.f;
                }
                if (a.vec_ok) store4<OUT_DT>(a.o, ob + d0, out);
                else
#pragma unroll
                    for (int c = 0; c < 4; ++c) st_dt<OUT_DT>(a.o, ob + d0 + c, out[c]);
            }
    }
}

// One KB global -> LDS, 16 bytes per lane, without registers; the wave's own s_waitcnt vmcnt covers it.
__device__ __forceinline__ void dma16(uint32_t lds_dst, uint32_t lane_off, const void* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_dst), "v"(lane_off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ float swap32_max(float x) {   // maximum of a lane and lane ^ 32
    const auto r = __builtin_amdgcn_permlane32_swap(f2u(x), f2u(x), false, false);
    return fmax_nn(u2f(r[0]), u2f(r[1]));
}
__device__ __forceinline__ float swap32_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(f2u(x), f2u(x), false, false);
    return u2f(r[0]) + u2f(r[1]);
}

// First key tile of part p.  The second of two halves is shorter by two tiles, or by one where their number is odd, so that it has
// mostly written its result when the first one ends, which then keeps its own in registers.
__device__ __forceinline__ int part_bound(int kb, int parts, int p) { return kb * p / parts + (parts == 2 && p == 1 ? 1 : 0); }
// Two floats to and from memory past the caches that XCDs do not share: agent-scope stores are written through and acknowledged where
// every XCD sees them, agent-scope loads are not served from a stale line.  So a part's result needs a wait for its own stores ahead
// of its counter, and no write-back of the whole L2 (a __threadfence per part costs more than the parts gain).
__device__ __forceinline__ void store_agent(float* p, int i, float x, float y) {
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p) + i, (uint64_t)f2u(x) | ((uint64_t)f2u(y) << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 load_agent(const float* p, int i) {
    const uint64_t v = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p) + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float2(u2f((uint32_t)v), u2f((uint32_t)(v >> 32)));
}

// A score is at most 128^3 (head dim 128), a product with V 255 * 128 * 128: both fit sum_value.
__device__ __forceinline__ v16i sum_one() {
    constexpr int z = kSumOne;
    return v16i{z, z, z, z, z, z, z, z, z, z, z, z, z, z, z, z};
}

// The attention without a key bias, head dims 64 and 128: attn_int8_kernel's arithmetic with the work of two tiles overlapped.
// It is bound by vector instruction issue (at 4608 tokens x 24 heads of 128: about 470 per wave and tile beside 32 MFMAs; by the
// counters the vector pipes are busy 73 % of its cycles and the matrix pipes 31 %, at 2 x 4096 x 10 x 64 86 and 18 %).
//   * K runs a tile ahead of V through the two LDS stages: as soon as a key block's probabilities are packed, the next tile's
//     scores go into its registers, one MFMA behind every fourth of the next block's probabilities; the products with V go
//     an output block at a time with the fold of the block before between them.  (All scores, then all probabilities, then
//     all products: the two waves of a SIMD want the same pipe at the same time.)
//   * the DMA instructions of the next tiles go between the probabilities, one behind every four of a lane (all at the start of a
//     tile: 860 us instead of 852 at 2 x 8192 x 16 x 128, 55.4 instead of 53.7 at 2048 x 10 x 128).
//   * the key scales of the next tile are loaded ahead of its DMA.  Loaded where they are used, their wait is a wait for the
//     whole tile that has just been asked for, since the counter runs in order.
//   * numerator and denominator are relative to a base that all but never moves (below), which takes the multiplication
//     of every output by its rescale factor out of every tile.
//   * DMA addresses are scalar, the exchange with lane ^ 32 is a row swap.
//   * the first output block's V fragments and column sums are read under the last probabilities, the others' under the products of the
//     block before; the last key block's scores go between the first block's products; integer sums become floats by a subtraction
//     (sum_value); V lies in LDS a half of its 32 bytes at a time (2-way bank conflicts, a fifth of the LDS cycles, before).
//     Together 4608 x 24 x 128 255.4 -> 250.0 us a call, 2 x 4096 x 10 x 64 117.1 -> 116.4.
//   * SPLIT: the keys of the row blocks that do not fill the CUs once more are shared by several workgroups (key_parts, with the
//     figures): each part has its own base, and the last to finish brings all of them to the largest.
// 250 -> 230 us at that shape by the kernel trace, 141 -> 129 us at SDXL's 2 x 4096 x 10 x 64, before the last of these.  A workgroup of eight waves
// (half the DMA per wave, one workgroup per CU) measured the same for 128 and 30 % slower for 64.
template <int OUT_DT, int CK, int D, bool SPLIT>
__global__ __launch_bounds__(256, 2) void attn_int8_pipe_kernel(AttnArgs a) {
    constexpr int NB = CK / 32, NS = D / 32, KV = CK * D, STAGE = 2 * KV + D * 4;
    static_assert(128 * 128 * D < kSumRoom && 255 * 128 * CK < kSumRoom, "scores and products with V stay within sum_value's range");
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, hh = lane >> 5;
    int hi = blockIdx.y, bi = blockIdx.z, rblk = blockIdx.x;
    int parts = 1, part = 0, t0 = 0, t1 = a.kb;   // the workgroup's key tiles
    if constexpr (SPLIT) {   // the first `whole` row blocks as they are, the others in parts
        if (rblk >= a.whole) {
            parts = a.parts;
            const int i = rblk - a.whole;
            rblk = a.whole + i / parts;
            part = i % parts;
            t0 = part_bound(a.kb, parts, part);
            t1 = part_bound(a.kb, parts, part + 1);
        }
        const int nqb = (a.lq + 127) / 128, head = rblk / nqb;
        bi = head / a.h;
        hi = head - bi * a.h;
        rblk -= head * nqb;
    }
    const int row0 = rblk * 128 + wave * 32;
    const int64_t bh = (int64_t)bi * a.h + hi, kvh = (int64_t)bi * a.hk + hi / a.rep;
    const int r = row0 + l32, rc = r < a.lq ? r : a.lq - 1;   // rows past lq are computed on a clamped row and never stored
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem, lane16 = lane * 16;
    const uint32_t v_lane = l32 * 32 + hh * 16;   // V: a KB of 32 channels, both halves' 16 bytes side by side; in LDS a half at a time
    const int8_t *kt = a.ki + kvh * a.nblk * (32 * D), *vt = a.vt + kvh * a.nblk * (32 * D);
    const int* vst = a.vsum + kvh * a.kb * D;
    // scalar bases and 32-bit lane offsets
    const uint8_t *kst = (const uint8_t*)(a.ks + kvh * a.kb * 4), *vs8 = (const uint8_t*)vst;
    const uint32_t k_lane = hh * 8;
    const auto key_scales = [&](int t) { return *reinterpret_cast<const float2*>(kst + (int64_t)t * 16 + k_lane); };

    // The DMA of a wave's share of K tile tk (j < NF) and V tile tv.  A K tile past the end fetches the last one, into the stage that
    // a tile tk would have: nothing reads that stage any more, while the last tile's own stage is being read.
    constexpr int NF = KV / 4096;
    auto dma = [&](int j, int tk, int tv) {
        const int c = (wave + 4 * (j % NF)) * 1024;
        if (j < NF) dma16(lds0 + (tk & 1) * STAGE + c, lane16, kt + (int64_t)(tk < a.kb ? tk : a.kb - 1) * KV + c);
        else dma16(lds0 + (tv & 1) * STAGE + KV + c, v_lane, vt + (int64_t)tv * KV + c);
    };
    // The column sums go through a register, where they get the bias kSumOne.  Every wave takes 64 of them (at 128 two waves the same
    // ones, at 64 all): no branch in the tile loop.
    const int vcol = (D == 128 ? (wave & 1) * 64 : 0) + lane;
    auto put_sums = [&](int tv, int sum) { reinterpret_cast<int*>(smem + (tv & 1) * STAGE + 2 * KV)[vcol] = sum + kSumOne; };
    const auto get_sums = [&](int tv) { return *reinterpret_cast<const int*>(vs8 + (int64_t)tv * (D * 4) + (uint32_t)(vcol * 4)); };
    const int sum0 = get_sums(t0);
#pragma unroll
    for (int j = 0; j < 2 * NF; ++j) dma(j, t0, t0);
#pragma unroll
    for (int j = 0; j < NF; ++j) dma(j, t0 + 1, 0);

    v4i qf[NS];
    {
        const int8_t* qrow = a.qi + (bh * a.lq + rc) * D + hh * 16;
#pragma unroll
        for (int s = 0; s < NS; ++s) qf[s] = *reinterpret_cast<const v4i*>(qrow + s * 32);
    }
    const float q_scale = a.qs[(bh * a.qg + r / 32) * 8 + (r & 7)];
    float k0 = key_scales(t0).x, k1 = key_scales(t0).y;

    float ro[NS][16];
#pragma unroll
    for (int x = 0; x < NS; ++x)
#pragma unroll
        for (int i = 0; i < 16; ++i) ro[x][i] = 0.f;
    float m = -50000.f, dsum = !SPLIT || part == 0 ? 1.f : 0.f, dsum2 = 0.f;
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
    put_sums(t0, sum0);
    __syncthreads();

    v16i S[NB], one = sum_one();
    if constexpr (D == 64) asm("" : "+v"(one));   // kept in registers: made anew, it is eight instructions of a tile's 280
    auto load_kf = [&](v4i (&kf)[NS], int t, int blk) {
        const uint8_t* st = smem + (t & 1) * STAGE + blk * (32 * D) + lane * 16;
#pragma unroll
        for (int s = 0; s < NS; ++s) kf[s] = *reinterpret_cast<const v4i*>(st + s * 1024);
    };
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
        v4i kf[NS];
        load_kf(kf, t0, blk);
        S[blk] = one;
#pragma unroll
        for (int s = 0; s < NS; ++s) S[blk] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[s], qf[s], S[blk], 0, 0, 0);
    }
    __syncthreads();   // the first K stage may be fetched into

    auto tile = [&](const int t, auto last_tag) {
        constexpr bool last = decltype(last_tag)::value;
        const uint8_t* st = smem + (t & 1) * STAGE;
        const int key0 = t * CK;
        float n0 = 0.f, n1 = 0.f;
        int next_sum = 0;
        if constexpr (!last) {
            const float2 n = key_scales(t + 1);
            n0 = n.x;
            n1 = n.y;
            next_sum = get_sums(t + 1);
        }
        const float gs0 = a.sm * (q_scale * k0), gs1 = a.sm * (q_scale * k1);
        int i0 = last ? kSumOne - 50000 : INT_MIN, i1 = i0;
#pragma unroll
        for (int blk = 0; blk < NB; ++blk)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                int sv = S[blk][i];
                if constexpr (last) {
                    const int key = key0 + blk * 32 + (i / 4) * 8 + hh * 4 + (i % 4);
                    sv = key < a.lk ? sv : INT_MIN;
                }
                if ((i % 4) < 2) i0 = max(i0, sv);
                else i1 = max(i1, sv);
            }
        const float tile_m = swap32_max(fmax_nn(fmaf(sum_value(i0), gs0, -kU8Offset), fmaf(sum_value(i1), gs1, -kU8Offset)));
        // The running base m only moves when a tile's maximum has outgrown it by 2^60 (and at the first tile): numerator and
        // denominator are both relative to it, so any base gives the same quotient, and the outputs need no rescaling here.
        if (__builtin_amdgcn_ballot_w64(tile_m - m > 60.f)) {
            // in two factors (the second is 1 down to 2^-120): what the base lags behind is in the outputs, so that one factor can
            // be below fp32's range where the product is not
            const float step = tile_m > m ? m - tile_m : 0.f, most = fmax_nn(step, -120.f);
            const float f = __builtin_amdgcn_exp2f(most), f2 = __builtin_amdgcn_exp2f(step - most);
            m = fmax_nn(m, tile_m);
            dsum = dsum * f * f2;
            dsum2 = dsum2 * f * f2;
#pragma unroll
            for (int x = 0; x < NS; ++x)
#pragma unroll
                for (int i = 0; i < 16; ++i) ro[x][i] = ro[x][i] * f * f2;
        }
        // a NaN maximum (every key scale of the tile infinite): the tile's probabilities are 0 and its factor 1, so that it drops out
        const float t_scale = tile_m == tile_m ? __builtin_amdgcn_exp2f(tile_m - m) : 1.f;

        v4i pf[NB], vf[2][NB];
        v16i acc[2];
        // the fragments of V for output block x, and the column sums that its products start from
        auto load_vf = [&](int x, int blk) {
            vf[x & 1][blk] = *reinterpret_cast<const v4i*>(st + KV + (blk * D + x * 32) * 32 + lane16);
        };
        auto load_sums = [&](int x) {
            const int* vsp = reinterpret_cast<const int*>(st + 2 * KV) + x * 32 + hh * 4;
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const v4i c4 = *reinterpret_cast<const v4i*>(vsp + g4 * 8);
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[x & 1][g4 * 4 + c] = c4[c];
            }
        };
        uint32_t psum = 0;
#pragma unroll
        for (int rg = 0; rg < NB; ++rg) {
            // region rg: probabilities of key block rg, and under them the next tile's scores into the block before it
            v4i kf[NS];
            if constexpr (!last)
                if (rg > 0) load_kf(kf, t + 1, rg - 1);
            float e[4][4];
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                uint32_t packed = 0u;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    e[g4][c] = __builtin_amdgcn_exp2f(fmaf(sum_value(S[rg][g4 * 4 + c]), c < 2 ? gs0 : gs1, -tile_m));
                    if constexpr (last) {
                        const int key = key0 + rg * 32 + g4 * 8 + hh * 4 + c;
                        e[g4][c] = key < a.lk ? e[g4][c] : 0.f;
                    }
                    packed = __builtin_amdgcn_cvt_pk_u8_f32(e[g4][c], c, packed);
                }
                if constexpr (!last) psum = __builtin_amdgcn_sad_u8(packed, 0u, psum);
                pf[rg][g4] = (int)(packed ^ 0x80808080u);
                if constexpr (!last) {
                    if (rg * 4 + g4 >= 1 && rg * 4 + g4 <= 2 * NF) dma(rg * 4 + g4 - 1, t + 2, t + 1);
                    if (rg > 0 && g4 % (4 / NS) == 0) {
                        const int s = g4 / (4 / NS);
                        if (s == 0) S[rg - 1] = one;
                        S[rg - 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[s], qf[s], S[rg - 1], 0, 0, 0);
                    }
                }
                if (rg == NB - 1) {   // what the products begin with
                    if (g4 == 1) load_sums(0);
                    if (g4 >= 2)
#pragma unroll
                        for (int blk = (g4 - 2) * NB / 2; blk < (g4 - 1) * NB / 2; ++blk) load_vf(0, blk);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (last) {   // the unrounded probabilities, in the reference's per-thread partials
#pragma unroll
                for (int fk = 0; fk < 2; ++fk) {
                    dsum += ((e[2 * fk][0] + e[2 * fk][1]) + (e[2 * fk + 1][0] + e[2 * fk + 1][1])) * t_scale;
                    dsum2 += ((e[2 * fk][2] + e[2 * fk][3]) + (e[2 * fk + 1][2] + e[2 * fk + 1][3])) * t_scale;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (!last) dsum = fmaf((float)psum, t_scale, dsum);

        // P.V, an output block at a time; the fold of a block rides between the products of the next, the fragments of the block after
        // that are read under them, and the last key block's scores go between the first block's products
        v4i kf[NS];
        if constexpr (!last) load_kf(kf, t + 1, NB - 1);
        if constexpr (!last) S[NB - 1] = one;
#pragma unroll
        for (int x = 0; x <= NS; ++x) {
#pragma unroll
            for (int blk = 0; blk < NB; ++blk) {
                if (x < NS) acc[x & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf[x & 1][blk], pf[blk], acc[x & 1], 0, 0, 0);
                if constexpr (!last)
                    if (x == 0)
#pragma unroll
                        for (int s = blk * NS / NB; s < (blk + 1) * NS / NB; ++s)
                            S[NB - 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[s], qf[s], S[NB - 1], 0, 0, 0);
                if (x > 0) {
#pragma unroll
                    for (int i = blk * (16 / NB); i < (blk + 1) * (16 / NB); ++i)
                        ro[x > 0 ? x - 1 : 0][i] = fmaf(sum_value(acc[(x + 1) & 1][i]), t_scale, ro[x > 0 ? x - 1 : 0][i]);
                }
                if (x + 1 < NS) {
                    load_vf(x + 1, blk);
                    if (blk == NB - 1) load_sums(x + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (!last) {
            k0 = n0;
            k1 = n1;
            __builtin_amdgcn_s_waitcnt(0x0f70);   // this wave's share of the next tiles has landed
            put_sums(t + 1, next_sum);
            __syncthreads();
        }
    };
    if constexpr (SPLIT) {
        // a part that ends before the last keys also multiplies the K tile behind it, which saves a third form of the tile
        for (int t = t0; t < t1 && t + 1 < a.kb; ++t) tile(t, std::false_type{});
        if (t1 == a.kb) tile(t1 - 1, std::true_type{});
    } else {
        for (int t = 0; t + 1 < a.kb; ++t) tile(t, std::false_type{});
        tile(a.kb - 1, std::true_type{});
    }

    float dtot = swap32_sum(dsum + dsum2);
    if (SPLIT && parts > 1) {
        // whoever finishes last of a row block's parts adds all of them, each rescaled to the largest base
        constexpr int SLOT = 64 * (NS * 16 + 2);
        const int64_t rb = bh * ((a.lq + 127) / 128) + rblk - a.whole;
        float* slots = a.part + (rb * parts * 4 + wave) * SLOT;
        uint32_t* done = a.done + rb;
        int* verdict = reinterpret_cast<int*>(smem);
        __syncthreads();   // the stages are read
        if (threadIdx.x == 0) *verdict = (int)__hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
        __syncthreads();
        bool mine = *verdict != 0;
        if (!mine) {
            float* w = slots + part * (4 * SLOT);
#pragma unroll
            for (int x = 0; x < NS; ++x)
#pragma unroll
                for (int i = 0; i < 8; ++i) store_agent(w, (x * 8 + i) * 64 + lane, ro[x][2 * i], ro[x][2 * i + 1]);
            store_agent(w, NS * 8 * 64 + lane, m, dtot);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the stores are where every XCD sees them
            __syncthreads();
            if (threadIdx.x == 0) *verdict = (int)__hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == parts - 1;
            __syncthreads();
            mine = *verdict != 0;
        }
        if (!mine) return;
        // in the order of the parts, whoever merges: the same bits in every call
        const auto head = [&](int v) { return v == part ? make_float2(m, dtot) : load_agent(slots + v * (4 * SLOT), NS * 8 * 64 + lane); };
        float base = m, d = 0.f, sum[NS][16];
        for (int v = 0; v < parts; ++v) base = fmax_nn(base, head(v).x);
#pragma unroll
        for (int x = 0; x < NS; ++x)
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[x][i] = 0.f;
        for (int v = 0; v < parts; ++v) {
            const float2 md = head(v);
            const float f = __builtin_amdgcn_exp2f(md.x - base);
            d = fmaf(md.y, f, d);
            const float* w = slots + v * (4 * SLOT);
#pragma unroll
            for (int x = 0; x < NS; ++x)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float2 o = v == part ? make_float2(ro[x][2 * i], ro[x][2 * i + 1]) : load_agent(w, (x * 8 + i) * 64 + lane);
                    sum[x][2 * i] = fmaf(o.x, f, sum[x][2 * i]);
                    sum[x][2 * i + 1] = fmaf(o.y, f, sum[x][2 * i + 1]);
                }
        }
        m = base;
        dtot = d;
#pragma unroll
        for (int x = 0; x < NS; ++x)
#pragma unroll
            for (int i = 0; i < 16; ++i) ro[x][i] = sum[x][i];
    }
    // `sink` more keys of score zero and value zero: each adds exp2(0 - m) to the denominator, nothing to the output.  The base can
    // be 60 below the largest score, which would take that out of fp32's range where the score's own distance from zero does not.
    if (a.sink != 0.f) {
        if (m < -64.f) {
            const float f = __builtin_amdgcn_exp2f(m + 64.f);
            m = -64.f;
            dtot *= f;
#pragma unroll
            for (int x = 0; x < NS; ++x)
#pragma unroll
                for (int i = 0; i < 16; ++i) ro[x][i] *= f;
        }
        dtot = fmaf(a.sink, __builtin_amdgcn_exp2f(-m), dtot);
    }
    const float rcp = 1.f / dtot;
    if (r < a.lq) {
        const int64_t ob = bi * a.o_bs + (int64_t)r * a.o_rs + hi * a.o_hs;
#pragma unroll
        for (int x = 0; x < NS; ++x)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d0 = x * 32 + g4 * 8 + hh * 4;
                const float4 s4 = *reinterpret_cast<const float4*>(a.vs + kvh * D + d0);
                float out[4] = {ro[x][g4 * 4] * rcp * s4.x, ro[x][g4 * 4 + 1] * rcp * s4.y, ro[x][g4 * 4 + 2] * rcp * s4.z,
                                ro[x][g4 * 4 + 3] * rcp * s4.w};
                if (a.vec_ok) store4<OUT_DT>(a.o, ob + d0, out);
                else
#pragma unroll
                    for (int c = 0; c < 4; ++c) st_dt<OUT_DT>(a.o, ob + d0 + c, out[c]);
            }
    }
}

int cta_k_for(int lk, int d) { return lk > 1024 && d != 64 ? 128 : 64; }   // csrc/attn_int8.cu:56

// The caller's per-key bias, prepared once per call (csrc/vendor/sage/sage_attn_launcher.cu:343-391; attn_utils.cuh:
// 466-515 for the per-key form): bias * log2e per key of every tile, -inf where the bias is not finite and for the
// padding past lk; for 128-key tiles also the value all keys of a tile share (times log2e), NaN when they differ.
template <int CK>
__global__ __launch_bounds__(CK) void attn_key_bias_kernel(const float* bias, int lk, float* kbias, float* tbias) {
    __shared__ float lo_s[CK / 64], hi_s[CK / 64];
    const int tid = threadIdx.x, key = blockIdx.x * CK + tid;
    float raw = key < lk ? bias[key] : -__builtin_inff();
    if (!__builtin_isfinite(raw)) raw = -__builtin_inff();
    kbias[key] = raw * 1.44269504088896340736f;
    if constexpr (CK == 128) {
        float lo = raw, hi = raw;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            lo = fminf(lo, __shfl_xor(lo, o));
            hi = fmaxf(hi, __shfl_xor(hi, o));
        }
        if ((tid & 63) == 0) { lo_s[tid >> 6] = lo; hi_s[tid >> 6] = hi; }
        __syncthreads();
        if (tid == 0) {
            lo = fminf(lo_s[0], lo_s[1]);
            hi = fmaxf(hi_s[0], hi_s[1]);
            tbias[blockIdx.x] = lo == hi ? hi * 1.44269504088896340736f : __builtin_nanf("");
        }
    }
}

struct Plan {
    int64_t qi, ki, qs, ks, vt, vs, anchors, vmax, vsum, done, part, whole, total;
    int ck, kb, qg, nblk, parts;
};

// What `parts` workgroups per row block of the tail take off a call, in us: the key tiles that a CU has less to go through, minus a fixed
// cost, one per part and one for the CUs that write parts at the same time.  Fitted to 1300 calls of 256 to 5000 keys against the same
// calls unshared, within about 1 us; of 800 others 77 took more than 3 % longer shared by the relative costs of key_parts alone, with
// this 3.  It leaves few keys unshared where those see a gain: 2 x 492 x 9 x 128 31.8 us unshared and 37.0 in halves, 516 x 20 x 128 35.0
// and 38.4, 602 x 19 x 64 27.0 and 28.8.  1849 queries, 877 keys x 2 x 128 stay in thirds (36.6 and 33.5), 2 x 300 queries, 1859 keys x
// 15 x 64 in fifths (51.9 and 45.4).
double parts_gain_us(int64_t tail, int64_t kb, int ck, int D, bool lone, int parts) {
    struct Cost { double tile, fixed, part, busy; };
    static constexpr Cost c[3][2] = {{{1.06, -0.3, 2.2, 4.0}, {0.77, 2.35, 0.47, 0.54}},    // head dim 64; [1]: behind whole row blocks
                                     {{1.75, -2.4, 4.85, 5.5}, {1.4, 0.4, 2.8, 1.7}},       // 128 with tiles of 64 keys
                                     {{1.66, 0.83, 1.73, 3.1}, {1.34, -2.0, 1.32, 5.0}}};   // and of 128
    const Cost& k = c[D == 64 ? 0 : ck == 64 ? 1 : 2][lone ? 0 : 1];
    const double busy = (double)(tail * parts) / 256.;
    const int n = (int)((tail * parts + 255) / 256);   // parts of the busiest CU
    // their time, of a part that has a CU for itself: two at once 1.6 to 1.7; of head dim 128 only two fit, and a third gains nothing
    const double time = !lone ? n : n == 1 ? 1. : D == 64 ? n - 0.43 : n == 2 ? 1.7 : n + 1.;
    return k.tile * (double)kb * (1. - time / parts) - (k.fixed + k.part * parts + k.busy * (lone && busy > 1. ? 1. : busy));
}

// How the pipelined kernel's row blocks (128 rows of a head) go to the CUs.  What is left over a multiple of the CUs keeps some of them
// busy for a whole row block's time, 55 us at 4608 keys, while the others idle; the keys of those row blocks are shared by P
// workgroups each.  P is what leaves a CU the least, in row blocks: ceil(tail * P / CUs) parts of 1 / P each (a part alone on a CU
// takes 1.3 times as long: 125 us for a row block of 8192 keys, 196 for two at once), plus about 3 us per part for writing and
// merging it, which is 2 to 5 key tiles; and parts_gain_us has to see a gain.  Calls in us, P = 1 and chosen: 4608 tokens x 24 heads 256 -> 231 (96 of 864 row blocks in
// halves; in fifths 240), 2 x 4096 x 10 x 64 138 -> 115 (128 of 640 in halves), 2500 x 20 x 64 75 -> 64 (thirds; halves 71), 2048 x
// 10 56 -> 52 (thirds; halves 55), 1024 x 10 45 -> 40.  Splitting every row block of the first costs 263: 57 MB of parts.
// Fewer than 8 row blocks stay whole: which keys are summed together then depends on nothing but the key tiles.  From 8 on it depends on
// the number of row blocks, so a row's last bits can change with the batch and the head count (its error does not).
int key_parts(int64_t row_blocks, int64_t kb, int ck, int D, int64_t& whole) {
    constexpr int64_t CUS = 256;   // not the present device's: the workspace's size and the call have to agree
    whole = row_blocks;
    const int64_t tail = row_blocks % CUS;
    if (D == 256 || row_blocks < 8 || tail == 0) return 1;
    const bool lone = row_blocks < CUS;
    const double merge = (D == 64 ? 5.0 : ck == 64 ? 4.0 : 2.0) / (double)kb;
    double least = (lone ? 1.3 : 1.0) - 0.05;
    int best = 1;
    for (int p = 2; p <= 8 && kb / p >= 4; ++p) {
        const double n = (double)((tail * p + CUS - 1) / CUS), cost = (lone && n == 1 ? 1.3 : n) / p + n * merge;
        if (cost < least) { least = cost - 0.05; best = p; }
    }
    if (best == 1 || parts_gain_us(tail, kb, ck, D, lone, best) < 0.15) return 1;
    whole = row_blocks - tail;
    return best;
}

Plan plan_for(int64_t b, int64_t h, int64_t hk, int64_t lq, int64_t lk, int D) {
    Plan p;
    p.ck = cta_k_for((int)lk, D);
    p.kb = (int)((lk + p.ck - 1) / p.ck);
    p.qg = (int)((lq + 127) / 128 * (128 / q_block_rows(D)));   // row blocks of the Q quantizer, eight scale groups each
    p.nblk = p.kb * (p.ck / 32);
    int64_t n = 0;
    auto add = [&](int64_t bytes) { const int64_t at = n; n += (bytes + 255) / 256 * 256; return at; };
    p.qi = add(b * h * lq * D);
    p.ki = add(b * hk * (int64_t)p.nblk * 32 * D);
    p.qs = add(b * h * p.qg * 8 * 4);
    p.ks = add(b * hk * p.kb * 4 * 4);
    p.vt = add(b * hk * (int64_t)p.nblk * D * 32);
    p.vs = add(b * hk * D * 4);
    p.anchors = add(b * hk * 4);
    p.vmax = add(b * hk * v_chunks((int)lk) * D * 4);
    p.vsum = add(b * hk * (int64_t)p.kb * D * 4);
    const int64_t row_blocks = b * h * ((lq + 127) / 128);
    p.parts = key_parts(row_blocks, p.kb, p.ck, D, p.whole);
    p.done = add((row_blocks - p.whole) * 4);
    p.part = add((row_blocks - p.whole) * p.parts * 4 * 64 * (D / 2 + 2) * 4);
    p.total = n;
    return p;
}

template <auto KERN>
int launch_tiles(const AttnArgs& a, dim3 grid, int lds, hipStream_t st) {
    if (lds > 64 * 1024) {   // has to be allowed once per kernel and device
        static PerDeviceOnce once;
        if (allow_dynamic_lds(reinterpret_cast<const void*>(KERN), lds, once) != 0) return -401;
    }
    KERN<<<grid, 256, lds, st>>>(a);
    return hipGetLastError() == hipSuccess ? 0 : -401;
}
template <int DT, int CK, bool MASK, bool FD, int D>
int launch_attn(const AttnArgs& a, hipStream_t st) {
    return launch_tiles<attn_int8_kernel<DT, CK, MASK, FD, D>>(a, dim3((a.lq + 127) / 128, a.h, a.b), 2 * (2 * CK * D + D * 4), st);
}
template <int DT, int CK, int D>
int launch_pipe(const AttnArgs& a, hipStream_t st) {
    if (a.parts > 1) return launch_tiles<attn_int8_pipe_kernel<DT, CK, D, true>>(a, dim3((unsigned)(a.whole + ((int64_t)((a.lq + 127) / 128) * a.h * a.b - a.whole) * a.parts)), 2 * (2 * CK * D + D * 4), st);
    return launch_tiles<attn_int8_pipe_kernel<DT, CK, D, false>>(a, dim3((a.lq + 127) / 128, a.h, a.b), 2 * (2 * CK * D + D * 4), st);
}

template <int DT, int D>
int run(AttnArgs a, hipStream_t st) {
    constexpr int GPB = 4 * q_groups_per_wave(D);   // scale groups per workgroup of the Q quantizer
    const int tiles = v_tiles(a.ck, D);
    const int64_t n1 = (int64_t)a.hk * a.b * (1 + v_chunks(a.lk)) + (int64_t)a.h * ((a.qg * 8 + GPB - 1) / GPB) * a.b;
    const int64_t n2 = (int64_t)a.hk * a.b * (a.kb + (a.kb + tiles - 1) / tiles);
    if (n1 > 0x7fffffff || n2 > 0x7fffffff) return -400;
    const auto stages = [&](auto nm) {
        constexpr int NM = decltype(nm)::value;
        attn_stage1_kernel<DT, D, NM><<<dim3((unsigned)n1), 256, 0, st>>>(a);
        if (a.ck == 64) attn_stage2_kernel<DT, 64, D, NM><<<dim3((unsigned)n2), stage2_threads(64), 0, st>>>(a);
        else if constexpr (D != 64) attn_stage2_kernel<DT, 128, D, NM><<<dim3((unsigned)n2), stage2_threads(128), 0, st>>>(a);
    };
    if constexpr (D == 128 && DT == DT_BF16) {   // the only form with a norm
        if (!a.q_norm && !a.k_norm) stages(std::integral_constant<int, NORM_NONE>{});
        else if (a.nr_vec && a.rope_mode != 2) stages(std::integral_constant<int, NORM_PAIRS>{});
        else stages(std::integral_constant<int, NORM_ANY>{});
    } else {
        stages(std::integral_constant<int, NORM_NONE>{});
    }
    if (hipGetLastError() != hipSuccess) return -401;
    if constexpr (D == 128) {
        if (a.bias) {
            if (a.ck == 64) {
                attn_key_bias_kernel<64><<<dim3(a.kb), 64, 0, st>>>(a.bias, a.lk, a.kbias, a.tbias);
                return launch_attn<DT, 64, true, false, D>(a, st);
            }
            attn_key_bias_kernel<128><<<dim3(a.kb), 128, 0, st>>>(a.bias, a.lk, a.kbias, a.tbias);
            return launch_attn<DT, 128, true, false, D>(a, st);
        }
    }
    // f16 outputs with at most 512 keys: the reference's build takes its unfused probability path in every tile
    if (DT == DT_F16 && a.lk <= 512 && a.ck == 64) return launch_attn<DT_F16, 64, false, true, D>(a, st);
    if constexpr (D != 256) {
        if (a.ck == 64) return launch_pipe<DT, 64, D>(a, st);
        if constexpr (D != 64) return launch_pipe<DT, 128, D>(a, st);
    } else {
        if (a.ck == 64) return launch_attn<DT, 64, false, false, D>(a, st);
        return launch_attn<DT, 128, false, false, D>(a, st);
    }
    return -400;
}

// Per-head RMSNorm and RoPE for q and k, applied on the way into the quantizer (csrc/attn_int8.cu:69-76).  A null kw
// takes K as it is (csrc/vendor/sage/quant_qk_int8.cu:1264-1268).
struct QkNorm {
    const float* qw;
    const float* kw;
    const float* rope;
    float eps;
    int rope_mode;
};

int int8_attn(const void* q, const void* k, const void* v, void* o, void* ws, int b, int lq, int lk, int h, int hk, int Dh,
              int64_t q_bs, int64_t q_rs, int64_t q_hs, int64_t k_bs, int64_t k_rs, int64_t k_hs, int64_t v_bs, int64_t v_rs,
              int64_t v_hs, int64_t o_bs, int64_t o_rs, int64_t o_hs, float scale, int dt, void* stream, float sink = 0.f,
              const QkNorm* norm = nullptr, const float* bias = nullptr) {
    const char* why = nullptr;
    if (Dh != 64 && Dh != 128 && Dh != 256) why = "head dim must be 64, 128 or 256";
    else if ((norm || bias) && (dt != DT_BF16 || Dh != 128)) why = "fused q/k norm and key bias need bf16 head dim 128";   // csrc/attn_int8.cu:135
    else if (norm && (norm->rope_mode < 0 || norm->rope_mode > 2)) why = "rope_mode must be 0, 1 or 2";   // quant_qk_int8.cu:1279
    else if (!q || !k || !v || !o || !ws) why = "null pointer";
    else if (b <= 0 || lq <= 0 || lk <= 0 || h <= 0 || hk <= 0 || h % hk != 0) why = "bad sizes";
    else if (b > 65535 || h > 65535 || lq > (1 << 20) || lk > (1 << 20)) why = "batch, head count or length beyond the grid limits";
    else if (((uintptr_t)ws & 255) != 0) why = "workspace must be 256-byte aligned";
    if (why) {
        fprintf(stderr, "int8 attention: %s\n", why);
        return -400;
    }
    const Plan p = plan_for(b, h, hk, lq, lk, Dh);
    char* w = (char*)ws;
    AttnArgs a;
    a.q = q; a.k = k; a.v = v; a.o = o;
    a.qi = (int8_t*)(w + p.qi); a.ki = (int8_t*)(w + p.ki); a.vt = (int8_t*)(w + p.vt);
    a.qs = (float*)(w + p.qs); a.ks = (float*)(w + p.ks); a.vs = (float*)(w + p.vs);
    a.anchors = (int*)(w + p.anchors); a.vmax = (float*)(w + p.vmax); a.vsum = (int*)(w + p.vsum);
    a.b = b; a.lq = lq; a.lk = lk; a.h = h; a.hk = hk; a.rep = h / hk;
    a.parts = p.parts; a.whole = (int)p.whole; a.done = (uint32_t*)(w + p.done); a.part = (float*)(w + p.part);
    a.qg = p.qg; a.kb = p.kb; a.ck = p.ck; a.nblk = p.nblk;
    a.q_bs = q_bs; a.q_rs = q_rs; a.q_hs = q_hs; a.k_bs = k_bs; a.k_rs = k_rs; a.k_hs = k_hs;
    a.v_bs = v_bs; a.v_rs = v_rs; a.v_hs = v_hs; a.o_bs = o_bs; a.o_rs = o_rs; a.o_hs = o_hs;
    a.sm = scale * 1.44269504088896340736f;
    a.rot4 = lk <= 256 ? 1 : 0;
    a.sink = sink;
    a.use_anchor = sink == 0.f ? 1 : 0;   // with a sink a zero key's score must stay zero: no shift (csrc/attn_int8.cu:134-141)
    a.vec_ok = ((o_bs | o_rs | o_hs) % 4 == 0 && ((uintptr_t)o & 7) == 0) ? 1 : 0;
    const auto vec_of = [](int64_t strides, uintptr_t base) { return strides % 8 == 0 && (base & 15) == 0 ? 2 : strides % 4 == 0 && (base & 7) == 0 ? 1 : 0; };
    a.v_vec = vec_of(v_bs | v_rs | v_hs, (uintptr_t)v);
    a.in_vec = vec_of(q_bs | q_rs | q_hs | k_bs | k_rs | k_hs, (uintptr_t)q | (uintptr_t)k);
    a.bias = bias;
    a.kbias = (float*)(w + p.total);   // the key-bias form's workspace is this much longer
    a.tbias = a.kbias + (int64_t)p.kb * p.ck;
    a.qw = a.kw = a.rope = nullptr;
    a.eps = 0.f;
    a.q_norm = a.k_norm = a.rope_mode = 0;
    if (norm) {
        a.qw = norm->qw;
        a.kw = norm->kw;
        a.rope = (norm->rope && norm->rope_mode != 0) ? norm->rope : nullptr;
        a.eps = norm->eps;
        a.rope_mode = norm->rope_mode;
        a.q_norm = 1;
        a.k_norm = norm->kw ? 1 : 0;
    }
    a.nr_vec = (((uintptr_t)a.qw | (uintptr_t)a.kw | (uintptr_t)a.rope) & 15) == 0 ? 1 : 0;
    hipStream_t st = (hipStream_t)stream;
    if (Dh == 64) return dt == DT_F16 ? run<DT_F16, 64>(a, st) : run<DT_BF16, 64>(a, st);
    if (Dh == 256) return dt == DT_F16 ? run<DT_F16, 256>(a, st) : run<DT_BF16, 256>(a, st);
    return dt == DT_F16 ? run<DT_F16, 128>(a, st) : run<DT_BF16, 128>(a, st);
}

}  // namespace

GPU_API int64_t gpu_int8_attn_workspace_d(int b, int h, int hk, int lq, int lk, int head_dim) {
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return 0;
    if (b <= 0 || h <= 0 || hk <= 0 || lq <= 0 || lk <= 0) return 0;
    return plan_for(b, h, hk, lq, lk, head_dim).total;
}

GPU_API int64_t gpu_int8_attn_workspace(int b, int h, int hk, int lq, int lk) {
    return gpu_int8_attn_workspace_d(b, h, hk, lq, lk, 128);
}

GPU_API int gpu_int8_attn_d(const void* q, const void* k, const void* v, void* o, void* ws, int b, int lq, int lk, int h,
                            int hk, int head_dim, int64_t q_bs, int64_t q_rs, int64_t q_hs, int64_t k_bs, int64_t k_rs,
                            int64_t k_hs, int64_t v_bs, int64_t v_rs, int64_t v_hs, int64_t o_bs, int64_t o_rs, int64_t o_hs,
                            float scale, void* stream) {
    return int8_attn(q, k, v, o, ws, b, lq, lk, h, hk, head_dim, q_bs, q_rs, q_hs, k_bs, k_rs, k_hs, v_bs, v_rs, v_hs, o_bs,
                     o_rs, o_hs, scale, DT_BF16, stream);
}

GPU_API int gpu_int8_attn_f16(const void* q, const void* k, const void* v, void* o, void* ws, int b, int lq, int lk, int h,
                              int hk, int head_dim, int64_t q_bs, int64_t q_rs, int64_t q_hs, int64_t k_bs, int64_t k_rs,
                              int64_t k_hs, int64_t v_bs, int64_t v_rs, int64_t v_hs, int64_t o_bs, int64_t o_rs,
                              int64_t o_hs, float scale, void* stream) {
    return int8_attn(q, k, v, o, ws, b, lq, lk, h, hk, head_dim, q_bs, q_rs, q_hs, k_bs, k_rs, k_hs, v_bs, v_rs, v_hs, o_bs,
                     o_rs, o_hs, scale, DT_F16, stream);
}

GPU_API int gpu_int8_attn(const void* q, const void* k, const void* v, void* o, void* ws, int b, int lq, int lk, int h,
                          int hk, int64_t q_bs, int64_t q_rs, int64_t q_hs, int64_t k_bs, int64_t k_rs, int64_t k_hs,
                          int64_t v_bs, int64_t v_rs, int64_t v_hs, int64_t o_bs, int64_t o_rs, int64_t o_hs, float scale,
                          void* stream) {
    return int8_attn(q, k, v, o, ws, b, lq, lk, h, hk, 128, q_bs, q_rs, q_hs, k_bs, k_rs, k_hs, v_bs, v_rs, v_hs, o_bs, o_rs,
                     o_hs, scale, DT_BF16, stream);
}

GPU_API int gpu_int8_attn_sink(const void* q, const void* k, const void* v, void* o, void* ws, int b, int lq, int lk, int h,
                               int hk, int64_t q_bs, int64_t q_rs, int64_t q_hs, int64_t k_bs, int64_t k_rs, int64_t k_hs,
                               int64_t v_bs, int64_t v_rs, int64_t v_hs, int64_t o_bs, int64_t o_rs, int64_t o_hs, float scale,
                               float sink, const float* qw, float eps, void* stream) {
    const QkNorm norm{qw, nullptr, nullptr, eps, 0};   // a non-null qw normalizes q; k is taken as it is (csrc/attn_int8.cu:198-201)
    return int8_attn(q, k, v, o, ws, b, lq, lk, h, hk, 128, q_bs, q_rs, q_hs, k_bs, k_rs, k_hs, v_bs, v_rs, v_hs, o_bs, o_rs,
                     o_hs, scale, DT_BF16, stream, sink, qw ? &norm : nullptr);
}

// gpu_int8_attn with q and k taken through the per-head RMSNorm, weight and RoPE of gpu_qk_norm_rope first, inside the
// quantizers; q and k in memory are left as they are (csrc/attn_int8.cu:163-174).  Head dim 128, bf16.
GPU_API int gpu_int8_attn_norm_rope(const void* q, const void* k, const void* v, void* o, void* ws, int b, int lq, int lk,
                                    int h, int hk, int64_t q_bs, int64_t q_rs, int64_t q_hs, int64_t k_bs, int64_t k_rs,
                                    int64_t k_hs, int64_t v_bs, int64_t v_rs, int64_t v_hs, int64_t o_bs, int64_t o_rs,
                                    int64_t o_hs, float scale, const float* qw, const float* kw, float eps,
                                    const float* rope, int rope_mode, void* stream) {
    const QkNorm norm{qw, kw, rope, eps, rope_mode};
    return int8_attn(q, k, v, o, ws, b, lq, lk, h, hk, 128, q_bs, q_rs, q_hs, k_bs, k_rs, k_hs, v_bs, v_rs, v_hs, o_bs, o_rs,
                     o_hs, scale, DT_BF16, stream, 0.f, &norm);
}

// sage's prepared key mask row for lk keys: each key's bias, then one value per 128-key tile (csrc/attn_int8.cu:178-182).
// The layout kept here (bias * log2e per key of every tile, then one value per 128-key tile) fits the same size.
static int64_t key_mask_width(int lk) {
    const int64_t tiles = (lk + 127) / 128;
    return (tiles * 129 + 3) / 4 * 4;
}

GPU_API int64_t gpu_int8_attn_key_bias_workspace(int b, int h, int hk, int lq, int lk) {
    if (b <= 0 || h <= 0 || hk <= 0 || lq <= 0 || lk <= 0) return 0;
    return gpu_int8_attn_workspace_d(b, h, hk, lq, lk, 128) + (key_mask_width(lk) * 4 + 255) / 256 * 256;
}

// gpu_int8_attn with bias (f32 [lk], the same for every batch item, query and head) added to each key's logits, as an
// additive attention mask; a bias that is not finite masks its key (csrc/attn_int8.cu:184-223).  bf16.
GPU_API int gpu_int8_attn_key_bias(const void* q, const void* k, const void* v, void* o, void* ws, int b, int lq, int lk, int h,
                                   int hk, int64_t q_bs, int64_t q_rs, int64_t q_hs, int64_t k_bs, int64_t k_rs, int64_t k_hs,
                                   int64_t v_bs, int64_t v_rs, int64_t v_hs, int64_t o_bs, int64_t o_rs, int64_t o_hs, float scale,
                                   const float* bias, void* stream) {
    if (!bias) {
        fprintf(stderr, "int8 attention: null key bias\n");
        return -400;
    }
    return int8_attn(q, k, v, o, ws, b, lq, lk, h, hk, 128, q_bs, q_rs, q_hs, k_bs, k_rs, k_hs, v_bs, v_rs, v_hs, o_bs, o_rs,
                     o_hs, scale, DT_BF16, stream, 0.f, nullptr, bias);
}

// Test hook: y[i] = v_cvt_pk_u8_f32(x[i]) into byte 0 of zero, so that a test can hold the instruction to
// round-to-nearest-even with saturation, which the probabilities rely on.
namespace {
__global__ void cvt_pk_u8_probe_kernel(const float* x, uint32_t* y, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = __builtin_amdgcn_cvt_pk_u8_f32(x[i], 0, 0u);
}
}  // namespace
GPU_API int gpu_internal_cvt_pk_u8_probe(const float* x, uint32_t* y, int n, void* stream) {
    if (!x || !y || n <= 0) return -400;
    cvt_pk_u8_probe_kernel<<<dim3((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(x, y, n);
    return hipGetLastError() == hipSuccess ? 0 : -401;
}

// Test hook: the sum of squares of rows of 128 floats as the fused norm takes it (eight lanes per row, sumsq128) and as
// the anchor search takes it (one thread, sumsq128_serial).  out[2 * row] and out[2 * row + 1]; rows a multiple of 8.
namespace {
__global__ void __launch_bounds__(64) sumsq_probe_kernel(const float* x, float* out, int split) {
    const int lane = threadIdx.x, o8 = block_of_lane<128>(lane & 7), row = blockIdx.x * 8 + (lane >> 3);
    float v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = x[row * 128 + o8 * 16 + e];
    const float ss = sumsq128(v, o8, split != 0);
    if (o8 == (row & 7)) out[2 * row] = ss;          // any of the eight lanes holds it: take a different one per row
    if (o8 == 0) out[2 * row + 1] = sumsq128_serial(x + row * 128, split != 0);
}
}  // namespace
GPU_API int gpu_internal_attn_sumsq_probe(const float* x, float* out, int rows, int split, void* stream) {
    if (!x || !out || rows <= 0 || rows % 8) return -400;
    sumsq_probe_kernel<<<dim3(rows / 8), 64, 0, (hipStream_t)stream>>>(x, out, split);
    return hipGetLastError() == hipSuccess ? 0 : -401;
}

// Test hook: where the pieces of the workspace lie (byte offsets), and the tiling.  out[0..9] = qi, ki, qs, ks, vt, vs,
// anchors, vsum, key tile length, key tiles.
GPU_API int gpu_internal_attn_layout_d(int b, int h, int hk, int lq, int lk, int head_dim, int64_t* out) {
    if (b <= 0 || h <= 0 || hk <= 0 || lq <= 0 || lk <= 0 || !out || (head_dim != 64 && head_dim != 128 && head_dim != 256)) return -400;
    const Plan p = plan_for(b, h, hk, lq, lk, head_dim);
    const int64_t v[10] = {p.qi, p.ki, p.qs, p.ks, p.vt, p.vs, p.anchors, p.vsum, p.ck, p.kb};
    for (int i = 0; i < 10; ++i) out[i] = v[i];
    return 0;
}
GPU_API int gpu_internal_attn_layout(int b, int h, int hk, int lq, int lk, int64_t* out) {
    return gpu_internal_attn_layout_d(b, h, hk, lq, lk, 128, out);
}
