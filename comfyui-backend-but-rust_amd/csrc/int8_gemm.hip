// int8 x int8 -> int32 GEMM on gfx950 MFMA with the dequant epilogue fused, D = Out(acc * xs[m] * ws[n] + bias[n]).
//
// Semantics follow the reference's fused CUTLASS kernel (csrc/vendor/cutlass_gemm_int8.cu:84-95 plain epilogue,
// :149-161 residual epilogue, :348-388 argument handling); the design is for CDNA4: A[M,K] and W[N,K] are both
// K-contiguous, which is exactly the operand shape of v_mfma_i32_32x32x32_i8 (each lane feeds 16 consecutive K bytes of
// one row), so tiles go global -> LDS as 16-byte chunks with an XOR swizzle and come back as ds_read_b128 fragments.
// W rides in src0 and A in src1, which leaves every lane holding runs of four consecutive n for one m: the epilogue
// stores 8-byte (bf16/f16) or 16-byte (f32) vectors straight from the accumulators.
#include <atomic>
#include <cstdio>

#include "common.hpp"
#include "kept_buffers.hpp"

// Nothing is scheduled across this point: it pins hand-interleaved instruction orders and keeps live ranges short.
#define SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

namespace {

__device__ __forceinline__ void store16_untracked(void* ptr, uint4 v);
__device__ __forceinline__ void store16_untracked_at(const void* base, uint32_t off, uint4 v);
__device__ __forceinline__ void store16_through_at(const void* base, uint32_t off, uint4 v);
__device__ __forceinline__ void store16_cached_at(const void* base, uint32_t off, uint4 v);
// A 64-bit value that is the same in every lane, moved to scalar registers.
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

enum { EPI_PLAIN = 0, EPI_RESID = 1, EPI_ACC = 2 };

// How whole wave tiles are stored: as the compiler does it; or by stores that it does not count, past the caches, through the L2, by the
// caches' default policy.  A kernel of its own for each: a choice in the store loop costs scalar registers, up to 1.8 % of a short call.
enum { STORE_TRACKED = -1, STORE_PAST, STORE_THROUGH, STORE_CACHED };
struct GemmArgs {
    const int8_t* A;
    const int8_t* W;
    const float* xs;
    const float* ws;
    const void* bias;
    const void* rscale;
    const void* resid;
    void* D;
    int M, N, K;
    int tiles_m, tiles_n;
    uint32_t magic;   // panel_magic(tiles_m, tiles_n), for tile_of_block
    int kslice;   // K of a split-K slice (a multiple of 128), 0 = no split
    int n_first;  // two-group kernel: the first column of these tiles
};

template <int BM_, int BN_, int BK_, int WGM_, int WGN_, int OCC_>
struct Cfg {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, WGM = WGM_, WGN = WGN_, OCC = OCC_;
    static constexpr int NT = 64 * WGM * WGN;
    static constexpr int WTM = BM / WGM, WTN = BN / WGN;   // wave tile
    static constexpr int TM = WTM / 32, TN = WTN / 32;     // 32x32 MFMA tiles per wave
    static constexpr int CPR = BK / 16;                    // 16-byte chunks per tile row
    static constexpr int A_CHUNKS = BM * CPR / NT, W_CHUNKS = BN * CPR / NT;
    static constexpr int STAGE = (BM + BN) * BK;           // bytes per LDS stage
    static constexpr int SMEM = 2 * STAGE;
    static_assert(BM % (32 * WGM) == 0 && BN % (32 * WGN) == 0, "wave tile must be a multiple of 32x32");
    static_assert((BM * CPR) % NT == 0 && (BN * CPR) % NT == 0, "chunks must divide over the threads");
    static_assert(BK == 64 || BK == 128, "swizzle is written for 64- and 128-byte rows");
};

// Chunk swizzle.  The LDS of gfx950 has 64 banks of 4 bytes, and a ds_read_b128 is served 16 lanes (256 bytes) at a
// time: a fragment read takes 16 consecutive rows at one chunk column, so those 16 rows must land on 16 distinct
// 16-byte bank groups.  Rows are BK bytes apart: with 128-byte rows an even/odd row pair already covers the two halves
// of the bank space, so the chunk index is XORed with bits 1..3 of the row; with 64-byte rows four rows span the banks
// and bits 2..3 are used.  (Measured: XOR with the low row bits instead costs 25 % of the read bandwidth.)
// The lane number from the execution mask counters: two instructions, and no register held across a loop for it.
__device__ __forceinline__ int hw_lane() {
    int l = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(l));
    return l;
}

template <int BK> __device__ __forceinline__ int swz(int row, int chunk) {
    return BK == 64 ? (chunk ^ ((row >> 2) & 3)) : (chunk ^ ((row >> 1) & 7));
}

// The epilogue arithmetic for one value.  t0 = float(acc)*xs; then fma(t0, ws, bias): the reference composes a
// multiply node and an add node (csrc/vendor/cutlass_gemm_int8.cu:90-93) that its compiler is free to contract; this
// kernel always contracts, and likewise for z*rscale + resid (:156-159).
template <int OUT_DT, int EPI>
__device__ __forceinline__ float epi_value(int acc, float xs, float ws, float b, float rs, float res) {
    const float t = __builtin_fmaf((float)acc * xs, ws, b);
    if (EPI == EPI_RESID) return __builtin_fmaf(rnd_dt<OUT_DT>(t), rs, res);
    return t;
}

// Epilogue of one wave tile whose origin is (mb, nb).  acc[in][im][4*rb + j] is the accumulator of
// (m = mb + 32*im + lane%32, n = nb + 32*in + 8*rb + 4*(lane/32) + j): four consecutive n per lane and register group.
template <int TM, int TN, int OUT_DT, int EPI>
__device__ __forceinline__ void epilogue_store(const GemmArgs& p, v16i (&acc)[TN][TM], int mb, int nb, int lane, bool vec_ok) {
    const int frow = lane & 31, fhalf = lane >> 5;
#pragma unroll
    for (int im = 0; im < TM; ++im) {
        const int m = mb + im * 32 + frow;
        if (m >= p.M) continue;
        const float xs = EPI == EPI_ACC ? 0.f : p.xs[m];
#pragma unroll
        for (int in = 0; in < TN; ++in) {
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                const int n = nb + in * 32 + rb * 8 + fhalf * 4;
                if (n >= p.N) continue;
                const int64_t o = (int64_t)m * p.N + n;
                if (EPI == EPI_ACC) {
                    int* d = (int*)p.D + o;
                    if (vec_ok) {
                        *reinterpret_cast<v4i*>(d) = v4i{acc[in][im][4 * rb], acc[in][im][4 * rb + 1], acc[in][im][4 * rb + 2], acc[in][im][4 * rb + 3]};
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j) if (n + j < p.N) d[j] = acc[in][im][4 * rb + j];
                    }
                    continue;
                }
                float ws[4], b[4] = {0.f, 0.f, 0.f, 0.f}, rs[4] = {0.f, 0.f, 0.f, 0.f}, res[4] = {0.f, 0.f, 0.f, 0.f}, out[4];
                if (vec_ok) {
                    const float4 w4 = *reinterpret_cast<const float4*>(p.ws + n);
                    ws[0] = w4.x; ws[1] = w4.y; ws[2] = w4.z; ws[3] = w4.w;
                    if (p.bias) load4<OUT_DT>(p.bias, n, b);
                    if (EPI == EPI_RESID) { load4<OUT_DT>(p.rscale, n, rs); load4<OUT_DT>(p.resid, o, res); }
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (n + j >= p.N) { ws[j] = 0.f; continue; }
                        ws[j] = p.ws[n + j];
                        if (p.bias) b[j] = ld_dt<OUT_DT>(p.bias, n + j);
                        if (EPI == EPI_RESID) { rs[j] = ld_dt<OUT_DT>(p.rscale, n + j); res[j] = ld_dt<OUT_DT>(p.resid, o + j); }
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) out[j] = epi_value<OUT_DT, EPI>(acc[in][im][4 * rb + j], xs, ws[j], b[j], rs[j], res[j]);
                if (vec_ok) {
                    store4<OUT_DT>(p.D, o, out);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) if (n + j < p.N) st_dt<OUT_DT>(p.D, o + j, out[j]);
                }
            }
        }
    }
}

// The constants of a wave tile's epilogue in a lane's registers: column scales and raw bias words of its runs of four columns, row
// scales.  (runs: per 32 columns; halves: per 32 rows; see L at epilogue_shuffle)
template <int TM, int TN, int OUT_DT, int EPI, int L>
struct EpiConst {
    static constexpr int SZ = (EPI == EPI_ACC || OUT_DT == DT_F32) ? 4 : 2, BW = SZ == 4 ? 4 : 2;   // 32-bit words holding 4 bias values
    static constexpr int NRB = L == 32 ? 4 : 2, NHM = L == 32 ? 1 : 2;
    float wsr[TN][NRB][4];
    uint32_t braw[TN][NRB][BW];
    float xsr[TM][NHM];
    // In one batch, no branches between the loads, so a single wait covers them.  Columns past N read the last valid vector.
    __device__ __forceinline__ void load_columns(const GemmArgs& p, int nb, int lane) {
        const int fhalf = lane / L;
#pragma unroll
        for (int in = 0; in < TN; ++in)
#pragma unroll
            for (int rb = 0; rb < NRB; ++rb) {
                int n = nb + in * 32 + (L == 32 ? rb * 8 : rb * 16) + fhalf * 4;
                n = n < p.N ? n : p.N - 4;
                const float4 w4 = *reinterpret_cast<const float4*>(p.ws + n);
                wsr[in][rb][0] = w4.x; wsr[in][rb][1] = w4.y; wsr[in][rb][2] = w4.z; wsr[in][rb][3] = w4.w;
                if (p.bias) {
                    if (SZ == 4) {
                        const uint4 b4 = *reinterpret_cast<const uint4*>((const uint8_t*)p.bias + (int64_t)n * 4);
                        braw[in][rb][0] = b4.x; braw[in][rb][1] = b4.y; braw[in][rb][BW - 2] = b4.z; braw[in][rb][BW - 1] = b4.w;
                    } else {
                        const uint2 b2 = *reinterpret_cast<const uint2*>((const uint8_t*)p.bias + (int64_t)n * 2);
                        braw[in][rb][0] = b2.x; braw[in][rb][1] = b2.y;
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < BW; ++j) braw[in][rb][j] = 0u;
                }
            }
    }
    __device__ __forceinline__ void load_rows(const GemmArgs& p, int mb, int lane) {
#pragma unroll
        for (int im = 0; im < TM; ++im)
#pragma unroll
            for (int hm = 0; hm < NHM; ++hm) {
                const int mrow = mb + im * 32 + hm * 16 + (lane & (L - 1));
                xsr[im][hm] = (EPI == EPI_ACC || mrow >= p.M) ? 0.f : p.xs[mrow];
            }
    }
};

// Coalesced epilogue: the accumulator layout (lane = one m, four consecutive n per register group) would store 16-byte
// pieces scattered over 32 rows per instruction.  Instead each wave rounds its values to the output type, passes a
// 32-row piece of its tile through a private LDS region (XOR-swizzled 16-byte chunks, conflict-free both ways) and
// writes whole rows: 16 bytes per lane, consecutive lanes on consecutive addresses.  For the residual form the LDS
// holds z = Out(acc*xs*ws + bias), exactly the intermediate the reference rounds, and fma(z, rscale, resid) is applied
// on the way out.  Needs row starts of D (and resid) 16-byte aligned; the caller falls back to epilogue_store otherwise.
// L: the MFMA shape the accumulators come from.  32: v16i acc[TN][TM], a lane holds row lane % 32 of a 32x32 tile and
// the columns 8*rb + 4*(lane / 32) + j.  16: v4i acc[2*TN][2*TM] of 16x16 tiles, a lane holds row lane % 16 and the
// columns 4*(lane / 16) + j; the 32x32 block (in, im) is then the four tiles (2*in + rb, 2*im + hm).
// EARLY: the constants are in `own` already; else they are loaded here.
template <int TM, int TN, int OUT_DT, int EPI, int PW, int STORE, int L, bool EARLY, class Acc>
__device__ __forceinline__ void epilogue_shuffle_with(const GemmArgs& p, Acc& acc, int mb, int nb, int lane, uint8_t* wl, uint8_t* wl2,
                                                      EpiConst<TM, TN, OUT_DT, EPI, L>& own) {
    // a piece is 32 rows x PW columns of the wave tile: PW*SZ bytes per LDS row, 32*PW*SZ bytes per wave
    constexpr int SZ = (EPI == EPI_ACC || OUT_DT == DT_F32) ? 4 : 2;
    constexpr int WTN = TN * 32, NP = WTN / PW, TNP = PW / 32;
    constexpr int ROWB = PW * SZ, CPRW = ROWB / 16, MASK = CPRW - 1;
    constexpr int EPC = 16 / SZ;                  // elements per 16-byte chunk
    constexpr int RPI = 64 / CPRW, PASSES = 32 / RPI;
    static_assert(PW % 32 == 0 && WTN % PW == 0, "piece width");
    static_assert((CPRW & MASK) == 0 && CPRW <= 64 && CPRW >= 2, "chunks per row must be a power of two");
    // Everything below is a function of the lane number only, so in a persistent kernel the compiler would hoist dozens
    // of addresses out of the tile loop, keep them live across the K loop and spill them; the reloads then sit between
    // the stores, each behind a full memory wait.  Making the lane number opaque here keeps the address arithmetic local.
    asm volatile("" : "+v"(lane));
    constexpr int NRB = L == 32 ? 4 : 2, NHM = L == 32 ? 1 : 2;   // column runs per 32 columns, row halves per 32 rows
    const int frow = lane & (L - 1), fhalf = lane / L;            // row inside a tile; which four of every 8 (16) columns
    // first column of run rb inside a 32-column block; value j of run rb of block (in, im), row half hm
    auto run_col = [&](int rb) { return L == 32 ? rb * 8 + fhalf * 4 : rb * 16 + fhalf * 4; };
    auto val = [&](int in, int im, int rb, int hm, int j) -> int {
        if constexpr (L == 32) return acc[in][im][4 * rb + j];
        else return acc[2 * in + rb][2 * im + hm][j];
    };

    if (EPI != EPI_ACC && !EARLY) own.load_columns(p, nb, lane);
    const auto& wsr = own.wsr;
    const auto& braw = own.braw;
    // bias value j of (in, rb) as float: +0.0 for a null bias
    auto bias_f = [&](int in, int rb, int j) -> float {
        if (SZ == 4) return u2f(braw[in][rb][j]);
        const uint32_t w = braw[in][rb][j >> 1];
        if (OUT_DT == DT_BF16) return (j & 1) ? u2f(w & 0xffff0000u) : u2f(w << 16);
        return f16_to_f((uint16_t)((j & 1) ? (w >> 16) : (w & 0xffffu)));
    };
    const int rrow = lane / CPRW, rc = lane % CPRW;   // read phase: row within a pass, chunk
    // uniform per wave: the wave tile is wholly inside the matrix; where it starts; bytes per output row
    const bool full = __builtin_amdgcn_readfirstlane((int)(mb + TM * 32 <= p.M && nb + WTN <= p.N && p.N < (1 << 21))) != 0;
    const uint64_t row_bytes = (uint64_t)p.N * SZ;
    const uint64_t tile_base = uniform64((uint64_t)(uintptr_t)p.D + ((uint64_t)mb * p.N + nb) * SZ);
    const uint32_t lane_off = __umul24((uint32_t)rrow, (uint32_t)row_bytes) + (uint32_t)(rc * 16);   // both factors < 2^24 when `full`

    // Every global load is issued ahead of the stores that precede its use: the memory counter retires in order, so a
    // load issued after a store cannot be waited for without also waiting for that store to reach memory.
    auto& xsr = own.xsr;
    if (!EARLY) own.load_rows(p, mb, lane);
    float rs[NP][EPC];
    if (EPI == EPI_RESID) {
#pragma unroll
        for (int np = 0; np < NP; ++np) {
            const int ncol = nb + np * PW + rc * EPC;
#pragma unroll
            for (int h = 0; h < EPC / 4; ++h) {
                if (ncol < p.N) load4<OUT_DT>(p.rscale, ncol + 4 * h, rs[np] + 4 * h);
                else { rs[np][4 * h] = 0.f; rs[np][4 * h + 1] = 0.f; rs[np][4 * h + 2] = 0.f; rs[np][4 * h + 3] = 0.f; }
            }
        }
    }
    // residual rows of piece (im, np), in the read phase's layout
    auto load_resid = [&](int im, int np, uint4* rv) {
        const int ncol = nb + np * PW + rc * EPC;
#pragma unroll
        for (int t = 0; t < PASSES; ++t) {
            const int m = mb + im * 32 + t * RPI + rrow;
            if (m < p.M && ncol < p.N) rv[t] = *reinterpret_cast<const uint4*>((const uint8_t*)p.resid + ((int64_t)m * p.N + ncol) * SZ);
            else rv[t] = make_uint4(0, 0, 0, 0);
        }
    };

    // write phase of piece (im, np): this lane's rows of the piece into `buf`
    auto write_piece = [&](int im, int np, uint8_t* buf) {
#pragma unroll
        for (int hm = 0; hm < NHM; ++hm) {
            const float xs = xsr[im][hm];
            const int prow = hm * 16 + frow;   // row inside the 32-row piece
#pragma unroll
            for (int ip = 0; ip < TNP; ++ip)
#pragma unroll
                for (int rb = 0; rb < NRB; ++rb) {
                    const int in = np * TNP + ip;
                    const int byte = (ip * 32 + run_col(rb)) * SZ;
                    uint8_t* dst = buf + prow * ROWB + ((((byte >> 4) ^ prow) & MASK) << 4) + (byte & 15);
                    if (EPI == EPI_ACC) {
                        *reinterpret_cast<v4i*>(dst) = v4i{val(in, im, rb, hm, 0), val(in, im, rb, hm, 1), val(in, im, rb, hm, 2), val(in, im, rb, hm, 3)};
                    } else {
                        float o[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) o[j] = __builtin_fmaf((float)val(in, im, rb, hm, j) * xs, wsr[in][rb][j], bias_f(in, rb, j));
                        if (OUT_DT == DT_F32) {
                            *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
                        } else if (OUT_DT == DT_BF16) {
                            *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
                        } else {
                            *reinterpret_cast<uint2*>(dst) = make_uint2(pack_f16x2(o[0], o[1]), pack_f16x2(o[2], o[3]));
                        }
                    }
                }
        }
    };
    // read phase, first half: the piece's rows back from `buf`, 16 bytes per lane and pass, all passes in one batch
    auto read_piece = [&](const uint8_t* buf, uint4* v) {
#pragma unroll
        for (int t = 0; t < PASSES; ++t) {
            const int r = t * RPI + rrow;
            v[t] = *reinterpret_cast<const uint4*>(buf + r * ROWB + (((rc ^ r) & MASK) << 4));
        }
    };
    // read phase, second half: whole rows out.  A wave tile that lies wholly inside the matrix stores through one
    // scalar base per pass plus a 32-bit lane offset: no per-pass compares, branches or 64-bit vector address arithmetic
    // (a fifth of the vector instructions of an epilogue that is bound by them).
    auto finish = [&](int np, const uint4& z, const uint4& r) -> uint4 {
        if (EPI != EPI_RESID) return z;
        const uint32_t zw[4] = {z.x, z.y, z.z, z.w}, rw[4] = {r.x, r.y, r.z, r.w};
        uint32_t ow[4];
        if (OUT_DT == DT_F32) {
#pragma unroll
            for (int j = 0; j < 4; ++j) ow[j] = f2u(__builtin_fmaf(u2f(zw[j]), rs[np][j], u2f(rw[j])));
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float z0, z1, r0, r1;
                if (OUT_DT == DT_BF16) {
                    z0 = u2f(zw[j] << 16); z1 = u2f(zw[j] & 0xffff0000u); r0 = u2f(rw[j] << 16); r1 = u2f(rw[j] & 0xffff0000u);
                    ow[j] = pack_bf16x2(__builtin_fmaf(z0, rs[np][2 * j], r0), __builtin_fmaf(z1, rs[np][2 * j + 1], r1));
                } else {
                    unpack_f16x2(zw[j], z0, z1);
                    unpack_f16x2(rw[j], r0, r1);
                    ow[j] = pack_f16x2(__builtin_fmaf(z0, rs[np][2 * j], r0), __builtin_fmaf(z1, rs[np][2 * j + 1], r1));
                }
            }
        }
        return make_uint4(ow[0], ow[1], ow[2], ow[3]);
    };
    auto store_piece = [&](int im, int np, const uint4* v, const uint4* rv) {
        if (full) {
            const uint64_t piece = tile_base + (uint64_t)(im * 32) * row_bytes + (uint64_t)(np * PW * SZ);
#pragma unroll
            for (int t = 0; t < PASSES; ++t) {
                const uint64_t pass = piece + (uint64_t)(t * RPI) * row_bytes;
                const uint4 o = finish(np, v[t], rv[t]);
                if (STORE == STORE_TRACKED) *reinterpret_cast<uint4*>((uint8_t*)pass + lane_off) = o;
                else if (STORE == STORE_THROUGH) store16_through_at((const void*)pass, lane_off, o);
                else if (STORE == STORE_CACHED) store16_cached_at((const void*)pass, lane_off, o);
                else store16_untracked_at((const void*)pass, lane_off, o);
            }
            return;
        }
        int l = lane;
        asm volatile("" : "+v"(l));   // keeps this path's address arithmetic from being hoisted in front of the branch
        const int row = l / CPRW, ncol = nb + np * PW + (l % CPRW) * EPC;
        uint8_t* base = (uint8_t*)p.D + ((int64_t)(mb + im * 32 + row) * p.N + ncol) * SZ;
        const int64_t step = (int64_t)RPI * p.N * SZ;
#pragma unroll
        for (int t = 0; t < PASSES; ++t) {
            const int m = mb + im * 32 + t * RPI + row;
            if (m >= p.M || ncol >= p.N) continue;
            uint8_t* out = base + t * step;
            const uint4 o = finish(np, v[t], rv[t]);
            if (STORE != STORE_TRACKED) store16_untracked(out, o);
            else *reinterpret_cast<uint4*>(out) = o;
        }
    };

    // Pieces go through the LDS one after the other.  With a second region (wl2) the loop is software-pipelined: the
    // LDS reads of piece i are issued, then the arithmetic and LDS writes of piece i+1 (into the other region) cover
    // their latency, then piece i is stored.  The LDS queue runs one wave's accesses in program order, so a piece's
    // reads see its writes, and a region is rewritten only after the reads of its previous piece have returned (they
    // are waited for by the stores in between).  The residual rows of a piece are requested before its write phase.
    constexpr int NPIECE = TM * NP;
    uint8_t* bufs[2] = {wl, wl2 ? wl2 : wl};
    uint4 rv[2][PASSES];
    if (EPI == EPI_RESID) load_resid(0, 0, rv[0]);
    write_piece(0, 0, bufs[0]);
#pragma unroll
    for (int i = 0; i < NPIECE; ++i) {
        const int im = i / NP, np = i % NP;
        uint4 v[PASSES];
        asm volatile("" ::: "memory");
        read_piece(bufs[i & 1], v);
        asm volatile("" ::: "memory");
        if (wl2 && i + 1 < NPIECE) {
            if (EPI == EPI_RESID) load_resid((i + 1) / NP, (i + 1) % NP, rv[(i + 1) & 1]);
            write_piece((i + 1) / NP, (i + 1) % NP, bufs[(i + 1) & 1]);
        }
        store_piece(im, np, v, rv[i & 1]);
        if (!wl2 && i + 1 < NPIECE) {
            if (EPI == EPI_RESID) load_resid((i + 1) / NP, (i + 1) % NP, rv[(i + 1) & 1]);
            asm volatile("" ::: "memory");
            write_piece((i + 1) / NP, (i + 1) % NP, bufs[0]);
        }
    }
    asm volatile("" ::: "memory");
}
template <int TM, int TN, int OUT_DT, int EPI, int PW = TN * 32, int STORE = STORE_TRACKED, int L = 32, class Acc>
__device__ __forceinline__ void epilogue_shuffle(const GemmArgs& p, Acc& acc, int mb, int nb, int lane, uint8_t* wl) {
    EpiConst<TM, TN, OUT_DT, EPI, L> own;
    epilogue_shuffle_with<TM, TN, OUT_DT, EPI, PW, STORE, L, false>(p, acc, mb, nb, lane, wl, nullptr, own);
}

// Chooses the coalesced epilogue when row starts are 16-byte aligned.  Must be called by all waves of the workgroup:
// it begins with a workgroup barrier because the shuffle reuses the LDS of the K loop.
template <int OUT_DT, int EPI>
__host__ __device__ __forceinline__ void epilogue_alignment(const GemmArgs& p, bool& vec_ok, bool& aligned) {
    constexpr int SZ = (EPI == EPI_ACC || OUT_DT == DT_F32) ? 4 : 2;
    constexpr uintptr_t V4 = 4 * SZ - 1;   // mask of a 4-element vector of the output type
    const uintptr_t ptrs = EPI == EPI_ACC ? (uintptr_t)p.D
                                          : ((uintptr_t)p.D | (uintptr_t)p.bias | (uintptr_t)p.rscale | (uintptr_t)p.resid);
    vec_ok = (p.N & 3) == 0 && (ptrs & V4) == 0 && (EPI == EPI_ACC || (((uintptr_t)p.ws) & 15) == 0);
    aligned = vec_ok && (((int64_t)p.N * SZ) & 15) == 0 &&
              (((uintptr_t)p.D | (uintptr_t)p.resid | (uintptr_t)p.rscale) & 15) == 0;
}

template <int TM, int TN, int OUT_DT, int EPI>
__device__ __forceinline__ void epilogue(const GemmArgs& p, v16i (&acc)[TN][TM], int mb, int nb, int lane, int wave, uint8_t* smem) {
    constexpr int SZ = (EPI == EPI_ACC || OUT_DT == DT_F32) ? 4 : 2;
    constexpr int PIECE = 32 * TN * 32 * SZ;   // bytes of one wave's 32-row piece
    bool vec_ok, aligned;
    epilogue_alignment<OUT_DT, EPI>(p, vec_ok, aligned);
    if (aligned) {
        __syncthreads();
        epilogue_shuffle<TM, TN, OUT_DT, EPI>(p, acc, mb, nb, lane, smem + wave * PIECE);
    } else {
        epilogue_store<TM, TN, OUT_DT, EPI>(p, acc, mb, nb, lane, vec_ok);
    }
}

template <class C, int OUT_DT, int EPI>
__global__ void __launch_bounds__(C::NT, C::OCC) int8_gemm_kernel(GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int BM = C::BM, BN = C::BN, BK = C::BK, NT = C::NT, CPR = C::CPR;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / C::WGN, wn = wave % C::WGN;

    int tm, tn;
    tile_of_block(blockIdx.x, gridDim.x, p.tiles_m, p.tiles_n, tm, tn, p.magic);
    const int m0 = tm * BM, n0 = tn * BN;
    const int K = p.K;

    // per-thread global sources (rows clamped into range: out-of-range rows compute garbage that is never stored)
    const int8_t* ga[C::A_CHUNKS];
    const int8_t* gw[C::W_CHUNKS];
    int la[C::A_CHUNKS], lw[C::W_CHUNKS], ka[C::A_CHUNKS], kw[C::W_CHUNKS];
#pragma unroll
    for (int i = 0; i < C::A_CHUNKS; ++i) {
        const int c = tid + i * NT, row = c / CPR, kc = c % CPR;
        const int gr = m0 + row < p.M ? m0 + row : p.M - 1;
        ga[i] = p.A + (int64_t)gr * K + kc * 16;
        ka[i] = kc * 16;
        la[i] = row * BK + (swz<BK>(row, kc) << 4);
    }
#pragma unroll
    for (int i = 0; i < C::W_CHUNKS; ++i) {
        const int c = tid + i * NT, row = c / CPR, kc = c % CPR;
        const int gr = n0 + row < p.N ? n0 + row : p.N - 1;
        gw[i] = p.W + (int64_t)gr * K + kc * 16;
        kw[i] = kc * 16;
        lw[i] = BM * BK + row * BK + (swz<BK>(row, kc) << 4);
    }

    v16i acc[C::TN][C::TM];
#pragma unroll
    for (int in = 0; in < C::TN; ++in)
#pragma unroll
        for (int im = 0; im < C::TM; ++im)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[in][im][r] = 0;

    const int nk = (K + BK - 1) / BK;
    v4i ra[C::A_CHUNKS], rw[C::W_CHUNKS];

    // Only the last K tile can be partial (K % 16 == 0, so whole chunks are in or out); it takes the guarded path.
    auto load_global = [&](int kt) {
        const int k0 = kt * BK;
#pragma unroll
        for (int i = 0; i < C::A_CHUNKS; ++i) ra[i] = *reinterpret_cast<const v4i*>(ga[i] + k0);
#pragma unroll
        for (int i = 0; i < C::W_CHUNKS; ++i) rw[i] = *reinterpret_cast<const v4i*>(gw[i] + k0);
    };
    auto load_global_tail = [&](int kt) {
        const int k0 = kt * BK;
#pragma unroll
        for (int i = 0; i < C::A_CHUNKS; ++i) {
            const bool in = k0 + ka[i] < K;
            ra[i] = *reinterpret_cast<const v4i*>(in ? ga[i] + k0 : ga[i] - ka[i]);  // row start is always readable
            if (!in) ra[i] = v4i{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < C::W_CHUNKS; ++i) {
            const bool in = k0 + kw[i] < K;
            rw[i] = *reinterpret_cast<const v4i*>(in ? gw[i] + k0 : gw[i] - kw[i]);
            if (!in) rw[i] = v4i{0, 0, 0, 0};
        }
    };
    const bool tail = (K % BK) != 0;
    auto load_tile = [&](int kt) {
        if (tail && kt == nk - 1) load_global_tail(kt);
        else load_global(kt);
    };
    auto store_lds = [&](int stage) {
        uint8_t* s = smem + stage * C::STAGE;
#pragma unroll
        for (int i = 0; i < C::A_CHUNKS; ++i) *reinterpret_cast<v4i*>(s + la[i]) = ra[i];
#pragma unroll
        for (int i = 0; i < C::W_CHUNKS; ++i) *reinterpret_cast<v4i*>(s + lw[i]) = rw[i];
    };

    // fragment rows of this lane inside the tile
    const int frow = lane & 31, fhalf = lane >> 5;

    load_tile(0);
    store_lds(0);
    __syncthreads();

    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
        if (kt + 1 < nk) load_tile(kt + 1);
        const uint8_t* sa = smem + cur * C::STAGE;
        const uint8_t* sw = sa + BM * BK;
#pragma unroll
        for (int kk = 0; kk < BK / 32; ++kk) {
            v4i af[C::TM], wf[C::TN];
#pragma unroll
            for (int im = 0; im < C::TM; ++im) {
                const int r = wm * C::WTM + im * 32 + frow;
                af[im] = *reinterpret_cast<const v4i*>(sa + r * BK + (swz<BK>(r, kk * 2 + fhalf) << 4));
            }
#pragma unroll
            for (int in = 0; in < C::TN; ++in) {
                const int r = wn * C::WTN + in * 32 + frow;
                wf[in] = *reinterpret_cast<const v4i*>(sw + r * BK + (swz<BK>(r, kk * 2 + fhalf) << 4));
            }
#pragma unroll
            for (int in = 0; in < C::TN; ++in)
#pragma unroll
                for (int im = 0; im < C::TM; ++im)
                    acc[in][im] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[in], af[im], acc[in][im], 0, 0, 0);
        }
        if (kt + 1 < nk) store_lds(cur ^ 1);
        __syncthreads();
    }

    static_assert(4 * 32 * C::WTN * 4 <= C::SMEM || C::NT != 256, "epilogue shuffle needs 4 pieces of LDS");
    epilogue<C::TM, C::TN, OUT_DT, EPI>(p, acc, m0 + wm * C::WTM, n0 + wn * C::WTN, lane, wave, smem);
}

// 16-byte global store the compiler's wait-count bookkeeping does not see
__device__ __forceinline__ void store16_untracked(void* ptr, uint4 v) {
    const v4i d = v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
    // The trailing s_nop gives the two wait states this hardware needs between a store of more than 8 bytes and a
    // vector write to its data registers; the compiler inserts them for its own stores but cannot see into this one.
    asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 1" ::"v"(ptr), "v"(d) : "memory");
}
// The same with a scalar base and a 32-bit lane offset.
__device__ __forceinline__ void store16_untracked_at(const void* base, uint32_t off, uint4 v) {
    const v4i d = v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
    asm volatile("global_store_dwordx4 %0, %1, %2 nt\n\ts_nop 1" ::"v"(off), "v"(d), "s"(base) : "memory");
}
// The same, written through to the last-level cache (device scope), which keeps it: the L2 does not.
__device__ __forceinline__ void store16_through_at(const void* base, uint32_t off, uint4 v) {
    const v4i d = v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
    asm volatile("global_store_dwordx4 %0, %1, %2 sc1\n\ts_nop 1" ::"v"(off), "v"(d), "s"(base) : "memory");
}
// The same with the caches' default policy.
__device__ __forceinline__ void store16_cached_at(const void* base, uint32_t off, uint4 v) {
    const v4i d = v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
    asm volatile("global_store_dwordx4 %0, %1, %2\n\ts_nop 1" ::"v"(off), "v"(d), "s"(base) : "memory");
}

template <int N> __device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void wg_barrier() { asm volatile("s_barrier" ::: "memory"); }
__device__ __forceinline__ void wait_lgkmcnt0() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

template <int V> struct ic { static constexpr int value = V; };
// ---------------------------------------------------------------------------------------------------------------
// Shapes with too few 256x256 tiles for the CUs: 128 x (64 * TN) tiles, one per workgroup and CU.
//
// Four waves multiply (64 x (32 * TN) each, one per SIMD) and four fetch.  A DMA instruction holds the wave that issues it for about 68
// cycles, four times a 16x16x64 MFMA, and with one wave per SIMD nothing else would run meanwhile; here the multiplying waves
// issue none.  Their fragments are double-buffered by halves of a K step: the next half is read from LDS behind the first MFMAs of
// this one.  One barrier per step, between its halves: step s + 1 has landed, and stage s, whose second half is in registers, may be
// fetched into.  Four stages: a step has three to land.  The epilogue's constants are loaded ahead of the K loop and the
// residual's lines are brought into the L2 by the waves that are done fetching.
// Stamps at 8192 x 2560 -> 640 (256 tiles, us): 2.0 until the first MFMA, 0.53 per step (the MFMAs take 0.37), 2.1 for the epilogue,
// 1.2 of them with constants and residual loaded where they are used.
// Against what ran these shapes before (a ring kernel of four waves that fetched for themselves, 128 x 192 tiles; 256 x 96 tiles
// streaming the weights for up to 256 rows), us, weights from HBM: 8192 x 2560 -> 640 20.5 and 19.0, 2048 x 2048 -> 2048 16.7 and
// 12.6, 512 x 4096 -> 4096 27.3 and 15.4, 256 x 4096 -> 4096 19.3 and 15.3, 200 x 8192 -> 3072 24.7 and 16.6, 40 x 4096 -> 24576 32.7 and
// 22.3.  The rule is at fed_plan.
// ---------------------------------------------------------------------------------------------------------------
template <int TN_>
struct FedCfg {
    static constexpr int TN = TN_, TM = 2, BM = 128, BN = 64 * TN, BK = 128, NT = 512, NS = 4;
    static constexpr int STAGE = (BM + BN) * BK, W_BASE = BM * BK, SMEM = NS * STAGE;
    static constexpr int A_LD = BM / 32, W_LD = BN / 32, LD = A_LD + W_LD;   // DMA instructions per fetching wave and step
    static constexpr int piece_cols(int sz) { return TN * 32 % (128 / sz) == 0 ? 128 / sz : 32; }
    static_assert(SMEM <= 160 * 1024, "LDS budget");
};
template <class C, int OUT_DT, int EPI>
__global__ void __launch_bounds__(512, 1) int8_gemm_fed_kernel(GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int NS = C::NS, LD = C::LD, FM = 2 * C::TM, FN = 2 * C::TN, BK = C::BK;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), wq = wave & 3;
    // split K: workgroup row blockIdx.y multiplies its slice of K and writes its own int32 plane
    const int k0 = p.kslice ? (int)blockIdx.y * p.kslice : 0;
    const int nk = (p.kslice && k0 + p.kslice < p.K ? p.kslice : p.K - k0) / BK;
    if (p.kslice) p.D = (uint8_t*)p.D + (int64_t)blockIdx.y * p.M * p.N * 4;
    int tm, tn;
    tile_of_block((int)blockIdx.x, (int)gridDim.x, p.tiles_m, p.tiles_n, tm, tn, p.magic);
    const int m0 = tm * C::BM, n0 = tn * C::BN;

    if (wave >= 4) {
        const int l = hw_lane(), lr = l >> 3, lc = ((l & 7) ^ (((wq & 1) << 2) | (lr >> 1))) * 16;
        uint32_t ga[C::A_LD], gw[C::W_LD];
#pragma unroll
        for (int j = 0; j < C::A_LD; ++j) {
            const int row = m0 + (wq + 4 * j) * 8 + lr;
            ga[j] = (uint32_t)(row < p.M ? row : p.M - 1) * (uint32_t)p.K + lc;
        }
#pragma unroll
        for (int j = 0; j < C::W_LD; ++j) {
            const int row = n0 + (wq + 4 * j) * 8 + lr;
            gw[j] = (uint32_t)(row < p.N ? row : p.N - 1) * (uint32_t)p.K + lc;
        }
        const uint32_t lds_base = (uint32_t)(uintptr_t)smem + wq * 1024;
        // Weights streamed once: workgroups that all read the same columns of K of rows 4 KB apart meet in a few of the HBM's channels,
        // so each tile column starts at a step of its own and wraps (integer sums: any order).  Cold weights, all at step 0 and
        // staggered, us: 256 x 4096 -> 24576 34.7 and 32.0, 40 rows 26.0 and 22.6, 128 x 8192 -> 28672 55.6 and 48.5, 40 x 3072 -> 18432
        // 17.2 and 16.6.  Slices start apart already, and with more rows tiles that share A or W do best in step (2048 x
        // 2048 -> 2048 11.1 and 11.6).
        const int first = p.tiles_m <= 2 && !p.kslice ? tn % nk : 0;
        const auto fetch = [&](int step) {
            const uint32_t dst = lds_base + (step & (NS - 1)) * C::STAGE;
            const int at = k0 + (step + first < nk ? step + first : step + first - nk) * BK;
            const int8_t *ab = p.A + at, *wb = p.W + at;
#pragma unroll
            for (int j = 0; j < C::A_LD; ++j)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst + j * 4096), "v"(ga[j]), "s"(ab) : "memory", "m0");
#pragma unroll
            for (int j = 0; j < C::W_LD; ++j)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst + C::W_BASE + j * 4096), "v"(gw[j]), "s"(wb) : "memory", "m0");
        };
        fetch(0);
        if (nk > 1) { fetch(1); wait_vmcnt<LD>(); }
        else wait_vmcnt<0>();
        wg_barrier();                                        // step 0 has landed
        for (int s = 2; s < NS && s < nk; ++s) fetch(s);
        for (int s = 0; s < nk; ++s) {
            if (s + NS <= nk) wait_vmcnt<(NS - 2) * LD>();   // step s + 1 has landed
            else wait_vmcnt<0>();
            wg_barrier();                                    // ... and nobody reads stage s any more
            if (s + NS < nk) fetch(s + NS);
            else if (EPI == EPI_RESID && (s + NS == nk || (nk < NS && s == 0))) {
                // the residual's lines into this XCD's L2, which the epilogue would otherwise wait for: SZ * BN bytes of 128 rows
                constexpr int CPR = C::BN * EpiConst<1, 1, OUT_DT, EPI, 16>::SZ / 128;
                for (int i = wq * 64 + hw_lane(); i < 128 * CPR; i += 256) {
                    const int row = m0 + i / CPR, col = n0 + i % CPR * (128 / EpiConst<1, 1, OUT_DT, EPI, 16>::SZ);
                    if (row < p.M && col < p.N) {
                        const uint32_t v = *reinterpret_cast<const volatile uint32_t*>((const uint8_t*)p.resid + ((int64_t)row * p.N + col) * EpiConst<1, 1, OUT_DT, EPI, 16>::SZ);
                        asm volatile("" ::"v"(v));
                    }
                }
            }
        }
        return;
    }

    const int wm = wq >> 1, wn = wq & 1;
    EpiConst<C::TM, C::TN, OUT_DT, EPI, 16> cst;
    if (EPI != EPI_ACC) {
        cst.load_columns(p, n0 + wn * C::TN * 32, hw_lane());
        cst.load_rows(p, m0 + wm * 64, hw_lane());
    }
    v4i acc[FN][FM], f[2][FM + FN];
#pragma unroll
    for (int in = 0; in < FN; ++in)
#pragma unroll
        for (int im = 0; im < FM; ++im) acc[in][im] = v4i{0, 0, 0, 0};
    const int frow = hw_lane() & 15, fq = hw_lane() >> 4;
    const int x = frow * BK + ((fq ^ ((frow >> 1) & 7)) << 4);
    const int ao = wm * 64 * BK + x, wo = C::W_BASE + wn * C::TN * 32 * BK + x;
    const auto read = [&](int step, int kk, int j) {
        const uint8_t* st = smem + (step & (NS - 1)) * C::STAGE;
        f[kk][j] = j < FM ? *reinterpret_cast<const v4i*>(st + (ao ^ (kk << 6)) + j * 16 * BK)
                          : *reinterpret_cast<const v4i*>(st + (wo ^ (kk << 6)) + (j - FM) * 16 * BK);
    };
    // the MFMAs of K half kk; the fragments of the half that follows are read behind the first of them
    const auto half = [&](auto kk_tag, int next_step) {
        constexpr int kk = decltype(kk_tag)::value;
#pragma unroll
        for (int in = 0; in < FN; ++in)
#pragma unroll
            for (int im = 0; im < FM; ++im) {
                acc[in][im] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f[kk][FM + in], f[kk][im], acc[in][im], 0, 0, 0);
                SCHED_FENCE();
                if (in * FM + im < FM + FN) { read(next_step, 1 - kk, in * FM + im); SCHED_FENCE(); }
            }
    };
    wg_barrier();
#pragma unroll
    for (int j = 0; j < FM + FN; ++j) read(0, 0, j);
    for (int s = 0; s < nk; ++s) {
        half(ic<0>{}, s);
        wait_lgkmcnt0();
        wg_barrier();
        half(ic<1>{}, s + 1);   // past the last step: a stage of the ring, read and not used
    }
    wait_lgkmcnt0();
    constexpr int SZ = (EPI == EPI_ACC || OUT_DT == DT_F32) ? 4 : 2;
    constexpr int PW = C::piece_cols(SZ);
    wg_barrier();
    uint8_t* scratch = smem + wave * 16384;
    epilogue_shuffle_with<C::TM, C::TN, OUT_DT, EPI, PW, STORE_PAST, 16, true>(p, acc, m0 + wm * 64, n0 + wn * C::TN * 32, hw_lane(), scratch, scratch + 8192, cst);
}

// ---------------------------------------------------------------------------------------------------------------
// The two-group persistent kernel for large shapes.  A global_load_lds_dwordx4 keeps the wave that issues it busy for
// about 68 cycles (measured: one wave alone, 16 of them back to back, 1088 cycles), twice the 32 cycles of a
// v_mfma_i32_32x32x32_i8, so a wave that issues its own DMA between its MFMAs leaves the matrix pipe of its SIMD idle
// for part of each one.  Here a workgroup has eight waves, two per SIMD, in two groups of four: group g owns rows
// 128g..128g+127 of a 256x256 tile (wave tiles 128x64).  The groups alternate between two kinds of phase, with one
// workgroup barrier between phases:
//   compute: the 64 MFMAs (16x16x64, 16 cycles each) of one 128-deep K step, on fragments already in registers, and
//            nothing else;
//   memory:  the 24 fragment reads of the group's next K step and NLA + NLW = 8 DMA instructions per wave.
// While one wave of a SIMD is in its memory phase the other is in its compute phase, so the matrix pipe always has an
// MFMA to run and no MFMA waits behind a DMA.
//
// LDS (160 KB): three 32 KB stages of W (both groups read them) and two 16 KB stages of A for each group.  With global
// step s = tile * nk + k tile, group 0 computes step s in phase 2s and group 1 in phase 2s + 1.  Group 0's memory phase
// before step s fetches A of group 1 for step s + 1 and rows 0..127 of W for step s + 2; group 1's fetches A of group 0
// and rows 128..255 of W, both for step s + 2.  Every memory phase ends with a wait that leaves only its own NLA + NLW DMA
// instructions in flight, so what a phase fetches is visible to everybody two phases later, and each stage is refilled
// only after the barrier that follows its last reader.  Steps run straight through tile boundaries.
//
// End of a tile: group 0 runs its epilogue while group 1 multiplies its last step and then runs its own; the shuffle
// scratch is the W stage of that step (4 KB per wave), which no DMA in flight targets.  Group 0 follows its epilogue with
// the memory phase of the next tile's first step (under group 1's epilogue), one barrier, and the alternation resumes
// with group 0 multiplying.
// Requires K % 128 == 0, M*K and N*K < 2^32, and the coalesced epilogue's alignment.
// ---------------------------------------------------------------------------------------------------------------
// GM: rows of a group.  128 gives the 256x256 tile (wave tiles 128x64), 96 a 192x256 tile, 64 a 128x256 tile (wave tiles 64x64):
// half the work per tile, at a step that is bound by its 6 DMA instructions per wave (7 with 96 rows) rather than by its 32 MFMAs.
// pp_split says which run.
template <int GM_>
struct PpCfg {
    static constexpr int GM = GM_, BM = 2 * GM, BN = 256, BK = 128, NT = 512;
    static constexpr int TM = GM / 32, TN = 2, WTN = 64;                            // wave tile GM x 64
    static constexpr int W_STAGE = BN * BK, A_STAGE = GM * BK, NSW = 3, NSA = 2;
    static constexpr int A_BASE = NSW * W_STAGE;                                    // group g's A ring at A_BASE + g*NSA*A_STAGE
    static constexpr int SMEM = NSW * W_STAGE + 2 * NSA * A_STAGE;
    static constexpr int NLA = GM / 32, NLW = 4;       // DMA instructions per wave for a group's A half / a 128-row W half
    static_assert(GM % 32 == 0 && SMEM <= 160 * 1024, "tile shape; LDS fits");
    static constexpr int piece_cols(int sz) { return sz == 2 ? 64 : 32; }           // 4 KB shuffle pieces
};
using PpL = PpCfg<128>;
using PpM = PpCfg<96>;
using PpS = PpCfg<64>;

// The work of workgroup `bid` of `G` on problem p.
template <class C, int OUT_DT, int EPI, int STORE>
__device__ __forceinline__ void pp_gemm_tiles(const GemmArgs& p, uint8_t* smem, const int bid, const int G) {
    constexpr int BK = C::BK, TM = C::TM, TN = C::TN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, wq = wave & 3;            // group; wave within the group = its column quarter
    const int ld = p.K, nk = p.K / BK;
    const int ntiles = p.tiles_m * p.tiles_n;
    const int nt_b = (ntiles - bid + G - 1) / G;         // tiles of this workgroup: bid, bid + G, ...
    const int S = nt_b * nk;                             // steps of this workgroup
    auto tile_origin = [&](int i, int& m0, int& n0) {
        int tm, tn;
        tile_of_block(bid + i * G, ntiles, p.tiles_m, p.tiles_n, tm, tn, p.magic);
        m0 = tm * C::BM;
        n0 = p.n_first + tn * C::BN;
    };
    const uint32_t lds_base = (uint32_t)(uintptr_t)smem;
    auto dma = [&](uint32_t dst, uint32_t off, const int8_t* base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
    };

    // DMA streams of this wave.  A wave fetches 8-row blocks wq, wq + 4, ... of the OTHER group's A rows and of its own
    // half of the W tile (group 0: rows 0..127, group 1: rows 128..255).
    // Lane offsets carry the chunk swizzle (bits 1..3 of the row) on the global side, chunk c of row r at slot c ^ ((r >> 1) & 7).
    uint32_t ga[C::NLA], gw[C::NLW];
    // a stream's position: the (tile, k tile) it fetches next and the stage that goes to.  A stream stops on the last step
    // and keeps re-fetching it, into the stage it would have used, which nothing reads again.
    int a_tile, a_kt, a_stage, w_tile = 0, w_kt = 0, w_stage = 0;
    auto set_rows = [&](uint32_t* g, auto n, int origin, int limit) {
        const int l = hw_lane();
        const int lr = l >> 3, lc = ((l & 7) ^ (((wq & 1) << 2) | (lr >> 1))) * 16;
#pragma unroll
        for (int j = 0; j < decltype(n)::value; ++j) {
            const int row = origin + (wq + 4 * j) * 8 + lr;
            g[j] = (uint32_t)(row < limit ? row : limit - 1) * (uint32_t)ld + lc;
        }
    };
    auto set_a = [&](int tile) { int m0, n0; tile_origin(tile, m0, n0); set_rows(ga, ic<C::NLA>{}, m0 + (grp ^ 1) * C::GM, p.M); };
    // W: a wave fetches the four CONSECUTIVE 8-row blocks 4*wq .. 4*wq + 3 of its group's half, which are exactly the 4 KB
    // of the stage that serve as this wave's shuffle scratch in the epilogue: group 0 may then refill the stage right
    // after its own epilogue, while other waves are still in theirs.  (A block's parity, which the swizzle needs, is j's.)
    auto set_w = [&](int tile) {
        int m0, n0;
        tile_origin(tile, m0, n0);
        const int l = hw_lane();
        const int lr = l >> 3;
#pragma unroll
        for (int j = 0; j < C::NLW; ++j) {
            const int row = n0 + grp * 128 + (4 * wq + j) * 8 + lr;
            const int lc = ((l & 7) ^ (((j & 1) << 2) | (lr >> 1))) * 16;
            gw[j] = (uint32_t)(row < p.N ? row : p.N - 1) * (uint32_t)ld + lc;
        }
    };
    auto fetch_a = [&]() {
        const int8_t* base = p.A + (int64_t)a_kt * BK;
        const uint32_t dst = lds_base + C::A_BASE + ((grp ^ 1) * C::NSA + a_stage) * C::A_STAGE + wq * 1024;
#pragma unroll
        for (int j = 0; j < C::NLA; ++j) dma(dst + j * 4096, ga[j], base);
        a_stage = a_stage == C::NSA - 1 ? 0 : a_stage + 1;
        if (a_tile == nt_b - 1 && a_kt == nk - 1) return;
        if (++a_kt == nk) { a_kt = 0; set_a(++a_tile); }
    };
    auto fetch_w = [&]() {
        const int8_t* base = p.W + (int64_t)w_kt * BK;
        const uint32_t dst = lds_base + w_stage * C::W_STAGE + grp * 128 * BK + wq * 4096;
#pragma unroll
        for (int j = 0; j < C::NLW; ++j) dma(dst + j * 1024, gw[j], base);
        w_stage = w_stage == C::NSW - 1 ? 0 : w_stage + 1;
        if (w_tile == nt_b - 1 && w_kt == nk - 1) return;
        if (++w_kt == nk) { w_kt = 0; set_w(++w_tile); }
    };

    // The tiles are multiplied with v_mfma_i32_16x16x64_i8: as many operations per cycle as the 32x32x32 form and the same
    // fragment bytes per K, but an accumulator is touched once per 64 K instead of once per 32.  On this power-limited
    // part that is worth clock: a loop of nothing but MFMAs on random bits sustains 3.95 POP/s in this form against 3.4,
    // and this kernel ran 9-11 % faster with it.  A wave tile is FM x FN tiles of 16 x 16, four accumulator registers each.
    // Fragment addresses inside a stage: row r at r*128, chunk c at slot c ^ ((r>>1)&7); a lane reads row lane % 16,
    // chunk 4*kk + lane / 16 of K half kk (which flips bit 6).
    constexpr int FM = 2 * TM, FN = 2 * TN;
    v4i acc[FN][FM];
    v4i f[2][FM + FN];
    int ra_stage = 0, rw_stage = 0;   // stages this group's next fragments come from
    auto load_frags = [&]() {
        const int l = hw_lane();
        const int frow = l & 15, fq = l >> 4;
        const int x = frow * BK + ((fq ^ ((frow >> 1) & 7)) << 4);
        const uint8_t* sa = smem + C::A_BASE + (grp * C::NSA + ra_stage) * C::A_STAGE;
        const uint8_t* sw = smem + rw_stage * C::W_STAGE + wq * C::WTN * BK;
        ra_stage = ra_stage == C::NSA - 1 ? 0 : ra_stage + 1;
        rw_stage = rw_stage == C::NSW - 1 ? 0 : rw_stage + 1;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int xk = x ^ (kk << 6);
#pragma unroll
            for (int j = 0; j < FM; ++j) f[kk][j] = *reinterpret_cast<const v4i*>(sa + xk + j * 16 * BK);
#pragma unroll
            for (int j = 0; j < FN; ++j) f[kk][FM + j] = *reinterpret_cast<const v4i*>(sw + xk + j * 16 * BK);
        }
    };
    // a tile's first MFMAs take C = 0 instead of cleared accumulators
    auto compute = [&](bool first) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int in = 0; in < FN; ++in)
#pragma unroll
                for (int im = 0; im < FM; ++im) {
                    const v4i c = (first && kk == 0) ? v4i{0, 0, 0, 0} : acc[in][im];
                    acc[in][im] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f[kk][FM + in], f[kk][im], c, 0, 0, 0);
                    SCHED_FENCE();
                }
        __builtin_amdgcn_s_setprio(0);
    };
    // memory phase before this group's next step
    auto memory = [&]() {
        load_frags();
        SCHED_FENCE();
        fetch_a();
        fetch_w();
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::NLA + C::NLW) : "memory");   // everything but this phase's own DMA has landed
    };

    // prologue: every group fetches its OWN A for step 0 (group 0 also for step 1: group 1's first memory phase fetches
    // A0 of step 2) and its half of W for steps 0 and 1; then the streams move to where the memory phases expect them
    {
        int m0, n0;
        const int own_a = C::A_BASE + grp * C::NSA * C::A_STAGE;
        const int t1 = (nk == 1 && nt_b > 1) ? 1 : 0, k1 = nk > 1 ? 1 : 0;   // step 1 as (tile, k tile); step 0 again if S == 1
        tile_origin(0, m0, n0);
        set_rows(ga, ic<C::NLA>{}, m0 + grp * C::GM, p.M);
#pragma unroll
        for (int j = 0; j < C::NLA; ++j) dma(lds_base + own_a + (wq + 4 * j) * 1024, ga[j], p.A);
        if (grp == 0) {
            if (t1) { tile_origin(1, m0, n0); set_rows(ga, ic<C::NLA>{}, m0, p.M); }
#pragma unroll
            for (int j = 0; j < C::NLA; ++j) dma(lds_base + own_a + C::A_STAGE + (wq + 4 * j) * 1024, ga[j], p.A + (int64_t)k1 * BK);
        }
        set_w(0);
        fetch_w();
        fetch_w();
        // the A stream of the OTHER group's tile: group 0 starts at step 1, group 1 at step 2 (clamped to the last step)
        int st = grp == 0 ? 1 : 2;
        a_stage = st % C::NSA;
        if (st > S - 1) st = S - 1;
        a_tile = st / nk;
        a_kt = st - a_tile * nk;
        set_a(a_tile);
        wait_vmcnt<0>();
        wg_barrier();
    }

    constexpr int SZ = (EPI == EPI_ACC || OUT_DT == DT_F32) ? 4 : 2;
    constexpr int PW = C::piece_cols(SZ);
    auto run_epilogue = [&](int ti, int s_last) {
        int m0, n0;
        tile_origin(ti, m0, n0);
        uint8_t* scratch = smem + (s_last % C::NSW) * C::W_STAGE + wave * 4096;
        epilogue_shuffle<TM, TN, OUT_DT, EPI, PW, STORE, 16>(p, acc, m0 + grp * C::GM, n0 + wq * C::WTN, hw_lane(), scratch);
    };

    // Both groups run the same loop; group 1 is one phase behind (the barrier in front) and multiplies its last step of a
    // tile in the phase in which group 0 already runs its epilogue.  Group 0 goes from its epilogue straight into the
    // memory phase of the next tile's first step, while group 1 is still in its epilogue: what that phase reads landed
    // before the tile's last compute phases, and what it fetches goes to stages that neither epilogue uses (group 1's A
    // stage of the step before last, and the half of the last step's W stage that was group 0's own shuffle scratch).
    // After the one barrier that follows the epilogues group 0 multiplies at once and the alternation is back.
    if (grp == 1) wg_barrier();
    int s = 0;
    for (int ti = 0; ti < nt_b; ++ti) {
        for (int kt = 0; kt < nk; ++kt, ++s) {
            memory();
            wait_lgkmcnt0();
            wg_barrier();
            compute(kt == 0);
            if (grp == 0 || kt + 1 < nk) wg_barrier();
        }
        run_epilogue(ti, s - 1);
        // the barrier behind the epilogues; group 0 meets it after the next tile's first memory phase (the loop's first
        // barrier), so it skips this one when a tile follows
        if (grp == 1 || ti + 1 == nt_b) wg_barrier();
    }
    wait_vmcnt<0>();   // no DMA may still be writing this workgroup's LDS when it retires
}

// Workgroups 0 .. g_main-1 walk the tiles of `main`; the others walk the 128x256 tiles of `rest` (the rows or columns that
// whole rounds of large tiles leave over, everything, or nothing).  One launch: the hardware starts a workgroup of the second kind
// on each CU as its workgroup of the first kind retires, with no gap between two launches.
template <class Main, int OUT_DT, int EPI, int STORE>
__global__ void __launch_bounds__(PpL::NT, 1) int8_gemm_pp_kernel(GemmArgs main, GemmArgs rest, int g_main) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int bid = (int)blockIdx.x;
    if (bid < g_main) pp_gemm_tiles<Main, OUT_DT, EPI, STORE>(main, smem, bid, g_main);
    else pp_gemm_tiles<PpS, OUT_DT, EPI, STORE>(rest, smem, bid - g_main, (int)gridDim.x - g_main);
}

// ---------------------------------------------------------------------------------------------------------------
// Up to 128 rows: weights straight from HBM into the registers that the matrix instruction reads, rows of A through LDS.  The
// kernel with fetching waves takes weights and A into a CU's LDS through one load path, in tiles of 128 rows; here only the M
// rows there are, in 16-row tiles (MT of them), go that way, and the weights are most of what a CU takes in.
//   * Eight waves; a wave owns 16 columns and one of NWK interleaved parts of K, so a workgroup covers 128 / NWK columns
//     and walks K in panels of 512 * NWK (or 256).  The parts are added through LDS at the end.
//   * W: a load is 16 columns x 64 bytes, an MFMA operand as it arrives.  Two panels of them are always in flight, each
//     reissued as soon as its MFMAs have read it: 128 KB per CU (64), and no wait of one wave for another on the way.
//   * A: the panel's rows by DMA into one of two stages, [128-byte column block][8 rows][128 bytes] with the chunk swizzle of
//     the other kernels on the global side, a panel ahead; one barrier per panel.
// The wait ahead of that barrier counts: the reissued W loads may stay in flight, the DMA before them may not.
// Bound by HBM behind 5 us of launch and first trips.  us per call, weights from HBM, the kernel with fetching waves and this one:
// 16 rows 1024 -> 1024 5.9 and 6.5, 2048 -> 5120 8.1 and 6.6, 4096 -> 4096 10.4 and 8.8, 12288 -> 4096 16.5 and 16.3; 64 rows 2048 -> 4096
// 8.4 and 8.0, 3072 -> 4096 10.7 and 9.5, 5120 -> 640 9.2 and 8.1; 40 rows 4096 -> 24576 22.3 and 36.3.  The rule is at rows_kernel_wins.
// Eight steps of 64 per panel where two stages fit the LDS, else four: with NWK = 1 instead, 77 rows take 16.6 instead of 13.8 us
// for 4096 -> 4096.
template <int MT, int NWK>   // NWK 2, 4 or 8
struct RowsCfg {
    static constexpr int NT = 512, NWN = 8 / NWK, BN = 16 * NWN, RB = 2 * MT;
    static constexpr int SP = MT * NWK <= 8 ? 8 : 4;   // steps of 64 per wave and panel; two stages have to fit the LDS
    static constexpr int KP = 64 * SP * NWK, NLA = KP / 128 * RB / 8;
    static constexpr int STAGE = KP / 128 * RB * 1024, SMEM = 2 * STAGE;
};
template <int MT, int NWK, int OUT_DT, int EPI>
__global__ void __launch_bounds__(512, (MT * NWK <= 4 ? 4 : 2)) int8_gemm_rows_kernel(GemmArgs p, bool vec_ok) {
    using C = RowsCfg<MT, NWK>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, quarter = lane >> 4;
    const int wn = wave % C::NWN, wk = wave / C::NWN;
    const int kb0 = (int)blockIdx.y * p.kslice;
    const int k1 = p.kslice && kb0 + p.kslice < p.K ? kb0 + p.kslice : p.K;
    const int nb = (int)blockIdx.x * C::BN + wn * 16;
    const int wrow = nb + l16 < p.N ? nb + l16 : p.N - 1;   // columns past the end read the last one and are not stored
    const uint32_t woff = (uint32_t)wrow * (uint32_t)p.K + quarter * 16;
    const int np = (k1 - kb0 + C::KP - 1) / C::KP;
    const uint32_t lds_base = (uint32_t)(uintptr_t)smem;

    uint32_t ga[C::NLA];
#pragma unroll
    for (int j = 0; j < C::NLA; ++j) {
        const int rb = (wave + 8 * j) % C::RB;
        const int row = rb * 8 + (lane >> 3) < p.M ? rb * 8 + (lane >> 3) : p.M - 1;
        ga[j] = (uint32_t)row * (uint32_t)p.K + (((lane & 7) ^ ((rb & 1) * 4 + (lane >> 4))) * 16);
    }
    const auto fetch_a = [&](int panel) {
#pragma unroll
        for (int j = 0; j < C::NLA; ++j) {
            const int blk = wave + 8 * j;
            const int k = kb0 + panel * C::KP + blk / C::RB * 128;   // a block past the end is fetched from the last one and not used
            const int8_t* base = p.A + (k < k1 ? k : k1 - 128);
            const uint32_t dst = lds_base + (panel & 1) * C::STAGE + blk * 1024;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(ga[j]), "s"(base) : "memory", "m0");
        }
    };
    const auto fetch_w = [&](int panel, int i) {
        const int k = kb0 + panel * C::KP + (wk * C::SP + i) * 64;
        return *reinterpret_cast<const v4i*>(p.W + (k < k1 ? k : k1 - 64) + (uint64_t)woff);
    };
    v4i w[2][C::SP], acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = v4i{0, 0, 0, 0};
    // the epilogue's constants first, so that their trip is over when they are used; then the longest trips
    const int n = nb + 4 * quarter;   // a lane ends up with the columns n..n+3 of row lane % 16 of the row tiles
    typedef uint32_t raw4 __attribute__((ext_vector_type(dt_size<OUT_DT>::value)));   // four outputs' worth, as it lies in memory
    float4 ws4 = make_float4(0.f, 0.f, 0.f, 0.f);
    raw4 b4 = 0, rs4 = 0;
    float xs[MT];
    if (EPI != EPI_ACC) {
        if (vec_ok && n < p.N) {
            ws4 = *reinterpret_cast<const float4*>(p.ws + n);
            if (p.bias) b4 = *reinterpret_cast<const raw4*>((const uint8_t*)p.bias + (int64_t)n * dt_size<OUT_DT>::value);
            if (EPI == EPI_RESID) rs4 = *reinterpret_cast<const raw4*>((const uint8_t*)p.rscale + (int64_t)n * dt_size<OUT_DT>::value);
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) xs[t] = p.xs[t * 16 + l16 < p.M ? t * 16 + l16 : p.M - 1];
    }
    SCHED_FENCE();
#pragma unroll
    for (int i = 0; i < C::SP; ++i) w[0][i] = fetch_w(0, i);
    SCHED_FENCE();
    fetch_a(0);
    SCHED_FENCE();
#pragma unroll
    for (int i = 0; i < C::SP; ++i) w[1][i] = fetch_w(1, i);
    SCHED_FENCE();
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(C::SP) : "memory");

    const auto panel_step = [&](int panel, auto set_tag, auto whole_tag) {
        constexpr int set = decltype(set_tag)::value, whole = decltype(whole_tag)::value;
        if (panel + 1 < np) fetch_a(panel + 1);
        SCHED_FENCE();
        const uint8_t* st = smem + set * C::STAGE + (l16 >> 3) * 1024 + (l16 & 7) * 128;
#pragma unroll
        for (int i = 0; i < C::SP; ++i) {
            const int ks = wk * C::SP + i;
            if (whole || kb0 + panel * C::KP + ks * 64 < k1) {
                const uint8_t* f = st + (ks >> 1) * (C::RB * 1024) + ((((i & 1) * 4 + quarter) ^ (l16 >> 1)) * 16);
                v4i a[MT];
#pragma unroll
                for (int t = 0; t < MT; ++t) a[t] = *reinterpret_cast<const v4i*>(f + t * 2048);
                SCHED_FENCE();   // one trip to LDS for all of them
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[set][i], a[t], acc[t], 0, 0, 0);
            }
            if constexpr (whole) {
                SCHED_FENCE();
                w[set][i] = fetch_w(panel + 2, i);
                SCHED_FENCE();
            }
        }
        if constexpr (whole) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::SP) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        SCHED_FENCE();
    };
    // whole panels in pairs without a way out between them, which would cost the compiler its count of the loads in flight
    int panel = 0;
    for (const int pairs_end = (k1 - kb0) / C::KP & ~1; panel < pairs_end; panel += 2) {
        panel_step(panel, ic<0>{}, ic<1>{});
        panel_step(panel + 1, ic<1>{}, ic<1>{});
    }
    if (panel < np) {
        panel_step(panel, ic<0>{}, ic<0>{});
        if (panel + 1 < np) panel_step(panel + 1, ic<1>{}, ic<0>{});
    }

    const auto finish = [&](const v4i& sum, int t, float x) {
        const int m = t * 16 + l16;
        if (m >= p.M || n >= p.N) return;
        const int64_t o = (int64_t)m * p.N + n;
        if (EPI == EPI_ACC) {
            int* d = (int*)p.D + (int64_t)blockIdx.y * p.M * p.N + o;
            if (vec_ok) *reinterpret_cast<v4i*>(d) = sum;
            else
#pragma unroll
                for (int j = 0; j < 4; ++j) if (n + j < p.N) d[j] = sum[j];
            return;
        }
        float ws[4] = {ws4.x, ws4.y, ws4.z, ws4.w}, b[4] = {0.f, 0.f, 0.f, 0.f}, rs[4] = {0.f, 0.f, 0.f, 0.f}, res[4] = {0.f, 0.f, 0.f, 0.f}, out[4];
        if (vec_ok) {
            load4<OUT_DT>(&b4, 0, b);
            load4<OUT_DT>(&rs4, 0, rs);
            if (EPI == EPI_RESID) load4<OUT_DT>(p.resid, o, res);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (n + j >= p.N) continue;
                ws[j] = p.ws[n + j];
                if (p.bias) b[j] = ld_dt<OUT_DT>(p.bias, n + j);
                if (EPI == EPI_RESID) { rs[j] = ld_dt<OUT_DT>(p.rscale, n + j); res[j] = ld_dt<OUT_DT>(p.resid, o + j); }
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = epi_value<OUT_DT, EPI>(sum[j], x, ws[j], b[j], rs[j], res[j]);
        if (vec_ok) store4<OUT_DT>(p.D, o, out);
        else
#pragma unroll
            for (int j = 0; j < 4; ++j) if (n + j < p.N) st_dt<OUT_DT>(p.D, o + j, out[j]);
    };
    v4i* red = reinterpret_cast<v4i*>(smem) + lane;   // [part of K][16 columns][row tile][lane]
#pragma unroll
    for (int t = 0; t < MT; ++t) red[(wave * MT + t) * 64] = acc[t];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        if (t % NWK != wk) continue;
        v4i sum = red[(wn * MT + t) * 64];
#pragma unroll
        for (int q = 1; q < NWK; ++q) sum += red[((q * C::NWN + wn) * MT + t) * 64];
        finish(sum, t, EPI == EPI_ACC ? 0.f : xs[t]);
    }
}

// Sum of the int32 planes of a split-K run, then the epilogue.  planes[s][M][N]; four consecutive n per thread.
template <int OUT_DT, int EPI>
__global__ void __launch_bounds__(256) splitk_epilogue_kernel(GemmArgs p, const int* planes, int slices) {
    const int64_t nvec = (int64_t)p.M * p.N / 4, plane = (int64_t)p.M * p.N;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nvec; i += (int64_t)gridDim.x * 256) {
        const int64_t o = i * 4;
        const int m = (int)(o / p.N), n = (int)(o - (int64_t)m * p.N);
        // the planes' loads go out in batches of four with nothing between them: one trip to memory instead of `slices`
        const int* src = planes + o;
        v4i acc = *reinterpret_cast<const v4i*>(src);
        int s = 1;
        for (; s + 3 < slices; s += 4) {
            const v4i a0 = *reinterpret_cast<const v4i*>(src + s * plane), a1 = *reinterpret_cast<const v4i*>(src + (s + 1) * plane);
            const v4i a2 = *reinterpret_cast<const v4i*>(src + (s + 2) * plane), a3 = *reinterpret_cast<const v4i*>(src + (s + 3) * plane);
            acc += (a0 + a1) + (a2 + a3);
        }
        for (; s < slices; ++s) acc += *reinterpret_cast<const v4i*>(src + s * plane);
        if (EPI == EPI_ACC) {   // the caller asked for the accumulators themselves: no scales to apply
            *reinterpret_cast<v4i*>((int*)p.D + o) = acc;
            continue;
        }
        const float xs = p.xs[m];
        const float4 w4 = *reinterpret_cast<const float4*>(p.ws + n);
        const float ws[4] = {w4.x, w4.y, w4.z, w4.w};
        float b[4] = {0.f, 0.f, 0.f, 0.f}, rs[4] = {0.f, 0.f, 0.f, 0.f}, res[4] = {0.f, 0.f, 0.f, 0.f}, out[4];
        if (p.bias) load4<OUT_DT>(p.bias, n, b);
        if (EPI == EPI_RESID) { load4<OUT_DT>(p.rscale, n, rs); load4<OUT_DT>(p.resid, o, res); }
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = epi_value<OUT_DT, EPI>(acc[j], xs, ws[j], b[j], rs[j], res[j]);
        store4<OUT_DT>(p.D, o, out);
    }
}

// Tile shapes of the register-staged kernel, the fallback for K % 128 != 0, unaligned outputs and small problems.
// M: 128x128, two workgroups per CU.  S: 64x64 for small M or N.
using CfgM = Cfg<128, 128, 64, 2, 2, 2>;
using CfgS = Cfg<64, 64, 64, 2, 2, 4>;

// Kernel family forced by the test hook (-1 = choose by shape), or 7000 + 100 * width + slices: the kernel with fetching waves on
// tiles of 64 * width columns and so many slices of K, or 9000 + 10 * kind + split: the two-group kernel (kind: 256, 192 or 128
// rows; split: none, rows, columns).  Process-wide and only meant for tests and benchmarks:
// relaxed atomic, so a concurrent call sees either the old or the new value, never a torn one.
std::atomic<int> g_force_cfg{-1};

template <class C, int OUT_DT, int EPI>
int launch_cfg(GemmArgs a, hipStream_t st) {
    a.tiles_m = (a.M + C::BM - 1) / C::BM;
    a.tiles_n = (a.N + C::BN - 1) / C::BN;
    a.magic = panel_magic(a.tiles_m, a.tiles_n);
    const int64_t nblocks = (int64_t)a.tiles_m * a.tiles_n;
    if (nblocks > 0x7fffffff) return -1;
    auto kern = int8_gemm_kernel<C, OUT_DT, EPI>;
    if (C::SMEM > 48 * 1024) {
        static PerDeviceOnce once;
        if (const int e = allow_dynamic_lds((const void*)kern, C::SMEM, once)) return e;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(C::NT), C::SMEM, st, a);
    KCHECK();
    return 0;
}

// Rows [row0, row0 + rows) of the problem as a problem of its own.
template <int OUT_DT, int EPI>
GemmArgs row_band(const GemmArgs& a, int64_t row0, int64_t rows) {
    constexpr int SZ = (EPI == EPI_ACC || OUT_DT == DT_F32) ? 4 : 2;
    GemmArgs b = a;
    b.A = a.A + row0 * a.K;
    b.xs = a.xs ? a.xs + row0 : nullptr;
    b.D = (uint8_t*)a.D + row0 * a.N * SZ;
    b.resid = a.resid ? (const uint8_t*)a.resid + row0 * a.N * SZ : nullptr;
    b.M = (int)rows;
    return b;
}

// Large shapes on the two-group kernel.  A launch takes whole rounds of one tile per CU, and what counts is how little of the last
// round is idle: tiles of 256, 192 or 128 rows by 256 columns, and where the tiles of 256 or 192 rows fill whole rounds and some
// more, the tile rows or tile columns that fill the whole ones, with the rest as 128 x 256 tiles by further workgroups of the same
// launch.  The smallest sum of rounds runs, a round of the smaller tiles counted as 0.78 and 0.67 of one of 256 rows: three
// quarters and half of the work, but a step of theirs is bound by its DMA instructions.  kCost is what chose best over 260 shapes of 512 to
// 8192 rows timed in all seven forms; over 720 others, weights from HBM and outputs in turn, it is 0.8 % slower than the best of them, 256-row
// tiles with rows left over alone 10 %.  us, those and the present choice, weights from HBM (from the last-level cache): 2048 x 14336 -> 5376
// 134.4 and 123.8 (125.2 and 122.2; 192 rows: 231 tiles instead of 168), 3000 x 2048 -> 7168 46.7 and 43.7 (45.2 and 42.3), 6000 x 1024 -> 3072
// 28.6 and 26.3 (28.4 and 26.0), 8192 x 640 -> 5120 39.2 and 39.5 (35.3 and 35.1; columns left over; bound by the chip's writes beside the MFMAs).
struct PpSplit {
    int rows;                          // of a tile of the first kind: 256 or 192; 128: there are only tiles of the second
    int64_t main_tm, main_tn, small;   // the grid of those tiles, and how many of the second kind
    bool columns;                      // the second kind takes the columns that are left, not the rows
    double rounds;                     // rounds of 256 x 256 tiles in all
};
PpSplit pp_split(int64_t M, int64_t N, int64_t cus) {
    static constexpr double kCost[3] = {1.0, 0.78, 0.67};
    const int64_t tn = (N + 255) / 256;
    const auto rounds = [&](int64_t tiles) { return (double)((tiles + cus - 1) / cus); };
    const int force = g_force_cfg.load(std::memory_order_relaxed) - 9000;
    PpSplit best{256, 0, 0, 0, false, 1e30};
    for (int kind = 0; kind < 3; ++kind) {
        if (force >= 0 && force < 30 && kind != force / 10) continue;
        const int bm = 256 - 64 * kind;
        const int64_t tm = (M + bm - 1) / bm, full = tm * tn / cus;
        const double whole = kCost[kind] * rounds(tm * tn);
        PpSplit form[3] = {kind == 2 ? PpSplit{bm, 0, 0, tm * tn, false, whole} : PpSplit{bm, tm, tn, 0, false, whole}, best, best};
        int forms = 1;
        if (kind < 2 && full >= 1 && tm > 1 && tn > 1 && tm * tn % cus != 0) {
            const int64_t rows = full * cus / tn < tm ? full * cus / tn : tm - 1, cols = full * cus / tm < tn ? full * cus / tm : tn - 1;
            const int64_t by_rows = (M - rows * bm + 127) / 128 * tn, by_cols = (M + 127) / 128 * (tn - cols);
            form[1] = {bm, rows, tn, by_rows, false, rows > 0 ? kCost[kind] * rounds(rows * tn) + kCost[2] * rounds(by_rows) : 1e30};
            form[2] = {bm, tm, cols, by_cols, true, cols > 0 ? kCost[kind] * rounds(tm * cols) + kCost[2] * rounds(by_cols) : 1e30};
            forms = 3;
        }
        if (force >= 0 && force < 30) return form[force % 10 < forms ? force % 10 : 0];
        for (int i = 0; i < forms; ++i)
            if (form[i].rounds < best.rounds - 0.005) best = form[i];
    }
    return best;
}

// How the two-group kernel stores outputs of 40 to 100 MB, which the last-level cache (256 MB) can hold beside the operands for whoever reads
// them next; all others go past the caches.  us with weights from HBM and outputs in turn in 0.6 to 0.9 GB.
//   * Rows of whole 64 bytes are written through to that cache, the L2 (32 MB) keeps nothing.  Past the caches and this way, alone and with the
//     quantizer that reads the output behind it: 84 MB 8192 x 640 -> 5120 35.0 and 37.3, 66.9 and 64.6; 4096 x 1280 -> 10240 53.7 and 54.4, 88.1 and
//     86.2; 67 MB of floats 2048 x 512 -> 8192 19.7 and 19.5, 46.9 and 41.2; 43 MB 4420 x 1024 -> 4864 25.7 and 26.7, 43.0 and 42.2.  51 such shapes:
//     alone 0.973 where the same output buffer comes again and 1.018 where it does not (1.06 at most), with the reader 0.976 and 0.973 (1.015 at
//     most, 47 MB 1034 x 5376 -> 22528).  By the caches' default policy the L2 keeps such lines until the kernel's end writes them back: 39.5
//     and 60.2 alone in the first two, and nothing gained with the reader (67.6 and 90.5; 42 MB 2048 x 1280 -> 10240 50.3 and 54.7).
//   * Other rows end in the middle of 64 bytes, which memory writes with a read ahead of it unless the L2 has brought the two rows' parts
//     together: the default policy.  0.85 of the time past the caches (45 shapes, 16-bit; 0.78 in floats), written through 1.15 (bf16 5114 x 256 -> 4976
//     24.1 past the caches, 34.5 through; 6385 x 256 -> 7000, one output buffer, with the quantizer of its rows 56 past them, 31 this way).
//   * The range ends where the default policy had been seen to lose.  60 shapes of 20 to 40 MB written through have 1.008 alone and 0.978 with
//     the reader, 19 of 100 to 150 MB 1.011 and 0.961, but 14 MB 520 x 256 -> 13312 8.3 and 8.8 alone, 134 MB 8192 x 512 -> 8192 45.8 and 59.9: left as it
//     was.  The residual form has no gain (4608 x 12288 -> 3072 127.3 and 127.5, by the default policy) and keeps the one way.
int store_policy(int64_t M, int64_t row_bytes, uintptr_t D) {
    const double bytes = (double)M * (double)row_bytes;
    if (bytes < 40e6 || bytes > 100e6) return STORE_PAST;
    return (((uintptr_t)row_bytes | D) & 63) == 0 ? STORE_THROUGH : STORE_CACHED;
}

template <class Main, int OUT_DT, int EPI, int STORE>
int launch_pp_as(const GemmArgs& main, const GemmArgs& rest, int g_main, int g_rest, hipStream_t st) {
    auto kern = int8_gemm_pp_kernel<Main, OUT_DT, EPI, STORE>;
    static PerDeviceOnce once;
    if (const int e = allow_dynamic_lds((const void*)kern, PpL::SMEM, once)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)(g_main + g_rest)), dim3(PpL::NT), PpL::SMEM, st, main, rest, g_main);
    KCHECK();
    return 0;
}
template <int OUT_DT, int EPI>
int launch_pp(GemmArgs a, hipStream_t st) {
    bool vec_ok, aligned;
    epilogue_alignment<OUT_DT, EPI>(a, vec_ok, aligned);
    if (!aligned) return launch_cfg<CfgM, OUT_DT, EPI>(a, st);   // this kernel has only the coalesced epilogue
    const int64_t G = device_cu_count();
    const PpSplit sp = pp_split(a.M, a.N, G);
    constexpr int SZ = EPI == EPI_ACC || OUT_DT == DT_F32 ? 4 : 2;
    const int policy = EPI == EPI_RESID ? (int)STORE_PAST : store_policy(a.M, (int64_t)a.N * SZ, (uintptr_t)a.D);
    GemmArgs main = a, rest = a;
    const int64_t n_main = sp.main_tm * sp.main_tn, n_rest = sp.small, tn = (a.N + 255) / 256;
    if (n_main > 0x7fffffff || n_rest > 0x7fffffff) return -1;
    if (n_main && n_rest) {
        if (sp.columns) {
            rest.n_first = (int)sp.main_tn * 256;
        } else {
            main = row_band<OUT_DT, EPI>(a, 0, sp.main_tm * sp.rows);
            rest = row_band<OUT_DT, EPI>(a, sp.main_tm * sp.rows, a.M - sp.main_tm * sp.rows);
        }
    }
    main.tiles_m = (int)sp.main_tm;
    main.tiles_n = (int)sp.main_tn;
    rest.tiles_m = (rest.M + PpS::BM - 1) / PpS::BM;
    rest.tiles_n = (int)(sp.columns ? tn - sp.main_tn : tn);
    main.magic = n_main ? panel_magic(main.tiles_m, main.tiles_n) : 0;
    rest.magic = panel_magic(rest.tiles_m, rest.tiles_n);
    const int g_main = (int)(n_main < G ? n_main : G), g_rest = (int)(n_rest < G ? n_rest : G);
    const auto as = [&](auto store) {
        constexpr int S = decltype(store)::value;
        return sp.rows == PpM::BM ? launch_pp_as<PpM, OUT_DT, EPI, S>(main, rest, g_main, g_rest, st)
                                  : launch_pp_as<PpL, OUT_DT, EPI, S>(main, rest, g_main, g_rest, st);
    };
    if constexpr (EPI != EPI_RESID) {
        if (policy == STORE_THROUGH) return as(ic<STORE_THROUGH>{});
        if (policy == STORE_CACHED) return as(ic<STORE_CACHED>{});
    }
    return as(ic<STORE_PAST>{});
}

// ---------------------------------------------------------------------------------------------------------------
// Scratch of the entry point that allocates nothing (gpu_int8_gemm_static): the int32 planes of a split-K run live in
// this file-scope device array instead of a stream-ordered allocation.  Every GPU the library runs on holds its own
// copy at its own address until the process ends; the array's name is only a host-side handle, so the device address
// is looked up once per device and host code uses that pointer from then on.  24 MiB covers every shape that is split on a
// GPU with up to 256 CUs: slices * tiles <= 256, and no tile of int32 is larger than 128 x 192.
// ---------------------------------------------------------------------------------------------------------------
constexpr size_t kStaticScratchBytes = (size_t)24 << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];   // device address of `scratch` on each device, null until looked up

// Device address of the scratch array on the current device; 0 and a hipError_t / -210 in *rc on failure.
void* static_scratch(int* rc) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) { *rc = (int)e; return nullptr; }
    if (dev < 0 || dev >= kMaxDevices) { *rc = -210; return nullptr; }
    void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));   // the current device's copy
        if (e != hipSuccess || !ptr) { *rc = e != hipSuccess ? (int)e : -210; return nullptr; }
        g_scratch_ptr[dev].store(ptr, std::memory_order_release);   // every thread finds the same address
    }
    *rc = 0;
    return ptr;
}

// Set by gpu_int8_gemm_static around its dispatch: split-K planes go to this buffer instead of a stream-ordered
// allocation.  Thread-local, so calls from other threads through the other entry points are not affected.
thread_local void* tl_scratch = nullptr;
thread_local size_t tl_scratch_bytes = 0;

// Keep freed scratch in the device's default pool instead of returning it to the driver at every synchronization, as
// the reference's runtime layer does at start-up (src/cuda.rs:88-97): otherwise each call that needs scratch pays a
// fresh allocation.
void retain_pool_memory() {
    static PerDeviceOnce once;
    const int dev = PerDeviceOnce::current();
    if (dev < 0 || once.is_done(dev)) return;
    hipMemPool_t pool;
    uint64_t keep = ~(uint64_t)0;
    if (hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess && hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep) == hipSuccess)
        once.mark(dev);
}

// Split-K planes of the allocating entry points: one buffer per (device, stream), made on that stream's first split
// call and kept until the process ends.  Work on one stream is ordered, so its calls can share a buffer (kept_buffers.hpp: also
// those of several host threads, since a call queues both its launches under the buffer's lock), and a stream-ordered
// allocation per call costs about 7 us on the stream's timeline (measured: 31 against 24 us per call at
// M=256, K=12288, N=4096).  The buffer has the one size every shape that the dispatcher splits fits into (slices * tiles <= CUs, and
// no tile of int32 is larger than 128 x 192: 24 MiB on 256 CUs) and is never grown or
// freed, so a captured graph that holds its address stays valid.  At most eight streams per process are served;
// a call on any further stream, a first call made under capture, or a shape beyond the size (a forced configuration)
// falls back to a stream-ordered allocation, and so does hipStreamPerThread (one handle for a different stream in every
// thread).  A stream handle that the runtime reuses after hipStreamDestroy inherits
// the destroyed stream's buffer; work still queued on the destroyed stream at that moment would share it.
constexpr size_t kPlanesPerCu = 128 * 192 * sizeof(int);
KeptBuffers<8> g_planes;

bool is_capturing(hipStream_t st) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) == hipSuccess) return cs != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;   // not known: taken as one
}

// A run on `slices` slices of kslice values of K: `body` writes the int32 planes, a second kernel adds them (exact, so the order of
// the sum does not matter) and applies the epilogue.
template <int OUT_DT, int EPI, class Body>
int launch_split(const GemmArgs& a, int slices, int kslice, hipStream_t st, Body body) {
    const size_t need = (size_t)slices * a.M * a.N * sizeof(int);
    const auto queue = [&](void* planes) -> int {   // every plane element is written before it is read: nothing to clear
        GemmArgs pa = a;
        pa.D = planes;
        pa.kslice = kslice;
        if (const int rc = body(pa)) return rc;
        const int64_t nvec = (int64_t)a.M * a.N / 4;
        const unsigned grid = (unsigned)((nvec + 255) / 256 < 4096 ? (nvec + 255) / 256 : 4096);
        hipLaunchKernelGGL((splitk_epilogue_kernel<OUT_DT, EPI>), dim3(grid), dim3(256), 0, st, a, (const int*)planes, slices);
        return (int)hipGetLastError();
    };
    if (tl_scratch != nullptr) {
        if (need > tl_scratch_bytes) {
            fprintf(stderr, "gpu_int8_gemm_static: M=%d N=%d K=%d needs %zu bytes of split-K scratch, the static buffer has %zu\n",
                    a.M, a.N, a.K, need, tl_scratch_bytes);
            return -210;
        }
        return queue(tl_scratch);
    }
    int rc = 0, dev = 0;
    const auto make = [&](size_t bytes) -> void* {
        void* ptr = nullptr;
        if (is_capturing(st)) return nullptr;
        if (hipMalloc(&ptr, bytes) == hipSuccess) return ptr;
        (void)hipGetLastError();
        return nullptr;
    };
    // hipStreamPerThread: one handle, a different stream in every thread: nothing to key on
    if (st != hipStreamPerThread && hipGetDevice(&dev) == hipSuccess &&
        g_planes.with(dev, st, need, (size_t)device_cu_count() * kPlanesPerCu, make, [&](void* planes) { rc = queue(planes); }))
        return rc;
    void* planes = nullptr;   // from the stream-ordered pool, and back to it
    retain_pool_memory();
    hipError_t e = hipMallocAsync(&planes, need, st);
    if (e != hipSuccess) return (int)e;
    rc = queue(planes);
    e = hipFreeAsync(planes, st);
    return rc == 0 ? (int)e : rc;
}

template <class C, int OUT_DT, int EPI>
int launch_fed_cfg(GemmArgs a, int slices, hipStream_t st) {
    a.tiles_m = (a.M + C::BM - 1) / C::BM;
    a.tiles_n = (a.N + C::BN - 1) / C::BN;
    a.magic = panel_magic(a.tiles_m, a.tiles_n);
    const int64_t ntiles = (int64_t)a.tiles_m * a.tiles_n;
    if (ntiles > 0x7fffffff) return -1;
    auto kern = int8_gemm_fed_kernel<C, OUT_DT, EPI>;
    static PerDeviceOnce once;
    if (const int e = allow_dynamic_lds((const void*)kern, C::SMEM, once)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)ntiles, (unsigned)slices), dim3(C::NT), C::SMEM, st, a);
    KCHECK();
    return 0;
}
template <int OUT_DT, int EPI>
int launch_fed_as(const GemmArgs& a, int width, int slices, hipStream_t st) {
    return width == 1   ? launch_fed_cfg<FedCfg<1>, OUT_DT, EPI>(a, slices, st)
           : width == 2 ? launch_fed_cfg<FedCfg<2>, OUT_DT, EPI>(a, slices, st)
                        : launch_fed_cfg<FedCfg<3>, OUT_DT, EPI>(a, slices, st);
}

// Tile width (of 64 columns) and K slices of the kernel with fetching waves, and its estimated time: rounds of one tile per CU, so many
// us each and per step of 128, more per step where tiles have all their 128 rows of A to fetch and where a CU has several tiles in
// a row (the clock goes down), or the weights' trip from HBM, which a CU cannot take in faster than about 32 bytes per ns.  A split
// pays for its planes and the launch that adds them, and some more where the slices start whole KB apart: their rows then meet in the
// same of HBM's channels (24 x 3072 -> 2048 in eight 9.5 us, in five 8.2).  Tiles of 192 columns share 128-byte lines of outputs
// whose rows are not whole ones (3490 x 512 -> 6536 43.6 us on them, 31.6 on 128 columns).
// The constants are fitted to 3000 shapes of 1 to 8192 rows (K 256 to 14208, N 256 to 28000), calls in a row with weights that come
// from HBM and not from the last-level cache (3 GiB of them in turn).  The choice is 1.1 % slower than the best of all
// widths and slices on the average; constants fitted to weights that had stayed in that cache split K too rarely: 2.7 %, and 128 x 5120
// -> 3072 in one slice 22.9 us, in five 13.4.
struct FedPlan { int width, slices, per; double us; };   // per: K of a slice
FedPlan fed_plan(int64_t M, int64_t N, int64_t K, int num_cu, bool may_split) {
    // fixed, per round, per step, per step with 128 rows, per step and round after the first
    static constexpr double c[3][5] = {{0.89, 2.20, 0.30, 0.07, 0.35}, {1.02, 3.12, 0.50, 0.01, 0.43}, {-0.69, 4.99, 0.89, -0.20, 0.63}};
    const int steps = (int)(K / 128), cus = num_cu;
    const double rows = M < 128 ? (double)M / 128. : 1., hbm = (double)N * (double)K / 32490., plane = 0.05 + (double)M * (double)N * 1.69e-6;
    FedPlan best{3, 1, (int)K, 1e30};
    for (int w = 1; w <= 3; ++w) {
        const int64_t all = (M + 127) / 128 * ((N + 64 * w - 1) / (64 * w));
        const int tiles = all < 1 << 24 ? (int)all : 1 << 24;
        const double* k = c[w - 1];
        const double step = k[2] + rows * k[3];
        if (tiles * 2 > cus || !may_split || steps < 6) {   // nothing to split
            const double n = (double)((tiles + cus - 1) / cus), trip = 3.86 + hbm / (tiles < cus ? tiles : cus);
            double us = k[0] + n * k[1] + (step + (n - 1.) * k[4]) * steps + (w == 3 && N % 64 != 0 ? 1.6 * n : 0.);
            if (us < trip) us = trip;
            if (us < best.us) best = {w, 1, steps * 128, us};
            continue;
        }
        // no more tiles than CUs: one round, however K is split
        const int most = cus / tiles < steps / 3 ? cus / tiles : steps / 3;
        const double fixed = k[0] + k[1] + (w == 3 && N % 64 != 0 ? 1.6 : 0.), per_tile = hbm / tiles;
        int before = 0;
        for (const int asked : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24}) {
            if (asked > most) break;
            const int per = (steps + asked - 1) / asked;
            if (per == before) continue;
            before = per;
            const int s = per * (asked - 1) < steps ? asked : (steps + per - 1) / per;   // no empty slice
            const double trip = 3.86 + per_tile / s;
            double us = fixed + step * per;
            if (s > 1) us += 3.4 + s * plane + (per % 8 == 0 ? 0.29 : 0.);
            if (us < trip) us = trip;
            if (us < best.us) best = {w, s, per * 128, us};
        }
    }
    return best;
}
// Whether the two-group kernel is estimated to be faster than that.  Its time on the same scale is fitted to 260 shapes (8.5 % rms).  `wide`:
// outputs of 32 bits.  In one round of 128-row tiles a CU's epilogue has nothing beside it, and with 32 bits it writes twice as much there as in
// the smaller tiles of the other kernel: up to K = 1024 1.05 times as long as that (93 shapes; 5377 x 768 -> 1112 17.8 us and 15.6,
// 2433 x 768 -> 2648 18.9 and 16.8), from there on 0.97 (45).  Weights from HBM, outputs in turn: the choice is 0.6 % slower than the faster
// of the two kernels over 790 shapes with 16-bit outputs, 0.45 % over 1490 with 32-bit ones (0.75 % without that line).
bool pp_wins(int64_t M, int64_t N, int64_t K, int cus, bool wide) {
    const PpSplit sp = pp_split(M, N, cus);
    if (wide && sp.rows == PpS::BM && sp.small <= cus && K <= 1024) return false;
    return 1.1 + sp.rounds * (7.2 + 1.25 * (double)(K / 128)) < fed_plan(M, N, K, cus, true).us;
}

// Whether a call may split K over workgroups.  Captured graphs and the static entry point do so only for the shapes that always did
// there: elsewhere a graph holds no address of the stream's planes, so that it may be replayed on any stream, and the static
// entry point leaves its buffer alone.
bool fed_may_split(int64_t M, int64_t N, int64_t K, hipStream_t st) {
    if (M <= 256 && K >= 4096 && N >= 1024 && N <= (M > 64 ? 8192 : 4096)) return true;
    return tl_scratch == nullptr && !is_capturing(st);
}


FedPlan fed_plan_or_forced(int64_t M, int64_t N, int64_t K, bool may_split) {
    const int force = g_force_cfg.load(std::memory_order_relaxed) - 7000, width = force / 100;
    if (force < 0 || width < 1 || width > 3) return fed_plan(M, N, K, device_cu_count(), may_split);
    const int steps = (int)(K / 128), asked = !may_split || force % 100 < 1 ? 1 : force % 100 < steps ? force % 100 : steps, per = (steps + asked - 1) / asked;
    return {width, (steps + per - 1) / per, per * 128, 0.};
}

template <int OUT_DT, int EPI>
int launch_fed(GemmArgs a, hipStream_t st) {
    bool vec_ok, aligned;
    epilogue_alignment<OUT_DT, EPI>(a, vec_ok, aligned);
    if (!aligned) return launch_cfg<CfgM, OUT_DT, EPI>(a, st);   // only a forced family
    FedPlan p = fed_plan_or_forced(a.M, a.N, a.K, true);
    if (p.slices > 1 && !fed_may_split(a.M, a.N, a.K, st)) p = fed_plan_or_forced(a.M, a.N, a.K, false);
    a.kslice = 0;
    if (p.slices == 1) return launch_fed_as<OUT_DT, EPI>(a, p.width, 1, st);
    return launch_split<OUT_DT, EPI>(a, p.slices, p.per, st, [&](const GemmArgs& pa) { return launch_fed_as<DT_F32, EPI_ACC>(pa, p.width, p.slices, st); });
}

template <int MT, int NWK, int OUT_DT, int EPI>
int launch_rows_cfg(const GemmArgs& a, bool vec_ok, int slices, hipStream_t st) {
    using C = RowsCfg<MT, NWK>;
    auto kern = int8_gemm_rows_kernel<MT, NWK, OUT_DT, EPI>;
    static PerDeviceOnce once;
    if (const int e = allow_dynamic_lds((const void*)kern, C::SMEM, once)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)((a.N + C::BN - 1) / C::BN), (unsigned)slices), dim3(C::NT), C::SMEM, st, a, vec_ok);
    KCHECK();
    return 0;
}
template <int OUT_DT_, int EPI>
int launch_rows_as(const GemmArgs& a, int mt, int nwk, bool vec_ok, int slices, hipStream_t st) {
    constexpr int OUT_DT = EPI == EPI_ACC ? DT_F32 : OUT_DT_;   // int32 sums have no output type
    switch (mt * 10 + nwk) {
        case 12: return launch_rows_cfg<1, 2, OUT_DT, EPI>(a, vec_ok, slices, st);
        case 14: return launch_rows_cfg<1, 4, OUT_DT, EPI>(a, vec_ok, slices, st);
        case 18: return launch_rows_cfg<1, 8, OUT_DT, EPI>(a, vec_ok, slices, st);
        case 22: return launch_rows_cfg<2, 2, OUT_DT, EPI>(a, vec_ok, slices, st);
        case 24: return launch_rows_cfg<2, 4, OUT_DT, EPI>(a, vec_ok, slices, st);
        case 42: return launch_rows_cfg<4, 2, OUT_DT, EPI>(a, vec_ok, slices, st);
        case 44: return launch_rows_cfg<4, 4, OUT_DT, EPI>(a, vec_ok, slices, st);
        case 62: return launch_rows_cfg<6, 2, OUT_DT, EPI>(a, vec_ok, slices, st);
        default: return launch_rows_cfg<8, 2, OUT_DT, EPI>(a, vec_ok, slices, st);
    }
}

// K that a split over workgroups has to take off each of them to be worth the planes and the second launch, about 4 us (rows
// 77, us unsplit and split: 1536 -> 4608 9.1 and 11.2, 3072 -> 3072 15.0 and 12.1; rows 64: 3072 -> 3072 in two 9.3 and 10.9,
// 4096 -> 4096 in two 12.3 and 11.7).
constexpr int kSplitRowsK = 1800;

// M <= 128.  The widest split of K inside the workgroup that still gives every CU at most one workgroup; where even that
// leaves CUs without one, K is split over workgroups as well.
struct RowsPlan { int mt, nwk, tiles, slices, per; };   // per: K of a slice
RowsPlan rows_plan(int64_t M, int64_t N, int64_t K, int cus, bool may_split) {
    const int mt = M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : M <= 96 ? 6 : 8;
    const auto tiles = [&](int nwk) { return (int)((N * nwk + 127) / 128); };
    const int most = mt == 1 ? 8 : mt <= 4 ? 4 : 2;
    int nwk = 2;
    while (nwk < most && tiles(2 * nwk) <= cus) nwk *= 2;
    if (mt == 1 && tiles(2) > cus) nwk = 4;   // several rounds: the smaller tiles fill the last one better
    const int unit = 64 * nwk * (mt * nwk <= 8 ? 8 : 4), panels = (int)((K + unit - 1) / unit);
    int slices = may_split ? cus / tiles(nwk) : 1;
    if (slices > panels) slices = panels;
    if (slices > 1 && K / slices * (slices - 1) < kSplitRowsK) slices = 1;
    if (slices <= 1) return {mt, nwk, tiles(nwk), 1, (int)K};
    const int per = (panels + slices - 1) / slices;
    return {mt, nwk, tiles(nwk), (panels + per - 1) / per, per * unit};   // no empty slice
}

template <int OUT_DT, int EPI>
int launch_rows(GemmArgs a, hipStream_t st) {
    bool vec_ok, aligned;
    epilogue_alignment<OUT_DT, EPI>(a, vec_ok, aligned);
    const RowsPlan p = rows_plan(a.M, a.N, a.K, device_cu_count(), vec_ok);
    if (p.slices == 1) {
        a.kslice = 0;
        return launch_rows_as<OUT_DT, EPI>(a, p.mt, p.nwk, vec_ok, 1, st);
    }
    // Under capture (fed_may_split has the reason) and in the static entry point outputs that are narrow, or whose rows or pointers are
    // not whole 16 bytes, do not split K, nor do more rows with shorter K.
    if ((a.N < 1024 || !aligned || (a.M <= 16 ? a.K < 2560 : a.K < 3072 || a.N > 1280)) && (tl_scratch != nullptr || is_capturing(st)))
        return aligned ? launch_fed<OUT_DT, EPI>(a, st) : a.N < 1024 ? launch_cfg<CfgS, OUT_DT, EPI>(a, st) : launch_cfg<CfgM, OUT_DT, EPI>(a, st);
    return launch_split<OUT_DT, EPI>(a, p.slices, p.per, st, [&](const GemmArgs& pa) { return launch_rows_as<DT_F32, EPI_ACC>(pa, p.mt, p.nwk, true, p.slices, st); });
}

// Whether the kernel for up to 128 rows runs a shape.  For outputs of whole 16 bytes: up to 64 rows and 8192 columns, from the K on
// from which it is faster than the kernel with fetching waves up to where that one splits K better.  Its time over the other's by
// 6000 shapes with weights from HBM, calls in a row:
//   1 to 16 rows: 0.6 to 0.98 from K = 1408 to 4000, 0.6 to 1.1 above (1.05 to 1.3 for 1280 to 2048 columns from K = 8192 on), 1.0 and
//     more below.  Beyond 8192 columns, where it takes one more round: 0.91 up to K = 1920, 1.06 to 1.13 up to 3300, 0.8 to 1.07 above (from
//     9 rows on also 1.04 to 1.11 up to 9500 columns from K = 10240 on), but 0.9 to 1.2 there where weight rows are whole 4 KB (from 9 rows
//     on: whole 2 KB), which the other kernel's staggered starts suit.
//   17 to 32: 0.77 to 1.0 from K = 1920 to 4096.  Above, 0.81 to 1.15 up to 1280 columns; 1.0 to 1.45 from there to 5120, where this kernel
//     splits K over workgroups too or leaves CUs without one; 0.76 to 1.05 beyond (from K = 8192 on: beyond 6144), where its 160 to 256
//     workgroups take all of K and the other kernel has planes to add.
//   33 to 64: 0.88 to 1.0 from K = 1024 to 2304 and 0.84 to 1.0 from 2816 to 4096, but 1.0 to 1.16 between with few columns (its panels of
//     1024 end half empty) and from 3072 to 4096 columns above K = 3584.  From K = 4096 on 0.8 to 1.0 up to 1280 columns, 1.0 to 1.38 from
//     there to 6144, 0.85 to 1.08 beyond, up to K = 10240.
//   65 to 128: 1.0 to 1.6.
// Other outputs have the register-staged tiles beside them, which have less to start (128 rows 1152 -> 512 8.5 and 7.5 us; but 128
// rows 1280 -> 640 8.5 and 9.2).
bool rows_kernel_wins(int64_t M, int64_t N, int64_t K, bool aligned) {
    if (aligned && M <= 16) {
        if (N <= 8192) return K >= 1408;
        return N <= 16384 && K >= 1408 && (K <= 1920 || (K >= 3328 && (M <= 8 ? K % 4096 != 0 : K % 2048 != 0 && (K <= 10240 || N > 9500))));
    }
    if (aligned && M <= 32) return N <= 8192 && K >= 1920 && (K <= 4096 || N <= 1280 || N > (K < 8192 ? 5120 : 6144));
    if (aligned && M <= 64) {
        if (N > 8192 || K < 1024) return false;
        if (K <= 3584) return K <= 2304 || K > 2816 || N > 3072;
        return K < 4096 ? N <= 3072 || N > 4096 : N <= 1280 || (N > 6144 && K <= 10240);
    }
    if (aligned) return false;
    if (K < (M > 96 ? 1024 : 768) || (M > 16 && N > 16384)) return false;
    if (K < 896) return !(N < 1152 && (M <= 32 || M > 64));
    return !(M > 64 && K >= 1024 && K < (M > 96 ? 1408 : 1280) && N < (K < 1152 ? 1024 : 640));
}

// `start`: the low four bits of A's and W's addresses together.  The kernel for up to 128 rows asks for 16-byte starts (its weight
// loads and its DMA).  The other DMA kernels take operands from any 4-byte address, the alignment that a DMA of several
// dwords needs; an operand that starts there but not at 16 bytes (a view into a larger buffer) goes to them from the sizes on from which
// such calls always did, and to the register-staged tiles below.  Other starts always take the register-staged tiles, whose
// ordinary loads may be unaligned.  `aligned` as epilogue_alignment has it, `wide` as pp_wins.
int choose_cfg(int64_t M, int64_t N, int64_t K, int start, bool aligned, bool wide) {
    const int force = g_force_cfg.load(std::memory_order_relaxed);
    const bool tiles_ok = M * K < ((int64_t)1 << 32) && N * K < ((int64_t)1 << 32) && (K % 128) == 0;   // 32-bit lane offsets, whole steps
    const bool dma_ok = tiles_ok && (start & 3) == 0;
    if (force == 5) return tiles_ok && start == 0 && M <= 128 ? 5 : 1;
    if (force == 7 || force / 1000 == 7) return dma_ok ? 7 : 1;
    if (force == 9 || force / 1000 == 9) return dma_ok ? 9 : 1;
    if (force == 1 || force == 2) return force;
    if (tiles_ok && start == 0 && M <= 128 && rows_kernel_wins(M, N, K, aligned)) return 5;
    const int cus = device_cu_count();
    // one or two steps of K and little to store: 512 threads and 96 KB of LDS to start cost more than they give (500 shapes, register-
    // staged tiles over fetching waves: K = 128 0.93 to 1.0, K = 256 0.94 to 1.0, K = 384 0.97 to 1.1; K = 256 with 1 << 21 outputs 1.1; one step
    // and more columns than the CUs take at once in tiles of 64, 25 x 24784 4.4 us and 5.1, but 73 x 10368 4.4 and 3.8)
    const bool tiny = K <= 256 && (M * N <= 1 << 19 || (K <= 128 && M * N <= 1 << 20 && N > 64 * cus));
    const int large = !dma_ok || !aligned ? 1 : M >= 512 && N >= 512 && pp_wins(M, N, K, cus, wide) ? 9 : 7;
    if (dma_ok && aligned && start == 0 && !tiny) return large;
    // the register-staged tiles: large ones, or for operands off 16 bytes the DMA kernels, as soon as there is work for them
    if (M <= 256 && N >= 1024 && tiles_ok && K >= 512) return K >= 1536 || (M > 128 && N >= 8192) ? large : 2;
    const int64_t tiles_s = ((M + 127) / 128) * ((N + 191) / 192);
    if (M >= 512 && N >= 512 && tiles_s > cus) return large;
    if (tiles_ok && M > 128 && N >= 192 && (tiles_s >= 96 || (tiles_s >= 40 && K >= 2048) || (M <= 512 && N >= 1024 && K >= 8192))) return large;
    const int64_t tiles_m = ((M + 127) / 128) * ((N + 127) / 128);
    if (M > 64 && N > 64 && tiles_m >= 256) return 1;
    return 2;
}

template <int OUT_DT, int EPI>
int dispatch_cfg(const GemmArgs& a, hipStream_t st) {
    bool vec_ok, aligned;
    epilogue_alignment<OUT_DT, EPI>(a, vec_ok, aligned);
    switch (choose_cfg(a.M, a.N, a.K, (int)(((uintptr_t)a.A | (uintptr_t)a.W) & 15), aligned, EPI == EPI_ACC || OUT_DT == DT_F32)) {
        case 5: return launch_rows<OUT_DT, EPI>(a, st);
        case 7: return launch_fed<OUT_DT, EPI>(a, st);
        case 9: return launch_pp<OUT_DT, EPI>(a, st);
        case 1: return launch_cfg<CfgM, OUT_DT, EPI>(a, st);
        default: return launch_cfg<CfgS, OUT_DT, EPI>(a, st);
    }
}

template <int EPI>
int dispatch_dt(const GemmArgs& a, int out_dt, hipStream_t st) {
    switch (out_dt) {
        case DT_F32: return dispatch_cfg<DT_F32, EPI>(a, st);
        case DT_F16: return dispatch_cfg<DT_F16, EPI>(a, st);
        case DT_BF16: return dispatch_cfg<DT_BF16, EPI>(a, st);
        default: return -1;
    }
}

bool shape_ok(int64_t M, int64_t N, int64_t K) {
    return M <= 0x7fffffff && N <= 0x7fffffff && K <= 0x7fffffff - 8 && (K % 8) == 0 && M * N < (int64_t)1 << 40;
}

// K % 16 == 8 (the reference's alignment-8 tile configurations, csrc/vendor/cutlass_gemm_int8.cu:191,237-247,265): the
// kernels here read 16-byte vectors of K, so such a call runs on copies of A and W whose rows carry eight more zero
// bytes, which leave every int32 sum as it was.  The copies live in one stream-ordered allocation for the length of
// the call.  No model in the reference's tree has such a K; the path exists so that the call is not refused.
__global__ void __launch_bounds__(256) pad_k_rows_kernel(const int8_t* src, int8_t* dst, int64_t rows, int k8) {
    const int64_t n = rows * (k8 + 1);   // 8-byte pieces of the destination
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / (k8 + 1);
        const int c = (int)(i - r * (k8 + 1));
        uint2 v = make_uint2(0u, 0u);
        if (c < k8) v = *reinterpret_cast<const uint2*>(src + (r * k8 + c) * 8);
        *reinterpret_cast<uint2*>(dst + i * 8) = v;
    }
}

struct PaddedK {
    int8_t* buf = nullptr;
    hipStream_t st;
    int rc = 0;
    // replaces A, W and K by the padded copies when K % 16 != 0
    PaddedK(const int8_t*& A, const int8_t*& W, int64_t M, int64_t N, int64_t& K, hipStream_t stream) : st(stream) {
        if ((K % 16) == 0) return;
        if ((((uintptr_t)A | (uintptr_t)W) & 7) != 0) { rc = -1; return; }
        const int64_t k16 = K + 8;
        retain_pool_memory();
        hipError_t e = hipMallocAsync((void**)&buf, (size_t)((M + N) * k16), st);
        if (e != hipSuccess) { buf = nullptr; rc = (int)e; return; }
        const int8_t* src[2] = {A, W};
        int8_t* dst[2] = {buf, buf + M * k16};
        const int64_t rows[2] = {M, N};
        for (int i = 0; i < 2; ++i) {
            const int64_t pieces = rows[i] * (k16 / 8);
            const unsigned grid = (unsigned)((pieces + 255) / 256 < 8192 ? (pieces + 255) / 256 : 8192);
            hipLaunchKernelGGL(pad_k_rows_kernel, dim3(grid), dim3(256), 0, st, src[i], dst[i], rows[i], (int)(K / 8));
        }
        hipError_t le = hipGetLastError();
        if (le != hipSuccess) rc = (int)le;
        A = dst[0];
        W = dst[1];
        K = k16;
    }
    ~PaddedK() { if (buf) (void)hipFreeAsync(buf, st); }
};

__global__ void mfma_layout_probe_kernel(int* out) {
    const int lane = threadIdx.x;
    v16i di, dj;
#pragma unroll
    for (int r = 0; r < 16; ++r) { di[r] = 0; dj[r] = 0; }
    const bool k0 = lane < 32;                       // lanes that feed the first 16 K bytes
    const v4i row = v4i{k0 ? (lane & 31) : 0, 0, 0, 0};  // byte 0 = row index
    const v4i one = v4i{k0 ? 1 : 0, 0, 0, 0};
    di = __builtin_amdgcn_mfma_i32_32x32x32_i8(row, one, di, 0, 0, 0);  // D[i][j] = i
    dj = __builtin_amdgcn_mfma_i32_32x32x32_i8(one, row, dj, 0, 0, 0);  // D[i][j] = j
#pragma unroll
    for (int r = 0; r < 16; ++r) out[lane * 16 + r] = di[r] * 32 + dj[r];
}

// Nothing but v_mfma_i32_32x32x32_i8: four waves per CU, sixteen independent accumulator tiles per wave (the register
// shape of the GEMM kernels), operands held in registers.  What this loop sustains is the matrix pipes' ceiling under
// the chip's power management for the given operand bits; the shader-clock count per workgroup gives the clock.
__global__ void __launch_bounds__(256, 1) mfma_ceiling_kernel(int iters, int random_bits, int form, long long* cycles, int* sink) {
    const uint32_t tid = threadIdx.x + blockIdx.x * 256u;
    auto hash = [](uint32_t x) { x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16; return x; };
    v4i a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            a[i][r] = random_bits ? (int)hash(tid * 977u + i * 17u + r) : 0;
            b[i][r] = random_bits ? (int)hash(tid * 613u + i * 29u + r + 99991u) : 0;
        }
    if (form == 16) {   // v_mfma_i32_16x16x64_i8: 32 accumulator tiles with their own operand pairs, the same operations per iteration
        v4i c4[32];
        v4i a2[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) a2[i][r] = random_bits ? (int)hash(tid * 331u + i * 41u + r + 77777u) : 0;
#pragma unroll
        for (int i = 0; i < 32; ++i) c4[i] = v4i{0, 0, 0, 0};
        const long long t0 = (long long)__builtin_readcyclecounter();
        for (int it = 0; it < iters; ++it) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int i = 0; i < 32; ++i) {
                    c4[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[(i >> 2) & 3], i < 16 ? a[i & 3] : a2[i & 3], c4[i], 0, 0, 0);
                    SCHED_FENCE();
                }
        }
        const long long t1 = (long long)__builtin_readcyclecounter();
        int s = 0;
#pragma unroll
        for (int i = 0; i < 32; ++i) s += c4[i][0] + c4[i][1] + c4[i][2] + c4[i][3];
        if (s == 0x7fffffff) sink[0] = s;   // keeps the accumulators alive
        if (threadIdx.x == 0) cycles[blockIdx.x] = t1 - t0;
        return;
    }
    v16i acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0;
    const long long t0 = (long long)__builtin_readcyclecounter();
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[i >> 2], a[i & 3], acc[i], 0, 0, 0);
                SCHED_FENCE();
            }
    }
    const long long t1 = (long long)__builtin_readcyclecounter();
    int s = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) s += acc[i][r];
    if (s == 0x7fffffff) sink[0] = s;   // keeps the accumulators alive
    if (threadIdx.x == 0) cycles[blockIdx.x] = t1 - t0;
}

}  // namespace

GPU_API int gpu_int8_gemm(const int8_t* A, const int8_t* W, const float* xs, const float* ws, const void* bias, void* D,
                          int64_t M, int64_t N, int64_t K, int out_dt, void* stream) {
    if (M == 0 || N == 0 || K == 0) return 0;  // csrc/vendor/cutlass_gemm_int8.cu:377
    if (out_dt < DT_F32 || out_dt > DT_BF16 || M < 0 || N < 0 || K < 0 || !shape_ok(M, N, K)) return -200;
    PaddedK pad(A, W, M, N, K, (hipStream_t)stream);
    if (pad.rc != 0) return pad.rc < 0 ? -200 : pad.rc;
    GemmArgs a{A, W, xs, ws, bias, nullptr, nullptr, D, (int)M, (int)N, (int)K, 0, 0, 0, 0};
    const int rc = dispatch_dt<EPI_PLAIN>(a, out_dt, (hipStream_t)stream);
    return rc < 0 ? -200 : rc;
}

GPU_API int gpu_int8_gemm_residual(const int8_t* A, const int8_t* W, const float* xs, const float* ws, const void* bias,
                                   const void* rscale, const void* resid, void* D, int64_t M, int64_t N, int64_t K,
                                   int out_dt, void* stream) {
    if (M == 0 || N == 0) return 0;                       // csrc/vendor/cutlass_gemm_int8.cu:353
    if (K == 0 || !rscale || !resid) return -201;         // :355-357
    if (out_dt < DT_F32 || out_dt > DT_BF16 || M < 0 || N < 0 || K < 0 || !shape_ok(M, N, K)) return -201;
    PaddedK pad(A, W, M, N, K, (hipStream_t)stream);
    if (pad.rc != 0) return pad.rc < 0 ? -201 : pad.rc;
    GemmArgs a{A, W, xs, ws, bias, rscale, resid, D, (int)M, (int)N, (int)K, 0, 0, 0, 0};
    const int rc = dispatch_dt<EPI_RESID>(a, out_dt, (hipStream_t)stream);
    return rc < 0 ? -201 : rc;
}

GPU_API int gpu_int8_gemm_static(const int8_t* A, const int8_t* W, const float* xs, const float* ws, const void* bias, void* D,
                                 int64_t M, int64_t N, int64_t K, int out_dt, void* stream) {
    if (M == 0 || N == 0 || K == 0) return 0;
    if (out_dt < DT_F32 || out_dt > DT_BF16 || M < 0 || N < 0 || K < 0 || !shape_ok(M, N, K)) return -200;
    if ((K % 16) != 0) return -200;   // the K % 16 == 8 path allocates its padded copies
    int rc = 0;
    void* ptr = static_scratch(&rc);
    if (!ptr) return rc;
    GemmArgs a{A, W, xs, ws, bias, nullptr, nullptr, D, (int)M, (int)N, (int)K, 0, 0, 0, 0};
    tl_scratch = ptr;
    tl_scratch_bytes = kStaticScratchBytes;
    rc = dispatch_dt<EPI_PLAIN>(a, out_dt, (hipStream_t)stream);
    tl_scratch = nullptr;
    tl_scratch_bytes = 0;
    return rc == -210 ? -210 : rc < 0 ? -200 : rc;
}

GPU_API int64_t gpu_int8_gemm_static_limit(void) { return (int64_t)kStaticScratchBytes; }

GPU_API int gpu_int8_gemm_acc(const int8_t* A, const int8_t* W, int32_t* acc, int64_t M, int64_t N, int64_t K, void* stream) {
    if (M == 0 || N == 0 || K == 0) return 0;
    if (M < 0 || N < 0 || K < 0 || !shape_ok(M, N, K)) return -200;
    PaddedK pad(A, W, M, N, K, (hipStream_t)stream);
    if (pad.rc != 0) return pad.rc < 0 ? -200 : pad.rc;
    GemmArgs a{A, W, nullptr, nullptr, nullptr, nullptr, nullptr, acc, (int)M, (int)N, (int)K, 0, 0, 0, 0};
    const int rc = dispatch_cfg<DT_F32, EPI_ACC>(a, (hipStream_t)stream);
    return rc < 0 ? -200 : rc;
}

// Test hook: force a kernel family (1 = 128x128, 2 = 64x64 register-staged tiles; 5 = up to 128 rows; 7 = waves that
// fetch for others, 7000 + 100 * width + slices = those with that tile width (of 64 columns) and split; 9 = two-group
// kernel, 9000 + 10 * kind + split = that with one of its tile grids; -1 or anything else = automatic).
GPU_API int gpu_int8_gemm_force_config(int cfg) {
    g_force_cfg.store(cfg, std::memory_order_relaxed);
    return 0;
}

// Test hook: what a call outside capture runs, for operands that start `start` bytes behind 16-byte addresses and outputs of whole 16
// bytes or not.  out[0] = family as above, out[1] = tile width (family 7; of 64 columns), 16-row tiles (5) or store policy of outputs from
// a whole line on (9); out[2] = slices of K.  Outputs are 16-bit ones, with aligned = 3 32-bit ones.
GPU_API int gpu_internal_int8_gemm_plan(int64_t M, int64_t N, int64_t K, int start, int aligned, int32_t* out) {
    if (M <= 0 || N <= 0 || K <= 0 || !shape_ok(M, N, K) || !out) return -200;
    const bool wide = aligned == 3;
    out[0] = choose_cfg(M, N, K, start & 15, aligned != 0, wide);
    out[1] = 0;
    out[2] = 1;
    if (out[0] == 7 && aligned) {
        const FedPlan p = fed_plan_or_forced(M, N, K, true);
        out[1] = p.width;
        out[2] = p.slices;
    } else if (out[0] == 5) {
        const RowsPlan p = rows_plan(M, N, K, device_cu_count(), (N & 3) == 0);
        out[1] = p.mt;
        out[2] = p.slices;
    } else if (out[0] == 9) {
        out[1] = store_policy(M, N * (wide ? 4 : 2), 0);
    }
    return 0;
}

GPU_API int gpu_mfma_ceiling_probe(int iters, int random_bits, int64_t* cycles, int32_t* sink, void* stream) {
    if (iters <= 0) return 0;
    // random_bits: 0 = zero operands, 1 = random; + 2 = the 16x16x64 form of the instruction instead of 32x32x32
    hipLaunchKernelGGL(mfma_ceiling_kernel, dim3((unsigned)device_cu_count()), dim3(256), 0, (hipStream_t)stream, iters, random_bits & 1,
                       (random_bits & 2) ? 16 : 32, (long long*)cycles, (int*)sink);
    KCHECK();
    return 0;
}

GPU_API int gpu_mfma_layout_probe(int32_t* out, void* stream) {
    hipLaunchKernelGGL(mfma_layout_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, out);
    KCHECK();
    return 0;
}
