// The LoRA bottlenecks of RWKV6TimeMix in two forward and two backward passes, for MI355X
// (gfx950).  Sequence-first [T,B,C] bf16, N = T*B token rows n = t*B + b.
//
// Reference (/root/reference/rwkv_megatron/rwkv6_layer_specs.py):
//   bottleneck(x) = tanh(x W_down) W_up + bias                  :177-195
//   token shift:  E = 5, R = 32, on xxx = x + (shift(x) - x) maa  :440-452 (LERP below)
//   decay:        E = 1, R = 64, on the decay's mix               :454
// Weights are read as the module holds them, W_down [C, E*R] and W_up [E*R, C], bf16 or fp32
// (fp32 is rounded to bf16 on the way into LDS).
//
//   rwkv6_lora_down_kernel  neck = tanh(xxx W_down) (xxx formed on the way, never stored)
//   (rwkv6_lora_up_kernel of lora.hip consumes neck: the mixes, or the decay)
//   rwkv6_lora_dpre_kernel  d_pre = (sum_c dm_e W_up_e) (1 - neck^2), dm_e = d_out_e (shift(x) - x)
//                           (LERP) or d_out: every channel of a token tile in one workgroup
//   rwkv6_lora_grads_kernel everything else, a 64-channel column per workgroup walking token
//                           tiles: d_xxx = d_pre W_down^T, dx, and the weight, bias and maa
//                           gradients accumulated over the tiles in MFMA accumulators
//   rwkv6_lora_reduce_kernel sums the workgroups' partial parameter gradients in order
//
// Why two backward passes over d_out: d_pre needs all channels of a token, the weight gradients
// all tokens of a channel.  Reading d_out and x twice (12 x 2C bytes a token) and recomputing
// m = neck W_up costs less than passing dm ([5,N,C]), the two lerp sums, xxx and d_xxx through
// HBM between a kernel per step and the library's batched GEMMs of 32 columns.  Measured at N =
// 16384, C = 2048, forward and backward: the token shift 718 -> 390 us (18 -> 5 launches), the
// decay 391 -> 127 us (16 -> 5); the general path (other ranks) is in timemix.py.
#include <algorithm>
#include <utility>

#include "common.h"
#include "../../include/rwkv6_amd.h"

#define LF_THR 512        // 8 waves
#define LF_TT 64          // token rows of a tile
#define LF_TS 72          // row stride (elements) of a 64-channel bf16 tile in LDS
#define LF_MS 68          // row stride (floats) of a 64-channel fp32 tile
// the bottlenecks the kernels are compiled for: the token shift's and the decay's
#define LF_E_MIX 5
#define LF_R_MIX 32
#define LF_R_DECAY 64

namespace {

// q or zeros, component by component (a select of whole vectors goes through memory)
__device__ __forceinline__ uint4 keep4(bool c, uint4 q) {
    return make_uint4(c ? q.x : 0u, c ? q.y : 0u, c ? q.z : 0u, c ? q.w : 0u);
}
__device__ __forceinline__ float4 ld_f4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ void ld_f8(const float* p, float* f) {
    const float4 a = ld_f4(p), b = ld_f4(p + 4);
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
    f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}
__device__ __forceinline__ void st_f8(float* p, const float* f) {
    *reinterpret_cast<float4*>(p) = make_float4(f[0], f[1], f[2], f[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(f[4], f[5], f[6], f[7]);
}
// Sum of v[0..7] over the wave's 8 token rows (lane bits 3-5), transposing: lane (rw, cg) gets
// the sum of element 4 b3 + 2 b4 + b5 of column group cg.  row_ror:8 for bit 3, then the row
// swaps for bits 4 and 5 (their two results sum to the even row's A value plus the odd one's in
// the even rows and to the B values in the odd ones); a fixed order.  Overwrites v.
__device__ __forceinline__ float lf_rows8(float* v, int lane) {
    const bool up = lane & 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (up ? v[i + 4] : v[i]) + lane_xor8(up ? v[i] : v[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 2]), false, false);
        v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[1]), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// raw parameters (bf16 or fp32 by `dtype`), two unconditional 16-byte loads as load_param8
struct PRaw { uint4 a, b; };
__device__ __forceinline__ PRaw p_load(const void* p, int dtype, int64_t off) {
    const bool h = dtype == RWKV6_BF16;
    const char* c = reinterpret_cast<const char*>(p) + (h ? off * 2 : off * 4);
    return {*reinterpret_cast<const uint4*>(c), *reinterpret_cast<const uint4*>(c + (h ? 0 : 16))};
}
__device__ __forceinline__ void p_f32(const PRaw& r, int dtype, float* f) {
    float hf[8];
    unpack8(r.a, hf);
    const unsigned w[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
#pragma unroll
    for (int s = 0; s < 8; ++s) f[s] = dtype == RWKV6_BF16 ? hf[s] : __builtin_bit_cast(float, w[s]);
}

}  // namespace

// neck[n][r] = tanh(sum_c xxx[n][c] W_down[c][r]), xxx = x + (shift(x) - x) maa rounded to bf16
// (LERP) or x.  Workgroup = TT token rows x all ER columns, 64 channels a step through double-
// buffered LDS tiles (one barrier a step), the loads of two steps ahead in registers.  The
// product is formed transposed (W_down^T as the A operand), so a lane ends with four adjacent
// columns of one token.  Wave (tt, hh) takes tokens 16 tt.. and the column tiles 2i + hh.
template <int ER, bool LERP, bool WF32, int TT>
__global__ void __launch_bounds__(8 * TT)
rwkv6_lora_down_kernel(const uint16_t* __restrict__ x, const void* __restrict__ maa, int mdt,
                       const void* __restrict__ wd, uint16_t* __restrict__ neck, int64_t N,
                       int64_t B, int64_t C) {
    constexpr int WS = ER + 8, THR = 8 * TT, NP = 64 * ER / 8, NPT = (NP + THR - 1) / THR, NA = ER / 32;
    __shared__ __attribute__((aligned(16))) uint16_t xs[2][TT][LF_TS];
    __shared__ __attribute__((aligned(16))) uint16_t ws[2][64][WS];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, L = lane & 15, q = lane >> 4;
    const int tt = wv % (TT / 16), hh = wv / (TT / 16), row = tid >> 3, cg = tid & 7;
    const int64_t n0 = (int64_t)blockIdx.x * TT, n = n0 + row < N ? n0 + row : N - 1;
    const uint16_t* xrow = x + n * C + 8 * cg;
    const uint16_t* prow = x + (n >= B ? n - B : n) * C + 8 * cg;
    const float keep = n >= B ? 1.f : 0.f;
    const int nk = (int)(C / 64);
    struct Step { uint4 x, p; PRaw m; WRaw<WF32> w[NPT]; };
    auto load = [&](Step& s, int k) {
        s.x = *reinterpret_cast<const uint4*>(xrow + 64 * k);
        if (LERP) {
            s.p = *reinterpret_cast<const uint4*>(prow + 64 * k);
            s.m = p_load(maa, mdt, 64 * k + 8 * cg);
        }
#pragma unroll
        for (int i = 0; i < NPT; ++i)          // the tile's 64 rows are contiguous; a piece past
            s.w[i] = w_load<WF32>(wd, (int64_t)64 * k * ER + 8 * min(tid + THR * i, NP - 1));  // the end repeats the last
    };
    f32x4 acc[NA] = {};
    auto step = [&](Step& s, int k) {
        uint16_t (*xt)[LF_TS] = xs[k & 1];
        uint16_t (*wt)[WS] = ws[k & 1];
        uint4 xq = s.x;
        if (LERP) {
            float xv[8], xp[8], mv[8];
            unpack8(s.x, xv);
            unpack8(s.p, xp);
            p_f32(s.m, mdt, mv);
#pragma unroll
            for (int j = 0; j < 8; ++j) xv[j] += (xp[j] * keep - xv[j]) * mv[j];
            xq = pack8(xv);
        }
        *reinterpret_cast<uint4*>(&xt[row][8 * cg]) = xq;
#pragma unroll
        for (int i = 0; i < NPT; ++i) {
            const int p = min(tid + THR * i, NP - 1);
            *reinterpret_cast<uint4*>(&wt[p / (ER / 8)][8 * (p % (ER / 8))]) = w_bf16<WF32>(s.w[i]);
        }
        __syncthreads();
        load(s, min(k + 2, nk - 1));
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const bf16x8 b = ld_bf16x8(&xt[16 * tt + L][32 * ks + 8 * q]);
#pragma unroll
            for (int i = 0; i < NA; ++i)
                acc[i] = mfma32(lds_tr8(&wt[0][0], WS, 32 * ks, 16 * (2 * i + hh), lane), b, acc[i]);
        }
    };
    Step s0, s1;
    load(s0, 0);
    load(s1, min(1, nk - 1));
    for (int k = 0; k < nk; k += 2) {
        step(s0, k);
        if (k + 1 < nk) step(s1, k + 1);
    }
    const int64_t t = n0 + 16 * tt + L;
    if (t < N) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
            *reinterpret_cast<uint2*>(neck + t * ER + 16 * (2 * i + hh) + 4 * q) =
                make_uint2(pk2(tanhf(acc[i][0]), tanhf(acc[i][1])), pk2(tanhf(acc[i][2]), tanhf(acc[i][3])));
    }
}

// d_pre[n][e R + r] = (sum_c dm_e[n][c] W_up[e][r][c]) (1 - neck^2), dm_e = d_out_e (shift(x) -
// x) rounded to bf16 (LERP; the MFMA operand the weight gradient uses too) or d_out_e.
// Workgroup = TT token rows x all channels, as the down kernel; per step the dm tiles of all
// mixes and W_up's 64 columns go to LDS.  Bound by reading d_out and x: the mixes load two steps
// ahead (N = 16384, C = 2048: 105 -> 90 us against one step), the decay's smaller step four.
template <int E, int R, int TT>
struct DpreSmem {
    uint16_t dm[2][E][TT][LF_TS];
    uint16_t w[2][E * R][LF_TS];
};
template <int E, int R, bool LERP, bool WF32, int DEPTH, int TT>
__global__ void __launch_bounds__(8 * TT)
rwkv6_lora_dpre_kernel(const uint16_t* __restrict__ x, InPtrs<E> dout,
                       const uint16_t* __restrict__ neck, const void* __restrict__ wup,
                       uint16_t* __restrict__ dpre, int64_t N, int64_t B, int64_t C) {
    constexpr int ER = E * R, THR = 8 * TT, NP = ER * 8, NPT = (NP + THR - 1) / THR, NA = ER / 32;
    extern __shared__ __attribute__((aligned(16))) unsigned char lf_smem[];
    DpreSmem<E, R, TT>& sm = *reinterpret_cast<DpreSmem<E, R, TT>*>(lf_smem);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, L = lane & 15, q = lane >> 4;
    const int tt = wv % (TT / 16), hh = wv / (TT / 16), row = tid >> 3, cg = tid & 7;
    const int64_t n0 = (int64_t)blockIdx.x * TT, n = n0 + row < N ? n0 + row : N - 1;
    const int64_t xo = n * C + 8 * cg, po = (n >= B ? n - B : n) * C + 8 * cg;
    const float keep = n >= B ? 1.f : 0.f;
    const int nk = (int)(C / 64);
    struct Step { uint4 x, p; u32x4_t d[E]; WRaw<WF32> w[NPT]; };
    auto load = [&](Step& s, int k) {
#pragma unroll
        for (int i = 0; i < NPT; ++i) {
            const int p = min(tid + THR * i, NP - 1);
            s.w[i] = w_load<WF32>(wup, (int64_t)(p >> 3) * C + 64 * k + 8 * (p & 7));
        }
        if (LERP) {
            s.x = *reinterpret_cast<const uint4*>(x + xo + 64 * k);
            s.p = *reinterpret_cast<const uint4*>(x + po + 64 * k);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) s.d[e] = *reinterpret_cast<const u32x4_t*>(dout.p[e] + xo + 64 * k);
    };
    f32x4 acc[NA] = {};
    auto step = [&](Step& s, int k) {
        const int bf = k & 1;
#pragma unroll
        for (int i = 0; i < NPT; ++i) {
            const int p = min(tid + THR * i, NP - 1);
            *reinterpret_cast<uint4*>(&sm.w[bf][p >> 3][8 * (p & 7)]) = w_bf16<WF32>(s.w[i]);
        }
        if (LERP) {
            float dl[8], xv[8];
            unpack8(s.x, xv);
            unpack8(s.p, dl);
#pragma unroll
            for (int j = 0; j < 8; ++j) dl[j] = dl[j] * keep - xv[j];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float v[8];
                unpack8(__builtin_bit_cast(uint4, s.d[e]), v);
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] *= dl[j];
                *reinterpret_cast<uint4*>(&sm.dm[bf][e][row][8 * cg]) = pack8(v);
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) *reinterpret_cast<u32x4_t*>(&sm.dm[bf][e][row][8 * cg]) = s.d[e];
        }
        __syncthreads();
        load(s, min(k + DEPTH, nk - 1));
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const int rt = 2 * i + hh;                       // its mix: 16 rt / R
                const bf16x8 b = ld_bf16x8(&sm.dm[bf][R == 32 ? i : 32 * i / R][16 * tt + L][32 * ks + 8 * q]);
                acc[i] = mfma32(ld_bf16x8(&sm.w[bf][16 * rt + L][32 * ks + 8 * q]), b, acc[i]);
            }
    };
    static_assert(DEPTH == 1 || DEPTH == 2 || DEPTH == 4, "ring of one, two or four steps");
    Step s0, s1, s2, s3;
    load(s0, 0);
    if constexpr (DEPTH >= 2) load(s1, min(1, nk - 1));
    if constexpr (DEPTH == 4) {
        load(s2, min(2, nk - 1));
        load(s3, min(3, nk - 1));
    }
    for (int k = 0; k < nk; k += DEPTH) {
        step(s0, k);
        if constexpr (DEPTH >= 2) {
            if (k + 1 < nk) step(s1, k + 1);
        }
        if constexpr (DEPTH == 4) {
            if (k + 2 < nk) step(s2, k + 2);
            if (k + 3 < nk) step(s3, k + 3);
        }
    }
    const int64_t t = n0 + 16 * tt + L;
    if (t < N) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int64_t o = t * ER + 16 * (2 * i + hh) + 4 * q;
            float nv[4];
            unpack4(*reinterpret_cast<const uint2*>(neck + o), nv);
            float y[4];
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) y[rr] = acc[i][rr] * (1.f - nv[rr] * nv[rr]);
            *reinterpret_cast<uint2*>(dpre + o) = make_uint2(pk2(y[0], y[1]), pk2(y[2], y[3]));
        }
    }
}

// The rest of the backward.  Workgroup (pidx, cb): the 64 channels c0 = 64 cb of one range of the token
// tiles.  A tile is 64 rows of all tokens; LERP, 64 consecutive tokens t of one batch column b, so that
// the shift is one row, or (T <= 32) `cpt` whole columns of T rows each, row r being token t = r mod T of
// column r / T.  A range walks its tiles across the columns' ends, so that the number of ranges, each of
// which writes a full set of partial gradients, follows the device and not the batch (a range per column
// wrote 684 MB at [64, 256, 2048] and took 833 us forward and backward; now 21 MB and 398 us; [1, 4096,
// 2048] 7157 -> 139 us).  Per tile
//   m_e = neck_e W_up_e (LERP), d_xxx = d_pre W_down^T                     [MFMA, to fp32 tiles]
//   dm_e = d_out_e (shift(x) - x),  d_delta = sum_e d_out_e (m_e + bias_e) + d_xxx maa
//   dx[t] = sum_e d_out_e + d_xxx - d_delta[t] + d_delta[t+1]   (E = 1: dx = d_xxx)
//   dW_up_e += neck_e^T dm_e,  dW_down += xxx^T d_pre                       [MFMA]
//   d_bias_e += sum_t dm_e,  d_maa += sum_t d_xxx (shift(x) - x)            [fp32]
// LERP tiles overlap by one token (step 63): the 64th row only supplies d_delta[t+1], so no tile
// waits for another.  A token that another tile counts (`cnt` false) is zeroed in the operands
// of the sums.  The thread of row `row` and channels 8 cg.. makes all global accesses (8 rows
// of 128 contiguous bytes an instruction) and the elementwise work; m and d_xxx reach it
// through fp32 LDS tiles, and dm_e overwrites the bytes of m_e that the same thread has read
// (16 of every 32 bytes: dm_piece below).  Waves (ct, hh): channel tile ct of every product.
template <int E, int R, bool LERP>
struct GradsSmem {
    float m[LERP ? E : 1][LF_TT][LF_MS];          // m_e, then dm_e (bf16, in place); E = 1: d_out (bf16)
    float dx[LF_TT][LF_MS];                       // d_xxx, then d_delta
    uint16_t nk[LF_TT][E * R + 8], dp[LF_TT][E * R + 8];
    uint16_t xx[LF_TT][LF_TS];                    // xxx
    float bias[E][64], maa[64];
};
static_assert(sizeof(GradsSmem<LF_E_MIX, LF_R_MIX, true>) <= 160 * 1024, "one workgroup per CU");
static_assert(2 * sizeof(GradsSmem<1, LF_R_DECAY, false>) <= 160 * 1024, "two workgroups per CU");
static_assert(sizeof(DpreSmem<LF_E_MIX, LF_R_MIX, 64>) <= 160 * 1024, "one workgroup per CU");
// partial parameter gradients of one workgroup range: dW_up [ER][C], dW_down [C][ER], d_bias
// [E][C], d_maa [C] (LERP)
__host__ __device__ constexpr int64_t lf_cols(int64_t E, int64_t R, int64_t C, bool lerp) {
    return (2 * E * R + E + (lerp ? 1 : 0)) * C;
}

template <int E, int R, bool LERP, bool WF32>
__global__ void __launch_bounds__(LF_THR) __attribute__((amdgpu_waves_per_eu(LERP ? 2 : 4)))
rwkv6_lora_grads_kernel(const uint16_t* __restrict__ x, const void* __restrict__ maa, int mdt,
                        InPtrs<E> dout, const uint16_t* __restrict__ neck,
                        const uint16_t* __restrict__ dpre, const void* __restrict__ wup,
                        const void* __restrict__ wd, const void* __restrict__ bias, int bdt,
                        uint16_t* __restrict__ dxo, float* __restrict__ part, int64_t T, int64_t B,
                        int64_t C, int ntiles, int cpt, int tiles, int tpr, int np) {
    constexpr int ER = E * R, WS = ER + 8, NA = ER / 32, KS = R / 32;
    constexpr int STEP = LERP ? LF_TT - 1 : LF_TT;
    constexpr int NP = LF_TT * ER / 8, NPT = (NP + LF_THR - 1) / LF_THR;
    extern __shared__ __attribute__((aligned(16))) unsigned char lf_smem[];
    GradsSmem<E, R, LERP>& sm = *reinterpret_cast<GradsSmem<E, R, LERP>*>(lf_smem);
    // workgroups go round-robin over the 8 XCDs: XCD x takes the ranges x, x + 8, ... with all
    // their channel blocks, so neck and d_pre of a range are read into one L2
    const int ncb = (int)(C / 64), id = blockIdx.x, pidx = (id >> 3) / ncb * 8 + (id & 7), cb = (id >> 3) % ncb;
    if (pidx >= np) return;
    const int t_lo = pidx * tpr, t_hi = min(tiles, t_lo + tpr);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, L = lane & 15, q = lane >> 4;
    const int ct = wv & 3, hh = wv >> 2, cg = tid & 7;
    const int64_t c0 = 64 * (int64_t)cb;

    // ---- per-block constants ----
    bf16x8 wua[LERP ? E * KS : 1], wda[NA];
    if (LERP) {
        // W_up's 64 columns through LDS (the m tiles' space) into A operands: rows = channels
        uint16_t* st = reinterpret_cast<uint16_t*>(&sm.m[0][0][0]);
        for (int p = tid; p < ER * 8; p += LF_THR)
            *reinterpret_cast<uint4*>(st + (p >> 3) * LF_TS + 8 * (p & 7)) =
                w_bf16<WF32>(w_load<WF32>(wup, (int64_t)(p >> 3) * C + c0 + 8 * (p & 7)));
        if (tid < 8 * E) {
            float f[8];
            load_param8(bias, bdt, (tid >> 3) * C + c0 + 8 * (tid & 7), f);
            st_f8(&sm.bias[tid >> 3][8 * (tid & 7)], f);
        } else if (tid < 8 * E + 8) {
            float f[8];
            load_param8(maa, mdt, c0 + 8 * (tid - 8 * E), f);
            st_f8(&sm.maa[8 * (tid - 8 * E)], f);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < E * KS; ++i) wua[i] = lds_tr8(st, LF_TS, 32 * i, 16 * ct, lane);
    }
#pragma unroll
    for (int ks = 0; ks < NA; ++ks)
        wda[ks] = __builtin_bit_cast(bf16x8, w_bf16<WF32>(w_load<WF32>(wd, (c0 + 16 * ct + L) * ER + 32 * ks + 8 * q)));

    // Tile g: its first token t0 and column b0, its rows, and whether the sequences end in it.
    struct Tile { int64_t t0, b0; int rows; bool end; };
    auto tile = [&](int g) {
        const int col = LERP ? g / ntiles : 0, ti = g - col * ntiles;
        const int64_t t0 = (int64_t)ti * STEP, b0 = (int64_t)col * cpt;
        const int rows = LERP && cpt > 1 ? min(cpt, (int)(B - b0)) * (int)T : (int)min<int64_t>(LF_TT, T - t0);
        return Tile{t0, b0, rows, ti == ntiles - 1};
    };
    // (column, token) of a tile's row, after b0 and t0: r / T by a factor rounded up, exact for r < 64
    const unsigned inv = LERP && cpt > 1 ? (65536u + (unsigned)T - 1) / (unsigned)T : 0u;
    auto col_of = [&](int r) { return LERP ? (int)((unsigned)r * inv >> 16) : 0; };
    // Addresses: a wave-uniform base per tile plus 32-bit byte offsets of the thread (B*C is
    // bounded by lf_supported, so that 64 token rows fit); rows past the end read the last token.
    uint4 xr, pr, dq[E], nkr[NPT], dpr[NPT];
    const unsigned rs = (unsigned)(B * C) * 2, rsn = (unsigned)B * ER * 2;
    auto at = [](const uint16_t* p, unsigned bytes) {
        return *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(p) + bytes);
    };
    auto load_rows = [&](const Tile& tl, int tid) {          // neck, d_pre
        const int64_t base = (tl.t0 * B + tl.b0) * ER;
#pragma unroll
        for (int i = 0; i < NPT; ++i) {
            const int p = min(tid + LF_THR * i, NP - 1), rw = p / (ER / 8), r = min(rw, tl.rows - 1), c = col_of(r);
            const unsigned o = (unsigned)(r - c * (int)T) * rsn + (unsigned)c * (2 * ER) + 16 * (p - rw * (ER / 8));
            nkr[i] = at(neck + base, o);
            dpr[i] = at(dpre + base, o);
        }
    };
    auto load_acts = [&](const Tile& tl, int tid) {
        const int cg = tid & 7, r = min(tid >> 3, tl.rows - 1), c = col_of(r), t = r - c * (int)T;
        const int64_t base = (tl.t0 * B + tl.b0) * C + c0;
        const unsigned o = (unsigned)t * rs + (unsigned)c * (2 * (unsigned)C) + 16 * cg;
        xr = at(x + base, o);
        // token t - 1; token 0 reads itself (and its shift is zeroed where it is used)
        if (LERP) pr = at(x + (tl.t0 > 0 ? base - B * C : base), tl.t0 > 0 || t == 0 ? o : o - rs);
#pragma unroll
        for (int e = 0; e < E; ++e) dq[e] = at(dout.p[e] + base, o);
    };
    f32x4 aup[NA] = {}, adn[NA] = {};
    // d_bias, d_maa: a lane's running sum of one channel (lf_rows8)
    float ab[E], am = 0.f;
#pragma unroll
    for (int e = 0; e < E; ++e) ab[e] = 0.f;
    constexpr int DMR = LERP ? LF_MS * 4 : LF_TS * 2;         // bytes of a dm row
    if (t_lo < t_hi) {
        const Tile tl = tile(t_lo);
        load_rows(tl, threadIdx.x);
        load_acts(tl, threadIdx.x);
    }
    for (int ti = t_lo; ti < t_hi; ++ti) {
        // the lane indices from an opaque copy per tile: hoisted out of the walk, the addresses
        // derived from them do not fit the registers
        int tid;
        asm volatile("" : "=v"(tid) : "0"((int)threadIdx.x));
        const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), L = lane & 15, q = lane >> 4;
        const int ct = wv & 3, hh = wv >> 2, row = tid >> 3, cg = tid & 7;
        // byte offset of the 4-channel chunk 4 (L & 3) of channel tile ct in a dm row
        const int dmc = LERP ? (2 * ct + ((L & 3) >> 1)) * 32 + (L & 1) * 8 : (16 * ct + 4 * (L & 3)) * 2;
        const Tile tl = tile(ti);
        const int col = col_of(row), tw = row - col * (int)T;
        const int64_t tr = tl.t0 + tw;
        // counted here: the tile's own tokens (all of them in the sequence's last tile)
        const bool cnt = row < tl.rows && (!LERP || row < STEP || tl.end);
        __syncthreads();                             // the previous tile's operands are read
#pragma unroll
        for (int i = 0; i < NPT; ++i) {
            const int p = min(tid + LF_THR * i, NP - 1);
            *reinterpret_cast<uint4*>(&sm.nk[p / (ER / 8)][8 * (p % (ER / 8))]) = nkr[i];
            *reinterpret_cast<uint4*>(&sm.dp[p / (ER / 8)][8 * (p % (ER / 8))]) = dpr[i];
        }
        if (!LERP) {
            const uint4 xz = keep4(cnt, xr), dz = keep4(cnt, dq[0]);
            *reinterpret_cast<uint4*>(&sm.xx[row][8 * cg]) = xz;
            *reinterpret_cast<uint4*>(reinterpret_cast<char*>(&sm.m[0][0][0]) + row * DMR + 16 * cg) = dz;
            float v[8];
            unpack8(dz, v);
            ab[0] += lf_rows8(v, lane);
        }
        __syncthreads();
        // ---- m and d_xxx, transposed (channels as rows): lane (q, L) holds four adjacent
        // channels of token L ----
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int tok = 16 * (2 * hh + k) + L;
            if (LERP) {
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    f32x4 a = {};
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        a = mfma32(wua[e * KS + ks], ld_bf16x8(&sm.nk[tok][e * R + 32 * ks + 8 * q]), a);
                    *reinterpret_cast<f32x4*>(&sm.m[e][tok][16 * ct + 4 * q]) = a;
                }
            }
            f32x4 a = {};
#pragma unroll
            for (int ks = 0; ks < NA; ++ks) a = mfma32(wda[ks], ld_bf16x8(&sm.dp[tok][32 * ks + 8 * q]), a);
            *reinterpret_cast<f32x4*>(&sm.dx[tok][16 * ct + 4 * q]) = a;
        }
        __syncthreads();
        float dxv[8];
        if (LERP) {
            float xv[8], dl[8], dx[8], dd[8], mv[8], sv[8];
            unpack8(xr, xv);
            unpack8(pr, dl);
            ld_f8(&sm.dx[row][8 * cg], dx);
            ld_f8(&sm.maa[8 * cg], mv);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                dl[j] = (tr > 0 ? dl[j] : 0.f) - xv[j];
                xv[j] += dl[j] * mv[j];                              // xxx
                dd[j] = dx[j] * mv[j];
                sv[j] = cnt ? dx[j] * dl[j] : 0.f;
                dxv[j] = dx[j];
            }
            am += lf_rows8(sv, lane);
            *reinterpret_cast<uint4*>(&sm.xx[row][8 * cg]) = keep4(cnt, pack8(xv));
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float v[8], m[8], bb[8];
                unpack8(dq[e], v);
                ld_f8(&sm.m[e][row][8 * cg], m);
                ld_f8(&sm.bias[e][8 * cg], bb);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    dd[j] += v[j] * (m[j] + bb[j]);
                    dxv[j] += v[j];
                    v[j] = cnt ? v[j] * dl[j] : 0.f;                 // dm
                }
                *reinterpret_cast<uint4*>(&sm.m[e][row][8 * cg]) = pack8(v);
                ab[e] += lf_rows8(v, lane);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) dxv[j] -= dd[j];
            st_f8(&sm.dx[row][8 * cg], dd);                          // d_delta
            __syncthreads();
        } else {
            ld_f8(&sm.dx[row][8 * cg], dxv);
        }
        // the next tile's loads (the last tile reloads itself), then this tile's weight-gradient
        // products and dx
        const Tile tn = tile(min(ti + 1, t_hi - 1));
        load_rows(tn, tid);
        load_acts(tn, tid);
        if (LERP) {
            float nd[8];
            const int rn = min(row + 1, LF_TT - 1);
            ld_f8(&sm.dx[rn][8 * cg], nd);
#pragma unroll
            for (int j = 0; j < 8; ++j) dxv[j] += tr + 1 < T ? nd[j] : 0.f;
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const bf16x8 xa = lds_tr8(&sm.xx[0][0], LF_TS, 32 * ks, 16 * ct, lane);
            bf16x8 dmb;
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const int r0 = 16 * (2 * i + hh);
                if (LERP || i == 0) {
                    const char* p = reinterpret_cast<const char*>(&sm.m[LERP ? (R == 32 ? i : 32 * i / R) : 0][0][0]) +
                                    (32 * ks + 8 * q + (L >> 2)) * DMR + dmc;
                    dmb = cat_bf16x8(lds_tr16(reinterpret_cast<const uint16_t*>(p)),
                                 lds_tr16(reinterpret_cast<const uint16_t*>(p + 4 * DMR)));
                }
                aup[i] = mfma32(lds_tr8(&sm.nk[0][0], WS, 32 * ks, r0, lane), dmb, aup[i]);
                adn[i] = mfma32(xa, lds_tr8(&sm.dp[0][0], WS, 32 * ks, r0, lane), adn[i]);
            }
        }
        if (cnt)
            store8(dxo + (tl.t0 * B + tl.b0) * C + c0 + (size_t)((unsigned)tw * (rs / 2) + (unsigned)col * (unsigned)C + 8 * cg),
                   dxv);
    }
    // ---- partial parameter gradients of the range ----
    float* po = part + (int64_t)pidx * lf_cols(E, R, C, LERP);
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int r0 = 16 * (2 * i + hh);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
            po[(int64_t)(r0 + 4 * q + rr) * C + c0 + 16 * ct + L] = aup[i][rr];
            po[(int64_t)ER * C + (c0 + 16 * ct + 4 * q + rr) * ER + r0 + L] = adn[i][rr];
        }
    }
    // the eight waves' row sums, in order
    __syncthreads();
    constexpr int NV = E + (LERP ? 1 : 0);
    float* red = &sm.m[0][0][0];                                     // [8 waves][NV][64]
    {
        const int ch = 8 * cg + 4 * ((lane >> 3) & 1) + 2 * ((lane >> 4) & 1) + (lane >> 5);
#pragma unroll
        for (int e = 0; e < NV; ++e) red[(wv * NV + e) * 64 + ch] = LERP && e == E ? am : ab[e < E ? e : 0];
    }
    __syncthreads();
    for (int i = tid; i < NV * 64; i += LF_THR) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) v += red[w * NV * 64 + i];
        po[2 * (int64_t)ER * C + (int64_t)(i >> 6) * C + c0 + (i & 63)] = v;
    }
}

// out[j] = sum_p part[p][j] over the workgroup ranges, in order; the columns are the parameter
// gradients one after the other, each with its own output and dtype.  Four columns a thread
// (every gradient's size is a multiple of 64).  P = 0 writes zeros.
struct LoraOuts { void* p[4]; int64_t end[4]; int dt[4]; };
__global__ void __launch_bounds__(256)
rwkv6_lora_reduce_kernel(const float* __restrict__ part, int P, int64_t n, LoraOuts out) {
    const int64_t j = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (j >= n) return;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p0 = 0; p0 < P; p0 += 8) {
        float4 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = ld_f4(part + (int64_t)min(p0 + k, P - 1) * n + j);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (p0 + k < P) { a.x += v[k].x; a.y += v[k].y; a.z += v[k].z; a.w += v[k].w; }
    }
    int s = 0;
    while (s < 3 && j >= out.end[s]) ++s;
    const int64_t o = j - (s ? out.end[s - 1] : 0);
    if (out.dt[s] == RWKV6_BF16)
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out.p[s]) + o) = make_uint2(pk2(a.x, a.y), pk2(a.z, a.w));
    else
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(out.p[s]) + o) = a;
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
namespace {

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline size_t lf_round(size_t n) { return (n + 255) & ~(size_t)255; }
inline bool dt_ok(int d) { return d == RWKV6_F32 || d == RWKV6_BF16; }
inline int launch_status() { return hipGetLastError() == hipSuccess ? RWKV6_OK : RWKV6_ERR_LAUNCH; }
// What the kernels take, the same for the forward, the backward and its workspace: their bottlenecks;
// 64 token rows of a batch column within 32-bit byte offsets; a grid of 32-token workgroups of 256
// threads below the launch's 2^32 threads.
inline bool lf_supported(int64_t T, int64_t B, int64_t C, int64_t E, int64_t R, bool lerp) {
    return (lerp ? E == LF_E_MIX && R == LF_R_MIX : E == 1 && R == LF_R_DECAY) && C % 64 == 0 && C <= (1 << 23) &&
           B <= (1 << 23) / C && T <= ((int64_t)1 << 28) / B;
}
// Token rows of a workgroup of the down and d_pre kernels.  Each workgroup reads the whole weight,
// so the mixes' 64 rows halve that traffic once 64 rows a workgroup still give half the CUs one
// (N = 16384, C = 2048: d_pre 88 against 106 us, down 42 against 45.5); below that, and for the
// decay's smaller weight, 32 rows spread a short walk over twice the CUs (N = 1024, C = 512:
// mixes 18 -> 12.4 and 13.4 -> 10.9 us, decay 6.9 -> 5.0 and 9.1 -> 5.5).
inline int lf_tile(int64_t N, bool lerp) { return lerp && N > 8192 ? 64 : 32; }
// Tiles of the gradient kernel: `ntiles` a batch column (or a group of `cpt` columns of at most 32 tokens,
// which fill a tile together), `tiles` in all, `np` ranges of `tpr`.  The time is the rounds of workgroups
// over the device times the tiles of a range; the fewest rounds (and so the least partial traffic) win
// ties.  `slots`: workgroups the device holds at once (LDS: one LERP workgroup of 157 KB a CU, two of the
// decay's).  At most 64 ranges for each of up to four columns: more are not measured.
struct LfPlan { int ntiles, cpt, tiles, tpr, np; };
inline LfPlan lf_plan(int64_t T, int64_t B, int64_t C, bool lerp) {
    if (T * B == 0) return {0, 1, 0, 1, 0};
    const int64_t ncb = C / 64, slots = lerp ? 256 : 512;
    const int64_t cpt = lerp && T <= LF_TT / 2 ? std::min(B, LF_TT / T) : 1, groups = lerp ? (B + cpt - 1) / cpt : 1;
    const int64_t nt = lerp ? (T > 1 ? (T - 1 + LF_TT - 2) / (LF_TT - 1) : 1) : (T * B + LF_TT - 1) / LF_TT;
    const int64_t tiles = groups * nt, most = std::min(tiles, 64 * (lerp ? std::min<int64_t>(B, 4) : 1));
    int64_t best = 1, cost = INT64_MAX;
    for (int64_t k = 1; k <= 4; ++k) {
        const int64_t np = std::max<int64_t>(1, std::min(most, k * slots / ncb));
        const int64_t c = ((ncb * np + slots - 1) / slots) * ((tiles + np - 1) / np + 1);
        if (c < cost) { cost = c; best = np; }
    }
    const int64_t tpr = (tiles + best - 1) / best;
    return {(int)nt, (int)cpt, (int)tiles, (int)tpr, (int)((tiles + tpr - 1) / tpr)};
}

}  // namespace

extern "C" {

int rwkv6_lora_down_fwd(const void* x, const void* maa, int maa_dtype, const void* w_down,
                        int w_dtype, void* neck, int64_t T, int64_t B, int64_t C, int64_t E,
                        int64_t R, void* stream) {
    if (T < 0 || B < 1 || C < 1 || E < 1 || R < 1) return RWKV6_ERR_INVALID_ARG;
    if (!dt_ok(w_dtype) || (maa && !dt_ok(maa_dtype))) return RWKV6_ERR_INVALID_ARG;
    const bool lerp = maa != nullptr, f32 = w_dtype == RWKV6_F32;
    if (!lf_supported(T, B, C, E, R, lerp)) return RWKV6_ERR_UNSUPPORTED;
    if (T == 0) return RWKV6_OK;
    if (!x || !w_down || !neck) return RWKV6_ERR_INVALID_ARG;
    if (!al16(x) || !al16(maa) || !al16(w_down) || !al16(neck)) return RWKV6_ERR_ALIGNMENT;
    const int64_t N = T * B;
    if (any_alias({{neck, (size_t)(N * E * R) * 2}},
                  {{x, (size_t)(N * C) * 2}, {maa, (size_t)C * param_bytes(maa_dtype)},
                   {w_down, (size_t)(C * E * R) * param_bytes(w_dtype)}}))
        return RWKV6_ERR_INVALID_ARG;
    constexpr int MIX = LF_E_MIX * LF_R_MIX, DEC = LF_R_DECAY;
    const int tt = lf_tile(N, lerp);
    auto kern = !lerp ? (f32 ? rwkv6_lora_down_kernel<DEC, false, true, 32> : rwkv6_lora_down_kernel<DEC, false, false, 32>)
                : tt == 64 ? (f32 ? rwkv6_lora_down_kernel<MIX, true, true, 64> : rwkv6_lora_down_kernel<MIX, true, false, 64>)
                           : (f32 ? rwkv6_lora_down_kernel<MIX, true, true, 32> : rwkv6_lora_down_kernel<MIX, true, false, 32>);
    hipLaunchKernelGGL(kern, dim3((unsigned)((N + tt - 1) / tt)), dim3(8 * tt), 0,
                       reinterpret_cast<hipStream_t>(stream), (const uint16_t*)x, maa, maa_dtype, w_down,
                       (uint16_t*)neck, N, B, C);
    return launch_status();
}

size_t rwkv6_lora_bwd_workspace_bytes(int64_t T, int64_t B, int64_t C, int64_t E, int64_t R) {
    if (T < 0 || B < 1 || C < 1 || !lf_supported(T, B, C, E, R, E != 1)) return 0;
    const LfPlan p = lf_plan(T, B, C, E != 1);
    return lf_round((size_t)(T * B * E * R) * 2) + (size_t)(std::max(p.np, 1) * lf_cols(E, R, C, E != 1)) * 4;
}

}  // extern "C"

namespace {

// The two kernels and the reduction of one backward.
template <int E, int R, bool LERP, bool WF32, int DEPTH>
int lora_bwd_launch(const uint16_t* x, const void* maa, int mdt, const InPtrs<E>& dout,
                    const uint16_t* neck, const void* wd, const void* wup, const void* bias, int bdt,
                    uint16_t* dx, const LoraOuts& outs, void* workspace, int64_t T, int64_t B,
                    int64_t C, hipStream_t s) {
    const LfPlan p = lf_plan(T, B, C, LERP);
    const int64_t N = T * B, n = lf_cols(E, R, C, LERP);
    uint16_t* dpre = reinterpret_cast<uint16_t*>(workspace);
    float* part = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + lf_round((size_t)(N * E * R) * 2));
    if (N > 0) {
        const int tt = lf_tile(N, LERP);
        auto kp64 = rwkv6_lora_dpre_kernel<E, R, LERP, WF32, DEPTH, LERP ? 64 : 32>;
        auto kp32 = rwkv6_lora_dpre_kernel<E, R, LERP, WF32, DEPTH, 32>;
        auto kg = rwkv6_lora_grads_kernel<E, R, LERP, WF32>;
        static DeviceOnce once[kMaxDevices];
        int dev = 0, cur = 0, st = stream_device(s, &dev, &cur);
        if (st != RWKV6_OK) return st;
        st = device_once(once[dev], dev, cur, [&] {
            const std::pair<const void*, size_t> list[] = {
                {reinterpret_cast<const void*>(kp64), sizeof(DpreSmem<E, R, LERP ? 64 : 32>)},
                {reinterpret_cast<const void*>(kp32), sizeof(DpreSmem<E, R, 32>)},
                {reinterpret_cast<const void*>(kg), sizeof(GradsSmem<E, R, LERP>)}};
            hipError_t e = hipSuccess;
            for (const auto& x : list)
                if (e == hipSuccess)
                    e = hipFuncSetAttribute(x.first, hipFuncAttributeMaxDynamicSharedMemorySize, (int)x.second);
            return e;
        });
        if (st != RWKV6_OK) return st;
        hipLaunchKernelGGL(tt == 64 ? kp64 : kp32, dim3((unsigned)((N + tt - 1) / tt)), dim3(8 * tt),
                           tt == 64 ? sizeof(DpreSmem<E, R, 64>) : sizeof(DpreSmem<E, R, 32>), s, x, dout, neck, wup,
                           dpre, N, B, C);
        hipLaunchKernelGGL(kg, dim3((unsigned)(8 * ((p.np + 7) / 8) * (C / 64))), dim3(LF_THR),
                           sizeof(GradsSmem<E, R, LERP>), s, x, maa, mdt, dout, neck, (const uint16_t*)dpre, wup, wd,
                           bias, bdt, dx, part, LERP ? T : N, LERP ? B : (int64_t)1, C, p.ntiles, p.cpt, p.tiles, p.tpr, p.np);
    }
    hipLaunchKernelGGL(rwkv6_lora_reduce_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s,
                       (const float*)part, p.np, n, outs);
    return launch_status();
}

}  // namespace

extern "C" {

int rwkv6_lora_bwd(const void* x, const void* maa, int maa_dtype, const void* const* d_out,
                   const void* neck, const void* w_down, const void* w_up, int w_dtype,
                   const void* bias, int bias_dtype, void* dx, void* d_maa, void* d_w_down,
                   int d_w_down_dtype, void* d_w_up, int d_w_up_dtype, void* d_bias,
                   void* workspace, int64_t T, int64_t B, int64_t C, int64_t E, int64_t R,
                   void* stream) {
    if (T < 0 || B < 1 || C < 1 || E < 1 || R < 1) return RWKV6_ERR_INVALID_ARG;
    if (!dt_ok(w_dtype) || !dt_ok(bias_dtype) || !dt_ok(d_w_down_dtype) || !dt_ok(d_w_up_dtype) ||
        (maa && !dt_ok(maa_dtype)))
        return RWKV6_ERR_INVALID_ARG;
    const bool lerp = maa != nullptr, f32 = w_dtype == RWKV6_F32;
    if (!lf_supported(T, B, C, E, R, lerp)) return RWKV6_ERR_UNSUPPORTED;
    if (!w_down || !w_up || !bias || !d_w_down || !d_w_up || !d_bias || !workspace || (!d_maa != !maa) ||
        (T > 0 && (!x || !neck || !dx || !d_out)))
        return RWKV6_ERR_INVALID_ARG;
    InPtrs<LF_E_MIX> dm{};
    for (int e = 0; e < (int)E && T > 0; ++e) {
        if (!d_out[e]) return RWKV6_ERR_INVALID_ARG;
        if (!al16(d_out[e])) return RWKV6_ERR_ALIGNMENT;
        dm.p[e] = (const uint16_t*)d_out[e];
    }
    if (!al16(x) || !al16(maa) || !al16(neck) || !al16(w_down) || !al16(w_up) || !al16(bias) || !al16(dx) ||
        !al16(d_maa) || !al16(d_w_down) || !al16(d_w_up) || !al16(d_bias) || !al16(workspace))
        return RWKV6_ERR_ALIGNMENT;
    {
        const size_t act = (size_t)(T * B * C) * 2, w = (size_t)(E * R * C);
        if (any_alias({{dx, act}, {d_maa, (size_t)C * param_bytes(maa_dtype)},
                       {d_w_down, w * param_bytes(d_w_down_dtype)}, {d_w_up, w * param_bytes(d_w_up_dtype)},
                       {d_bias, (size_t)(E * C) * param_bytes(bias_dtype)},
                       {workspace, rwkv6_lora_bwd_workspace_bytes(T, B, C, E, R)}},
                      {{x, act}, {maa, (size_t)C * param_bytes(maa_dtype)}, {neck, (size_t)(T * B * E * R) * 2},
                       {w_down, w * param_bytes(w_dtype)}, {w_up, w * param_bytes(w_dtype)},
                       {bias, (size_t)(E * C) * param_bytes(bias_dtype)}, {dm.p[0], act}, {dm.p[1], act},
                       {dm.p[2], act}, {dm.p[3], act}, {dm.p[4], act}}))
            return RWKV6_ERR_INVALID_ARG;
    }
    LoraOuts o;
    const int64_t w = E * R * C;
    void* ptr[4] = {d_w_up, d_w_down, d_bias, d_maa};
    const int dt[4] = {d_w_up_dtype, d_w_down_dtype, bias_dtype, maa_dtype};
    const int64_t end[4] = {w, 2 * w, 2 * w + E * C, 2 * w + (E + 1) * C};
    for (int i = 0; i < 4; ++i) { o.p[i] = ptr[i]; o.dt[i] = dt[i]; o.end[i] = end[i]; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const uint16_t *xp = (const uint16_t*)x, *np = (const uint16_t*)neck;
    if (lerp) {
        auto go = f32 ? lora_bwd_launch<LF_E_MIX, LF_R_MIX, true, true, 2> : lora_bwd_launch<LF_E_MIX, LF_R_MIX, true, false, 2>;
        return go(xp, maa, maa_dtype, dm, np, w_down, w_up, bias, bias_dtype, (uint16_t*)dx, o, workspace, T, B, C, s);
    }
    InPtrs<1> d1;
    d1.p[0] = dm.p[0];
    auto go = f32 ? lora_bwd_launch<1, LF_R_DECAY, false, true, 4> : lora_bwd_launch<1, LF_R_DECAY, false, false, 4>;
    return go(xp, maa, maa_dtype, d1, np, w_down, w_up, bias, bias_dtype, (uint16_t*)dx, o, workspace, T, B, C, s);
}

}  // extern "C"
