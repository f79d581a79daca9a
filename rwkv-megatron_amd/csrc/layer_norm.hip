// LayerNorm over the channels of bf16 token rows for MI355X (gfx950), forward and backward, with
// the parameters as the module holds them (bf16 or fp32).
//
// Reference: the LayerNorms around the time and channel mix and of the model
// (/root/reference/rwkv_megatron/rwkv6_layer_specs.py:543-547, rwkv6_model.py:34-37).
//   y = (x - mean) rstd gamma + beta, statistics over the C channels of a row, fp32 inside
//   dx = rstd (g - mean(g) - xhat mean(g xhat)), g = dy gamma, xhat = (x - mean) rstd
//   dgamma = sum_rows dy xhat, dbeta = sum_rows dy     (two stages, fixed order)
// A wave owns a row, held in registers (16-byte pieces, lane by lane), so x and dy are read once.
// Bound by those reads at many rows and by the launch at few, where the library's kernels need
// casts of fp32 parameters before (two launches), three launches in the backward and two casts of
// the parameters' gradients after.  Measured with fp32 parameters, us, library -> here,
// forward and forward + backward (graph replays): 1024 x 512 15 -> 10 and 28 -> 18; 4096 x 2048 24 ->
// 13 and 65 -> 42; 16384 x 2048 52 -> 28 and 171 -> 86 (4.7 TB/s and 3.9 TB/s); 16384 x 4096 75 -> 49
// and 400 -> 229; bf16 ones 11 -> 12 and 20 -> 18, 18 -> 13 and 56 -> 42, 44 -> 28 and 156 -> 85, 68
// -> 50 and 391 -> 222.
#include "common.h"
#include "../../include/rwkv6_amd.h"

#define LN_THR 256        // 4 rows at a time
#define LN_PART 512       // row ranges of the backward at most
#define LN_MAX_C 4096

namespace {

__device__ __forceinline__ float ln_wave_sum(float v) {
    v = sum8lanes(v);
    v += dpp_mov<0x140>(v);                       // row_mirror: the other 8 lanes of the row
    const RowSums r = row_sums(v);
    return r.lo + r.hi;
}
// The lane's pieces of a row: channels 8 (lane + 64 i).., zeros past the end.
template <int NV>
__device__ __forceinline__ void ln_load(const uint16_t* row, int C, int lane, uint4* q) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = 8 * (lane + 64 * i);
        q[i] = c < C ? *reinterpret_cast<const uint4*>(row + c) : make_uint4(0u, 0u, 0u, 0u);
    }
}

}  // namespace

// grid: ceil(N / 4); `gcopy` (nullable) receives gamma in fp32 for the backward
template <int NV>
__global__ void __launch_bounds__(LN_THR)
rwkv6_layer_norm_fwd_kernel(const uint16_t* __restrict__ x, const void* __restrict__ gamma,
                            const void* __restrict__ beta, int pdt, float eps, uint16_t* __restrict__ y,
                            float* __restrict__ mean_out, float* __restrict__ rstd_out,
                            float* __restrict__ gcopy, int64_t N, int C) {
    const int lane = threadIdx.x & 63;
    const int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (n >= N) return;
    // Short rows have the parameters in flight with x; long ones read them when the statistics are
    // known: their 128 registers left two waves a SIMD (16384 x 4096: 72 -> 49 us).
    constexpr bool EARLY = NV <= 2;
    uint4 q[NV];
    float ga[EARLY ? NV : 1][8], be[EARLY ? NV : 1][8];
    ln_load<NV>(x + n * C, C, lane, q);
    if (EARLY)
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = 8 * (lane + 64 * i);
            if (c < C) {
                load_param8(gamma, pdt, c, ga[EARLY ? i : 0]);
                load_param8(beta, pdt, c, be[EARLY ? i : 0]);
            }
        }
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        float v[8];
        unpack8(q[i], v);
#pragma unroll
        for (int j = 0; j < 8; ++j) s += v[j];
    }
    const float inv = 1.f / (float)C, mean = ln_wave_sum(s) * inv;
    float var = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        float v[8];
        unpack8(q[i], v);
        if (8 * (lane + 64 * i) < C)
#pragma unroll
            for (int j = 0; j < 8; ++j) var += (v[j] - mean) * (v[j] - mean);
    }
    const float rstd = rsqrtf(ln_wave_sum(var) * inv + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = 8 * (lane + 64 * i);
        if (c >= C) continue;
        const int ip = EARLY ? i : 0;
        if (!EARLY) {
            load_param8(gamma, pdt, c, ga[ip]);
            load_param8(beta, pdt, c, be[ip]);
        }
        float v[8];
        unpack8(q[i], v);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (v[j] - mean) * rstd * ga[ip][j] + be[ip][j];
        store8(y + n * C + c, v);
        if (gcopy && n == 0)
#pragma unroll
            for (int j = 0; j < 8; ++j) gcopy[c + j] = ga[ip][j];
    }
    if (lane == 0) {
        mean_out[n] = mean;
        rstd_out[n] = rstd;
    }
}

// Block p: rows [p rpb, (p + 1) rpb), a wave every fourth of them, the next one's loads in flight;
// part[p][2][C] = its sums of dgamma and dbeta (part null: dx only).
template <int NV>
__global__ void __launch_bounds__(LN_THR)
rwkv6_layer_norm_bwd_kernel(const uint16_t* __restrict__ x, const void* __restrict__ gamma, int pdt,
                            const float* __restrict__ mean_in, const float* __restrict__ rstd_in,
                            const uint16_t* __restrict__ dy, uint16_t* __restrict__ dx,
                            float* __restrict__ part, int64_t N, int C, int64_t rpb) {
    extern __shared__ __attribute__((aligned(16))) float ln_red[];            // [2][C]
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t n0 = (int64_t)blockIdx.x * rpb, n1 = min(N, n0 + rpb);
    const float inv = 1.f / (float)C;
    float ag[NV][8], ab[NV][8];
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) ag[i][j] = ab[i][j] = 0.f;
    uint4 xq[NV], gq[NV];
    float mean = 0.f, rstd = 0.f;
    auto load = [&](int64_t n) {
        ln_load<NV>(x + n * C, C, lane, xq);
        ln_load<NV>(dy + n * C, C, lane, gq);
        mean = mean_in[n];
        rstd = rstd_in[n];
    };
    if (n0 + wv < n1) load(n0 + wv);
    for (int64_t n = n0 + wv; n < n1; n += 4) {
        uint4 xc[NV], gc[NV];
        const float m = mean, r = rstd;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            xc[i] = xq[i];
            gc[i] = gq[i];
        }
        load(min(n + 4, n1 - 1));
        float s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = 8 * (lane + 64 * i);
            if (c >= C) continue;
            float xh[8], g[8], ga[8];
            unpack8(xc[i], xh);
            unpack8(gc[i], g);
            load_param8(gamma, pdt, c, ga);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                xh[j] = (xh[j] - m) * r;
                ag[i][j] += g[j] * xh[j];
                ab[i][j] += g[j];
                s1 += g[j] * ga[j];
                s2 += g[j] * ga[j] * xh[j];
            }
        }
        s1 = ln_wave_sum(s1) * inv;
        s2 = ln_wave_sum(s2) * inv;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = 8 * (lane + 64 * i);
            if (c >= C) continue;
            float xh[8], g[8], ga[8];
            unpack8(xc[i], xh);
            unpack8(gc[i], g);
            load_param8(gamma, pdt, c, ga);
#pragma unroll
            for (int j = 0; j < 8; ++j) g[j] = r * (g[j] * ga[j] - s1 - (xh[j] - m) * r * s2);
            store8(dx + n * C + c, g);
        }
    }
    if (!part) return;
    // the four waves' sums, in order
    for (int w = 0; w < 4; ++w) {
        if (wv == w) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = 8 * (lane + 64 * i);
                if (c >= C) continue;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    ln_red[c + j] = (w ? ln_red[c + j] : 0.f) + ag[i][j];
                    ln_red[C + c + j] = (w ? ln_red[C + c + j] : 0.f) + ab[i][j];
                }
            }
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < 2 * C; i += LN_THR) part[(int64_t)blockIdx.x * 2 * C + i] = ln_red[i];
}

namespace {
inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline int ln_check(int64_t N, int64_t C, int pdt) {
    if (N < 0 || C < 1) return RWKV6_ERR_INVALID_ARG;
    if (pdt != RWKV6_F32 && pdt != RWKV6_BF16) return RWKV6_ERR_INVALID_ARG;
    // rows: a grid of 256 threads for four of them stays below the launch's 2^32 threads
    if (C % 8 || C > LN_MAX_C || N > ((int64_t)1 << 26) - 4) return RWKV6_ERR_UNSUPPORTED;
    return RWKV6_OK;
}
// Row ranges of the backward: 8 rows (two a wave) at least, so that few rows still spread over the
// CUs, and LN_PART ranges at most, which bounds the partial sums to 2 x 512 rows of C.
inline int64_t ln_rows(int64_t N) {
    const int64_t r = (N + LN_PART - 1) / LN_PART;
    return r < 8 ? 8 : r;
}
inline int64_t ln_parts(int64_t N) { return (N + ln_rows(N) - 1) / ln_rows(N); }
inline int launch_status() { return hipGetLastError() == hipSuccess ? RWKV6_OK : RWKV6_ERR_LAUNCH; }
}  // namespace

extern "C" {

int rwkv6_layer_norm_fwd(const void* x, const void* gamma, const void* beta, int param_dtype, float eps,
                         void* y, float* mean, float* rstd, float* gamma_copy, int64_t N, int64_t C,
                         void* stream) {
    const int st = ln_check(N, C, param_dtype);
    if (st) return st;
    if (N == 0) return RWKV6_OK;
    if (!x || !gamma || !beta || !y || !mean || !rstd) return RWKV6_ERR_INVALID_ARG;
    if (!al16(x) || !al16(gamma) || !al16(beta) || !al16(y)) return RWKV6_ERR_ALIGNMENT;
    const size_t act = (size_t)(N * C) * 2, par = (size_t)C * param_bytes(param_dtype);
    if (any_alias({{y, act}, {mean, (size_t)N * 4}, {rstd, (size_t)N * 4}, {gamma_copy, (size_t)C * 4}},
                  {{x, act}, {gamma, par}, {beta, par}}))
        return RWKV6_ERR_INVALID_ARG;
    auto k = C <= 512 ? rwkv6_layer_norm_fwd_kernel<1> : C <= 1024 ? rwkv6_layer_norm_fwd_kernel<2>
           : C <= 2048 ? rwkv6_layer_norm_fwd_kernel<4> : rwkv6_layer_norm_fwd_kernel<8>;
    hipLaunchKernelGGL(k, dim3((unsigned)((N + 3) / 4)), dim3(LN_THR), 0, reinterpret_cast<hipStream_t>(stream),
                       (const uint16_t*)x, gamma, beta, param_dtype, eps, (uint16_t*)y, mean, rstd, gamma_copy,
                       N, (int)C);
    return launch_status();
}

size_t rwkv6_layer_norm_bwd_workspace_bytes(int64_t N, int64_t C) {
    if (ln_check(N, C, RWKV6_F32)) return 0;
    return (size_t)((N > 0 ? ln_parts(N) : 1) * 2 * C) * sizeof(float);
}

int rwkv6_layer_norm_bwd(const void* x, const void* gamma, int gamma_dtype, const float* mean, const float* rstd,
                         const void* dy, void* dx, void* dgamma, void* dbeta, int param_dtype, void* workspace,
                         int64_t N, int64_t C, void* stream) {
    int st = ln_check(N, C, gamma_dtype);
    if (!st) st = ln_check(N, C, param_dtype);
    if (st) return st;
    const bool sums = dgamma || dbeta;
    if (!gamma || (!dgamma != !dbeta) || (sums && !workspace) || (N > 0 && (!x || !mean || !rstd || !dy || !dx)))
        return RWKV6_ERR_INVALID_ARG;
    if (!al16(x) || !al16(gamma) || !al16(dy) || !al16(dx) || !al16(workspace)) return RWKV6_ERR_ALIGNMENT;
    const size_t act = (size_t)(N * C) * 2, par = (size_t)C * param_bytes(param_dtype), st4 = (size_t)N * 4;
    if (any_alias({{dx, act}, {dgamma, par}, {dbeta, par},
                   {sums ? workspace : nullptr, rwkv6_layer_norm_bwd_workspace_bytes(N, C)}},
                  {{x, act}, {gamma, (size_t)C * param_bytes(gamma_dtype)}, {mean, st4}, {rstd, st4}, {dy, act}}))
        return RWKV6_ERR_INVALID_ARG;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    float* part = sums ? (float*)workspace : nullptr;
    if (N > 0) {
        auto k = C <= 512 ? rwkv6_layer_norm_bwd_kernel<1> : C <= 1024 ? rwkv6_layer_norm_bwd_kernel<2>
               : C <= 2048 ? rwkv6_layer_norm_bwd_kernel<4> : rwkv6_layer_norm_bwd_kernel<8>;
        hipLaunchKernelGGL(k, dim3((unsigned)ln_parts(N)), dim3(LN_THR), (size_t)(2 * C) * 4, s, (const uint16_t*)x,
                           gamma, gamma_dtype, mean, rstd, (const uint16_t*)dy, (uint16_t*)dx, part, N, (int)C,
                           ln_rows(N));
    }
    if (sums) launch_partials_reduce(part, N > 0 ? ln_parts(N) : (int64_t)0, 2 * C, param_dtype, dgamma, dbeta, C, s);
    return launch_status();
}

}  // extern "C"
