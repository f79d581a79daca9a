// y = x W^T for few tokens with a weight held in fp32, for MI355X (gfx950): the projections of
// RWKV6TimeMix and RWKV6ChannelMix (/root/reference/rwkv_megatron/rwkv6_layer_specs.py:395-421,
// :484-505) of a model whose parameters are fp32.
//
// The weight is rounded to bf16 on the way into LDS (and written out once where a backward will
// want it), so no cast runs before the product: at a few hundred tokens the two launches and the
// weight's trip through memory took longer than the arithmetic.  Measured, us, cast and library
// product -> here, N tokens: O x I = 512 x 512: 8.0 -> 5.7 (N = 1), 11 -> 6.6 (777); 1792 x 512: 14 ->
// 10 (777); 512 x 1792: 13.7 -> 11.8 (777; 13.2 with four waves); 1024 x 1024: 13.4 -> 8.8 (512), 13.7
// -> 12.1 (1024); 2048 x 2048: 15.6 -> 11.8 (1), 18.7 -> 13.2 (256).  Past 2^30 multiplications the
// library's larger tiles win: 2048 x 2048 25 -> 30 (1024), 7168 x 2048 34 -> 50 (512).
#include "common.h"
#include "../../include/rwkv6_amd.h"

#define LIN_O 64          // outputs of a workgroup
#define LIN_AHEAD 3       // steps whose loads are in flight

// Workgroup (o tile, token tile): TN tokens x 64 outputs, 4 KG waves; wave (w, kg) forms the outputs
// 16 w.. of all tokens over every KG-th 64 inputs, transposed (W's rows as the product's rows), so
// that a lane ends with four adjacent outputs of a token; the KG sums meet in LDS at the end.  64 KG
// inputs a step through double-buffered LDS tiles, one barrier a step, LIN_AHEAD steps of loads in
// registers: bound by the latency of the chain of steps, which KG = 2 halves.
// Workgroups go round-robin over the 8 XCDs and the output tile is the faster index, so with a
// multiple of 8 of them the token tiles that read one piece of W share an L2.
template <int TN, int KG>
__global__ void __launch_bounds__(256 * KG)
rwkv6_linear_f32_kernel(const uint16_t* __restrict__ x, const float* __restrict__ w, uint16_t* __restrict__ y,
                        uint16_t* __restrict__ wc, int64_t N, int O, int I, int otiles) {
    constexpr int XP = TN / 32, LIN_K = 64 * KG, LIN_S = LIN_K + 8;   // XP: pieces of x a thread and step
    __shared__ __attribute__((aligned(16))) uint16_t xs[2][TN][LIN_S];
    __shared__ __attribute__((aligned(16))) uint16_t ws[2][LIN_O][LIN_S];
    const int tid = threadIdx.x, lane = tid & 63, wv = (tid >> 6) & 3, kg = tid >> 8, L = lane & 15, q = lane >> 4;
    const int ot = blockIdx.x % otiles;
    const int64_t n0 = (int64_t)(blockIdx.x / otiles) * TN;
    const int o0 = ot * LIN_O, row = tid / (8 * KG), col = 8 * (tid % (8 * KG));
    const int nk = (I + LIN_K - 1) / LIN_K;
    // rows past the end read the last one (their products are not stored)
    const uint16_t* xr[XP];
    const float* wr[2];
#pragma unroll
    for (int i = 0; i < XP; ++i) xr[i] = x + (n0 + row + 32 * i < N ? n0 + row + 32 * i : N - 1) * I + col;
#pragma unroll
    for (int i = 0; i < 2; ++i) wr[i] = w + (int64_t)min(o0 + row + 32 * i, O - 1) * I + col;
    struct Step { uint4 x[XP]; WRaw<true> w[2]; };
    // a piece past the last input is read at the row's start instead and zeroed where it is used
    auto load = [&](Step& s, int k) {
        const int c = k * LIN_K + col < I ? k * LIN_K : -col;
#pragma unroll
        for (int i = 0; i < XP; ++i) s.x[i] = *reinterpret_cast<const uint4*>(xr[i] + c);
#pragma unroll
        for (int i = 0; i < 2; ++i) s.w[i] = w_load<true>(wr[i], c);
    };
    f32x4 acc[TN / 16] = {};
    const bool keep = wc != nullptr && n0 == 0;
    auto step = [&](Step& s, int k) {
        const int bf = k & 1;
        const bool in = k * LIN_K + col < I;
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const uint4 v = s.x[i];
            *reinterpret_cast<uint4*>(&xs[bf][row + 32 * i][col]) =
                make_uint4(in ? v.x : 0u, in ? v.y : 0u, in ? v.z : 0u, in ? v.w : 0u);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint4 v = w_bf16<true>(s.w[i]);
            *reinterpret_cast<uint4*>(&ws[bf][row + 32 * i][col]) =
                make_uint4(in ? v.x : 0u, in ? v.y : 0u, in ? v.z : 0u, in ? v.w : 0u);
            if (keep && in && o0 + row + 32 * i < O)
                *reinterpret_cast<uint4*>(wc + (int64_t)(o0 + row + 32 * i) * I + k * LIN_K + col) = v;
        }
        __syncthreads();
        load(s, min(k + LIN_AHEAD, nk - 1));
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int c = 64 * kg + 32 * ks + 8 * q;
            const bf16x8 a = ld_bf16x8(&ws[bf][16 * wv + L][c]);
#pragma unroll
            for (int t = 0; t < TN / 16; ++t) acc[t] = mfma32(a, ld_bf16x8(&xs[bf][16 * t + L][c]), acc[t]);
        }
    };
    Step s0, s1, s2;
    load(s0, 0);
    load(s1, min(1, nk - 1));
    load(s2, min(2, nk - 1));
    for (int k = 0; k < nk; k += 3) {
        step(s0, k);
        if (k + 1 < nk) step(s1, k + 1);
        if (k + 2 < nk) step(s2, k + 2);
    }
    const int o = o0 + 16 * wv + 4 * q;
    if constexpr (KG == 2) {
        f32x4* red = reinterpret_cast<f32x4*>(&ws[0][0][0]);               // [TN / 16][4 waves][64]
        static_assert(sizeof(f32x4) * (TN / 16) * 256 <= sizeof(ws), "the sums fit");
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TN / 16; ++t)
            if (kg) red[(t * 4 + wv) * 64 + lane] = acc[t];
        __syncthreads();
        if (kg) return;
#pragma unroll
        for (int t = 0; t < TN / 16; ++t) acc[t] += red[(t * 4 + wv) * 64 + lane];
    }
#pragma unroll
    for (int t = 0; t < TN / 16; ++t) {
        const int64_t n = n0 + 16 * t + L;
        if (n < N && o < O)
            *reinterpret_cast<uint2*>(y + n * O + o) = make_uint2(pk2(acc[t][0], acc[t][1]), pk2(acc[t][2], acc[t][3]));
    }
}

extern "C" int rwkv6_linear_f32(const void* x, const float* w, void* y, void* w_bf16, int64_t N, int64_t O,
                                int64_t I, void* stream) {
    if (N < 0 || O < 1 || I < 1) return RWKV6_ERR_INVALID_ARG;
    if (O % 4 || I % 8 || O > (1 << 24) || I > (1 << 24)) return RWKV6_ERR_UNSUPPORTED;
    if (N == 0) return RWKV6_ERR_UNSUPPORTED;                     // no workgroup would write w_bf16
    if (!w || !x || !y) return RWKV6_ERR_INVALID_ARG;
    for (const void* p : {x, (const void*)w, (const void*)y, (const void*)w_bf16})
        if (reinterpret_cast<uintptr_t>(p) & 15u) return RWKV6_ERR_ALIGNMENT;
    if (any_alias({{y, (size_t)(N * O) * 2}, {w_bf16, (size_t)(O * I) * 2}}, {{x, (size_t)(N * I) * 2}, {w, (size_t)(O * I) * 4}}))
        return RWKV6_ERR_INVALID_ARG;
    const int64_t ot = (O + LIN_O - 1) / LIN_O;
    // Workgroups of 32 tokens in eight waves while they leave CUs idle, then of 64 tokens (half the
    // reads of W) where those still give every CU one.
    const int64_t n32 = (N + 31) / 32, n64 = (N + 63) / 64;
    const bool split = ot * n32 <= 256, wide = !split && ot * n64 >= 256;
    const int64_t nt = wide ? n64 : n32;
    if (ot * nt > 0x7fffffff) return RWKV6_ERR_UNSUPPORTED;
    auto k = split ? rwkv6_linear_f32_kernel<32, 2> : wide ? rwkv6_linear_f32_kernel<64, 1> : rwkv6_linear_f32_kernel<32, 1>;
    hipLaunchKernelGGL(k, dim3((unsigned)(ot * nt)), dim3(split ? 512 : 256),
                       0, reinterpret_cast<hipStream_t>(stream), (const uint16_t*)x, w, (uint16_t*)y, (uint16_t*)w_bf16, N,
                       (int)O, (int)I, (int)ot);
    return hipGetLastError() == hipSuccess ? RWKV6_OK : RWKV6_ERR_LAUNCH;
}
