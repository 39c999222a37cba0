// The reference's FP4Linear numerics (qwen38_inf2/model.py:198-208): bf16 x [T, K] against an MXFP4 weight, the inputs of
// even and odd index summed apart in float32, each sum rounded to bf16, the two added and rounded again.
//
// Both sums come from one pass over the weight: lane by lane a weight tile's MFMA words 2p and 2p + 1 (8 nibbles each, of
// one MX block) are regrouped into a word of their even and a word of their odd inputs, three bit operations each, so that
// every MFMA takes inputs of one parity only, and the activation tiles are written in the same order. That is the work of
// one ordinary projection, with twice the accumulators.
#include <algorithm>

#include "kernels.h"

typedef uint32_t u4 __attribute__((ext_vector_type(4)));

namespace {

// bf16 activation tiles [T / 32][K / 64][2 p + parity][64][8]: lane l of tile (i, k) holds of token 32 i + l % 32 the inputs
// of that parity among the 16 from 64 k + 32 p + 16 (l / 32), in the order 0, 8, 2, 10, ... (1, 9, 3, 11, ...).
__global__ __launch_bounds__(256) void act_planes_kernel(const bf16_t* x, int T, int K, bf16_t* act) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;  // 16 inputs of a token
    const int per = K / 16;
    if (i >= (size_t)T * per) return;
    const int t = (int)(i / per), g = (int)(i % per);  // g: K-step g / 4, block p = g / 2 % 2, lane half g % 2
    const uint2* src = (const uint2*)(x + (size_t)t * K + g * 16);
    uint2 r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = src[j];
    const uint32_t lo[4] = {r[0].x, r[0].y, r[1].x, r[1].y}, hi[4] = {r[2].x, r[2].y, r[3].x, r[3].y};
    u4 even, odd;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        even[j] = (lo[j] & 0xffffu) | hi[j] << 16;
        odd[j] = lo[j] >> 16 | (hi[j] & 0xffff0000u);
    }
    bf16_t* dst = act + ((size_t)(t >> 5) * (K >> 6) + (g >> 2)) * 2048 + ((g >> 1) & 1) * 1024 + ((t & 31) + (g & 1) * 32) * 8;
    *(u4*)dst = even;
    *(u4*)(dst + 512) = odd;
}

struct PlanesArgs {
    const uint8_t* w;   // weight tiles [N/32][K/64][4][64][4]
    const uint8_t* ws;  // scales [N/32][K/64][32][2]
    const bf16_t* act;  // act_planes_kernel's tiles
    bf16_t* out;        // [T][N]
    int T, K, N, blocks;  // blocks of 32 TT tokens
};

// A workgroup of KW waves takes 32 FR features x 32 TT tokens; its waves split K and add up through LDS at the end, a feature
// tile and a parity at a time, so nothing is shared before that: every operand goes straight to registers, D K-steps
// ahead, without a barrier. Bound by the L2 at 64 tokens per block (FR = 4: 12 KB per K-step for 32 MFMAs), by HBM's
// weights and the launches at few tokens. With the tiles' preparation, 200 rows of 5120 -> 5120 take 22.5 us a call among
// others (0.47 PFLOP/s), 1,024 of 5120 -> 14336 176 us (0.85 PFLOP/s); as a projection per parity, the other parity's inputs
// zero, in 256 x 256 tiles, they took 148 and 287 us. Without the scheduling barrier the compiler moves the 128 x 64
// tile's loads to their use (31.4 against 25.4 us in a sweep that waited for each call).
template <int FR, int TT, int KW, int D>
__global__ __launch_bounds__(KW * 64) __attribute__((amdgpu_waves_per_eu(KW / 4))) void fp4_planes_kernel(const PlanesArgs a) {
    constexpr int G = TT * 4, GW = (G + KW - 1) / KW;  // (token tile, quarter of the rows) quads of a feature tile, per wave
    __shared__ __attribute__((aligned(16))) float red[KW * G * 256];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int KS = a.K >> 6, group = 8 * a.blocks, in = blockIdx.x % group;
    // A feature tile's token blocks 8 ids apart, on one XCD: its weights come from HBM once.
    const int fb = blockIdx.x / group * 8 + in % 8, tb = in / 8;
    if (fb >= a.N / (32 * FR)) return;
    const int k0 = (int)((long)wave * KS / KW), k1 = (int)((long)(wave + 1) * KS / KW), klast = max(k1 - 1, 0);

    struct Step {
        uint32_t w[FR][4];
        u4 x[TT][4];
        uint16_t sc[FR];
    };
    Step st[D];
    auto load = [&](int k, Step& s) __attribute__((always_inline)) {
        k = min(k, klast);  // past the range: loaded, never used
        const uint8_t* wp = a.w + ((size_t)(fb * FR) * KS + k) * 1024 + lane * 4;
        const uint8_t* sp = a.ws + ((size_t)(fb * FR) * KS + k) * 64 + (lane & 31) * 2;
        const bf16_t* xp = a.act + ((size_t)(tb * TT) * KS + k) * 2048 + lane * 8;
#pragma unroll
        for (int f = 0; f < FR; ++f) {
            s.sc[f] = *(const uint16_t*)(sp + (size_t)f * KS * 64);
#pragma unroll
            for (int m = 0; m < 4; ++m) s.w[f][m] = *(const uint32_t*)(wp + (size_t)f * KS * 1024 + m * 256);
        }
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int m = 0; m < 4; ++m) s.x[t][m] = *(const u4*)(xp + (size_t)t * KS * 2048 + m * 512);
    };
    v16f acc[2][FR][TT];  // even, odd
#pragma unroll
    for (int f = 0; f < FR; ++f)
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[0][f][t][i] = acc[1][f][t][i] = 0.0f;
    auto compute = [&](const Step& s) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int f = 0; f < FR; ++f) {
                const float scale = __uint_as_float((uint32_t)(p ? s.sc[f] >> 8 : s.sc[f] & 0xff) << 23);
                const uint32_t w0 = s.w[f][2 * p], w1 = s.w[f][2 * p + 1];
                const v8bf16 even = widen_e2m1((w0 & 0x0f0f0f0fu) | (w1 & 0x0f0f0f0fu) << 4, scale);
                const v8bf16 odd = widen_e2m1((w0 >> 4 & 0x0f0f0f0fu) | (w1 & 0xf0f0f0f0u), scale);
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    acc[0][f][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(even, __builtin_bit_cast(v8bf16, s.x[t][2 * p]), acc[0][f][t], 0, 0, 0);
                    acc[1][f][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(odd, __builtin_bit_cast(v8bf16, s.x[t][2 * p + 1]), acc[1][f][t], 0, 0, 0);
                }
            }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load(k0 + d, st[d]);
    int k = k0;
    for (; k + D <= k1; k += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            compute(st[d]);
            load(k + D + d, st[d]);
            __builtin_amdgcn_sched_barrier(0);  // the loads stay D - 1 K-steps ahead of their use
        }
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (k + d < k1) compute(st[d]);

    // Wave w holds quads w, w + KW, ...: features 8 q + 4 (l / 32) + [0, 4) of token 32 t + l % 32 for quad 4 t + q.
#pragma unroll
    for (int f = 0; f < FR; ++f) {
        v4f sum[2][GW];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            __syncthreads();  // the last reads of red are done
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *(v4f*)(red + ((wave * G + t * 4 + q) * 64 + lane) * 4) =
                        (v4f){acc[h][f][t][4 * q], acc[h][f][t][4 * q + 1], acc[h][f][t][4 * q + 2], acc[h][f][t][4 * q + 3]};
            __syncthreads();
#pragma unroll
            for (int j = 0; j < GW; ++j) {
                const int g = wave + j * KW;
                if (g >= G) continue;
                v4f x[KW];
#pragma unroll
                for (int w = 0; w < KW; ++w) x[w] = *(const v4f*)(red + ((w * G + g) * 64 + lane) * 4);
#pragma unroll
                for (int w = 1; w < KW; ++w) x[0] += x[w];
                sum[h][j] = x[0];
            }
        }
#pragma unroll
        for (int j = 0; j < GW; ++j) {
            const int g = wave + j * KW, tok = (tb * TT + (g >> 2)) * 32 + (lane & 31);
            if (g >= G || tok >= a.T) continue;
            const int col = (fb * FR + f) * 32 + (g & 3) * 8 + (lane >> 5) * 4;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = rbf(sum[0][j][e]) + rbf(sum[1][j][e]);
            *(uint2*)(a.out + (size_t)tok * a.N + col) = make_uint2(pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3]));
        }
    }
}

template <int FR, int TT, int KW, int D>
hipError_t launch(PlanesArgs a, hipStream_t stream) {
    a.blocks = (a.T + 32 * TT - 1) / (32 * TT);
    const int groups = (a.N / (32 * FR) + 7) / 8;
    hipLaunchKernelGGL((fp4_planes_kernel<FR, TT, KW, D>), dim3(groups * 8 * a.blocks), dim3(KW * 64), 0, stream, a);
    return hipGetLastError();
}

}  // namespace

hipError_t q38_fp4_planes(const bf16_t* x, int T, int K, const uint8_t* tiles, const uint8_t* scales, int N, bf16_t* act,
                          bf16_t* out, int cus, hipStream_t stream) {
    if (N % 256 || K % 64) return hipErrorInvalidValue;
    const size_t pieces = (size_t)T * (K / 16);
    hipLaunchKernelGGL(act_planes_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream, x, T, K, act);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const PlanesArgs a = {tiles, scales, act, out, T, K, N, 0};
    // The largest tile that still leaves no CU without one: operands weigh less the larger it is (us with 32 x 32, 64 x 32,
    // 64 x 64 and 128 x 64 features x tokens). 6144 -> 5120: 13.3, 15.7, -, - at 1 row (160, 80 tiles); 20.8, 17.1, 20.8, 26.7
    // at 50 (320, 160, 80, 40); 5120 -> 14336: 20.5, 16.4, -, - at 1 row (448, 224), 34.9, 27.0, 20.9, 26.2 at 50 (896, 448,
    // 224, 112). A 128 x 64 workgroup has its CU to itself, a 64 x 64 one shares it, so between these the line is at half
    // the CUs: 5120 -> 5120 16.7 against 22.6 us at 100 rows (80 of the larger tiles), 29.8 against 25.4 at 200 (160).
    const long t32 = (T + 31) / 32, t64 = (T + 63) / 64;
    if (N / 32 * t32 <= cus) return launch<1, 1, 8, 4>(a, stream);
    if (T <= 32 || N / 64 * t32 <= cus) return launch<2, 1, 8, 4>(a, stream);
    if (N / 128 * t64 * 2 <= cus) return launch<2, 2, 4, 3>(a, stream);
    return launch<4, 2, 4, 2>(a, stream);
}
