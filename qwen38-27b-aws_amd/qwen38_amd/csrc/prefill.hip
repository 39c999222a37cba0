// Prefill form of the verify path's layers: one chunk of L tokens of one row (`slot`) from position `start`, tokens
// from `n_valid` on being padding (reference qwen38_inf2/model.py:476-521 for the gated delta net, 704-799 for
// attention, 843-855 for the MTP layer's cache-only form).
//
// Gated delta net, after the qkvz GEMM and the gates kernel over the chunk:
//   gdn_prefill_prep   (32 tokens, key head): conv over the chunk with the row's conv history (bf16 tap products summed
//                      by bf16 additions, model.py:514), SiLU, l2 norms of q and k, the gates times `valid`; the
//                      state-independent matrices of the delta rule over these tokens
//   gdn_prefill_scan   (value head, 32 state columns): the gated delta rule (per token S = e^g S, delta = (v - S^T k)
//                      beta, S += k delta^T, o = S^T q) in chunks of 32 tokens from the row's state (times `start > 0`), in
//                      float32 on the matrix cores
//   gdn_prefill_finish (4 tokens, 4 value heads): gated RMS norm of bf16 o times SiLU(z), e5m2 tiles for out_proj
//   gdn_prefill_carry  the row's new conv state: the three inputs from n_valid on of [history, chunk]
//
// Attention, after the qkv GEMM over the chunk:
//   attn_prefill_prep  (token): q and k RMS norms and RoPE in bf16 (model.py:565-577), q times 1/16 (exact) to scratch;
//                      the chunk's keys and values into row slot's cache at start .. start + L - 1 (model.py:791-799;
//                      the other rows' junk writes at the cache's end are left out: nothing reads them)
//   attn_prefill_widen an FP8 cache's row widened to bf16 once
//   attn_prefill_max, attn_prefill, attn_prefill_finish: blocked_attention (model.py:170-191) over the row's cached
//                      positions before `start` and the chunk's own tokens causally, in the reference's blocks of 2048
//                      positions of [cache, chunk]: per block the running max, e^(s - max) summed in float32, the
//                      weights in bf16 times V on the MFMA (float32 sums, rounded to bf16 once per block, as the
//                      reference's bf16 matmul), output and sum rescaled across blocks; then out / sum, the gate, e5m2.
//                      Positions a row cannot see are skipped: the reference gives them weights of exactly zero.
#include <algorithm>
#include <type_traits>

#include "kernels.h"

namespace {

constexpr int GC = PREFILL_GDN_CHUNK;  // tokens of one chunk of the delta rule

__device__ __forceinline__ float conv_window(const PrefillGdnArgs& a, const bf16_t* hist, float keep, int c, int w) {
    // Input w of channel c's window: the row's conv history (times keep) for w < 3, then the chunk's inputs.
    return w < 3 ? bf2f(hist[(size_t)c * 3 + w]) * keep : bf2f(a.qkv[(size_t)(w - 3) * a.C + c]);
}

__device__ __forceinline__ v4f mfma16(float x, float y, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }

// e^x of a 64-bit x, to expf's error without x's own rounding (|x| ulps of the result).
__device__ __forceinline__ double exp_of(double x) {
    const float hi = (float)x;
    const double e = expf(hi);
    return e + e * (x - hi);
}

__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }

// This wave's LDS accesses are done; then meet the other waves (loads from global memory stay in flight).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace

// Grid (32 tokens, key head): conv, SiLU, l2 norms and gates of the tokens, then what a chunk of the delta rule needs that
// does not depend on the state. With c_t the log decays summed from the chunk's start, k . k and q . k on the float64 MFMA, and per
// value head M_ts = beta_t e^(c_t - c_s) k_t . k_s (s < t), T = (I + M)^-1 by forward substitution (a column per lane),
// P_ts = e^(c_t - c_s) q_t . k_s (s <= t).
// Bounds: the conv's and SiLU's arithmetic (about 40 instructions per input at a bf16 rounding after each operation; the
// memory traffic, 145 MB for 2,048 tokens of the 27B layer, is half its time). Wave w takes tokens 8 w .. 8 w + 7 of one
// head after another, a lane two channels, each input loaded once for the four taps, the next head's meanwhile: 60 us
// with the matrices (67 since these are 64-bit sums), where one token and channel per thread took 152 us for the conv and norms alone.
__global__ __launch_bounds__(256) void gdn_prefill_prep_kernel(const PrefillGdnArgs a) {
    constexpr int D = 128, GMAX = 8, KP = D + 4, MP = GC + 4;
    __shared__ __attribute__((aligned(16))) float sk[GC][KP], sq[GC][KP], sm[4][GC][MP];
    __shared__ float sb[4][GC];
    __shared__ double sc[4][GC];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ch = blockIdx.x, t0 = ch * GC, kh = blockIdx.y;
    const int Hk = a.Hk, Hv = a.Hv, C = a.C, rep = Hv / Hk;
    const int slot = *a.slot, nv = *a.n_valid;
    if (slot < 0 || slot >= a.rows) return;
    const float keep = *a.start > 0 ? 1.0f : 0.0f;
    const bf16_t* hist = a.conv + (size_t)slot * C * 3;

    const int tw = t0 + 8 * wave;  // this wave's first token
    // Inputs of head hd (q, k, then the value heads): the window of this wave's tokens, a word of two channels each, and the
    // taps; the next head's load while this one's are used.
    auto channel = [&](int hd) {
        return (hd == 0 ? kh * D : hd == 1 ? Hk * D + kh * D : 2 * Hk * D + (kh * rep + hd - 2) * D) + 2 * lane;
    };
    uint32_t xw[11];
    uint4 cw;
    auto load = [&](int hd) {
        const int c = channel(hd);
#pragma unroll
        for (int j = 0; j < 11; ++j)
            xw[j] = j < 3 && tw == 0 ? pk_bf16(conv_window(a, hist, keep, c, j), conv_window(a, hist, keep, c + 1, j))
                                     : *(const uint32_t*)(a.qkv + (size_t)(tw + j - 3) * C + c);
        cw = *(const uint4*)(a.conv_w + (size_t)c * 4);
    };
    load(0);
    for (int hd = 0; hd < 2 + rep; ++hd) {
        float x[11][2];
#pragma unroll
        for (int j = 0; j < 11; ++j) x[j][0] = lo_bf(xw[j]), x[j][1] = hi_bf(xw[j]);
        const float w[2][4] = {{lo_bf(cw.x), hi_bf(cw.x), lo_bf(cw.y), hi_bf(cw.y)}, {lo_bf(cw.z), hi_bf(cw.z), lo_bf(cw.w), hi_bf(cw.w)}};
        if (hd + 1 < 2 + rep) load(hd + 1);
        float y[8][2];
        auto round2 = [](float& p, float& q) {  // both to bf16 and back, one conversion
            const uint32_t r = pk_bf16(p, q);
            p = lo_bf(r);
            q = hi_bf(r);
        };
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            float m[2];
#pragma unroll
            for (int j = 0; j < 4; ++j) {  // bf16 tap products summed by bf16 additions (model.py:514)
                float p[2] = {x[t + j][0] * w[0][j], x[t + j][1] * w[1][j]};
                round2(p[0], p[1]);
                m[0] = j ? m[0] + p[0] : p[0];
                m[1] = j ? m[1] + p[1] : p[1];
                if (j) round2(m[0], m[1]);
            }
            float g[2] = {sigmoidf_(m[0]), sigmoidf_(m[1])};
            round2(g[0], g[1]);
            y[t][0] = m[0] * g[0];
            y[t][1] = m[1] * g[1];
            round2(y[t][0], y[t][1]);
        }
        if (hd < 2) {
            float ss[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) ss[t] = y[t][0] * y[t][0] + y[t][1] * y[t][1];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
#pragma unroll
                for (int t = 0; t < 8; ++t) ss[t] += __shfl_xor(ss[t], o);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const float rs = 1.0f / sqrtf(ss[t] + 1e-6f);
                const float2 v = hd ? make_float2(y[t][0] * rs, y[t][1] * rs)
                                    : make_float2((y[t][0] * rs) / 11.313708498984761f, (y[t][1] * rs) / 11.313708498984761f);
                *(float2*)((hd ? a.kn : a.qn) + ((size_t)(tw + t) * Hk + kh) * D + 2 * lane) = v;
                *(float2*)&(hd ? sk : sq)[8 * wave + t][2 * lane] = v;
            }
        } else {
            const int h = kh * rep + hd - 2;
#pragma unroll
            for (int t = 0; t < 8; ++t) *(uint32_t*)(a.v + ((size_t)(tw + t) * Hv + h) * D + 2 * lane) = pk_bf16(y[t][0], y[t][1]);
        }
    }
    __syncthreads();

    // k . k and q . k, a 16 x 16 quarter per wave (rows t, columns s; the quarter above the diagonal stays zero): four
    // MFMA steps per 16-byte read, the same order of inputs in both operands. In 64 bits: as float32 chains of 128 their
    // rounding was most of the delta rule's error.
    const int wr = wave >> 1, wc = wave & 1, lr = lane & 15, lq = lane >> 4;
    typedef double v4d __attribute__((ext_vector_type(4)));
    v4d kk = {0.0, 0.0, 0.0, 0.0}, qk = kk;  // element i: row 16 wr + 4 i + lq, column 16 wc + lr
    if (wr >= wc)
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const v4f kt = *(const v4f*)&sk[16 * wr + lr][16 * g + 4 * lq], qt = *(const v4f*)&sq[16 * wr + lr][16 * g + 4 * lq];
            const v4f ks = *(const v4f*)&sk[16 * wc + lr][16 * g + 4 * lq];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                kk = __builtin_amdgcn_mfma_f64_16x16x4f64(kt[e], ks[e], kk, 0, 0, 0);
                qk = __builtin_amdgcn_mfma_f64_16x16x4f64(qt[e], ks[e], qk, 0, 0, 0);
            }
        }
    for (int r0 = 0; r0 < rep; r0 += 4) {  // value heads, four at a time
        const int nh = min(4, rep - r0);
        // Gates (model.py:333-337, 499-500), then the chunk's cumulative log decays: a half wave per head.
        if (tid < 32 * nh) {
            const int r = tid >> 5, t = t0 + (tid & 31), h = kh * rep + r0 + r, O = 2 * Hv;
            const float valid = t < nv ? 1.0f : 0.0f;
            float sum[2] = {0.0f, 0.0f};
#pragma unroll
            for (int gi = 0; gi < GMAX; ++gi)
                if (gi < a.gate_groups) {
                    const float* p = a.gate_part + ((size_t)gi * a.L + t) * O + h;
                    sum[0] += p[0];
                    sum[1] += p[Hv];
                }
            const float beta = rbf(sigmoidf_(rbf(sum[0]))) * valid;
            const float g = -expf(bf2f(a.a_log[h])) * softplusf_(rbf(sum[1]) + bf2f(a.dt_bias[h])) * valid;
            // Summed in 64 bits: the factors are e to differences of these sums, often small ones of large ones. No term is
            // below -200, whose e^g is zero in float32 as well, so that the differences after it keep their digits.
            double c = g < -200.0f ? -200.0f : g;
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) {
                const double up = __shfl_up(c, o, 32);
                if ((tid & 31) >= o) c += up;
            }
            sb[r][tid & 31] = beta;
            sc[r][tid & 31] = c;
            const double last = __shfl(c, 31, 32) - c;
            float* f = a.decay + (((size_t)ch * Hv + h) * 3) * GC + (tid & 31);
            f[0] = beta;
            f[GC] = (float)exp_of(c);
            f[2 * GC] = (float)exp_of(last);
        }
        __syncthreads();
        for (int r = 0; r < nh; ++r) {
            float* P = a.pt + ((size_t)ch * Hv + kh * rep + r0 + r) * 2 * GC * GC + GC * GC;
            const int s = 16 * wc + lr;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = 16 * wr + 4 * i + lq;
                const double e = t >= s ? exp_of(sc[r][t] - sc[r][s]) : 0.0;
                sm[r][t][s] = (float)(sb[r][t] * e * kk[i]);
                P[t * GC + s] = t >= s ? (float)(e * qk[i]) : 0.0f;  // not 0 q . k: a token's NaN is not an earlier one's
            }
        }
        __syncthreads();
        if (wave < nh && lane < GC) {  // column `lane` of T
            float* T = a.pt + ((size_t)ch * Hv + kh * rep + r0 + wave) * 2 * GC * GC;
            float col[GC];
#pragma unroll
            for (int i = 0; i < GC; ++i) {
                float v = i == lane ? 1.0f : 0.0f;
#pragma unroll
                for (int s4 = 0; s4 < i; s4 += 4) {
                    const v4f m = *(const v4f*)&sm[wave][i][s4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (s4 + e < i) v -= m[e] * col[s4 + e];
                }
                col[i] = v;
                T[i * GC + lane] = v;
            }
        }
        if (r0 + 4 < rep) __syncthreads();  // sm, sb and sc are read before the next heads' are written
    }
}

// The delta rule over the chunks, grid (value head, group of 32 state columns), four waves. The state S (128 x 32 here)
// stays in registers, wave w rows 32 w .. 32 w + 31 as one 32x32 float32 accumulator, whose registers are at the same
// time the B operands of the next chunk's reads (MFMA i takes state rows drow(i, half)). Per chunk of 32 tokens:
//   k . S and q . S over the wave's rows, the four waves' parts added through LDS;  R = beta (v - e^c k . S)
//   Delta = T R;  o = e^c q . S + P Delta;  S = e^(c_last) S + (e^(c_last - c) k)^T Delta
// all in float32 on the float32 MFMA. The reference runs the same in pieces of 128 tokens (chunked_gated_delta,
// model.py:88-124); 32 keep T and P small, and the state's products, which are most of the work, do not depend on it.
// Bounds: the float32 matrix rate of the CUs that 4 Hv workgroups fill: per wave and chunk 32 + 16 MFMAs of 64 cycles and
// 16 of 32, with three LDS round trips between them. k, q, T, P, v and the gates of the next chunk load meanwhile.
// A value, token or decay that is not finite reaches the tokens after it and the state, as token by token: a chunk with such
// an R or Delta clears them before they meet the zeros of T and P (3 us for the tests; nothing else in a chunk without).
// 2,048 tokens of the 27B layer (64 chunks): 231 us, 46 TFLOP/s; token by token (one state column in 8 lanes, DPP
// sums) 781 us. Against 64 bits from the same k, q, v, beta and g, o before its rounding to bf16 is off by 7.6e-8 to 1.9e-7
// (512 tokens, decays from e^-5 to e^-0.002 per token; 7.9e-8 to 4.3e-7 token by token, and with k . k and q . k as float32
// chains 1.7e-7 to 2.3e-7, 10 us less in all), the state after its rounding by 1.64e-3 to 1.67e-3 in every form.
__global__ __launch_bounds__(256) void gdn_prefill_scan_kernel(const PrefillGdnArgs a) {
    constexpr int D = 128, KB = GC * D * 4, RP = 36;  // bytes of a chunk's k or q, floats per row of the 32 x 32 tiles
    __shared__ __attribute__((aligned(1024))) uint8_t ring[2][2][KB];  // [stage][k, q], 16-byte chunk c of row r at c ^ (r % 16)
    __shared__ __attribute__((aligned(16))) float red[4][2][4][64][4];
    __shared__ __attribute__((aligned(16))) float sR[GC][RP], sO[GC][RP], sD[GC][RP], sW[GC][RP];
    __shared__ int sbad[2][2];  // by chunk parity: whether an R, a Delta is not finite
    __shared__ int sfirst[GC];  // then, by column: the first such token
    __shared__ float sf[2][3 * GC];  // beta, e^c, e^(c_last - c), by chunk parity: a chunk's tail reads while the next's are written
    const int h = blockIdx.x, grp = blockIdx.y, tid = threadIdx.x, lane = tid & 63, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int Hk = a.Hk, Hv = a.Hv, kh = h / (Hv / Hk), nch = a.L / GC;
    const int slot = *a.slot;
    if (slot < 0 || slot >= a.rows) return;
    const float keep = *a.start > 0 ? 1.0f : 0.0f;
    bf16_t* st = a.state + ((size_t)slot * Hv + h) * D * D + grp * 32 + (lane & 31);
    auto row = [&](int i) { return 32 * wave + 8 * (i >> 2) + 4 * hf + (i & 3); };
    v16f S;
#pragma unroll
    for (int i = 0; i < 16; ++i) S[i] = bf2f(st[(size_t)row(i) * D]) * keep;

    // Loads of chunk c: k and q into stage c % 2 (a wave 8 rows of each, two per instruction), T's and P's rows of this
    // wave's quarter, the four v of this thread's tokens 8 w + 4 hf + e, and for threads 0..95 the tokens' factors.
    const int wr = wave >> 1, wc = wave & 1, lr = lane & 15, lq = lane >> 4;
    const uint32_t lds0 = (uint32_t)(uintptr_t)LDS_PTR(&ring[0][0][0]);
    v4f T[2], P[2];
    uint32_t vr[4];
    float gf = 0.0f;
    auto load = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint8_t* src = (const uint8_t*)(w ? a.qn : a.kn) + ((size_t)c * GC * Hk + kh) * D * 4;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = 8 * wave + 2 * j + hf;
                lds_quad(src, (uint32_t)(r * Hk * D * 4 + (((lane & 31) ^ (r & 15)) << 4)),
                         lds0 + ((c & 1) * 2 + w) * KB + (8 * wave + 2 * j) * D * 4);
            }
        }
        const float* pt = a.pt + ((size_t)c * Hv + h) * 2 * GC * GC + (16 * wr + lr) * GC + 4 * lq;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            T[g] = *(const v4f*)(pt + 16 * g);
            P[g] = *(const v4f*)(pt + GC * GC + 16 * g);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            vr[e] = a.v[((size_t)(c * GC + 8 * wave + 4 * hf + e) * Hv + h) * D + grp * 32 + (lane & 31)];
        if (tid < 3 * GC) gf = a.decay[((size_t)c * Hv + h) * 3 * GC + tid];
    };
    // A column's R or Delta from its first token that is not finite on (at `most` by then) become zero, so that earlier
    // tokens, whose rows of T and P multiply them by zero, stay as they are; sfirst says from where on the column is lost.
    auto clear_from_first = [&](float(*x)[RP], int most) {
        int first = most;
        for (int t = most - 1; t >= 0; --t) first = finite(x[t][tid]) ? first : t;
        for (int t = first; t < GC; ++t) x[t][tid] = 0.0f;
        sfirst[tid] = first;
    };
    load(0);
    for (int c = 0; c < nch; ++c) {
        // Everything but the last chunk's four output stores.
        if (c == 0)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        const float *sb = sf[c & 1], *se = sb + GC, *sw = sb + 2 * GC;
        if (tid < 3 * GC) sf[c & 1][tid] = gf;
        if (tid < 2) sbad[c & 1][tid] = 0;
        const v4f Tc[2] = {T[0], T[1]}, Pc[2] = {P[0], P[1]};
        float vc[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) vc[e] = __uint_as_float(vr[e] << 16);
        lds_barrier();  // the chunk's k, q and gates are in LDS; every wave is done with the chunk before
        // This wave's LDS operands of k . S, q . S and the state's update (rows of k down its 32 columns) in one go: read
        // one by one before their MFMAs they cost their latency each. The fences keep the reads here.
        const uint32_t kq = lds0 + (c & 1) * 2 * KB;
        auto piece = [&](uint32_t base, int g) __attribute__((always_inline)) {  // inputs 32 w + 8 g + 4 hf + [0, 4) of token lane % 32
            const int r = lane & 31;
            return *(const __attribute__((address_space(3))) v4f*)(uintptr_t)(base + r * D * 4 + (((8 * wave + 2 * g + hf) ^ (r & 15)) << 4));
        };
        v4f kp[4], qp[4];
        float kt[16];
#pragma unroll
        for (int g = 0; g < 4; ++g) kp[g] = piece(kq, g), qp[g] = piece(kq + KB, g);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int s = 2 * j + hf;
            kt[j] = *(const __attribute__((address_space(3))) float*)(uintptr_t)(
                kq + s * D * 4 + (((8 * wave + ((lane & 31) >> 2)) ^ (s & 15)) << 4) + (lane & 3) * 4);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (c + 1 < nch) load(c + 1);

        // k . S and q . S over this wave's 32 state rows; q . S, which goes straight into o, as two sums of 16.
        v16f ks, qs, qs2;
#pragma unroll
        for (int i = 0; i < 16; ++i) ks[i] = qs[i] = qs2[i] = 0.0f;
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ks = __builtin_amdgcn_mfma_f32_32x32x2f32(kp[g][e], S[4 * g + e], ks, 0, 0, 0);
                v16f& q = g < 2 ? qs : qs2;
                q = __builtin_amdgcn_mfma_f32_32x32x2f32(qp[g][e], S[4 * g + e], q, 0, 0, 0);
            }
        qs += qs2;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            *(v4f*)red[wave][0][q][lane] = (v4f){ks[4 * q], ks[4 * q + 1], ks[4 * q + 2], ks[4 * q + 3]};
            *(v4f*)red[wave][1][q][lane] = (v4f){qs[4 * q], qs[4 * q + 1], qs[4 * q + 2], qs[4 * q + 3]};
        }
        lds_barrier();
        {  // this thread: tokens 8 w + 4 hf + e, column lane % 32
            v4f kw[4], qw[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) kw[w] = *(const v4f*)red[w][0][wave][lane], qw[w] = *(const v4f*)red[w][1][wave][lane];
            __builtin_amdgcn_sched_barrier(0);
            const v4f k4 = (kw[0] + kw[1]) + (kw[2] + kw[3]), q4 = (qw[0] + qw[1]) + (qw[2] + qw[3]);
            float zero = 0.0f;  // NaN if a value is not finite
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 8 * wave + 4 * hf + e;
                const float R = sb[t] * (vc[e] - se[t] * k4[e]);
                sR[t][lane & 31] = R;
                sO[t][lane & 31] = se[t] * q4[e];
                zero += 0.0f * R;
            }
            if (zero != 0.0f) sbad[c & 1][0] = 1;
        }
        lds_barrier();
        // Delta, a 16 x 16 quarter per wave (T is lower triangular: the upper quarters sum 16 tokens).
        float rr[8];
        auto read_r = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 8; ++j) rr[j] = sR[16 * (j >> 2) + 4 * lq + (j & 3)][16 * wc + lr];
        };
        read_r();
        const bool bad_r = __builtin_amdgcn_readfirstlane(sbad[c & 1][0]) != 0;
        __builtin_amdgcn_sched_barrier(0);
        if (bad_r) {
            lds_barrier();  // every wave has read
            if (tid < GC) clear_from_first(sR, GC);
            lds_barrier();
            read_r();
        }
        v4f dl = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 4; ++e) dl = mfma16(Tc[0][e], rr[e], dl);
        if (wr)
#pragma unroll
            for (int e = 0; e < 4; ++e) dl = mfma16(Tc[1][e], rr[4 + e], dl);
        float zero = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = 16 * wr + 4 * lq + i;
            sD[t][16 * wc + lr] = dl[i];
            sW[t][16 * wc + lr] = dl[i] * sw[t];
            zero += 0.0f * dl[i];
        }
        if (zero != 0.0f) sbad[c & 1][1] = 1;
        const float es = se[GC - 1];
#pragma unroll
        for (int i = 0; i < 16; ++i) S[i] *= es;
        lds_barrier();
        // The state, and beside its chain the outputs.
        float dw[16], dd[8];
        v4f oq;
#pragma unroll
        for (int j = 0; j < 16; ++j) dw[j] = sW[2 * j + hf][lane & 31];
        auto read_d = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 8; ++j) dd[j] = sD[16 * (j >> 2) + 4 * lq + (j & 3)][16 * wc + lr];
        };
        read_d();
#pragma unroll
        for (int i = 0; i < 4; ++i) oq[i] = sO[16 * wr + 4 * lq + i][16 * wc + lr];
        const bool bad = bad_r || __builtin_amdgcn_readfirstlane(sbad[c & 1][1]) != 0;
        __builtin_amdgcn_sched_barrier(0);
        if (bad) {
            lds_barrier();
            if (tid < GC) clear_from_first(sD, bad_r ? sfirst[tid] : GC);
            lds_barrier();
            read_d();
        }
        v4f op[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) op[j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            S = __builtin_amdgcn_mfma_f32_32x32x2f32(kt[j], dw[j], S, 0, 0, 0);
            if (j < 8) op[j >> 1] = mfma16(Pc[j >> 2][j & 3], dd[j], op[j >> 1]);
        }
        v4f o = oq + ((op[0] + op[1]) + (op[2] + op[3]));
        if (bad) {
            const int from = sfirst[16 * wc + lr];
            const bool lost = sfirst[lane & 31] < GC;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = 16 * wr + 4 * lq + i < from ? o[i] : NAN;
#pragma unroll
            for (int i = 0; i < 16; ++i) S[i] = lost ? NAN : S[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a.o[((size_t)(c * GC + 16 * wr + 4 * lq + i) * Hv + h) * D + grp * 32 + 16 * wc + lr] = f2bf(o[i]);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) st[(size_t)row(i) * D] = f2bf(S[i]);
}

// The gated norm and out_proj's e5m2 tiles (model.py:339-345), grid (4 tokens, value heads / 4): wave w takes value head
// 4 blockIdx.y + w, 16 lanes per token, 8 dims per lane: whole cache lines of o and z, 8-byte tile stores (one byte at a
// time it took 40 us for 2,048 tokens of the 27B layer, 18 us now).
__global__ __launch_bounds__(256) void gdn_prefill_finish_kernel(const PrefillGdnArgs a) {
    constexpr int D = 128;
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (lane >> 4), d = (lane & 15) * 8;
    const int h = blockIdx.y * 4 + (threadIdx.x >> 6), Hv = a.Hv;
    const size_t at = ((size_t)t * Hv + h) * D + d;
    const uint4 ow = *(const uint4*)(a.o + at), zw = *(const uint4*)(a.z + at), nw = *(const uint4*)(a.norm_w + d);
    const uint32_t o2[4] = {ow.x, ow.y, ow.z, ow.w}, z2[4] = {zw.x, zw.y, zw.z, zw.w}, n2[4] = {nw.x, nw.y, nw.z, nw.w};
    float o[8], ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        o[e] = e & 1 ? hi_bf(o2[e >> 1]) : lo_bf(o2[e >> 1]);
        ss += o[e] * o[e];
    }
    const float r = 1.0f / sqrtf(group16_sum(ss) / 128.0f + a.eps);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float z = e & 1 ? hi_bf(z2[e >> 1]) : lo_bf(z2[e >> 1]), n = e & 1 ? hi_bf(n2[e >> 1]) : lo_bf(n2[e >> 1]);
        v[e] = rbf(rbf(n * rbf(o[e] * r)) * (z * sigmoidf_(z)));
    }
    *(uint2*)(a.act + act_offset(t, h * D + d, Hv * D)) = make_uint2(pk_e5m2(v[0], v[1], v[2], v[3]), pk_e5m2(v[4], v[5], v[6], v[7]));
}

// The row's new conv state (model.py:492-495): inputs n_valid .. n_valid + 2 of [history * keep, chunk].
__global__ __launch_bounds__(256) void gdn_prefill_carry_kernel(const PrefillGdnArgs a) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= a.C) return;
    const int slot = *a.slot, n = *a.n_valid;
    if (slot < 0 || slot >= a.rows || n < 1 || n > a.L) return;
    const float keep = *a.start > 0 ? 1.0f : 0.0f;
    bf16_t* hist = a.conv + (size_t)slot * a.C * 3;
    float w[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) w[q] = conv_window(a, hist, keep, c, n + q);
#pragma unroll
    for (int q = 0; q < 3; ++q) hist[(size_t)c * 3 + q] = f2bf(w[q]);
}

namespace {

constexpr int QP = 256;  // bf16 per scaled query row in the scratch

__device__ __forceinline__ int order_bits(float f) {  // floats in the order of signed ints
    const int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7fffffff;
}
__device__ __forceinline__ v8bf16 load8p(const bf16_t* p) { return *(const v8bf16*)p; }

// Wait until at most N of this wave's vector-memory operations are outstanding (its copies into the stage about to be
// read have landed) and its LDS reads have returned, then meet the other waves: after it the stage read one step
// before is free. The memory clobber keeps LDS reads after it.
template <int N>
__device__ __forceinline__ void ring_ready() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

}  // namespace

// Grid (token): wave w normalises and rotates rows w, w + 4, ...: query heads (scaled by 1/16 into qs), then the KV
// heads' keys (into the cache) and values (into the cache, transposed per 32 positions), as e4m3 bytes of value / scale
// with KV8. Lane l holds dims 4l .. 4l+3.
template <bool KV8>
__global__ __launch_bounds__(256) void attn_prefill_prep_kernel(const PrefillAttnArgs a) {
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int Hq = a.Hq, Hkv = a.Hkv, S = a.S, d0 = lane * 4;
    const int slot = *a.slot, p = *a.start + t;
    if (slot < 0 || slot >= a.rows) return;
    const int rows = a.keys_only ? 2 * Hkv : Hq + 2 * Hkv;
    const float ksc = KV8 ? bf2f(*a.k_scale) : 0.0f, vsc = KV8 ? bf2f(*a.v_scale) : 0.0f;
    float cs[4], sn[4];
    {
        const uint2 rc = *(const uint2*)(a.cos + (size_t)t * 64 + (d0 & 63));
        const uint2 rsn = *(const uint2*)(a.sin + (size_t)t * 64 + (d0 & 63));
        cs[0] = lo_bf(rc.x); cs[1] = hi_bf(rc.x); cs[2] = lo_bf(rc.y); cs[3] = hi_bf(rc.y);
        sn[0] = lo_bf(rsn.x); sn[1] = hi_bf(rsn.x); sn[2] = lo_bf(rsn.y); sn[3] = hi_bf(rsn.y);
    }
    for (int r0 = wave; r0 < rows; r0 += 4) {
        const int r = a.keys_only ? Hq + r0 : r0;  // 0..Hq-1 query heads, then keys, then values
        const bf16_t* src = r < Hq ? a.qkv + (size_t)t * a.ld + (size_t)r * 512
                                   : a.qkv + (size_t)t * a.ld + a.kv_col + (size_t)(r - Hq) * 256;
        const uint2 raw = *(const uint2*)(src + d0);
        float v[4] = {lo_bf(raw.x), hi_bf(raw.x), lo_bf(raw.y), hi_bf(raw.y)};
        if (r >= Hq + Hkv) {  // a value: stored as is
            const int kvh = r - Hq - Hkv;
            if (p < S) {
                const size_t vo = (((size_t)slot * Hkv + kvh) * S + (p & ~31)) * 256 + (p & 31);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (KV8)
                        ((uint8_t*)a.v_cache)[vo + (size_t)(d0 + e) * 32] = (uint8_t)kv_code(v[e], vsc);
                    else
                        a.v_cache[vo + (size_t)(d0 + e) * 32] = f2bf(v[e]);
                }
            }
            continue;
        }
        const bf16_t* nw = r < Hq ? a.q_norm : a.k_norm;
        const float ss = warp_sum(v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3]);
        const float rsq = 1.0f / sqrtf(ss / 256.0f + a.eps);
        float hn[4], out[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) hn[e] = rbf(v[e] * rsq * (1.0f + bf2f(nw[d0 + e])));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float part = __shfl_xor(hn[e], 8);
            const int d = d0 + e;
            out[e] = d < 64 ? rbf(rbf(hn[e] * cs[e]) + rbf((d < 32 ? -part : part) * sn[e])) : hn[e];
        }
        if (r < Hq) {
            for (int b = lane; b < a.nblk; b += 64)  // the row's block maxima start below every score
                a.mx[((size_t)r * a.nblk + b) * a.L + t] = order_bits(-INFINITY);
            *(uint2*)(a.qs + ((size_t)r * a.L + t) * QP + d0) =
                make_uint2(pk_bf16(out[0] * 0.0625f, out[1] * 0.0625f), pk_bf16(out[2] * 0.0625f, out[3] * 0.0625f));
        } else if (p < S) {
            const int kvh = r - Hq;
            const size_t ko = (((size_t)slot * Hkv + kvh) * S + p) * 256 + d0;
            if constexpr (KV8)
                *(uint32_t*)((uint8_t*)a.k_cache + ko) = kv_code(out[0], ksc) | kv_code(out[1], ksc) << 8 |
                                                         kv_code(out[2], ksc) << 16 | kv_code(out[3], ksc) << 24;
            else
                *(uint2*)(a.k_cache + ko) = make_uint2(pk_bf16(out[0], out[1]), pk_bf16(out[2], out[3]));
        }
    }
}

// ---- Attention over one chunk: attn_prefill_max, attn_prefill, attn_prefill_finish.
//
// A wave takes 64 tokens of one query head; a workgroup's four waves take four consecutive (64 tokens, query head) tiles
// of one KV head, heads fastest, so they see nearly the same positions, and each 32-position sub-block of K (and V) is
// copied into an LDS ring once and read by all four. 64 tokens per wave, because with 32 the waves' reads of the
// sub-blocks take the LDS as long as their MFMAs take the matrix cores (16 KB per 16 MFMAs and wave, 128 B a cycle).
// The 64 x 256 output (256 registers), the queries (128) and the scores then fill one wave per SIMD.
//
// The weights are the reference's bf16(e^(s - m)), m the running maximum through the end of the block of 2048 that
// holds the position, so m has to be known before a block's first weight: attn_prefill_max makes one pass over the
// scores for the blocks' maxima (two waves per SIMD), attn_prefill a second one for weights x V. Since every block's
// maximum is then known, a tile's positions need not be taken in order by one workgroup: the work is dealt out as items
// (tile of four waves, range of sub-blocks), as many ranges per tile as fill the CUs evenly (prefill_ranges), and
// attn_prefill_finish puts the blocks together in order.
//
// Bounds: the matrix cores, and in attn_prefill the weights' exponentials beside them. 2,048 tokens after 14,336 positions of
// the 27B layer (24 x 256 dims): 3 x 387 GFLOP in 310 + 1,120 + 110 us (0.75 PFLOP/s; two passes over the scores), before
// with 32 tokens a wave, 128 a workgroup and every tile's positions in one workgroup 3,669 us. Items that are whole blocks
// would save two thirds of the last kernel's reads, but leave the CUs idle: nine blocks over four items or less, 478 +
// 1,384 + 51 us.
namespace {

constexpr int PF_ROWS = 64;                  // tokens per wave
constexpr int PF_SUB = 32 * 256 * 2;         // bytes of one K or V sub-block in LDS

// e^x for x <= 0 (-inf and NaN included): x log2 e in two parts (the product and what its rounding left out), 2 to the
// power of their fraction, scaled by the whole part. Against 64 bits over all magnitudes from 5e-10 to 110 the largest
// and rms errors are expf's to the digit, 0.84 and 0.30 ulp, also below 2^-126; expf's tests for overflow and underflow
// are what is left out, which is half its time beside the MFMAs (attn_prefill over 16K positions: the layer 2,740 us, 2,850
// with expf; 2,600 with 2^(x log2 e) from the rounded product, which is off by 16 ulp at x = -20 and 0 below 2^-126).
__device__ __forceinline__ float exp_neg(float x) {
    constexpr float HI = 1.44269502162933349609375f, LO = 1.9259629911266175e-8f;  // log2 e
    const float p = fmaxf(x * HI, -300.0f), n = __builtin_rintf(p);  // past -300: r is as low, and the result zero
    const float r = (p - n) + __builtin_fmaf(x, LO, __builtin_fmaf(x, HI, -p));
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(r), (int)n);
}

// Sub-blocks (of 32 aligned cache positions) a tile sees: the cached positions [0, start) in order, then its own
// chunk's tokens 0 .. top, cut where the reference's blocks of [cache, chunk] end. Its blocks are numbered over those that
// hold a position the tile may see: the cached ones, then the own tokens', the first of which the last cached one may
// hold as well.
struct PrefillSpan {
    int S, start, n_c, first;  // first: own tokens before the first cut
    int cached, shared;        // blocks with cached positions; 1 if the last of them holds own tokens too
    __device__ __forceinline__ PrefillSpan(int S_, int start_)
        : S(S_), start(start_), n_c((start_ + 31) >> 5), first(2048 - (S_ & 2047)), cached((start_ + 2047) >> 11),
          shared(start_ > 0 && (start_ - 1) >> 11 == S_ >> 11) {}
    __device__ __forceinline__ int own(int lo, int end) const {  // sub-blocks of own tokens [lo, end)
        return end > lo ? ((start + end + 31) >> 5) - ((start + lo) >> 5) : 0;
    }
    __device__ __forceinline__ int count(int top) const {
        int n = n_c;
        for (int lo = 0, end = first; lo <= top; lo = end, end += 2048) n += own(lo, min(end, top + 1));
        return n;
    }
    __device__ __forceinline__ int block_id(int j) const { return j < cached ? j : (S >> 11) + j - cached + shared; }
    __device__ __forceinline__ int edge(int top, int j) const {  // the first sub-block of block j
        if (j < cached) return 64 * j;
        int n = n_c;
        for (int i = cached - shared, lo = 0, end = first; i < j && lo <= top; ++i, lo = end, end += 2048) n += own(lo, min(end, top + 1));
        return n;
    }
};

// One sub-block of a span: cache position p0, the positions [lo, hi) of it that belong to the span, whether they are
// the chunk's own (then token t sees those up to start + t), and its block of the reference.
struct PrefillSub {
    int p0, lo, hi, own, block;
};

__device__ __forceinline__ PrefillSub prefill_sub(const PrefillSpan& sp, int top, int u) {
    if (u < sp.n_c) return {u * 32, 0, sp.start, 0, u >> 6};
    u -= sp.n_c;
    int lo = 0, end = sp.first;
    for (;; lo = end, end += 2048) {
        const int n = sp.own(lo, min(end, top + 1));
        if (u < n || end > top) break;
        u -= n;
    }
    return {(((sp.start + lo) >> 5) + u) * 32, sp.start + lo, sp.start + min(end, top + 1), 1, (sp.S + lo) >> 11};
}

// Items (ranges of sub-blocks) per tile: the count up to ns_max that ends the last tile first when every CU takes items of
// 1 / count of the longest tile, each with a fixed cost of about six sub-blocks (queries, first loads, output).
__device__ __forceinline__ int prefill_ranges(const PrefillAttnArgs& a, const PrefillSpan& sp) {
    const int tiles = (a.Hq / a.Hkv * ((a.L + PF_ROWS - 1) / PF_ROWS) + 3) / 4 * a.Hkv, longest = sp.count(a.L - 1);
    int ns = 1, best = 0x7fffffff;
    for (int c = 1; c <= a.ns_max && (c == 1 || longest >= 4 * c); ++c) {
        const int cost = ((tiles * c + a.cus - 1) / a.cus) * ((longest + c - 1) / c + 6);
        if (cost < best) best = cost, ns = c;
    }
    return ns;
}

__device__ __forceinline__ int prefill_cut(int n, int z, int ns) { return z * n / ns; }  // where item z of n sub-blocks starts

__device__ __forceinline__ int prefill_top(const PrefillAttnArgs& a, int quad) {  // the last token of the quad's tiles
    const int G = a.Hq / a.Hkv, ntt = (a.L + PF_ROWS - 1) / PF_ROWS;
    return min((min(quad * 4 + 3, G * ntt - 1) / G) * PF_ROWS + PF_ROWS - 1, a.L - 1);
}

// The item of this workgroup: tile (KV head, four wave tiles), its range z of sub-blocks, [u0, u1). Workgroups start in id
// order and go to the XCDs in turn: ranges outermost, so that an XCD's workgroups stream the same part of one KV head
// (8 / Hkv XCDs per head) through its L2; the tiles with the latest tokens, the longest, first.
struct PrefillItem {
    int kvh, quad, top, u0, u1, z;
};

__device__ __forceinline__ bool prefill_item(const PrefillAttnArgs& a, const PrefillSpan& sp, int id, PrefillItem& it) {
    const int nq = (a.Hq / a.Hkv * ((a.L + PF_ROWS - 1) / PF_ROWS) + 3) / 4, ns = prefill_ranges(a, sp);
    int j;
    if (a.Hkv <= 8 && 8 % a.Hkv == 0) {
        const int per = 8 / a.Hkv, x = id & 7;
        it.kvh = x / per;
        j = (id >> 3) * per + x % per;
    } else {
        it.kvh = id % a.Hkv;
        j = id / a.Hkv;
    }
    if (j >= nq * ns) return false;
    it.z = j / nq;
    it.quad = nq - 1 - j % nq;
    it.top = prefill_top(a, it.quad);
    const int n = sp.count(it.top);
    it.u0 = prefill_cut(n, it.z, ns);
    it.u1 = prefill_cut(n, it.z + 1, ns);
    return true;
}

// Where a quad's sums go. A block that one item has all of: slot j (the block) of nblk, 4 waves x 64 tokens x 256 dims in
// bf16, rounded as the reference rounds each block's weights x V. A block that cuts divide: the parts' float32 sums, in two
// slots per cut between items: 2 (z - 1) + 1 for what item z begins with, 2 z for what it ends with (a part that begins
// and ends an item counts as its beginning). Beside each slot a float per token, its weight sum.
struct PrefillSlots {
    bf16_t* blocks;
    float *parts, *rows;  // [nblk + 2 (ns_max - 1)][4 waves][64 tokens]
    int nblk;
    __device__ __forceinline__ PrefillSlots(const PrefillAttnArgs& a, int kvh, int quad) : nblk(a.nblk) {
        const int nq = (a.Hq / a.Hkv * ((a.L + PF_ROWS - 1) / PF_ROWS) + 3) / 4, np = 2 * (a.ns_max - 1);
        const size_t q = (size_t)(kvh * nq + quad), one = 4 * PF_ROWS * 256;
        blocks = a.part + q * (a.nblk + 2 * np) * one;
        parts = (float*)(blocks + a.nblk * one);
        rows = a.part_rows + q * (a.nblk + np) * (4 * PF_ROWS);
    }
    // The part of a block that item z holds: `later` if a cut lies before it in the block.
    __device__ __forceinline__ static int part(int z, bool later) { return later ? 2 * z - 1 : 2 * z; }
};

__device__ __forceinline__ float order_float(int i) { return __int_as_float(i >= 0 ? i : i ^ 0x7fffffff); }

__device__ __forceinline__ v8bf16 lds_frag(uint32_t at) {
    return *(const __attribute__((address_space(3))) v8bf16*)(uintptr_t)at;
}

// A sub-block in LDS and how the MFMAs read it.
// K: row r holds cache position p0 + pi(r), pi swapping bits 2 and 3: with the keys as A and the queries as B, lane l
//    (token l % 32, half h = l / 32) then holds the scores of positions 16 (i / 8) + 8 h + i % 8, the eight consecutive
//    positions that MFMA step i / 8 of weights x V takes from a lane, so scores become operands without moving. Row r's
//    16-byte chunk c sits at c ^ (r % 16), which spreads a read of 32 rows over the banks.
// V: row d (dim) of 32 positions, its 16-byte chunk c at c ^ f(d), f(d) = (d / 2) % 4 ^ (d / 8) % 2.
struct SubCopy {
    const uint8_t *kg, *vg;
    uint32_t lane_k, lane_v, lds0;
    int wv;
    __device__ __forceinline__ void init(const bf16_t* k, const bf16_t* v, size_t head, int S, int lane, int wv_, uint32_t lds) {
        kg = (const uint8_t*)(k + head * S * 256);
        vg = (const uint8_t*)(v + head * S * 256);
        wv = wv_;
        lds0 = lds;
        lane_k = (lane >> 5) * 512 + (((lane & 31) ^ (2 * wv + (lane >> 5))) << 4);
        const int d = lane >> 2;
        lane_v = d * 64 + (((lane & 3) ^ (((d >> 1) & 3) ^ ((d >> 3) & 1))) << 4);
    }
    __device__ __forceinline__ void keys(int p0, uint32_t at) const {
        const uint8_t* src = kg + (size_t)p0 * 512;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 8 * j + 2 * wv, q = (r & ~12) | (r & 4) << 1 | (r & 8) >> 1;  // pi(r)
            lds_quad(src + q * 512, j & 1 ? lane_k ^ 128 : lane_k, at + r * 512);
        }
    }
    __device__ __forceinline__ void values(int p0, uint32_t at) const {
        const uint8_t* src = vg + (size_t)(p0 >> 5) * PF_SUB;
#pragma unroll
        for (int j = 0; j < 4; ++j) lds_quad(src + (j * 4 + wv) * 1024, lane_v, at + (j * 4 + wv) * 1024);
    }
};

// The wave's tile: query head and first token, and its queries in registers (zero past the chunk).
struct PrefillTile {
    int hq, t0;
    bool live;
};

__device__ __forceinline__ PrefillTile prefill_tile(const PrefillAttnArgs& a, int kvh, int id) {
    const int G = a.Hq / a.Hkv, t0 = (id / G) * PF_ROWS;
    return {kvh * G + id % G, t0, t0 < a.L};
}

__device__ __forceinline__ void prefill_queries(const PrefillAttnArgs& a, const PrefillTile& tl, int lane, v8bf16 (&qf)[2][16]) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const int t = min(tl.t0 + rt * 32, a.L - 32);  // past the chunk (L is a multiple of 32): its last tokens, never used
        const bf16_t* qp = a.qs + ((size_t)tl.hq * a.L + t + (lane & 31)) * QP + (lane >> 5) * 128;
#pragma unroll
        for (int m = 0; m < 16; ++m) qf[rt][m] = load8p(qp + m * 8);
    }
}

// Scores of the sub-block whose keys are at LDS address kl (this lane's row), operands read four MFMA pairs ahead. The
// fences hold that order: left alone, the compiler gathers all sixteen reads first, and spills.
__device__ __forceinline__ void prefill_scores(uint32_t kl, const v8bf16 (&qf)[2][16], v16f (&s)[2]) {
    v16f zero;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero[i] = 0.0f;
    v8bf16 kf[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) kf[m] = lds_frag(kl ^ (m << 4));
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        __builtin_amdgcn_sched_barrier(0);
        s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[m & 3], qf[0][m], m ? s[0] : zero, 0, 0, 0);
        s[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[m & 3], qf[1][m], m ? s[1] : zero, 0, 0, 0);
        if (m < 12) kf[m & 3] = lds_frag(kl ^ ((m + 4) << 4));
    }
    __builtin_amdgcn_sched_barrier(0);
}

// Scores of positions a lane's token does not see become -inf (weight zero): those outside [lo, hi), and of the
// chunk's own those after the token. Only sub-blocks at an edge need it.
__device__ __forceinline__ bool prefill_whole(const PrefillSub& sb, const PrefillTile& tl, int start) {
    return sb.p0 >= sb.lo && sb.p0 + 32 <= sb.hi && (!sb.own || sb.p0 + 31 <= start + tl.t0);
}
__device__ __forceinline__ void prefill_mask(const PrefillSub& sb, const PrefillTile& tl, int start, int lane, v16f (&s)[2]) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const int t = tl.t0 + rt * 32 + (lane & 31), h8 = (lane >> 5) * 8;
        const int hi = sb.own ? min(sb.hi, start + t + 1) : sb.hi;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int p = sb.p0 + 16 * (i >> 3) + h8 + (i & 7);
            if (p < sb.lo || p >= hi) s[rt][i] = -INFINITY;
        }
    }
}

}  // namespace

// Largest score of each token over each block of the reference, into mx [Hq][blocks][L] (ordered ints, reset by the
// prep kernel) by integer maxima, which do not depend on the order.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_prefill_max_kernel(const PrefillAttnArgs a) {
    __shared__ __attribute__((aligned(1024))) uint8_t ring[4][PF_SUB];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slot = *a.slot, start = *a.start;
    if (start < 0 || start + a.L > a.S || slot < 0 || slot >= a.rows) return;  // the host checks these too
    const PrefillSpan sp(a.S, start);
    PrefillItem it;
    if (!prefill_item(a, sp, blockIdx.x, it)) return;
    const int n = it.u1 - it.u0;
    if (n <= 0) return;
    const PrefillTile tl = prefill_tile(a, it.kvh, it.quad * 4 + wv);
    const uint32_t lds0 = (uint32_t)(uintptr_t)LDS_PTR(&ring[0][0]);
    SubCopy cp;
    cp.init(a.kw, a.vw, (size_t)(a.kw_slot ? slot : 0) * a.Hkv + it.kvh, a.S, lane, wv, lds0);
    v8bf16 qf[2][16];
    prefill_queries(a, tl, lane, qf);
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (i < n) cp.keys(prefill_sub(sp, it.top, it.u0 + i).p0, lds0 + i * PF_SUB);
    const uint32_t kl = (lane & 31) * 512 + (lane >> 5) * 256 + ((lane & 15) << 4);
    float mx[2] = {-INFINITY, -INFINITY};
    auto flush = [&](int block) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            // The largest bf16 score is the largest score in bf16.
            const float m = rbf(fmaxf(mx[rt], __shfl_xor(mx[rt], 32)));
            const int t = tl.t0 + rt * 32 + (lane & 31);
            if (lane < 32 && tl.live && t < a.L && m > -INFINITY) atomicMax(a.mx + ((size_t)tl.hq * a.nblk + block) * a.L + t, order_bits(m));
            mx[rt] = -INFINITY;
        }
    };
    PrefillSub sb = prefill_sub(sp, it.top, it.u0);
    for (int i = 0; i < n; ++i) {
        if (i + 2 < n)
            ring_ready<8>();
        else
            ring_ready<0>();
        if (i + 3 < n) cp.keys(prefill_sub(sp, it.top, it.u0 + i + 3).p0, lds0 + ((i + 3) & 3) * PF_SUB);
        v16f s[2];
        prefill_scores(lds0 + (i & 3) * PF_SUB + kl, qf, s);
        if (!prefill_whole(sb, tl, start)) prefill_mask(sb, tl, start, lane, s);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int e = 0; e < 16; ++e) mx[rt] = fmaxf(mx[rt], s[rt][e]);
        const int block = sb.block;
        if (i + 1 < n) sb = prefill_sub(sp, it.top, it.u0 + i + 1);
        if (i + 1 == n || sb.block != block) flush(block);
    }
}

// Weights x V of one item: per sub-block the scores again, the weights e^(s - m) with m the running maximum through the
// sub-block's block, their float32 sums, and the bf16 weights times V; at a block's end the block's sums go to its
// slot, a whole block's rounded to bf16. V as A and the weights as B, so that a lane holds four consecutive dims of one token
// (the order the activation tiles and the float4 partials want) and its row factors are its own. Sub-block i's
// weights x V run beside sub-block i + 1's scores, whose weights are formed beside them (the loop body has no branch
// but the edges), with the copies two sub-blocks ahead.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void attn_prefill_kernel(const PrefillAttnArgs a) {
    __shared__ __attribute__((aligned(1024))) uint8_t ring[4][2][PF_SUB];  // [stage][K, V]
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slot = *a.slot, start = *a.start;
    if (start < 0 || start + a.L > a.S || slot < 0 || slot >= a.rows) return;
    const PrefillSpan sp(a.S, start);
    PrefillItem it;
    if (!prefill_item(a, sp, blockIdx.x, it)) return;
    const int n = it.u1 - it.u0;
    if (n <= 0) return;
    const PrefillTile tl = prefill_tile(a, it.kvh, it.quad * 4 + wv);
    const uint32_t lds0 = (uint32_t)(uintptr_t)LDS_PTR(&ring[0][0][0]);
    SubCopy cp;
    cp.init(a.kw, a.vw, (size_t)(a.kw_slot ? slot : 0) * a.Hkv + it.kvh, a.S, lane, wv, lds0);
    v8bf16 qf[2][16];
    prefill_queries(a, tl, lane, qf);
    auto copy = [&](int i) {
        const int p0 = prefill_sub(sp, it.top, it.u0 + i).p0;
        const uint32_t at = lds0 + (i & 3) * 2 * PF_SUB;
        cp.keys(p0, at);
        cp.values(p0, at + PF_SUB);
    };
    for (int i = 0; i < min(n, 2); ++i) copy(i);
    const uint32_t kl = (lane & 31) * 512 + (lane >> 5) * 256 + ((lane & 15) << 4);
    const int fd = ((lane >> 1) & 3) ^ ((lane >> 3) & 1);
    const uint32_t vl = PF_SUB + (lane & 31) * 64 + (((lane >> 5) ^ fd) << 4);

    float nb[2] = {2.0f * -1e4f, 2.0f * -1e4f}, total[2] = {0.0f, 0.0f};
    int known = -1;  // blocks whose maxima nb holds
    auto raise = [&](int block) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const int* mp = a.mx + (size_t)tl.hq * a.nblk * a.L + min(tl.t0 + rt * 32, a.L - 32) + (lane & 31);
            if (tl.live)
                for (int b = known + 1; b <= block; ++b) nb[rt] = fmaxf(nb[rt], order_float(mp[(size_t)b * a.L]));
        }
        known = block;
    };
    v16f o[2][8];  // o[rt][db][e]: token 32 rt + l % 32, dim 32 db + 8 (e / 4) + 4 (l / 32) + e % 4
    v16f s[2];
    // Two of the sub-block's weights (x: token tile x / 8, MFMA step x / 4 % 2, word x % 4) into w.
    typedef uint32_t u4_ __attribute__((ext_vector_type(4)));
    auto weight2 = [&](int x, u4_ (&w)[2][2]) __attribute__((always_inline)) {
        const int rt = x >> 3, e = 2 * (x & 7);
        const uint32_t r = pk_bf16(s[rt][e], s[rt][e + 1]);
        const float e0 = exp_neg(lo_bf(r) - nb[rt]);
        const float e1 = exp_neg(hi_bf(r) - nb[rt]);
        total[rt] += e0;
        total[rt] += e1;
        w[rt][(x >> 2) & 1][x & 3] = pk_bf16(e0, e1);
    };
    u4_ pw[2][2];  // [token tile][MFMA step]: the sub-block's bf16 weights
    // Weights x V of sub-block i (MFMA step x: dims 32 (x / 2), positions 16 (x % 2) + [0, 16)), with the next
    // sub-block's weights formed beside the MFMAs.
    auto values = [&](int i, auto next) __attribute__((always_inline)) {
        const uint32_t va = lds0 + (i & 3) * 2 * PF_SUB + vl;
        auto frag = [&](int x) __attribute__((always_inline)) { return lds_frag((va ^ ((x & 1) << 5)) + (x >> 1) * 2048); };
        v8bf16 vf[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) vf[x] = frag(x);
        u4_ nw[2][2];
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
                o[rt][x >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[x & 3], __builtin_bit_cast(v8bf16, pw[rt][x & 1]),
                                                                       o[rt][x >> 1], 0, 0, 0);
            if (x < 12) vf[x & 3] = frag(x + 4);
            if constexpr (decltype(next)::value) weight2(x, nw);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(next)::value) {
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) pw[rt][ks] = nw[rt][ks];
        }
    };
    // Sub-block i landed (and every wave past sub-block i - 2's operands), sub-block i + 2's copies issued, i's scores.
    auto scores = [&](int i) __attribute__((always_inline)) {
        if (i + 1 < n)
            ring_ready<8>();
        else
            ring_ready<0>();
        if (i + 2 < n) copy(i + 2);
        prefill_scores(lds0 + (i & 3) * 2 * PF_SUB + kl, qf, s);
        asm volatile("" : "+v"(s[0]), "+v"(s[1]));  // in VGPRs, where the weights are formed; the AGPRs hold o
        const PrefillSub sb = prefill_sub(sp, it.top, it.u0 + i);
        if (!prefill_whole(sb, tl, start)) prefill_mask(sb, tl, start, lane, s);
    };
    // The sums of block j, or of a part of it, [wave][rt][db][e / 4][lane] of 4 dims, and per token its weight sum.
    const PrefillSlots slots(a, it.kvh, it.quad);
    auto store = [&](int j, bool whole, bool later) __attribute__((always_inline)) {
        const int part = PrefillSlots::part(it.z, later);
        const size_t at = (size_t)(whole ? j : part) * (4 * PF_ROWS * 256) + (size_t)wv * (PF_ROWS * 256) + lane * 4;
        if (whole) {
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int db = 0; db < 8; ++db)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *(uint2*)(slots.blocks + at + ((rt * 8 + db) * 4 + q) * 256) =
                            make_uint2(pk_bf16(o[rt][db][4 * q], o[rt][db][4 * q + 1]), pk_bf16(o[rt][db][4 * q + 2], o[rt][db][4 * q + 3]));
        } else {
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int db = 0; db < 8; ++db)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *(v4f*)(slots.parts + at + ((rt * 8 + db) * 4 + q) * 256) =
                            (v4f){o[rt][db][4 * q], o[rt][db][4 * q + 1], o[rt][db][4 * q + 2], o[rt][db][4 * q + 3]};
        }
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const float sum = total[rt] + __shfl_xor(total[rt], 32);
            if (lane < 32) slots.rows[(whole ? j : slots.nblk + part) * (4 * PF_ROWS) + wv * PF_ROWS + rt * 32 + lane] = sum;
        }
    };
    int j = 0;  // the block of the item's first sub-block
    while (sp.edge(it.top, j + 1) <= it.u0) ++j;
    for (int i = 0; i < n; ++j) {  // one block at a time
        const int e0 = sp.edge(it.top, j) - it.u0, e1 = sp.edge(it.top, j + 1) - it.u0, first = i, end = min(n, e1);
        raise(sp.block_id(j));
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            total[rt] = 0.0f;
#pragma unroll
            for (int db = 0; db < 8; ++db)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[rt][db][e] = 0.0f;
        }
        scores(i);
#pragma unroll
        for (int x = 0; x < 16; ++x) weight2(x, pw);
        for (; i < end - 1; ++i) {
            scores(i + 1);
            values(i, std::true_type{});
        }
        values(i++, std::false_type{});
        if (tl.live) store(j, first == e0 && end == e1, first > e0);
    }
}

// One wave tile's blocks put together as the reference does: from block to block the sums so far are rescaled to the running
// maximum and the block's weights x V, rounded to bf16, added in float32; then out / total in bf16, times bf16
// sigmoid(gate), e5m2 tiles for o_proj. Grid (wave tiles of 64 tokens x 4): wave w of block q takes 32 tokens and 64 dims, a
// lane 4 dims of one token at a time.
__global__ __launch_bounds__(256) void attn_prefill_finish_kernel(const PrefillAttnArgs a) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int slot = *a.slot, start = *a.start;
    if (start < 0 || start + a.L > a.S || slot < 0 || slot >= a.rows) return;
    const PrefillSpan sp(a.S, start);
    const int G = a.Hq / a.Hkv, ntt = (a.L + PF_ROWS - 1) / PF_ROWS;
    const int kvh = blockIdx.y, tile = blockIdx.x >> 2, quad = tile >> 2, w = tile & 3;
    if (tile >= G * ntt) return;
    const PrefillTile tl = prefill_tile(a, kvh, tile);
    const int rt = wv & 1, db0 = ((blockIdx.x & 3) * 2 + (wv >> 1)), t = tl.t0 + rt * 32 + (lane & 31);
    if (tl.t0 + rt * 32 >= a.L) return;
    const int top = prefill_top(a, quad);
    const int n = sp.count(top), ns = prefill_ranges(a, sp);
    const PrefillSlots slots(a, kvh, quad);
    const float* rows = slots.rows + w * PF_ROWS + rt * 32 + (lane & 31);
    const size_t at = (size_t)w * (PF_ROWS * 256) + (rt * 8 + db0) * 1024 + lane * 4;
    const int* mp = a.mx + (size_t)tl.hq * a.nblk * a.L + t;
    float best = 2.0f * -1e4f, total = 0.0f;
    v4f o[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    int z = 0;  // the item that holds the block's first sub-block
    for (int j = 0, e0 = 0; e0 < n; ++j) {
        const int e1 = sp.edge(top, j + 1);
        const float m = fmaxf(best, order_float(mp[(size_t)sp.block_id(j) * a.L])), f = exp_neg(best - m);
        best = m;
        float sum = 0.0f;
        v4f pv[4];
        while (prefill_cut(n, z + 1, ns) <= e0) ++z;
        if (prefill_cut(n, z + 1, ns) >= e1) {
            sum = rows[j * (4 * PF_ROWS)];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint2 v = *(const uint2*)(slots.blocks + (size_t)j * (4 * PF_ROWS * 256) + at + q * 256);
                pv[q] = (v4f){lo_bf(v.x), hi_bf(v.x), lo_bf(v.y), hi_bf(v.y)};
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) pv[q] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
            for (int y = z, u0 = prefill_cut(n, z, ns); u0 < e1; ++y) {
                const int u1 = prefill_cut(n, y + 1, ns), part = PrefillSlots::part(y, u0 > e0);
                if (u1 > u0) {  // else the item is empty
                    sum += rows[(slots.nblk + part) * (4 * PF_ROWS)];
#pragma unroll
                    for (int q = 0; q < 4; ++q) pv[q] += *(const v4f*)(slots.parts + (size_t)part * (4 * PF_ROWS * 256) + at + q * 256);
                }
                u0 = u1;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) pv[q][e] = rbf(pv[q][e]);
        }
        total = total * f + sum;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[q][e] = o[q][e] * f + pv[q][e];
        e0 = e1;
    }
    const int act_k = a.Hq * 256;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int d = db0 * 32 + q * 8 + (lane >> 5) * 4;
        const uint2 g = *(const uint2*)(a.qkv + (size_t)t * a.ld + (size_t)tl.hq * 512 + 256 + d);
        const float gt[4] = {lo_bf(g.x), hi_bf(g.x), lo_bf(g.y), hi_bf(g.y)};
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = rbf(o[q][e] / total);
            r[e] = rbf(v * rbf(sigmoidf_(gt[e])));
        }
        *(uint32_t*)(a.act + act_offset(t, tl.hq * 256 + d, act_k)) = pk_e5m2(r[0], r[1], r[2], r[3]);
    }
}

// An FP8 cache's row `slot` as bf16(e4m3 x scale), positions up to the chunk's end: the operands attn_prefill_max and
// attn_prefill read, widened once instead of by every tile. Grid (32 positions, KV head).
__global__ __launch_bounds__(256) void attn_prefill_widen_kernel(const PrefillAttnArgs a) {
    const int slot = *a.slot, start = *a.start, p0 = blockIdx.x * 32;
    if (start < 0 || start + a.L > a.S || slot < 0 || slot >= a.rows || p0 >= start + a.L) return;
    const size_t src = ((size_t)slot * a.Hkv + blockIdx.y) * a.S * 256 + (size_t)p0 * 256;
    const size_t dst = (size_t)blockIdx.y * a.S * 256 + (size_t)p0 * 256;
    const float ksc = bf2f(*a.k_scale), vsc = bf2f(*a.v_scale);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const size_t e = (size_t)(i * 256 + threadIdx.x) * 8;
        const uint2 k = *(const uint2*)((const uint8_t*)a.k_cache + src + e), v = *(const uint2*)((const uint8_t*)a.v_cache + src + e);
        *(v8bf16*)(a.k_wide + dst + e) = kv_widen8(k.x, k.y, ksc);
        *(v8bf16*)(a.v_wide + dst + e) = kv_widen8(v.x, v.y, vsc);
    }
}

hipError_t q38_attn_prefill(const PrefillAttnArgs& a0, hipStream_t stream) {
    PrefillAttnArgs a = a0;
    a.nblk = prefill_blocks(a.L, a.S);
    if (a.L < 1 || a.L % 32 || a.Hq % a.Hkv || a.S % 32) return hipErrorInvalidValue;
    if (a.kv8 && (!a.k_scale || !a.v_scale)) return hipErrorInvalidValue;
    if (a.kv8)
        hipLaunchKernelGGL(attn_prefill_prep_kernel<true>, dim3(a.L), dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL(attn_prefill_prep_kernel<false>, dim3(a.L), dim3(256), 0, stream, a);
    if (a.keys_only) return hipGetLastError();
    const int tiles = (a.Hq / a.Hkv) * ((a.L + PF_ROWS - 1) / PF_ROWS), quads = (tiles + 3) / 4 * a.Hkv;
    a.ns_max = prefill_ranges_max(quads);
    a.cus = q38_device_cus();
    if ((size_t)quads * (a.nblk + 4 * (a.ns_max - 1)) > a.part_slots) return hipErrorInvalidValue;
    a.kw = a.k_cache;
    a.vw = a.v_cache;
    a.kw_slot = 1;
    if (a.kv8) {
        hipLaunchKernelGGL(attn_prefill_widen_kernel, dim3(a.S / 32, a.Hkv), dim3(256), 0, stream, a);
        a.kw = a.k_wide;
        a.vw = a.v_wide;
        a.kw_slot = 0;
    }
    // Every item has an id: with 8 / Hkv XCDs per KV head the ids come in rounds of eight, one item per XCD.
    const int per_head = (tiles + 3) / 4 * a.ns_max;
    const int grid = a.Hkv <= 8 && 8 % a.Hkv == 0 ? (per_head + 8 / a.Hkv - 1) / (8 / a.Hkv) * 8 : per_head * a.Hkv;
    hipLaunchKernelGGL(attn_prefill_max_kernel, dim3(grid), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(attn_prefill_kernel, dim3(grid), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(attn_prefill_finish_kernel, dim3(tiles * 4, a.Hkv), dim3(256), 0, stream, a);
    return hipGetLastError();
}

hipError_t q38_gdn_prefill(const PrefillGdnArgs& a, hipStream_t stream) {
    if (a.L < 1 || a.gate_groups < 1 || a.gate_groups > 8 || a.Hv % a.Hk || a.Hv % 4 || a.C != 2 * a.Hk * 128 + a.Hv * 128)
        return hipErrorInvalidValue;
    if (a.L % GC || a.Hv % 4) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gdn_prefill_prep_kernel, dim3(a.L / GC, a.Hk), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(gdn_prefill_scan_kernel, dim3(a.Hv, 4), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(gdn_prefill_finish_kernel, dim3(a.L / 4, a.Hv / 4), dim3(256), 0, stream, a);
    hipLaunchKernelGGL(gdn_prefill_carry_kernel, dim3((a.C + 255) / 256), dim3(256), 0, stream, a);
    return hipGetLastError();
}
