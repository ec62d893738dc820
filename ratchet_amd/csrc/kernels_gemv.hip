// Streaming GEMV kernels for gfx950: y[i, j] = sum_k A[i, k] * x[j, k] (+ bias)
// for a tall weight operand A (rows of K, K contiguous) and a handful of
// activation vectors x[j] (j < 8).  The weight stream is read once, straight
// from HBM into registers with 128-bit loads and dequantized in registers;
// there is no LDS staging of weights.  One wavefront owns one row at a time
// and its 64 lanes stride the row in 16-byte chunks, so every load
// instruction of a wavefront covers 1 KiB of contiguous weights; Q8_0F
// weights have a workgroup per four rows (gemv_q8f_kernel).
//
// Roles in the reference: ops/gemv.rs:156-574 (the workgroup and subgroup
// GEMV generators) and, for 2..8 activation rows, the scalar QGEMM of
// ops/gemm.rs:342-492 which the reference uses for those shapes.
#include "device_common.h"

#include <algorithm>

namespace rt {

struct GemvArgs {
    const uint8_t *A;   // weight bytes (int8 stream / Q4_K blocks / f16 / f32)
    const void *scales; // Q8_0 scale stream
    const void *X;
    const void *bias;
    void *out;
    int64_t M, K;
    int64_t a_stack, b_stack;
    int64_t a_bs, a_rs; // stack and row stride of A in elements (float kernels)
    int64_t b_bs, b_js;
    int64_t o_bs, o_is, o_js;
    int has_bias, bias_on_rows, act;
    int64_t row_first; // gemv_q8f_kernel: this launch's first weight row
};

constexpr int kGemvThreads = 256;
constexpr int kGemvWaves = kGemvThreads / kWave;

template <typename AT, int NC>
__device__ __forceinline__ void gemv_store(const GemvArgs &g, int64_t s, int64_t row, int lane, const float *acc) {
    // lane j (< NC) writes column j.  acc[] is wave-uniform after the reduction.
    const AT *bias = (const AT *)g.bias;
    AT *out = (AT *)g.out;
#pragma unroll
    for (int j = 0; j < NC; j++) {
        if (lane == j) {
            float v = acc[j];
            if (g.has_bias) v += to_f32(bias[g.bias_on_rows ? row : (int64_t)j]);
            out[s * g.o_bs + row * g.o_is + j * g.o_js] = from_f32<AT>(rt_act(v, g.act));
        }
    }
}

// Loads 16 consecutive activations starting at x[k0] as floats.
__device__ __forceinline__ void load_x16(const half_t *x, float (&xf)[16]) {
    half8_t a = *(const half8_t *)x, b = *(const half8_t *)(x + 8);
#pragma unroll
    for (int i = 0; i < 8; i++) xf[i] = (float)a[i], xf[8 + i] = (float)b[i];
}
// ---------------------------------------------------------------------------
// Q8_0H weights x f16 activations (what the matrix-core kernels decline).  Chunk = 16 int8 (half a block) + the block's scale.
// ---------------------------------------------------------------------------
template <int NC, int U>
__global__ __launch_bounds__(kGemvThreads) void gemv_q8_kernel(GemvArgs g) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    const int64_t s = blockIdx.y;
    // an operand's stack is either the full stack or 1 (broadcast)
    const int64_t sa = g.a_stack == 1 ? 0 : s, sb = g.b_stack == 1 ? 0 : s;
    const int nchunks = (int)(g.K >> 4);
    const half_t *x = (const half_t *)g.X + sb * g.b_bs;
    for (int64_t row = (int64_t)blockIdx.x * kGemvWaves + wave; row < g.M; row += (int64_t)gridDim.x * kGemvWaves) {
        const int64_t rowel = (sa * g.M + row) * g.K;
        const uint8_t *q = g.A + rowel;
        const half_t *sc = (const half_t *)g.scales + (rowel >> 5);
        float acc[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) acc[j] = 0.f;
        for (int c0 = 0; c0 < nchunks; c0 += kWave * U) {
            uint4_t w[U];
            float d[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = c0 + u * kWave + lane;
                const bool ok = c < nchunks;
                w[u] = ok ? *(const uint4_t *)(q + 16 * (int64_t)c) : uint4_t{0, 0, 0, 0};
                d[u] = ok ? to_f32(sc[c >> 1]) : 0.f;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = c0 + u * kWave + lane;
                if (c < nchunks) {
                    float wf[16];
#pragma unroll
                    for (int i = 0; i < 16; i++) wf[i] = (float)(int8_t)(w[u][i >> 2] >> (8 * (i & 3)));
#pragma unroll
                    for (int j = 0; j < NC; j++) {
                        float xf[16];
                        load_x16(x + j * g.b_js + 16 * (int64_t)c, xf);
                        float part = 0.f;
#pragma unroll
                        for (int i = 0; i < 16; i++) part += wf[i] * xf[i];
                        acc[j] += d[u] * part;
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NC; j++) acc[j] = wave_sum(acc[j]);
        gemv_store<half_t, NC>(g, s, row, lane, acc);
    }
}

// ---------------------------------------------------------------------------
// Q8_0F weights x f32 activations.  A workgroup of four wavefronts takes four weight rows, wavefront w every fourth step of 256 k from the w-th
// on; a lane takes four codes of each row and the four activations of each vector beside them, so that both come in runs of consecutive bytes (with
// sixteen codes to a lane, its 64 bytes of activations are a line of their own in each of four loads, and every row asks
// for them again), and an activation is read once for four rows.  A block's scale is applied to the sum of four products.
// us at 1 / 2 / 4 / 8 vectors, with a row per wavefront and sixteen codes to a lane, and here: 10240 x 2560 10.6 / 17.0 / 31 / 62 and 7.1 / 9.0 / 12.1 / 17.8;
// 2560 x 10240 10.5 / 17.6 / 32 / 57 and 9.5 / 10.3 / 13.1 / 19.1; 5536 x 2080 6.8 / 11.0 / 18.0 / 33 and 5.2 / 5.9 / 7.9 / 10.4.  Bound by the weight's bytes (4.2 TB/s at one
// vector), then by the vector instructions: 84 for a lane's four codes of four rows against eight vectors, and by the loads of the activations.
// ---------------------------------------------------------------------------
constexpr int kQ8fRows = 4;
constexpr int kQ8fLongK = 1024; // from here on the sums are no less exact than the limb kernel's (gemv_q8f_chunks)
typedef float float4_u __attribute__((ext_vector_type(4), aligned(4))); // activations start at any f32: the loads take them as they are
template <int NC, int U>
__global__ __launch_bounds__(kGemvThreads) void gemv_q8f_kernel(GemvArgs g) {
    constexpr int R = kQ8fRows;
    __shared__ float red[kGemvWaves][R][NC];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int64_t s = blockIdx.y, sa = g.a_stack == 1 ? 0 : s, sb = g.b_stack == 1 ? 0 : s; // an operand's stack is either the full stack or 1 (broadcast)
    const float *x = (const float *)g.X + sb * g.b_bs;
    const int64_t row0 = g.row_first + (int64_t)blockIdx.x * R;
    const uint8_t *q[R];
    const float *sc[R];
#pragma unroll
    for (int r = 0; r < R; r++) { // rows past the end repeat the last one; never stored
        const int64_t el = (sa * g.M + min(row0 + r, g.M - 1)) * g.K;
        q[r] = g.A + el, sc[r] = (const float *)g.scales + (el >> 5);
    }
    float acc[R][NC];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int j = 0; j < NC; j++) acc[r][j] = 0.f;
    const int K = (int)g.K, last = K - 4;
    for (int k0 = 256 * wave; k0 < K; k0 += 256 * kGemvWaves * U) {
        uint32_t w[U][R];
        float d[U][R];
#pragma unroll
        for (int u = 0; u < U; u++) { // past the end: the row's last codes, left out below
            const uint32_t k = (uint32_t)min(k0 + 256 * kGemvWaves * u + 4 * lane, last);
#pragma unroll
            for (int r = 0; r < R; r++) w[u][r] = __builtin_nontemporal_load((const uint32_t *)(q[r] + k)), d[u][r] = sc[r][k >> 5];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = k0 + 256 * kGemvWaves * u + 4 * lane;
            if (k < K) {
                float wf[R][4];
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int e = 0; e < 4; e++) wf[r][e] = (float)(int8_t)(w[u][r] >> (8 * e));
#pragma unroll
                for (int j = 0; j < NC; j++) {
                    const float4_t xv = *(const float4_u *)(x + j * g.b_js + k);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        float p = wf[r][0] * xv[0];
#pragma unroll
                        for (int e = 1; e < 4; e++) p = fmaf(wf[r][e], xv[e], p);
                        acc[r][j] = fmaf(d[u][r], p, acc[r][j]);
                    }
                }
            }
        }
    }
    // the lanes' sums: halves and quarters of the wavefront swap, so that a quarter is left with one row, whose sixteen lanes then add up
    float v[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) {
        auto add = [](auto p) { return __builtin_bit_cast(float, (uint32_t)p[0]) + __builtin_bit_cast(float, (uint32_t)p[1]); };
        const float a = add(__builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, acc[0][j]), __builtin_bit_cast(uint32_t, acc[2][j]), false, false)); // rows 0 and 2
        const float b = add(__builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, acc[1][j]), __builtin_bit_cast(uint32_t, acc[3][j]), false, false)); // 1 and 3
        v[j] = add(__builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false));                          // quarter l / 16: row l / 16
        v[j] += wave_dpp<0x128>(v[j]); // row_ror:8, 4, 2, 1
        v[j] += wave_dpp<0x124>(v[j]);
        v[j] += wave_dpp<0x122>(v[j]);
        v[j] += wave_dpp<0x121>(v[j]);
        if ((lane & 15) == j) red[wave][lane >> 4][j] = v[j];
    }
    __syncthreads();
    if (t < R * NC) {
        const int r = t / NC, j = t - r * NC;
        if (row0 + r < g.M) {
            float o = (red[0][r][j] + red[1][r][j]) + (red[2][r][j] + red[3][r][j]);
            if (g.has_bias) o += ((const float *)g.bias)[g.bias_on_rows ? row0 + r : (int64_t)j];
            ((float *)g.out)[s * g.o_bs + (row0 + r) * g.o_is + j * g.o_js] = rt_act(o, g.act);
        }
    }
}

// ---------------------------------------------------------------------------
// Q4_K weights.  A lane takes 16 bytes of a super-block's qs: 16 low nibbles
// (sub-block 2c) and 16 high nibbles (sub-block 2c+1), plus the 16-byte header
// {d, dmin, scales[12]} of that super-block.
// ---------------------------------------------------------------------------
template <int NC>
__global__ __launch_bounds__(kGemvThreads) void gemv_q4k_kernel(GemvArgs g) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    const int64_t s = blockIdx.y;
    // an operand's stack is either the full stack or 1 (broadcast)
    const int64_t sa = g.a_stack == 1 ? 0 : s, sb = g.b_stack == 1 ? 0 : s;
    const int nsb = (int)(g.K >> 8);  // super-blocks per row
    const int npieces = nsb * 8;      // 16-byte qs pieces per row
    const half_t *x = (const half_t *)g.X + sb * g.b_bs;
    for (int64_t row = (int64_t)blockIdx.x * kGemvWaves + wave; row < g.M; row += (int64_t)gridDim.x * kGemvWaves) {
        const uint8_t *blk0 = g.A + ((sa * g.M + row) * nsb) * 144;
        float acc[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) acc[j] = 0.f;
        for (int p0 = 0; p0 < npieces; p0 += kWave) {
            const int p = p0 + lane;
            if (p < npieces) {
                const int sbi = p >> 3, piece = p & 7, c = piece >> 1, h = piece & 1;
                const uint8_t *blk = blk0 + (int64_t)sbi * 144;
                const uint4_t hdr = *(const uint4_t *)blk;
                const uint4_t qv = *(const uint4_t *)(blk + 16 + 16 * piece);
                half2_t dm = __builtin_bit_cast(half2_t, hdr[0]);
                const float d = (float)dm[0], dmin = (float)dm[1];
                uint8_t sbytes[12];
#pragma unroll
                for (int i = 0; i < 12; i++) sbytes[i] = (uint8_t)(hdr[1 + (i >> 2)] >> (8 * (i & 3)));
                int sc0, mn0, sc1, mn1;
                q4k_scale_min(2 * c, sbytes, sc0, mn0);
                q4k_scale_min(2 * c + 1, sbytes, sc1, mn1);
                const float d0 = d * (float)sc0, m0 = dmin * (float)mn0;
                const float d1 = d * (float)sc1, m1 = dmin * (float)mn1;
                const int64_t k_lo = (int64_t)sbi * 256 + 64 * c + 16 * h, k_hi = k_lo + 32;
#pragma unroll
                for (int j = 0; j < NC; j++) {
                    float xl[16], xh[16];
                    load_x16(x + j * g.b_js + k_lo, xl);
                    load_x16(x + j * g.b_js + k_hi, xh);
                    float part = 0.f;
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const uint32_t byte = (qv[i >> 2] >> (8 * (i & 3))) & 0xFFu;
                        // same evaluation as the dequantizer: w = d*sc*q - dmin*mn
                        const float wl = d0 * (float)(byte & 0xFu) - m0;
                        const float wh = d1 * (float)(byte >> 4) - m1;
                        part += wl * xl[i];
                        part += wh * xh[i];
                    }
                    acc[j] += part;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NC; j++) acc[j] = wave_sum(acc[j]);
        gemv_store<half_t, NC>(g, s, row, lane, acc);
    }
}

// ---------------------------------------------------------------------------
// f16 / f32 weights.  VEC selects 16-byte loads (aligned, K % 16 == 0 handled
// by a scalar tail) or a fully scalar walk for odd strides.
// ---------------------------------------------------------------------------
template <typename AT, int NC, bool VEC>
__global__ __launch_bounds__(kGemvThreads) void gemv_float_kernel(GemvArgs g) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    const int64_t s = blockIdx.y;
    // an operand's stack is either the full stack or 1 (broadcast)
    const int64_t sa = g.a_stack == 1 ? 0 : s, sb = g.b_stack == 1 ? 0 : s;
    const AT *x = (const AT *)g.X + sb * g.b_bs;
    const AT *Abase = (const AT *)g.A + sa * g.a_bs;
    constexpr int E = 16 / (int)sizeof(AT); // elements per 16-byte chunk
    for (int64_t row = (int64_t)blockIdx.x * kGemvWaves + wave; row < g.M; row += (int64_t)gridDim.x * kGemvWaves) {
        const AT *a = Abase + row * g.a_rs;
        float acc[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) acc[j] = 0.f;
        int64_t kdone = 0;
        if (VEC) {
            const int64_t nchunks = g.K / E;
            for (int64_t c = lane; c < nchunks; c += kWave) {
                const uint4_t raw = *(const uint4_t *)(a + c * E);
                float wf[E];
                if constexpr (sizeof(AT) == 2) {
                    half8_t hv = __builtin_bit_cast(half8_t, raw);
#pragma unroll
                    for (int i = 0; i < E; i++) wf[i] = (float)hv[i];
                } else {
                    float4_t fv = __builtin_bit_cast(float4_t, raw);
#pragma unroll
                    for (int i = 0; i < E; i++) wf[i] = fv[i];
                }
#pragma unroll
                for (int j = 0; j < NC; j++) {
                    const uint4_t xr = *(const uint4_t *)(x + j * g.b_js + c * E);
                    float part = 0.f;
                    if constexpr (sizeof(AT) == 2) {
                        half8_t hv = __builtin_bit_cast(half8_t, xr);
#pragma unroll
                        for (int i = 0; i < E; i++) part += wf[i] * (float)hv[i];
                    } else {
                        float4_t fv = __builtin_bit_cast(float4_t, xr);
#pragma unroll
                        for (int i = 0; i < E; i++) part += wf[i] * fv[i];
                    }
                    acc[j] += part;
                }
            }
            kdone = nchunks * E;
        }
        for (int64_t k = kdone + lane; k < g.K; k += kWave) {
            const float w = to_f32(a[k]);
#pragma unroll
            for (int j = 0; j < NC; j++) acc[j] += w * to_f32(x[j * g.b_js + k]);
        }
#pragma unroll
        for (int j = 0; j < NC; j++) acc[j] = wave_sum(acc[j]);
        gemv_store<AT, NC>(g, s, row, lane, acc);
    }
}

// ---------------------------------------------------------------------------
// Launch
// ---------------------------------------------------------------------------
static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

template <int NC> static void launch_q8f(dim3 grid, hipStream_t st, const GemvArgs &g) {
    hipLaunchKernelGGL((gemv_q8f_kernel<NC, (NC <= 4 ? 4 : 2)>), grid, dim3(kGemvThreads), 0, st, g);
}
template <int NC> static void launch_q8(dim3 grid, hipStream_t st, const GemvArgs &g) {
    hipLaunchKernelGGL((gemv_q8_kernel<NC, 4>), grid, dim3(kGemvThreads), 0, st, g);
}
template <int NC> static void launch_q4k(dim3 grid, hipStream_t st, const GemvArgs &g) {
    hipLaunchKernelGGL((gemv_q4k_kernel<NC>), grid, dim3(kGemvThreads), 0, st, g);
}
template <int NC> static void launch_float(int act_dt, bool vec, dim3 grid, hipStream_t st, const GemvArgs &g) {
    if (act_dt == RT_F16) {
        if (vec) hipLaunchKernelGGL((gemv_float_kernel<half_t, NC, true>), grid, dim3(kGemvThreads), 0, st, g);
        else hipLaunchKernelGGL((gemv_float_kernel<half_t, NC, false>), grid, dim3(kGemvThreads), 0, st, g);
    } else {
        if (vec) hipLaunchKernelGGL((gemv_float_kernel<float, NC, true>), grid, dim3(kGemvThreads), 0, st, g);
        else hipLaunchKernelGGL((gemv_float_kernel<float, NC, false>), grid, dim3(kGemvThreads), 0, st, g);
    }
}

#define RT_DISPATCH_NC(N, CALL)                                                                    \
    switch (N) {                                                                                   \
    case 1: { constexpr int NC = 1; CALL; } break;                                                 \
    case 2: { constexpr int NC = 2; CALL; } break;                                                 \
    case 3: { constexpr int NC = 3; CALL; } break;                                                 \
    case 4: { constexpr int NC = 4; CALL; } break;                                                 \
    case 5: { constexpr int NC = 5; CALL; } break;                                                 \
    case 6: { constexpr int NC = 6; CALL; } break;                                                 \
    case 7: { constexpr int NC = 7; CALL; } break;                                                 \
    case 8: { constexpr int NC = 8; CALL; } break;                                                 \
    default: return hipErrorInvalidValue;                                                          \
    }

// Tunable: non-zero keeps Q8_0H weights on the VALU kernel (for comparisons).
RT_TUNABLE(g_gemv_disable_mfma, 0);

// A few more activation vectors than one streaming launch takes: one launch per 16 of them.  Each
// launch streams the weights again (after the first mostly from the Infinity Cache), which still beats
// the tiled kernels while the MFMA work is small: measured at 8192 x 3072 Q4_K, 17 / 32 vectors take
// 12 / 14 us (48: 21) against 15 us tiled: the tiled kernels take over from 33.  (10240 x 2560 Q8_0H:
// 18 / 20 us, 48 / 64 vectors 29 / 38.)
hipError_t gemv_chunks(const Problem &p, const void *A, const void *B, const void *bias, void *out, hipStream_t stream, const DeviceInfo &dev) {
    const bool q8 = p.a_dt == RT_Q8_0H, q4 = p.a_dt == RT_Q4_K;
    if ((!q8 && !q4) || p.act_dt != RT_F16 || g_gemv_disable_mfma) return hipErrorNotSupported;
    if (p.N <= 16 || p.N > 32) return hipErrorNotSupported;
    for (int64_t j0 = 0; j0 < p.N; j0 += 16) {
        Problem c = p;
        c.N = p.N - j0 < 16 ? p.N - j0 : 16;
        c.kernel = q8 ? RT_KERNEL_GEMV_Q8 : RT_KERNEL_GEMV_Q4K;
        const half_t *Bc = (const half_t *)B + j0 * p.b_js;
        half_t *oc = (half_t *)out + j0 * p.o_js;
        const half_t *bc = bias && !p.bias_on_rows ? (const half_t *)bias + j0 : (const half_t *)bias;
        const hipError_t e = q8 ? launch_gemv_q8h_mfma(c, A, Bc, bc, oc, stream, dev) : launch_gemv_q4k_mfma(c, A, Bc, bc, oc, stream, dev);
        // a shape or alignment the kernel declines is declined on the first chunk (the later ones share
        // its strides and alignment); whatever a failed attempt wrote is overwritten by the kernel that runs instead
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Q8_0H weights that a kernel reads once are faster there: where their 64 x 64 tiles give half of the compute units a workgroup; and from a
// quarter on (with fewer the streaming launches stay ahead: 2560 x 2560 at 17 / 32 vectors 7.5 / 8.3 us here, 9.7 / 10.1 there) where
// launch_gemm_stream takes them (7680 x 2560 12.1 / 13.1 and 9.1 / 9.5, 5120 x 4096 13.5 / 16.4 and 10.2 / 10.6, 4096 x 1024 7.3 / 6.9 and 4.5), where the tiles
// share K (4352 x 4096 16.7 / 19.9 and 14.7 / 15.0) or where a K above 4096 makes these launches slow (4352 x 4352 22.1 / 27.3 and, K whole, 22.7
// / 22.7).  Between them they stay: 4352 x 1024 7.5 / 8.1 and 8.1 / 8.1, x 4096 without a workspace 16.7 / 19.9 and 21.4 / 21.4.  Those whose
// tiles could share K are left to launch_gemm_nt, which knows whether they do and calls gemv_chunks where not: what the families
// decline does not depend on the workspace, so that a plan, which asks first the one that ran last, runs what a call without a plan does.
static bool q8h_between(const Problem &p, const DeviceInfo &dev) {
    const int64_t tiles = (p.M + 63) / 64;
    return p.a_dt == RT_Q8_0H && p.K % 256 == 0 && p.K <= 4096 && p.stacks == 1 && tiles >= dev.num_cus / 4 && tiles < dev.num_cus / 2 && !gemm_stream_fills(p.M, dev);
}
bool gemv_chunks_unless_shared(const Problem &p, const DeviceInfo &dev) {
    return q8h_between(p, dev) && p.N > 16 && p.N <= 32 && gemm_nt_workspace_bytes(p, dev) > 0;
}
// 9 to 16 vectors against a small Q8_0F weight: two launches of the streaming kernel, each of which reads the weight at the rate of a launch of few
// bytes, where the limb kernel splits K over a workspace and merges, or without one walks all of it (us at 9 / 16 vectors, the limb kernel with a
// workspace, without, and two launches: 1001 x 4096 21.0 / 22.6, 69 and 8.9 / 11.0; 512 x 10240 21.0 / 22.1, 166 and 15.2 / 18.9; 4096 x 1280 12.9 / 13.1,
// 25 and 9.6 / 10.9; 384 x 1536 12.5, 28 and 6.8 / 7.7).  Beyond 4096 rows or five million codes that kernel fills the device and reads the codes
// once (4096 x 2560 15.4, here 12.6 / 17.1; 8192 x 640 13.5, here 11.3 / 14.7).  From K = 1024 on, since the sums are no less exact there (relative error
// against float64 at K = 800 / 1280 / 2048 / 4096 here 9.4e-8 / 9.5e-8 / 9.6e-8 / 9.9e-8, there 9.2e-8 / 9.8e-8 / 1.08e-7 / 1.29e-7).
bool gemv_q8f_chunks(const Problem &p) {
    return p.a_dt == RT_Q8_0F && p.act_dt == RT_F32 && p.N > kGemvMaxCols && p.N <= 2 * kGemvMaxCols && p.stacks == 1 && p.b_ks == 1 && p.K >= kQ8fLongK &&
           p.M <= 4096 && p.M * p.K <= 5 << 20;
}
hipError_t launch_gemv_chunked(const Problem &p, const void *A, const void *B, const void *bias, void *out, hipStream_t stream, const DeviceInfo &dev) {
    if (gemv_q8f_chunks(p)) {
        for (int64_t j0 = 0; j0 < p.N; j0 += kGemvMaxCols) {
            Problem c = p;
            c.N = std::min<int64_t>(p.N - j0, kGemvMaxCols), c.kernel = RT_KERNEL_GEMV_Q8;
            const float *bc = bias && !p.bias_on_rows ? (const float *)bias + j0 : (const float *)bias;
            // what it declines (a weight off 16 bytes) it declines on the first chunk
            if (const hipError_t e = launch_gemv(c, A, (const float *)B + j0 * p.b_js, bc, (float *)out + j0 * p.o_js, stream, dev); e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    if (p.a_dt == RT_Q8_0H && p.K % 256 == 0 && p.stacks == 1 && (p.M + 63) / 64 >= dev.num_cus / 4 &&
        (!q8h_between(p, dev) || gemv_chunks_unless_shared(p, dev)))
        return hipErrorNotSupported;
    return gemv_chunks(p, A, B, bias, out, stream, dev);
}

// Whether launch_gemv leaves 5..8 vectors against Q8_0H weights to the kernels behind it (see there); launch_gemm_nt takes those without a workspace only then
bool gemv_q8h_few_leave(const Problem &p, const DeviceInfo &dev) {
    if (p.K % 256 != 0 || gemv_q8h_mfma_well(p, dev)) return false;
    if (p.stacks == 1 && gemm_stream_fills(p.M, dev)) return true;
    return gemm_nt_q8h_few(p, dev) && p.workspace && !((uintptr_t)p.workspace & 15u) && p.workspace_bytes >= gemm_nt_workspace_bytes(p, dev);
}

// Returns hipErrorNotSupported when the operands do not meet the alignment the
// streaming kernels assume; the caller then takes the tiled GEMM, which has no
// such requirement.
hipError_t launch_gemv(const Problem &p, const void *A, const void *B, const void *bias, void *out,
                       hipStream_t stream, const DeviceInfo &dev) {
    // 5..8 vectors whose K is more than the matrix-core kernel does well or at all: one pass over the weight in launch_gemm_stream where it fills the device
    // (5120 x 10240 at 5 / 8 vectors 36 / 43 us here, 23 / 24 there), the tiles where they share K (gemm_nt_q8h_few)
    if (p.kernel == RT_KERNEL_GEMV_Q8 && p.a_dt == RT_Q8_0H && p.N >= 5 && p.b_ks == 1 && aligned16(A) && aligned16(B) && (p.b_js * 2) % 16 == 0 && (p.b_bs * 2) % 16 == 0 &&
        gemv_q8h_few_leave(p, dev))
        return hipErrorNotSupported;
    if (p.kernel == RT_KERNEL_GEMV_Q8 && p.a_dt == RT_Q8_0H && !g_gemv_disable_mfma) {
        // f16 activations, one or two vectors: the row-streaming kernel; three or four: the row-streaming kernel on
        // the 4x4x4 matrix instruction; then the matrix-core kernel; shapes all of them decline fall through
        hipError_t e = launch_gemv_q8h_rowdot(p, A, B, bias, out, stream, dev);
        if (e != hipErrorNotSupported) return e;
        e = launch_gemv_q8h_quad(p, A, B, bias, out, stream, dev);
        if (e != hipErrorNotSupported) return e;
        e = launch_gemv_q8h_mfma(p, A, B, bias, out, stream, dev);
        if (e != hipErrorNotSupported) return e;
    }
    // 5..8 vectors against Q8_0H rows that none of these take (K no multiple of 256), enough of them that 64-row tiles give half of the
    // compute units a workgroup: the tiled kernel (11392 x 352 at 5 / 8 vectors 11.3 / 17.2 us here, 6.2 / 6.0 there; 9088 x 2272
    // 15.8 / 24.6 and 15.2 / 14.6; with fewer rows 3840 x 1440 6.8 / 11.6 and 10.5)
    if (p.kernel == RT_KERNEL_GEMV_Q8 && p.a_dt == RT_Q8_0H && p.N >= 5 && p.stacks == 1 && p.K % 32 == 0 && (p.M + 63) / 64 >= dev.num_cus / 2 &&
        p.b_ks == 1 && aligned16(A) && aligned16(B) && (p.b_js * 2) % 16 == 0)
        return hipErrorNotSupported;
    if (p.kernel == RT_KERNEL_GEMV_Q4K) {
        if (p.N >= 3 && aligned16(A) && aligned16(B) && (p.b_js * 2) % 16 == 0 && (p.b_bs * 2) % 16 == 0 && gemm_q4k_few(p, dev)) return hipErrorNotSupported;
        // one vector: the row-streaming kernel; then the matrix-core kernel
        hipError_t e = launch_gemv_q4k_rowdot(p, A, B, bias, out, stream, dev);
        if (e != hipErrorNotSupported) return e;
        e = launch_gemv_q4k_mfma(p, A, B, bias, out, stream, dev);
        if (e != hipErrorNotSupported) return e;
    }
    if (p.kernel == RT_KERNEL_GEMV_FLOAT) { // up to four vectors, rows of whole 16-byte vectors: the row-streaming kernel
        hipError_t e = launch_gemv_float_rowdot(p, A, B, bias, out, stream, dev);
        if (e != hipErrorNotSupported) return e;
        // 5..8 vectors against an f16 weight with enough rows that 64-row tiles give half of the compute units a
        // workgroup: the weight-streaming GEMM, or the tiled kernel's 64 x 64 tiles (10240 x 2560, weights from HBM:
        // 12.7 / 16 us against 19 / 24 / 26 us at 5 / 7 / 8 vectors here), from 6 vectors on where K ends in half a 64 (8192 x 2016: 10.5 us
        // against 9.9 / 15.0 at 5 / 8 vectors; 16384 x 544: 6.0 against 10.7 / 15.6); the conditions are the ones under which
        // the tiled kernel takes the product.  With fewer rows, where launch_gemm_stream takes it (4096 x 2560 at 5 / 8 vectors 7.1 / 9.7 us here, 5.6
        // there, 3200 x 512 4.4 / 5.5 and 4.0 / 3.6, 5536 x 10240 26.9 / 38.4 and 20.6 / 21.4)
        if (p.a_dt == RT_F16 && p.act_dt == RT_F16 && p.N >= (p.K % 64 == 0 ? 5 : 6) && p.stacks == 1 && p.K > 256 && p.K % 32 == 0 &&
            ((p.M + 63) / 64 >= dev.num_cus / 2 || (gemm_stream_fills(p.M, dev) && p.K % 256 == 0 && p.a_rs == p.K)) && p.a_ks == 1 && p.b_ks == 1 && aligned16(A) && aligned16(B) &&
            (p.a_rs * 2) % 16 == 0 && (p.b_js * 2) % 16 == 0 && !(p.o_js == 1 && p.o_is != 1))
            // (a row-major output would make the tiled kernel exchange the operands, and with the weight as its
            // activation side it declines: such a product stays here)
            return hipErrorNotSupported;
    }
    if (p.N < 1 || p.N > kGemvMaxCols || p.stacks > 65535) return hipErrorNotSupported;
    const int64_t esz = p.act_dt == RT_F16 ? 2 : 4;
    GemvArgs g{};
    g.A = (const uint8_t *)A;
    g.X = B;
    g.bias = bias;
    g.out = out;
    g.M = p.M, g.K = p.K;
    g.a_stack = p.a_stack, g.b_stack = p.b_stack;
    g.a_bs = p.a_bs, g.a_rs = p.a_rs;
    g.b_bs = p.b_bs, g.b_js = p.N == 1 ? 0 : p.b_js; // a single vector has no column stride
    g.o_bs = p.o_bs, g.o_is = p.o_is, g.o_js = p.o_js;
    g.has_bias = p.has_bias, g.bias_on_rows = p.bias_on_rows, g.act = p.act;

    const int64_t row_blocks = (p.M + kGemvWaves - 1) / kGemvWaves;
    const int64_t cap = (int64_t)dev.num_cus * 16;
    dim3 grid((unsigned)(row_blocks < cap ? row_blocks : cap), (unsigned)p.stacks);
    // x rows must be 16-byte aligned for the vector loads.
    const bool x_ok = aligned16(B) && (g.b_js * esz) % 16 == 0 && (p.b_bs * esz) % 16 == 0;

    switch (p.kernel) {
    case RT_KERNEL_GEMV_Q8: {
        // gemv_q8f_kernel's loads take vectors at any f32: from K = 1024 on, as gemv_q8f_chunks, which asks for no workspace whatever the pointer (us, the
        // limb kernel and this: 10240 x 2560 at 1 / 8 vectors 44.6 and 7.6 / 17.9, 1001 x 4096 at 12, with a workspace there, 21.1 and 9.0)
        const bool any_f32 = p.a_dt == RT_Q8_0F && p.K >= kQ8fLongK && ((uintptr_t)B & 3u) == 0;
        if (!(x_ok || any_f32) || !aligned16(A) || p.K % 32 != 0) return hipErrorNotSupported;
        const uint64_t numel = (uint64_t)p.a_stack * p.M * p.K;
        g.scales = (const uint8_t *)A + rt_q8_0_scale_offset(numel);
        if (p.a_dt == RT_Q8_0F) {
            if (p.K > 0x7fffffff - 8192) return hipErrorNotSupported; // (its steps count in 32 bits)
            // a launch's threads along an axis are fewer than 2^32: 67 million rows and more go in several
            const int64_t groups = (p.M + kQ8fRows - 1) / kQ8fRows, most = 0xffffffffu / kGemvThreads;
            for (int64_t first = 0; first < groups; first += most) {
                grid.x = (unsigned)std::min(groups - first, most), g.row_first = first * kQ8fRows;
                RT_DISPATCH_NC(p.N, launch_q8f<NC>(grid, stream, g));
                if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
            }
            return hipSuccess;
        } else {
            RT_DISPATCH_NC(p.N, launch_q8<NC>(grid, stream, g));
        }
        break;
    }
    case RT_KERNEL_GEMV_Q4K: {
        if (!x_ok || !aligned16(A) || p.K % 256 != 0) return hipErrorNotSupported;
        RT_DISPATCH_NC(p.N, launch_q4k<NC>(grid, stream, g));
        break;
    }
    case RT_KERNEL_GEMV_FLOAT: {
        const bool vec = x_ok && aligned16(A) && (p.a_rs * esz) % 16 == 0;
        RT_DISPATCH_NC(p.N, launch_float<NC>(p.act_dt, vec, grid, stream, g));
        break;
    }
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

} // namespace rt
