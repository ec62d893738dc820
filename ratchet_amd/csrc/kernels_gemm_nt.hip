// MFMA GEMMs for the Linear / QK^T form, where both operands are K-contiguous:
//   C[s, i, j] = sum_k A[s, i, k] * B[s, j, k] (+ bias),  f16 in, f32 accumulate, f16 out.
// A is f16 or a Q8_0H weight; B is f16.  Six kernels, chosen by launch_gemm_nt:
//
//   gemm_nt_wide_kernel    f16 x f16, K % 64 == 0, many activation rows: 320 x 256 tiles, eight wavefronts that
//                          both load and multiply (half the operand bytes per product of the 160 x 128 tiles)
//   gemm_nt_dl_kernel      f16 x f16, K % 32 == 0: tiles of 64 x 64 to 160 x 128 (nt_choose), loaded global -> LDS
//                          directly into a ring of stages by two wavefronts that do nothing else,
//                          issue order pinned (the fast path for the Phi-2 prefill shape:
//                          10240 x 512 outputs = 256 workgroups, one per CU)
//   gemm_nt_q8w_kernel     Q8_0H x f16, K % 256 == 0: the same pipeline; four loading wavefronts widen the int8
//                          tile to f16 codes on its way into LDS, each block of 32 is multiplied from zero and
//                          its partial sums are folded into the accumulators with the block's scale in f32
//   gemm_nt_q8r_kernel     Q8_0H x f16, any other K
//   gemm_nt_shortk_kernel  f16 x f16, K <= 128 (attention scores): a resident strip of B rows,
//                          A tiles prefetched through registers, output written as it is produced
//   gemm_nt_kernel         f16 x f16 with a K that is no multiple of 32, or short and without a contiguous
//                          output axis: register-staged, two LDS stages
//
// Common to all: 2 x 2 multiplying wavefronts (the wide kernel: 2 x 4), v_mfma_f32_16x16x32_f16 with A rows on the MFMA's
// lane index, XOR-swizzled or odd-stride LDS rows so that fragment reads are conflict-free, an
// epilogue that transposes through LDS and stores 128 bits along the contiguous output axis, and
// workgroup ids remapped so that each of the 8 XCDs takes a block of neighbouring tiles, whose
// operands its L2 holds once (nt_tile_of).
//
// gemm_nt_kernel's pipeline per K tile of 64: global loads of tile t+2 into registers, MFMAs on LDS
// stage t, then the registers of tile t+1 -> the other LDS stage, one barrier.
//
// Roles in the reference: ops/gemm.rs:305-657 (GEMM generators), with Linear's
// W.gemm(x, b, false, true, true) (crates/ratchet-nn/src/linear.rs:17-24) and attention's
// Q.matmul(K, false, true) (phi3/attn.rs:142-158) as the callers.
#include "device_common.h"
#include <algorithm>
#include <utility>

namespace rt {

typedef uint32_t uint4_d __attribute__((ext_vector_type(4), aligned(4)));
typedef float float4_d __attribute__((ext_vector_type(4), aligned(4)));

struct GemmNtArgs {
    const void *A;       // f16 [.., M, K] or Q8_0H codes
    const half_t *scales; // Q8_0H scale stream of A, dwords in it (whole 256 bytes)
    int64_t scale_dwords;
    const half_t *B;     // f16 [.., N, K]
    const half_t *bias;
    half_t *out;
    int64_t M, N, K;
    int64_t a_stack, b_stack;
    int64_t a_bs, a_rs;  // elements
    int64_t b_bs, b_js;
    int64_t o_bs, o_is, o_js;
    int has_bias, bias_on_rows, act;
    int tiles_i, tiles_j;
    int xi, pj; // XCD-aware order of the tiles (nt_tile_of)
    int rows, cols, panels, xj_log2; // of an XCD's block
    int vec_epilogue; // o_is == 1 and rows of the output 16-byte aligned: LDS-staged 128-bit stores
    // split K (direct-to-LDS kernels): blockIdx.z owns K range [z * k_len, (z + 1) * k_len) and writes its
    // f32 sums to partial [stack][split][N][M]; a second kernel adds them up, then bias, activation, rounding
    int ksplit;
    int64_t k_len;
    float *partial;
};

// Which output tile a workgroup takes.  Workgroup ids go round the 8 XCDs, each with an L2 of its own.
// g.xi > 0: the grid of tiles is cut into xi x (8 / xi) equal blocks, one per XCD, and a block is walked in panels
// of g.pj columns, so that the 32 workgroups an XCD runs at a time share the fewest operand rows
// (nt_set_tiles chooses).  Otherwise XCD x takes the x-th of eight contiguous ranges of the tiles in row-major order, the first
// ntiles % 8 of them one longer (taken as they come, neighbours of a tile row would read its operands into eight L2s: f16, 300 rows x
// 2560 x 10240 in 60 tiles of 128 x 128 and 4 shares 39.6 -> 35.3 us, 1300 rows x 8192 x 4096 in 572 of 160 x 128 133.5 -> 101.5).  In 32 bits and with the block's sides from the host: every
// workgroup waits for this before its first load, and six 64-bit divisions were 0.3 us a launch (a 512-row prompt through
// a layer with Q8_0H weights, four products: 178.8 -> 176.6 us).
__device__ __forceinline__ void nt_tile_of(const GemmNtArgs &g, int64_t wg, int64_t &ti, int64_t &tj) {
    const uint32_t id = (uint32_t)wg; // < 2^31: launcher
    if (g.xi > 0) {
        const uint32_t x = id & 7, r = id >> 3, per = (uint32_t)(g.rows * g.pj);
        const uint32_t p = min(r / per, (uint32_t)(g.panels - 1)), q = r - p * per;
        const uint32_t w = min((uint32_t)g.pj, (uint32_t)g.cols - p * g.pj); // the last panel may be narrower
        const uint32_t qi = q / w;
        ti = (x >> g.xj_log2) * g.rows + qi, tj = (x & ((1u << g.xj_log2) - 1)) * g.cols + p * g.pj + (q - qi * w);
        return;
    }
    const uint32_t ntiles = (uint32_t)g.tiles_i * (uint32_t)g.tiles_j, x = id & 7, n = x * (ntiles >> 3) + min(x, ntiles & 7) + (id >> 3);
    ti = n / (uint32_t)g.tiles_j, tj = n - (uint32_t)ti * (uint32_t)g.tiles_j;
}

// Timing-only variants of gemm_nt_dl_kernel for the measurement probes (a bit mask: 1 no tile loads, 2 no MFMAs,
// 4 no fragment reads, 8 no output); the product is built with 0.
#ifndef RT_NT_ABLATION
#define RT_NT_ABLATION 0
#endif

constexpr int NT_BK = 64;
constexpr int NT_LDK = NT_BK;     // halfs per LDS row: 128 B = 8 vectors of 16 B, no padding
constexpr int NT_THREADS = 256;

// LDS tile layout: row r holds its 8 K-vectors at slots c ^ ((r >> 1) & 7).  Two
// consecutive rows cover all 64 banks, so a 16-lane group that writes two whole rows
// (the global-load order) and a 16-lane group that reads one vector from each of 16
// rows (the MFMA fragment order) are both free of bank conflicts.
__device__ __forceinline__ int nt_slot(int r, int c) { return (r * 8 + (c ^ ((r >> 1) & 7))) * 8; } // in halfs

__device__ __forceinline__ void nt_cvt_i8x4(uint32_t v, half2_t &lo, half2_t &hi) {
    v ^= 0x80808080u;
    const uint32_t a = __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u);
    const uint32_t b = __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u);
    const half2_t bias = {(half_t)1152.0f, (half_t)1152.0f};
    lo = __builtin_bit_cast(half2_t, a) - bias;
    hi = __builtin_bit_cast(half2_t, b) - bias;
}

// Output stage shared by the tiled kernels: accumulators (+ bias, activation) to f16.  In tile
// (a, b) lane l holds A row (l % 16) and B rows 4 * (l / 16) + r.  With vec_epilogue the A-row
// axis is contiguous in the output (o_is == 1): the wavefront's sub-tile is transposed through
// LDS (free once the main loop's last barrier has passed) so that every lane stores 8
// consecutive outputs (128 bits); otherwise bounds-checked scalar stores.
// PARTS: the transposition takes the B rows in that many parts, one after the other through the same LDS.
template <int TM, int TN, int WM, int WN, int PARTS = 1>
__device__ __forceinline__ void nt_epilogue(const GemmNtArgs &g, float4_t (&acc)[TM][TN], uint8_t *smem, int64_t s,
                                            int64_t i0, int64_t j0, int wi, int wj, int wave, int lane) {
    const int fr = lane & 15, fg = lane >> 4;
    if (g.ksplit > 1) {
        // this workgroup summed only its share of K: the sums go out as they are, [j][i] with i contiguous
        float *pt = g.partial + ((s * g.ksplit + blockIdx.z) * g.N) * g.M;
#pragma unroll
        for (int a = 0; a < TM; a++) {
            const int64_t i = i0 + wi * WM + a * 16 + fr;
#pragma unroll
            for (int b = 0; b < TN; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t j = j0 + wj * WN + b * 16 + 4 * fg + r;
                    if (i < g.M && j < g.N) pt[j * g.M + i] = acc[a][b][r];
                }
        }
        return;
    }
    half_t *out = g.out + s * g.o_bs;
    if (g.vec_epilogue) {
        constexpr int EROW = WM + 8;                       // halfs per staged B-row (+16 B pad)
        constexpr int TP = TN / PARTS, WP = WN / PARTS;    // MFMA tiles and B rows of a part
        static_assert(TN % PARTS == 0, "parts are whole MFMA tiles");
        half_t *es = (half_t *)smem + wave * (WP * EROW);
        float bi[TM]; // the bias of this lane's A rows, asked for once
#pragma unroll
        for (int a = 0; a < TM; a++) {
            const int64_t i = i0 + wi * WM + a * 16 + fr;
            bi[a] = g.has_bias && g.bias_on_rows && i < g.M ? (float)g.bias[i] : 0.f;
        }
#pragma unroll
        for (int h = 0; h < PARTS; h++) {
            const int64_t jh = j0 + wj * WN + h * WP;
            rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
                for (int a = 0; a < TM; a++) {
#pragma unroll
                    for (int b = 0; b < TP; b++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int jl = b * 16 + 4 * fg + r;
                            float v = acc[a][h * TP + b][r] + bi[a];
                            if (g.has_bias && !g.bias_on_rows) v += (float)g.bias[min(jh + jl, g.N - 1)];
                            v = rt_act_k<decltype(has_act)::value>(v);
                            es[jl * EROW + a * 16 + fr] = (half_t)v;
                        }
                }
            });
            asm volatile("" ::: "memory"); // same wavefront reads back below; DS operations complete in order
            constexpr int VPR = WM / 8;    // 128-bit vectors per staged row
            for (int v = lane; v < WP * VPR; v += 64) {
                const int jl = v / VPR, c = v - jl * VPR;
                const int64_t j = jh + jl, i = i0 + wi * WM + 8 * c;
                if (j < g.N) {
                    if (i + 8 <= g.M) {
                        __builtin_nontemporal_store(*(const uint4_t *)(es + jl * EROW + 8 * c), (uint4_t *)(out + j * g.o_js + i)); // written once, not read back here
                    } else {
                        for (int e = 0; e < 8; e++)
                            if (i + e < g.M) out[j * g.o_js + i + e] = es[jl * EROW + 8 * c + e];
                    }
                }
            }
            asm volatile("" ::: "memory");
        }
        return;
    }
    rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
        for (int a = 0; a < TM; a++) {
            const int64_t i = i0 + wi * WM + a * 16 + fr;
            float bi = 0.f;
            if (g.has_bias && g.bias_on_rows && i < g.M) bi = (float)g.bias[i];
#pragma unroll
            for (int b = 0; b < TN; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t j = j0 + wj * WN + b * 16 + 4 * fg + r;
                    if (i < g.M && j < g.N) {
                        float v = acc[a][b][r] + bi;
                        if (g.has_bias && !g.bias_on_rows) v += (float)g.bias[j];
                        v = rt_act_k<decltype(has_act)::value>(v);
                        out[i * g.o_is + j * g.o_js] = (half_t)v;
                    }
                }
        }
    });
}

// The same for accumulators of 32 x 32 MFMA tiles: lane l holds A row l % 32 and B rows 8 * (r / 4) + 4 * (l / 32) + r % 4.
template <int TM, int TN, int WM, int WN>
__device__ __forceinline__ void nt_epilogue32(const GemmNtArgs &g, float16_t (&acc)[TM][TN], uint8_t *smem, int64_t s, int64_t i0, int64_t j0, int wi, int wj,
                                              int wave, int lane) {
    const int fr = lane & 31, fh = lane >> 5;
    const int64_t iw = i0 + wi * WM, jw = j0 + wj * WN;
    if (g.ksplit > 1) { // this workgroup's share of K: the sums as they are, [j][i] with i contiguous
        float *pt = g.partial + ((s * g.ksplit + blockIdx.z) * g.N) * g.M;
#pragma unroll
        for (int a = 0; a < TM; a++) {
            const int64_t i = iw + a * 32 + fr;
#pragma unroll
            for (int b = 0; b < TN; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int64_t j = jw + b * 32 + 8 * (r >> 2) + 4 * fh + (r & 3);
                    if (i < g.M && j < g.N) pt[j * g.M + i] = acc[a][b][r];
                }
        }
        return;
    }
    half_t *out = g.out + s * g.o_bs;
    constexpr int EROW = WM + 8; // halfs per staged B row (+16 B pad)
    half_t *es = (half_t *)smem + wave * (WN * EROW);
    float bi[TM]; // the bias of this lane's A rows, asked for once
#pragma unroll
    for (int a = 0; a < TM; a++) {
        const int64_t i = iw + a * 32 + fr;
        bi[a] = g.has_bias && g.bias_on_rows && i < g.M ? (float)g.bias[i] : 0.f;
    }
    if (!g.vec_epilogue) {
        // rows that do not start on 16 bytes, or another axis contiguous: as they are, 32 values of a row per
        // instruction (through LDS and value by value 51865 x 448 x 64 took 80.5 us where these take 53.4; 3794 x 1036 x 288 19.3 and 14.9)
        rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
            for (int a = 0; a < TM; a++) {
                const int64_t i = iw + a * 32 + fr;
#pragma unroll
                for (int b = 0; b < TN; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int64_t j = jw + b * 32 + 8 * (r >> 2) + 4 * fh + (r & 3);
                        if (i < g.M && j < g.N) {
                            float v = acc[a][b][r] + bi[a];
                            if (g.has_bias && !g.bias_on_rows) v += (float)g.bias[j];
                            out[i * g.o_is + j * g.o_js] = (half_t)rt_act_k<decltype(has_act)::value>(v);
                        }
                    }
            }
        });
        return;
    }
    rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
            for (int b = 0; b < TN; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int jl = b * 32 + 8 * (r >> 2) + 4 * fh + (r & 3);
                    float v = acc[a][b][r] + bi[a];
                    if (g.has_bias && !g.bias_on_rows) v += (float)g.bias[min(jw + jl, g.N - 1)];
                    v = rt_act_k<decltype(has_act)::value>(v);
                    es[jl * EROW + a * 32 + fr] = (half_t)v;
                }
    });
    asm volatile("" ::: "memory"); // same wavefront reads back below; DS operations complete in order
    constexpr int VPR = WM / 8; // 128-bit vectors per staged row
    for (int v = lane; v < WN * VPR; v += 64) {
        const int jl = v / VPR, c = v - jl * VPR;
        const int64_t j = jw + jl, i = iw + 8 * c;
        if (j < g.N) {
            if (i + 8 <= g.M) {
                __builtin_nontemporal_store(*(const uint4_t *)(es + jl * EROW + 8 * c), (uint4_t *)(out + j * g.o_js + i)); // written once, not read back here
            } else {
                for (int e = 0; e < 8; e++)
                    if (i + e < g.M) out[j * g.o_js + i + e] = es[jl * EROW + 8 * c + e];
            }
        }
    }
}

// The output stage for rows that start on 4 bytes only (o_is == 1, o_js even): staged as nt_epilogue does, stored as pairs, consecutive ones by
// consecutive lanes, a lane's all read back before they are stored.
template <int TM, int TN, int WM, int WN>
__device__ __forceinline__ void nt_epilogue_pairs(const GemmNtArgs &g, float4_t (&acc)[TM][TN], uint8_t *smem, int64_t s, int64_t i0, int64_t j0, int wi,
                                                  int wj, int wave, int lane) {
    constexpr int EROW = WM + 8, NPAIR = WN * (WM / 2) / 64;
    static_assert(WN * (WM / 2) % 64 == 0, "whole instructions");
    const int fr = lane & 15, fg = lane >> 4;
    const int64_t iw = i0 + wi * WM, jw = j0 + wj * WN;
    half_t *es = (half_t *)smem + wave * (WN * EROW);
    rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
        for (int a = 0; a < TM; a++) {
            const float bi = g.has_bias && g.bias_on_rows ? (float)g.bias[min(iw + a * 16 + fr, g.M - 1)] : 0.f;
#pragma unroll
            for (int b = 0; b < TN; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int jl = b * 16 + 4 * fg + r;
                    float v = acc[a][b][r] + bi;
                    if (g.has_bias && !g.bias_on_rows) v += (float)g.bias[min(jw + jl, g.N - 1)];
                    es[jl * EROW + a * 16 + fr] = (half_t)rt_act_k<decltype(has_act)::value>(v);
                }
        }
    });
    asm volatile("" ::: "memory"); // same wavefront reads back below; DS operations complete in order
    const int jn = (int)min<int64_t>(WN, g.N - jw), in = (int)min<int64_t>(WM, g.M - iw); // rows and values inside
    half_t *o = g.out + s * g.o_bs + jw * g.o_js + iw;
    uint32_t x[NPAIR];
#pragma unroll
    for (int u = 0; u < NPAIR; u++) {
        const int v = u * 64 + lane, jl = v / (WM / 2), c = 2 * (v - jl * (WM / 2));
        x[u] = *(const uint32_t *)(es + jl * EROW + c);
    }
#pragma unroll
    for (int u = 0; u < NPAIR; u++) {
        const int v = u * 64 + lane, jl = v / (WM / 2), c = 2 * (v - jl * (WM / 2));
        if (jl >= jn || c >= in) continue;
        half_t *d = o + jl * g.o_js + c;
        if (c + 2 <= in) __builtin_nontemporal_store(x[u], (uint32_t *)d);
        else *d = __builtin_bit_cast(half2_t, x[u])[0];
    }
    asm volatile("" ::: "memory");
}

// KFULL: K is a multiple of the K step, so no load or store needs a bound.
template <int BM, int BN, bool KFULL>
__global__ __launch_bounds__(NT_THREADS, (BM * BN <= 128 * 64 ? 3 : 1)) void gemm_nt_kernel(GemmNtArgs g) {
    constexpr int WM = BM / 2, WN = BN / 2;      // wavefront sub-tile
    constexpr int TM = WM / 16, TN = WN / 16;    // MFMA tiles per wavefront
    static_assert(WM % 16 == 0 && WN % 16 == 0, "tile must split into 16x16 MFMA tiles");
    // 16-byte vectors per K tile row, and per thread
    constexpr int A_VPR = NT_BK / 8;
    constexpr int A_VEC = (BM * A_VPR + NT_THREADS - 1) / NT_THREADS;
    constexpr int B_VPR = NT_BK / 8;
    constexpr int B_VEC = (BN * B_VPR + NT_THREADS - 1) / NT_THREADS;

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    half_t *As = (half_t *)smem;                         // [2][BM][NT_LDK]
    half_t *Bs = As + 2 * BM * NT_LDK;                   // [2][BN][NT_LDK]

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wi = wave >> 1, wj = wave & 1;
    const int fr = lane & 15, fg = lane >> 4;            // fragment row / K group

    int64_t ti, tj;
    nt_tile_of(g, blockIdx.x, ti, tj); // XCD-aware tile order (see the file comment)
    const int64_t i0 = ti * BM, j0 = tj * BN;
    const int64_t s = blockIdx.y;
    const int64_t a_el = (g.a_stack == 1 ? 0 : s) * g.a_bs, b_el = (g.b_stack == 1 ? 0 : s) * g.b_bs;

    // two register sets: the loads of tile t+2 are in flight while tile t is multiplied
    uint4_t ra0[A_VEC], rb0[B_VEC], ra1[A_VEC], rb1[B_VEC];

    // Loads are unconditional (addresses past K are clamped to a valid one) so that no branch
    // separates them from the LDS store that consumes them and the hardware counters can let
    // the other register set's loads stay in flight; store_tiles zeroes what lies past K.
    auto load_tiles = [&](int64_t k0, uint4_t (&ra)[A_VEC], uint4_t (&rb)[B_VEC]) {
#pragma unroll
        for (int e = 0; e < A_VEC; e++) {
            const int v = min(e * NT_THREADS + t, BM * A_VPR - 1);
            const int r = v / A_VPR, c = v - r * A_VPR;
            const int64_t gr = min(i0 + r, g.M - 1); // rows past the end duplicate the last one; never stored
            const int64_t gk = KFULL ? k0 + 8 * c : min(k0 + 8 * c, g.K - 8);
            ra[e] = *(const uint4_t *)((const half_t *)g.A + a_el + gr * g.a_rs + gk);
        }
#pragma unroll
        for (int e = 0; e < B_VEC; e++) {
            const int v = min(e * NT_THREADS + t, BN * B_VPR - 1);
            const int r = v / B_VPR, c = v - r * B_VPR;
            const int64_t gr = min(j0 + r, g.N - 1);
            const int64_t gk = KFULL ? k0 + 8 * c : min(k0 + 8 * c, g.K - 8);
            rb[e] = *(const uint4_t *)(g.B + b_el + gr * g.b_js + gk);
        }
    };

    auto store_tiles = [&](int stage, int64_t k0, const uint4_t (&ra)[A_VEC], const uint4_t (&rb)[B_VEC]) {
        half_t *as = As + stage * BM * NT_LDK, *bs = Bs + stage * BN * NT_LDK;
        const uint4_t zero4 = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < A_VEC; e++) {
            const int v = e * NT_THREADS + t;
            if (v < BM * A_VPR) {
                const int r = v / A_VPR, c = v - r * A_VPR;
                *(uint4_t *)(as + nt_slot(r, c)) = (KFULL || k0 + 8 * c < g.K) ? ra[e] : zero4;
            }
        }
#pragma unroll
        for (int e = 0; e < B_VEC; e++) {
            const int v = e * NT_THREADS + t;
            if (v < BN * B_VPR) {
                const int r = v / B_VPR, c = v - r * B_VPR;
                *(uint4_t *)(bs + nt_slot(r, c)) = (KFULL || k0 + 8 * c < g.K) ? rb[e] : zero4;
            }
        }
    };

    float4_t acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};

    // Fragment addressing: lane (fr, fg) reads row base + 16 * tile + fr, K-vector kk * 4 + fg.  The
    // wavefront's row bases are multiples of 16, so the row's swizzle term depends on fr only.
    const int swz = (fr >> 1) & 7;
    struct Frags {
        half8_t fa[TM], fb[TN];
    };
    auto read_frags = [&](int stage, int kk, Frags &f) {
        const half_t *as = As + stage * BM * NT_LDK + (wi * WM + fr) * NT_LDK + (((kk * 4 + fg) ^ swz) << 3);
        const half_t *bs = Bs + stage * BN * NT_LDK + (wj * WN + fr) * NT_LDK + (((kk * 4 + fg) ^ swz) << 3);
#pragma unroll
        for (int a = 0; a < TM; a++) f.fa[a] = __builtin_bit_cast(half8_t, *(const uint4_t *)(as + a * 16 * NT_LDK));
#pragma unroll
        for (int b = 0; b < TN; b++) f.fb[b] = __builtin_bit_cast(half8_t, *(const uint4_t *)(bs + b * 16 * NT_LDK));
    };
    auto mma_step = [&](const Frags &f) {
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
            for (int b = 0; b < TN; b++)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.fb[b], f.fa[a], acc[a][b], 0, 0, 0);
    };

    // Software pipeline: tile t is multiplied from LDS stage t % 2 while tile t+1 sits in one
    // register set (written to the other stage after the MFMAs) and tile t+2 is being loaded
    // into the other register set.  Loads past the last tile re-read it (their data is unused),
    // which keeps the loop body free of branches around memory operations.  Within a tile the
    // second K step's fragments are requested before the first step's MFMAs are issued.
    const int64_t nk = (g.K + NT_BK - 1) / NT_BK;
    auto kclamp = [&](int64_t kt) { return min(kt, nk - 1) * NT_BK; };
    auto compute = [&](int stage) {
        Frags f0, f1;
        read_frags(stage, 0, f0);
        read_frags(stage, 1, f1);
        mma_step(f0);
        mma_step(f1);
    };
    if (nk > 0) {
        load_tiles(0, ra0, rb0);
        load_tiles(kclamp(1), ra1, rb1);
        store_tiles(0, 0, ra0, rb0);
    }
    __syncthreads();
    for (int64_t kt = 0; kt < nk; kt += 2) {
        // even tile: set 1 holds tile kt+1, set 0 is free for tile kt+2
        load_tiles(kclamp(kt + 2), ra0, rb0);
        compute(0);
        store_tiles(1, (kt + 1) * NT_BK, ra1, rb1);
        __syncthreads();
        if (kt + 1 >= nk) break;
        // odd tile: set 0 holds tile kt+2, set 1 is free for tile kt+3
        load_tiles(kclamp(kt + 3), ra1, rb1);
        compute(1);
        store_tiles(0, (kt + 2) * NT_BK, ra0, rb0);
        __syncthreads();
    }
    __syncthreads(); // every wavefront is done with the tile stages: the epilogue reuses them

    nt_epilogue<TM, TN, WM, WN>(g, acc, smem, s, i0, j0, wi, wj, wave, lane);
}

// ---------------------------------------------------------------------------
// f16 x f16 variant with direct-to-LDS loads (global_load_lds_dwordx4): tiles go
// from global memory straight into a three-stage LDS ring without passing through
// registers.  A wavefront's load instruction writes 1 KiB of LDS contiguously
// (lane l at base + 16 l), i.e. 8 whole rows of the swizzled tile; the swizzle is
// applied on the global side by choosing which K-vector each lane fetches.
// Requires K % 32 == 0; full tiles are not required (rows are clamped, and a last tile of 32 is multiplied as half a one).
//
// The loads are issued by wavefronts of their own.  A wavefront issues in order, one per SIMD
// here: when the memory pipeline pushes back on a load, the MFMAs behind it wait too, and with
// every wavefront loading its share the fill (16.5 us alone at the [512 x 2560] . [10240 x 2560]^T
// shape) and the MFMAs (12.8 us alone) nearly added up.  So wavefronts 0..3 only read fragments
// and multiply; LW further wavefronts only issue the ring's loads (chunks dealt round-robin) and
// meet the others at the one barrier per K tile: a stalled load stalls nobody else (40 -> 33 us).
//
// Iteration t, loading wavefronts: issue tile t + STAGES - 1 into the stage that was read for
// the last time before the barrier of iteration t - 1, wait until tile t + 1 has landed, barrier.
// Multiplying wavefronts: the first K step's MFMAs with the second step's fragment reads between
// them, barrier (every read has returned, tile t + 1 is visible), the second step's MFMAs with
// the reads of tile t + 1's first-step fragments between them.
// ---------------------------------------------------------------------------
template <int BM, int BN, int STAGES, int LW, bool TAIL>
__global__ __launch_bounds__(NT_THREADS + 64 * LW) void gemm_nt_dl_kernel(GemmNtArgs g) {
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 16, TN = WN / 16;
    constexpr int CH = (BM + BN) / 8;  // 8-row chunks of one K tile: the A rows, then the B rows
    constexpr int LCH = CH / LW;       // per loading wavefront
    static_assert(BM % 16 == 0 && BN % 8 == 0 && CH % LW == 0, "chunks must deal out evenly");
    static_assert((STAGES - 2) * LCH < 64, "the wait counter has six bits");
    constexpr int STAGE_HALFS = (BM + BN) * NT_LDK;

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    half_t *ring = (half_t *)smem; // [STAGES][BM + BN][64]

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);

    int64_t ti, tj;
    nt_tile_of(g, blockIdx.x, ti, tj); // XCD-aware tile order (see the file comment)
    const int64_t i0 = ti * BM, j0 = tj * BN;
    const int64_t s = blockIdx.y;
    const int64_t kbase = (int64_t)blockIdx.z * g.k_len;
    const int64_t a_el = (g.a_stack == 1 ? 0 : s) * g.a_bs + kbase, b_el = (g.b_stack == 1 ? 0 : s) * g.b_bs + kbase;
    const int kn = (int)min(g.k_len, g.K - kbase); // this workgroup's share of K: > 0, a multiple of 32 (launcher)
    const int nk = (kn + NT_BK - 1) / NT_BK;

    if (wave >= 4) {
        // ---- loading wavefront: lane l fills LDS row chunk * 8 + l / 8, slot l % 8, which must
        // hold K-vector (l % 8) ^ ((row >> 1) & 7); BM is a multiple of 16, so the swizzle of a B
        // row is the same counted from the top of the stage as from the top of the B tile
        const int lw = wave - 4;
        static_assert(LW % 2 == 0, "one K-vector per lane for all chunks");
        const int kv = 8 * ((lane & 7) ^ ((lw * 4 + (lane >> 4)) & 7)); // (lane % 8) ^ (row / 2 % 8)
        const half_t *gp[LCH];
#pragma unroll
        for (int c = 0; c < LCH; c++) {
            const int row = (lw + c * LW) * 8 + (lane >> 3);
            gp[c] = (row < BM ? (const half_t *)g.A + a_el + min(i0 + row, g.M - 1) * g.a_rs : g.B + b_el + min(j0 + (row - BM), g.N - 1) * g.b_js) + (TAIL ? 0 : kv);
        }
        auto issue_tile = [&](int stage, int tile) {
            const int kt = min(tile, nk - 1) * NT_BK; // past the last tile that one again
            const int k = TAIL ? min(kt + kv, kn - 8) : kt; // past the end of K its last vector: never used
            half_t *st = ring + stage * STAGE_HALFS;
            if (RT_NT_ABLATION & 1) return; // timing only: no tile loads
#pragma unroll
            for (int c = 0; c < LCH; c++)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(gp[c] + k),
                                                 (__attribute__((address_space(3))) void *)(st + (lw + c * LW) * 8 * NT_LDK),
                                                 16, 0, 0);
        };
        // all but the newest STAGES - 2 tiles have landed
        constexpr int kNew = (STAGES - 2) * LCH;
        constexpr int kWaitOlder = 0x0F70 | (kNew & 0xF) | (((kNew >> 4) & 0x3) << 14);
        auto publish = [&]() {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(kWaitOlder);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
#pragma unroll
        for (int st = 0; st < STAGES - 1; st++) issue_tile(st, st);
        publish(); // tile 0
        int wr = STAGES - 1;
        for (int kt = 0; kt < nk; kt++) {
            // stage wr was read for the last time before the barrier that ended iteration kt - 1
            issue_tile(wr, kt + STAGES - 1);
            publish(); // tile kt + 1
            wr = wr + 1 == STAGES ? 0 : wr + 1;
        }
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): nothing may land once the epilogue reuses the ring
        __syncthreads();
        return;
    }

    // ---- multiplying wavefronts
    const int wi = wave >> 1, wj = wave & 1;
    const int fr = lane & 15, fg = lane >> 4;
    const int swz = (fr >> 1) & 7;
    struct Frags {
        half8_t fa[TM], fb[TN];
    };
    auto read_one = [&](int stage, int kk, Frags &f, int i) {
        if (RT_NT_ABLATION & 4) return; // timing only: no fragment reads
        const half_t *as = ring + stage * STAGE_HALFS + (wi * WM + fr) * NT_LDK + (((kk * 4 + fg) ^ swz) << 3);
        const half_t *bs = ring + stage * STAGE_HALFS + BM * NT_LDK + (wj * WN + fr) * NT_LDK + (((kk * 4 + fg) ^ swz) << 3);
        if (i < TM)
            f.fa[i] = __builtin_bit_cast(half8_t, *(const uint4_t *)(as + i * 16 * NT_LDK));
        else
            f.fb[i - TM] = __builtin_bit_cast(half8_t, *(const uint4_t *)(bs + (i - TM) * 16 * NT_LDK));
    };
    float4_t acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
    // every fragment read has returned (the stage may be refilled after the barrier); no loads of its own
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    meet(); // tile 0 visible
#if RT_NT_ABLATION & 4
    Frags f0 = {}, f1 = {};
    asm volatile("" : "+v"(f0.fa[0]), "+v"(f1.fa[0]));
#else
    Frags f0, f1;
#endif
#pragma unroll
    for (int i = 0; i < TM + TN; i++) read_one(0, 0, f0, i);
    int cur = 0, nxt = 1;
    // a fragment read behind every second MFMA, or behind every one where the tile has too few of them
    constexpr int RS = TM * TN / 2 >= TM + TN ? 2 : 1;
    static_assert(TM * TN / RS >= TM + TN, "not enough MFMAs to spread the reads over");
    for (int kt = 0; kt < nk; kt++) {
#pragma unroll
        for (int m = 0; m < TM * TN; m++) {
            if (!(RT_NT_ABLATION & 2)) acc[m / TN][m % TN] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f0.fb[m % TN], f0.fa[m / TN], acc[m / TN][m % TN], 0, 0, 0);
            if (m % RS == RS - 1) {
                if (m / RS < TM + TN) read_one(cur, 1, f1, m / RS);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        meet(); // tile kt + 1 visible
        if (TAIL && kt + 1 == nk && kn % NT_BK) break; // K ends with the first half of this tile
#pragma unroll
        for (int m = 0; m < TM * TN; m++) {
            if (!(RT_NT_ABLATION & 2)) acc[m / TN][m % TN] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f1.fb[m % TN], f1.fa[m / TN], acc[m / TN][m % TN], 0, 0, 0);
            if (m % RS == RS - 1) {
                if (m / RS < TM + TN) read_one(nxt, 0, f0, m / RS);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        cur = nxt;
        nxt = nxt + 1 == STAGES ? 0 : nxt + 1;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __syncthreads();
    if (RT_NT_ABLATION & 8) { // timing only: no output (one store per lane keeps the accumulators alive)
        float v = 0.f;
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
            for (int b = 0; b < TN; b++) v += acc[a][b][0] + acc[a][b][1] + acc[a][b][2] + acc[a][b][3];
        if (RT_NT_ABLATION & 4) v += (float)f0.fa[0][0] + (float)f1.fb[0][0];
        if (v == 12345.678f) g.out[t] = (half_t)v;
        return;
    }
    nt_epilogue<TM, TN, WM, WN>(g, acc, smem, s, i0, j0, wi, wj, wave, lane);
}

// ---------------------------------------------------------------------------
// f16 x f16 with many activation rows: 320 x 256 outputs per workgroup, one workgroup per compute unit.
// A K step of 64 is 2560 cycles of MFMAs per SIMD against 74 KB of tiles to fetch (29 bytes per cycle;
// the 160 x 128 tile needs 58, more than the L2s deliver to all compute units at once) and 1792 of
// LDS fragment reads.  Eight wavefronts of 160 x 64 outputs, two per SIMD: 160 accumulator registers leave no
// room for a second fragment set of everything, so an A fragment is read for the next half step into the registers
// its last MFMA has just left, and only the B fragments and the last two A fragments are held twice.  Every
// wavefront loads an eighth of each tile (LDS-DMA, between its MFMAs): wavefronts that only load would halve the
// registers of the ones that multiply.
//
// Two LDS stages.  Per tile: half step 0 on the fragments in registers, reading half step 1's; then, all of the stage read
// and the next tile landed (its loads have had a whole tile's time), one barrier; half step 1, reading the next
// tile's first fragments and issuing the loads of the tile after it into the stage just left.
// 10240 x 2560 weights against 2048 / 4096 activation rows: 89.7 / 177.0 us (1.20 / 1.21 PFLOP/s) where the 160 x 128 tiles take
// 110.7 / 218.5; 12288 x 3072 against 1300 rows 102 for 148.
// ---------------------------------------------------------------------------
template <int BM, int BN, int WI, int WJ>
__global__ __launch_bounds__(64 * WI * WJ) void gemm_nt_wide_kernel(GemmNtArgs g) {
    constexpr int WAVES = WI * WJ, WM = BM / WI, WN = BN / WJ, TM = WM / 16, TN = WN / 16;
    constexpr int TD = 2, TS = TM - TD; // A fragments held twice (the last TD) and once
    constexpr int ACH = BM / 8 / WAVES, BCH = BN / 8 / WAVES; // 8-row chunks of a tile per wavefront
    constexpr int STAGE_BYTES = (BM + BN) * NT_LDK * 2;
    static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0 && TS >= TD + TN && ACH + BCH <= TM, "chunks must deal out evenly");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    int64_t ti, tj;
    nt_tile_of(g, blockIdx.x, ti, tj); // XCD-aware tile order (see the file comment)
    const int64_t i0 = ti * BM, j0 = tj * BN;
    const int64_t s = blockIdx.y;
    const half_t *A = (const half_t *)g.A + (g.a_stack == 1 ? 0 : s) * g.a_bs + i0 * g.a_rs;
    const half_t *B = g.B + (g.b_stack == 1 ? 0 : s) * g.b_bs + j0 * g.b_js;
    const int nk = (int)(g.K / NT_BK);
    const int a_last = (int)min<int64_t>(BM, g.M - i0) - 1, b_last = (int)min<int64_t>(BN, g.N - j0) - 1; // rows past them repeat the last

    // Chunk c of this wavefront: LDS rows 8 (wave + WAVES c) .. + 7 of the A rows, then of the B rows; lane l fills row l / 8,
    // slot l % 8, which holds K-vector (l % 8) ^ ((row >> 1) & 7).  Row offsets are computed at each use: the vector ALU has
    // time for it, the register file has no room to keep them.
    auto issue_chunk = [&](int c, uint32_t stage, int64_t k0) __attribute__((always_inline)) {
        const bool is_a = c < ACH;
        const int cc = is_a ? c : c - ACH;
        int l = lane;
        asm volatile("" : "+v"(l));
        const int row = (wave + WAVES * cc) * 8 + (l >> 3);
        const uint32_t kv = (uint32_t)((l & 7) ^ ((row >> 1) & 7));
        const uint32_t off = (uint32_t)min(row, is_a ? a_last : b_last) * (uint32_t)(2 * (is_a ? g.a_rs : g.b_js)) + 16u * kv; // < 2^32: launcher
        const uint8_t *base = (const uint8_t *)((is_a ? A : B) + k0); // wave-uniform
        const uint32_t dst = stage + (uint32_t)((is_a ? 0 : BM) + (wave + WAVES * cc) * 8) * (NT_LDK * 2);
        // as asm: behind the builtin the compiler waits for every load in flight before the next fragment read, which it
        // cannot tell from a read of what the load writes; no register is written, and the barrier's wait covers it
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "m0", "memory");
    };
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;

    const int wi = wave / WJ, wj = wave % WJ;
    const int fr = lane & 15, fg = lane >> 4;
    // byte addresses of this lane's first A and B fragments of half step 0 in stage 0 (half step 1: the slot's bit 2 flipped)
    const uint32_t slot = (uint32_t)((fg ^ ((fr >> 1) & 7)) << 4);
    const uint32_t ra0 = (uint32_t)(wi * WM + fr) * (NT_LDK * 2) + slot, rb0 = (uint32_t)(BM + wj * WN + fr) * (NT_LDK * 2) + slot;

    float4_t acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
    half8_t fs[TS], fd0[TD], fd1[TD], fb0[TN], fb1[TN];

    // One half step: the MFMAs of the fragments in hand, the next half step's read behind them from `ra`, `rb`.
    auto half_step = [&](half8_t (&fd)[TD], half8_t (&fb)[TN], half8_t (&fdn)[TD], half8_t (&fbn)[TN], uint32_t ra, uint32_t rb, auto Lc, uint32_t stage,
                         int64_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < TM; a++) {
#pragma unroll
            for (int b = 0; b < TN; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[b], a < TS ? fs[a < TS ? a : 0] : fd[a < TS ? 0 : a - TS], acc[a][b], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (a < TS) fs[a < TS ? a : 0] = __builtin_bit_cast(half8_t, *(const uint4_t *)(smem + ra + a * 16 * NT_LDK * 2));
            if (a < TN) fbn[a < TN ? a : 0] = __builtin_bit_cast(half8_t, *(const uint4_t *)(smem + rb + a * 16 * NT_LDK * 2));
            if (a >= TN && a < TN + TD) fdn[a >= TN && a < TN + TD ? a - TN : 0] = __builtin_bit_cast(half8_t, *(const uint4_t *)(smem + ra + (TS + a - TN) * 16 * NT_LDK * 2));
            if (decltype(Lc)::value && a < ACH + BCH) issue_chunk(a, stage, k0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto meet = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); // this wavefront's loads landed, its fragment reads done
        __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<bool, true> with_loads;
    const std::integral_constant<bool, false> no_loads;

#pragma unroll
    for (int c = 0; c < ACH + BCH; c++) issue_chunk(c, lds0, 0);
    meet(); // tile 0
#pragma unroll
    for (int c = 0; c < ACH + BCH; c++) issue_chunk(c, lds0 + STAGE_BYTES, (int64_t)min(1, nk - 1) * NT_BK);
#pragma unroll
    for (int a = 0; a < TS; a++) fs[a] = __builtin_bit_cast(half8_t, *(const uint4_t *)(smem + ra0 + a * 16 * NT_LDK * 2));
#pragma unroll
    for (int a = 0; a < TD; a++) fd0[a] = __builtin_bit_cast(half8_t, *(const uint4_t *)(smem + ra0 + (TS + a) * 16 * NT_LDK * 2));
#pragma unroll
    for (int b = 0; b < TN; b++) fb0[b] = __builtin_bit_cast(half8_t, *(const uint4_t *)(smem + rb0 + b * 16 * NT_LDK * 2));
    uint32_t cur = 0; // stage of tile kt, in bytes
    for (int kt = 0; kt < nk; kt++) {
        half_step(fd0, fb0, fd1, fb1, (ra0 ^ 64u) + cur, (rb0 ^ 64u) + cur, no_loads, 0, 0);
        meet(); // tile kt + 1 is whole, stage `cur` is free
        const uint32_t nxt = STAGE_BYTES - cur;
        // past the last tile: the last one again, into a stage nobody reads from before the loop has ended
        half_step(fd1, fb1, fd0, fb0, ra0 + nxt, rb0 + nxt, with_loads, lds0 + cur, (int64_t)min(kt + 2, nk - 1) * NT_BK);
        cur = nxt;
    }
    meet(); // nothing may land once the epilogue reuses the stages
    nt_epilogue<TM, TN, WM, WN, 2>(g, acc, smem, s, i0, j0, wi, wj, wave, lane);
}

// ---------------------------------------------------------------------------
// Q8_0H x f16.  Four loading wavefronts, one per SIMD, fetch the int8 tile into registers (a lane: 16 codes of
// one row), widen it to f16 (exact) and store f16 code tiles into the ring in the f16 kernel's swizzled layout;
// the activation tile goes global -> LDS directly.  The four multiplying wavefronts run the f16 kernel's
// fragment reads and, per block of 32, one MFMA from zero whose four sums per lane are folded into the
// accumulators with the block's f16 scale two MFMAs later (v_fma_mix: the f16 scale is an operand as it is).
// No weight is rounded.  Two earlier forms: the operand q * d itself, exactly, as the sum of two f16
// (hi = rn(q * d), lo = fma(q, d, -hi)) with two MFMAs per tile into the running accumulator, 64.5 us at
// [512 x 2560] . [10240 x 2560]^T; int8 tiles in LDS, widened by the multiplying wavefronts when they read their
// fragments (50 of their 153 vector instructions per K step), 43.2 us; this one 41.6: what is left is the
// fold, four fused multiply-adds per MFMA, which the multiplying wavefronts cannot hand to anyone.
// Rounding q * d to f16 (the reference's own shader does, ops/gemm.rs:547-548) would remove the fold, and was
// measured: the outputs near zero then miss the 2e-2 tolerance (0.115).  The hi / lo form was built once more on this
// pipeline (the loading wavefronts computing both tiles, two weight stages of hi and lo and four activation stages,
// the multiplying wavefronts issuing MFMAs only): 57.1 us against this kernel's 44.3 in the same harness.  The lo tile
// is subnormal f16 as a rule, which the matrix cores take at full speed (scaled into the normal range it ran the
// same); the form doubles the weight fragments read from LDS and the stores of the loading wavefronts.
//
// Ring of four stages of (BM + BN) x 64 halves.  Loading wavefront, iteration j: request the codes of tile
// j + 3 (registers, set (j + 3) % 4) and its activation rows (LDS-DMA into stage (j + 3) % 4, last read
// before the barrier that ended iteration j - 1); wait for the codes of tile j + 1, requested two
// iterations ago (everything older has landed with them, the activation rows of tile j + 1 included);
// widen and store them into stage (j + 1) % 4; barrier.  Requires K % 256 == 0 (scales in groups of 8).
// ---------------------------------------------------------------------------
template <int BM, int BN, int LW>
__global__ __launch_bounds__(NT_THREADS + 64 * LW) void gemm_nt_q8w_kernel(GemmNtArgs g) {
    constexpr int STAGES = 4, AHEAD = 2;
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 16, TN = WN / 16;
    constexpr int STAGE_HALFS = (BM + BN) * NT_LDK;
    constexpr int NREAD = TM + TN;
    static_assert(BM % 16 == 0 && BN % (8 * LW) == 0, "tile rows must fill whole chunks");
    static_assert(TM * TN >= NREAD, "not enough MFMAs to spread the reads over");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    half_t *ring = (half_t *)smem; // [STAGES][BM + BN][64]
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);

    int64_t ti, tj;
    nt_tile_of(g, blockIdx.x, ti, tj); // XCD-aware tile order (see the file comment)
    const int64_t i0 = ti * BM, j0 = tj * BN;
    const int64_t s = blockIdx.y;
    const int64_t kbase = (int64_t)blockIdx.z * g.k_len; // this workgroup's share of K (all of it without a split)
    const int64_t a_el = (g.a_stack == 1 ? 0 : s) * g.a_bs + kbase, b_el = (g.b_stack == 1 ? 0 : s) * g.b_bs + kbase;
    const int64_t nk = min(g.k_len, g.K - kbase) / NT_BK; // a multiple of 4

    if (wave >= 4) {
        const int lw = wave - 4;
        constexpr int ACH = BM / 16;            // 16-row pieces of the code tile (one load instruction each)
        constexpr int NA = (ACH + LW - 1) / LW; // per loading wavefront
        constexpr int LCHB = BN / 8 / LW;       // 8-row chunks of the activation tile per loading wavefront
        static_assert(AHEAD * (LCHB + NA) < 64, "the wait counter has six bits");
        const uint8_t *ga[NA];
        int adst[NA]; // this lane's row within the code tile
        bool alive[NA];
        const int piece = lane & 3;
#pragma unroll
        for (int c = 0; c < NA; c++) {
            const int ch = lw + c * LW;
            alive[c] = ch < ACH; // wave-uniform
            const int row = min(ch, ACH - 1) * 16 + (lane >> 2);
            ga[c] = (const uint8_t *)g.A + a_el + min(i0 + row, g.M - 1) * g.a_rs + 16 * piece;
            adst[c] = row;
        }
        const half_t *gb[LCHB];
#pragma unroll
        for (int c = 0; c < LCHB; c++) {
            const int row = (lw + c * LW) * 8 + (lane >> 3);
            const int kv = (lane & 7) ^ ((row >> 1) & 7);
            gb[c] = g.B + b_el + min(j0 + row, g.N - 1) * g.b_js + 8 * kv;
        }
        uint4_t ra[STAGES][NA];
        auto request = [&](int slot, int64_t tile) __attribute__((always_inline)) {
            const int64_t k0 = min(tile, nk - 1) * NT_BK; // past the last tile: re-read it, never used
            half_t *st = ring + slot * STAGE_HALFS + BM * NT_LDK;
#pragma unroll
            for (int c = 0; c < LCHB; c++)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(gb[c] + k0),
                                                 (__attribute__((address_space(3))) void *)(st + (lw + c * LW) * 8 * NT_LDK), 16, 0, 0);
            __builtin_amdgcn_sched_barrier(0); // the wait in widen_store counts the loads in this order
#pragma unroll
            for (int c = 0; c < NA; c++) ra[slot][c] = *(const uint4_t *)(ga[c] + k0);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto widen_store = [&](int slot) __attribute__((always_inline)) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0x0F70 | ((AHEAD * (LCHB + NA)) & 0xF) | ((((AHEAD * (LCHB + NA)) >> 4) & 0x3) << 14));
            half_t *st = ring + slot * STAGE_HALFS;
#pragma unroll
            for (int c = 0; c < NA; c++) {
                if (alive[c]) {
                    half2_t h[8];
#pragma unroll
                    for (int d = 0; d < 4; d++) nt_cvt_i8x4(ra[slot][c][d], h[2 * d], h[2 * d + 1]);
                    const uint4_t lo = {__builtin_bit_cast(uint32_t, h[0]), __builtin_bit_cast(uint32_t, h[1]),
                                        __builtin_bit_cast(uint32_t, h[2]), __builtin_bit_cast(uint32_t, h[3])};
                    const uint4_t hi = {__builtin_bit_cast(uint32_t, h[4]), __builtin_bit_cast(uint32_t, h[5]),
                                        __builtin_bit_cast(uint32_t, h[6]), __builtin_bit_cast(uint32_t, h[7])};
                    // the four lanes of a row store four of its eight slots, and two neighbouring rows have the same
                    // swizzle: odd rows store their odd slots first, so that eight consecutive lanes cover eight
                    // different 16-byte bank groups
                    const int flip = adst[c] & 1;
                    *(uint4_t *)(st + nt_slot(adst[c], 2 * piece + flip)) = flip ? hi : lo;
                    *(uint4_t *)(st + nt_slot(adst[c], 2 * piece + 1 - flip)) = flip ? lo : hi;
                }
            }
        };
        auto publish = [&]() __attribute__((always_inline)) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): the widened tile is in LDS
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        request(0, 0);
        request(1, 1);
        request(2, 2);
        widen_store(0);
        publish(); // tile 0
        for (int64_t kg = 0; kg < nk; kg += 4) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                request((u + 3) & 3, kg + u + 3); // into the stage that was read for the last time before the barrier of iteration kg + u - 1
                widen_store((u + 1) & 3);         // tile kg + u + 1
                publish();
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): nothing may land once the epilogue reuses the ring
        __syncthreads();
        return;
    }

    // ---- multiplying wavefronts: the f16 kernel's fragments, the Q8 fold
    const int wi = wave >> 1, wj = wave & 1;
    const int fr = lane & 15, fg = lane >> 4;
    const int swz = (fr >> 1) & 7;
    // this lane's scale rows: 16 bytes = the 8 blocks of four K tiles
    const half_t *sp[TM];
#pragma unroll
    for (int a = 0; a < TM; a++) {
        const int64_t gr = min(i0 + wi * WM + a * 16 + fr, g.M - 1);
        sp[a] = g.scales + ((a_el + gr * g.a_rs) >> 5);
    }
    struct Frags {
        half8_t a[TM], b[TN];
    };
    auto read_one = [&](int stage, int kk, Frags &f, int i) {
        const half_t *as = ring + stage * STAGE_HALFS + (wi * WM + fr) * NT_LDK + (((kk * 4 + fg) ^ swz) << 3);
        const half_t *bs = ring + stage * STAGE_HALFS + BM * NT_LDK + (wj * WN + fr) * NT_LDK + (((kk * 4 + fg) ^ swz) << 3);
        if (i < TM)
            f.a[i] = __builtin_bit_cast(half8_t, *(const uint4_t *)(as + i * 16 * NT_LDK));
        else
            f.b[i - TM] = __builtin_bit_cast(half8_t, *(const uint4_t *)(bs + (i - TM) * 16 * NT_LDK));
    };
    uint4_t sc_cur[TM], sc_nxt[TM];
#pragma unroll
    for (int a = 0; a < TM; a++) sc_cur[a] = *(const uint4_t *)sp[a];
    auto next_tile = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): this tile's fragment reads have returned
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    next_tile(); // tile 0

    Frags r0, r1;
#pragma unroll
    for (int i = 0; i < NREAD; i++) read_one(0, 0, r0, i);
    int cur = 0, nxt = 1;
    auto scale_of = [&](int a, int blk) -> half_t { return __builtin_bit_cast(half8_t, sc_cur[a])[blk]; };
    float accs[TM][TN][4]; // the accumulators as scalars: each is written by a vector instruction of its own
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) accs[a][b][r] = 0.f;
    // One K step (a block of 32): TM * TN MFMAs on the fragments in `rc` from zero, each folded into the
    // accumulators two MFMAs later with the scale of block `blk`; between them the fragment reads of the
    // following K step into `rn`.
    auto k_step = [&](const Frags &rc, Frags &rn, int blk, int rstage, int rkk) {
        const float4_t zero = {0.f, 0.f, 0.f, 0.f};
        float4_t P[3]; // partial sums of three tiles in flight: a tile is folded two MFMAs after its own
        int slot = 0;
#pragma unroll
        for (int idx = 0; idx < TM * TN + 2; idx++) {
            const int a = idx / TN, b = idx % TN;
            if (idx < TM * TN) {
                P[idx % 3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(rc.b[b], rc.a[a], zero, 0, 0, 0);
                asm volatile("" : "+v"(P[idx % 3])); // instruction selection lets results nobody orders float: this MFMA is issued here
                if (slot < NREAD) read_one(rstage, rkk, rn, slot++); // the fragments of the following K step
            }
            if (idx >= 2) {
                const int fa = (idx - 2) / TN, fb = (idx - 2) % TN;
                const float d = (float)scale_of(fa, blk);
#pragma unroll
                for (int r = 0; r < 4; r++) accs[fa][fb][r] = fmaf(d, P[(idx - 2) % 3][r], accs[fa][fb][r]);
                // ... and the sums are folded here, not gathered at the end of the loop body with every partial sum kept alive
                asm volatile("" : "+v"(accs[fa][fb][0]), "+v"(accs[fa][fb][1]), "+v"(accs[fa][fb][2]), "+v"(accs[fa][fb][3]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int64_t kg = 0; kg < nk; kg += 4) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (u == 0) {
                // scales of the next group of four tiles, a group ahead of their use
                const int64_t gn = min(kg + 4, nk - 4) >> 2;
#pragma unroll
                for (int a = 0; a < TM; a++) sc_nxt[a] = *(const uint4_t *)(sp[a] + 8 * gn);
            }
            k_step(r0, r1, 2 * u, cur, 1);
            next_tile();
            k_step(r1, r0, 2 * u + 1, nxt, 0);
            cur = nxt;
            nxt = nxt + 1 == STAGES ? 0 : nxt + 1;
        }
#pragma unroll
        for (int a = 0; a < TM; a++) sc_cur[a] = sc_nxt[a];
    }
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
    __syncthreads();
    float4_t acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = float4_t{accs[a][b][0], accs[a][b][1], accs[a][b][2], accs[a][b][3]};
    nt_epilogue<TM, TN, WM, WN>(g, acc, smem, s, i0, j0, wi, wj, wave, lane);
}

// ---------------------------------------------------------------------------
// Q8_0H x f16 for a K that is not a multiple of 256 (any whole number of blocks): the same division of work, with
//  - the scales of four tiles of K, whose 16 bytes then start at any multiple of two, loaded by the loading wavefronts (a dword-aligned
//    16-byte load, the dword behind it and a shift) and handed over through LDS;
//  - a K that ends in the middle of a tile of 64: loads repeat valid addresses past its end, and the multiplying wavefronts leave
//    the tile's second block out;
//  - 32 x 32 x 16 MFMAs, two chained from zero per block and tile, sixteen sums per lane folded while the next tile's run.
// The register-staged kernel that took these shapes had one tile size and one load in flight: 1373 rows x 1152 x 288 56.9 -> 19.5 us with the
// product behind it, 118 x 3488 x 2592 81.6 -> 20.0, 9 x 5000 x 1504 49.0 -> 10.7, 1633 x 10304 x 1568 with GELU 217 -> 123.
// For K % 256 == 0 the kernel above stays: one 16-byte load per row and four tiles goes straight to the wavefronts that use it
// ([512 x 2560] . [10240 x 2560]^T 46.2 us there, 47.0 with this kernel's form; 300 x 1024 x 1024 9.3 and 10.4).
// What bounds it is what bounds the kernel above: the fold beside the MFMAs, the fill and the LDS traffic add up.
//
// Ring of four stages.  Loading wavefront, iteration j: request tile j + 3 (codes and scales into registers, activation rows by
// LDS-DMA into stage (j + 3) % 4, last read before the barrier that ended iteration j - 1); wait for tile j + 1, requested two
// iterations ago; widen and store its codes into stage (j + 1) % 4; barrier.
// ---------------------------------------------------------------------------
template <int BM, int BN, int WI>
__global__ __launch_bounds__(2 * NT_THREADS) void gemm_nt_q8r_kernel(GemmNtArgs g) {
    constexpr int LW = 4, STAGES = 4, AHEAD = 2;
    constexpr int WJ = 4 / WI, WM = BM / WI, WN = BN / WJ, TM = WM / 32, TN = WN / 32, TILES = TM * TN;
    constexpr int ROW = NT_LDK * 2;                            // bytes of a staged row
    constexpr int STAGE = (BM + BN) * ROW;                     // codes, activations
    constexpr int SCALES = STAGES * STAGE;                     // behind the ring, twice: 16 bytes per row, the eight blocks' scales of four tiles
    static_assert(TM * 32 * WI == BM && TN * 32 * WJ == BN && BN % (8 * LW) == 0 && BM <= 64 * LW, "tile must split into 32 x 32 MFMA tiles and whole chunks");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[]; // [STAGES][STAGE], [2][64 * LW][16]
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    if (wave < 4) __builtin_amdgcn_s_setprio(3); // the multiplying wavefronts: 0.5 % over twelve products, each within 2 %

    int64_t ti, tj;
    nt_tile_of(g, blockIdx.x, ti, tj); // XCD-aware tile order (see the file comment)
    const int64_t i0 = ti * BM, j0 = tj * BN;
    const int64_t s = blockIdx.y;
    const int64_t kbase = (int64_t)blockIdx.z * g.k_len; // this workgroup's share of K (all of it without a split)
    const int64_t a_el = (g.a_stack == 1 ? 0 : s) * g.a_bs + kbase, b_el = (g.b_stack == 1 ? 0 : s) * g.b_bs + kbase;
    const int kn = (int)min(g.k_len, g.K - kbase);        // > 0, a multiple of 32: launcher
    const int nk = (kn + NT_BK - 1) / NT_BK;

    if (wave >= 4) {
        const int lw = wave - 4;
        constexpr int ACH = BM / 16;            // 16-row pieces of the code tile (one load instruction each)
        constexpr int NA = (ACH + LW - 1) / LW; // per loading wavefront
        constexpr int LCHB = BN / 8 / LW;       // 8-row chunks of the activation tile per loading wavefront
        constexpr int NL = LCHB + NA;           // load instructions of a request, without the scales' two
        static_assert(AHEAD * NL + 2 < 64, "the wait counter has six bits");
        const uint8_t *ga[NA];
        int adst[NA]; // this lane's row within the code tile
        bool alive[NA];
        const int piece = lane & 3;
#pragma unroll
        for (int c = 0; c < NA; c++) {
            const int ch = lw + c * LW;
            alive[c] = ch < ACH; // wave-uniform
            const int row = min(ch, ACH - 1) * 16 + (lane >> 2);
            ga[c] = (const uint8_t *)g.A + a_el + min(i0 + row, g.M - 1) * g.a_rs;
            adst[c] = row;
        }
        const half_t *gb[LCHB];
        const int kv = (lane & 7) ^ ((lw * 4 + (lane >> 4)) & 7); // of row (lw + c LW) 8 + lane / 8: the same for every c
#pragma unroll
        for (int c = 0; c < LCHB; c++) gb[c] = g.B + b_el + min(j0 + (lw + c * LW) * 8 + (lane >> 3), g.N - 1) * g.b_js;
        const int srow = lw * 64 + lane; // this lane's row of the scales
        // The scales of four tiles are 16 bytes that start at any multiple of two: a dword-aligned 16-byte load, the dword behind it,
        // and a shift by `off` values.  A row near the end of the stream (padded to 256 bytes) loads the last 16 bytes.
        const int64_t s0 = (a_el + min(i0 + min(srow, BM - 1), g.M - 1) * g.a_rs) >> 5;
        const int64_t s_last = g.scale_dwords - 4;
        uint4_t ra[STAGES][NA];
        uint4_t rs;
        uint32_t rs4;
        int off = 0;
        auto request = [&](int slot, int tile, bool scales) __attribute__((always_inline)) {
            const int k0 = min(tile, nk - 1) * NT_BK; // past the last tile: re-read it, never used ...
            const int to = tile < nk + 3 ? slot : nk & 3; // ... and not stored where the last one is read
            uint8_t *st = smem + to * STAGE + BM * ROW;
            const int kb = min(k0 + 8 * kv, kn - 8), ka = min(k0 + 16 * piece, kn - 16);
#pragma unroll
            for (int c = 0; c < LCHB; c++)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(gb[c] + kb),
                                                 (__attribute__((address_space(3))) void *)(st + (lw + c * LW) * 8 * ROW), 16, 0, 0);
            __builtin_amdgcn_sched_barrier(0); // the wait in widen_store counts whole requests
#pragma unroll
            for (int c = 0; c < NA; c++) ra[slot][c] = *(const uint4_t *)(ga[c] + ka);
            if (scales) { // tile is a multiple of four
                const int64_t at = s0 + (k0 >> 5), dw = min(at >> 1, s_last);
                off = (int)(at - 2 * dw); // 0 .. 7
                rs = *(const uint4_d *)((const uint32_t *)g.scales + dw);
                rs4 = ((const uint32_t *)g.scales)[min(dw + 4, s_last + 3)];
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto widen_store = [&](int slot, auto NEWER, bool scales, int group) __attribute__((always_inline)) { // NEWER: of the two requests behind this tile's, those with scales
            asm volatile("" ::: "memory");
            constexpr int left = AHEAD * NL + 2 * decltype(NEWER)::value;
            __builtin_amdgcn_s_waitcnt(0x0F70 | (left & 0xF) | (((left >> 4) & 0x3) << 14));
            uint8_t *st = smem + slot * STAGE;
#pragma unroll
            for (int c = 0; c < NA; c++) {
                if (alive[c]) {
                    half2_t h[8];
#pragma unroll
                    for (int d = 0; d < 4; d++) nt_cvt_i8x4(ra[slot][c][d], h[2 * d], h[2 * d + 1]);
                    const uint4_t lo = {__builtin_bit_cast(uint32_t, h[0]), __builtin_bit_cast(uint32_t, h[1]),
                                        __builtin_bit_cast(uint32_t, h[2]), __builtin_bit_cast(uint32_t, h[3])};
                    const uint4_t hi = {__builtin_bit_cast(uint32_t, h[4]), __builtin_bit_cast(uint32_t, h[5]),
                                        __builtin_bit_cast(uint32_t, h[6]), __builtin_bit_cast(uint32_t, h[7])};
                    // the four lanes of a row store four of its eight slots, and two neighbouring rows have the same
                    // swizzle: odd rows store their odd slots first, so that eight consecutive lanes cover eight
                    // different 16-byte bank groups
                    const int flip = adst[c] & 1;
                    *(uint4_t *)((half_t *)st + nt_slot(adst[c], 2 * piece + flip)) = flip ? hi : lo;
                    *(uint4_t *)((half_t *)st + nt_slot(adst[c], 2 * piece + 1 - flip)) = flip ? lo : hi;
                }
            }
            if (scales) {
                uint4_t v = rs;
                uint32_t w = rs4;
                if (off & 4) v = uint4_t{v[2], v[3], w, w}, w = 0;
                if (off & 2) v = uint4_t{v[1], v[2], v[3], w}, w = 0;
                const uint32_t sh = (uint32_t)(off & 1) << 4;
                v = uint4_t{__builtin_amdgcn_alignbit(v[1], v[0], sh), __builtin_amdgcn_alignbit(v[2], v[1], sh), __builtin_amdgcn_alignbit(v[3], v[2], sh),
                            __builtin_amdgcn_alignbit(w, v[3], sh)};
                *(uint4_t *)(smem + SCALES + (group & 1) * (64 * LW * 16) + 16 * srow) = v;
            }
        };
        auto publish = [&](bool meet) __attribute__((always_inline)) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): the widened tile is in LDS
            if (meet) __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        request(0, 0, true);
        request(1, 1, false);
        request(2, 2, false);
        widen_store(0, std::integral_constant<int, 0>{}, true, 0);
        publish(true); // tile 0
        auto iteration = [&](auto U, int j) __attribute__((always_inline)) { // U: j % 4
            constexpr int u = decltype(U)::value;
            request((u + 3) & 3, j + 3, u == 1); // into the stage that was read for the last time before the barrier of iteration j - 1
            widen_store((u + 1) & 3, std::integral_constant<int, u == 1 || u == 2>{}, u == 3, (j + 1) >> 2); // tile j + 1
            publish(j + 1 < nk);
        };
        const std::integral_constant<int, 0> u0;
        const std::integral_constant<int, 1> u1;
        const std::integral_constant<int, 2> u2;
        const std::integral_constant<int, 3> u3;
        // nk - 1 iterations, and up to three more without a barrier that nobody waits for but the end: whole turns of the ring without
        // a way out or around in between, with which the compiler drains every load
        for (int j = 0; j + 1 < nk; j += 4) iteration(u0, j), iteration(u1, j + 1), iteration(u2, j + 2), iteration(u3, j + 3);
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): nothing may land once the epilogue reuses the ring
        __syncthreads();
        return;
    }

    // ---- multiplying wavefronts
    const int wi = wave / WJ, wj = wave % WJ;
    const int fr = lane & 31, fh = lane >> 5;
    // 16 k of a row (half m of block kk) are K-vectors 4 kk + 2 m, + 1: this lane's is 4 kk + 2 m + fh.  Byte addresses of this lane's
    // first fragments in stage 0 for m = kk = 0; m flips bit 5 of them, kk bit 6.
    const uint32_t slot = (uint32_t)((fh ^ ((fr >> 1) & 7)) << 4);
    const uint32_t ra0 = (uint32_t)(wi * WM + fr) * ROW + slot, rb0 = (uint32_t)(BM + wj * WN + fr) * ROW + slot;
    const uint32_t rs0 = (uint32_t)(SCALES + (wi * WM + fr) * 16);
    auto frag = [&](uint32_t at) __attribute__((always_inline)) { return __builtin_bit_cast(half8_t, *(const uint4_t *)(smem + at)); };
    auto next_tile = [&]() __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): this tile's fragment reads have returned
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const float16_t zero = {};
    float16_t acc[TM][TN], P[2];
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++) acc[a][b] = zero;
    half8_t fa[TM][2], fb[2][TN][2];
    half2_t sc[TM], last = {(half_t)0.f, (half_t)0.f}; // scales of this tile's two blocks; of the tile before, its last rows'
    P[0] = P[1] = zero;
    next_tile(); // tile 0
#pragma unroll
    for (int a = 0; a < TM; a++) {
        fa[a][0] = frag(ra0 + a * 32 * ROW), fa[a][1] = frag((ra0 ^ 32u) + a * 32 * ROW);
        sc[a] = *(const half2_t *)(smem + rs0 + a * 512);
    }
#pragma unroll
    for (int b = 0; b < TN; b++) fb[0][b][0] = frag(rb0 + b * 32 * ROW), fb[0][b][1] = frag((rb0 ^ 32u) + b * 32 * ROW);

    // One block of 32: per MFMA tile two MFMAs, then the fold of the tile before.  The next block's fragments are read from `ra`, `rb`
    // behind their registers' last use (the activations', which all tiles of a column share, into a second set).
    auto block = [&](auto KK, uint32_t ra, uint32_t rb, uint32_t rs) __attribute__((always_inline)) {
        constexpr int kk = decltype(KK)::value;
#pragma unroll
        for (int idx = 0; idx < TILES; idx++) {
            const int a = idx / TN, b = idx % TN, p = (kk * TILES + idx) & 1;
            const int pa = idx ? (idx - 1) / TN : TM - 1, pb = idx ? (idx - 1) % TN : TN - 1;
            P[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[kk][b][0], fa[a][0], zero, 0, 0, 0);
            P[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[kk][b][1], fa[a][1], P[p], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (b == TN - 1) fa[a][0] = frag(ra + a * 32 * ROW), fa[a][1] = frag((ra ^ 32u) + a * 32 * ROW);
            if (idx < TN) fb[kk ^ 1][idx][0] = frag(rb + idx * 32 * ROW), fb[kk ^ 1][idx][1] = frag((rb ^ 32u) + idx * 32 * ROW);
            const float d = (float)(idx == 0 ? (kk ? sc[pa][0] : last[1]) : sc[pa][kk]);
#pragma unroll
            for (int r = 0; r < 16; r++) acc[pa][pb][r] = fmaf(d, P[p ^ 1][r], acc[pa][pb][r]);
            if (kk && idx && pb == TN - 1) sc[pa] = *(const half2_t *)(smem + rs + pa * 512);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (kk) last = sc[TM - 1], sc[TM - 1] = *(const half2_t *)(smem + rs + (TM - 1) * 512);
    };
    const std::integral_constant<int, 0> first_block;
    const std::integral_constant<int, 1> second_block;
    uint32_t cur = 0; // stage of tile kt, in bytes
    const bool half = kn % NT_BK != 0;
    for (int kt = 0; kt + 1 < nk; kt++) {
        block(first_block, (ra0 ^ 64u) + cur, (rb0 ^ 64u) + cur, 0);
        next_tile(); // tile kt + 1 is whole, stage `cur` is free
        cur = cur == (STAGES - 1) * STAGE ? 0 : cur + STAGE;
        block(second_block, ra0 + cur, rb0 + cur, rs0 + ((kt + 1) & 3) * 4 + ((kt + 1) >> 2 & 1) * (64 * LW * 16));
    }
    block(first_block, (ra0 ^ 64u) + cur, (rb0 ^ 64u) + cur, 0);
    if (!half) block(second_block, ra0 + cur, rb0 + cur, rs0); // (what it reads ahead is not used)
    {
        // the last tile's sums: of the second block, or of the first where K ends with it
        const float d = (float)(half ? sc[TM - 1][0] : last[1]);
        constexpr int p0 = (TILES - 1) & 1, p1 = (2 * TILES - 1) & 1;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[TM - 1][TN - 1][r] = fmaf(d, half ? P[p0][r] : P[p1][r], acc[TM - 1][TN - 1][r]);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __syncthreads();
    nt_epilogue32<TM, TN, WM, WN>(g, acc, smem, s, i0, j0, wi, wj, wave, lane);
}

// Second pass of a split-K launch: out = round(act(sum over the splits + bias)).  One thread per four
// consecutive i (the partial sums' contiguous axis); M need not be a multiple of four.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(GemmNtArgs g) {
    const int64_t s = blockIdx.y;
    const int64_t mq = (g.M + 3) >> 2, total = mq * g.N;
    const float *pt = g.partial + s * g.ksplit * g.N * g.M;
    const int64_t sstride = g.N * g.M;
    half_t *out = g.out + s * g.o_bs;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = idx / mq, i = (idx - j * mq) << 2;
        const int n = (int)min<int64_t>(4, g.M - i);
        // a row's last values end a group of four that begins in front of theirs: whole loads, at any multiple of four bytes
        // (value by value Q4_K 62 rows x 1059 x 7680 in 15 shares took 20.2 us for both kernels, 12.7 so; 323 x 1149 x 3072 in four 18.1 and 16.0)
        const int back = 4 - n;
        const float *src = pt + j * g.M + i - back;
        float4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int sp = 0; sp < g.ksplit; sp++) sum += *(const float4_d *)(src + sp * sstride);
        const float v[4] = {back & 2 ? (back & 1 ? sum[3] : sum[2]) : back ? sum[1] : sum[0], back & 2 ? sum[3] : back ? sum[2] : sum[1], back ? sum[3] : sum[2], sum[3]};
        half_t r[4];
        for (int e = 0; e < 4; e++) {
            float t = v[e];
            if (g.has_bias && e < n) t += (float)g.bias[g.bias_on_rows ? i + e : j];
            r[e] = (half_t)rt_act(t, g.act);
        }
        half_t *dst = out + i * g.o_is + j * g.o_js;
        if (n == 4 && g.vec_epilogue) {
            *(uint2_t *)dst = __builtin_bit_cast(uint2_t, half4_t{r[0], r[1], r[2], r[3]});
        } else {
            for (int e = 0; e < n; e++) dst[e * g.o_is] = r[e];
        }
    }
}

static hipError_t launch_splitk_reduce(const GemmNtArgs &g, int64_t stacks, hipStream_t st) {
    const int64_t total = ((g.M + 3) >> 2) * g.N;
    const unsigned gx = (unsigned)((total + 255) / 256 > 8192 ? 8192 : (total + 255) / 256);
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3(gx, (unsigned)stacks), dim3(256), 0, st, g);
    return hipGetLastError();
}

// The second pass for another file's kernel that left f32 sums of `ks` shares of problem p in `partial` [stack][share][N][M].
hipError_t launch_splitk_sums(const Problem &p, const void *bias, void *out, float *partial, int ks, hipStream_t st) {
    GemmNtArgs g{};
    g.bias = (const half_t *)bias, g.out = (half_t *)out, g.partial = partial, g.ksplit = ks;
    g.M = p.M, g.N = p.N;
    g.o_bs = p.o_bs, g.o_is = p.o_is, g.o_js = p.o_js;
    g.has_bias = p.has_bias, g.bias_on_rows = p.bias_on_rows, g.act = p.act;
    g.vec_epilogue = p.o_is == 1 && p.o_js % 8 == 0 && p.o_bs % 8 == 0 && ((uintptr_t)out & 15u) == 0;
    return launch_splitk_reduce(g, p.stacks, st);
}

template <int BM, int BN, int LW>
static hipError_t launch_nt_q8w(const GemmNtArgs &g, int64_t stacks, hipStream_t st) {
    const size_t lds = (size_t)4 * (BM + BN) * NT_LDK * 2;
    if (const hipError_t e = ensure_lds_limit<&gemm_nt_q8w_kernel<BM, BN, LW>>(); e != hipSuccess) return e;
    dim3 grid((unsigned)((int64_t)g.tiles_i * g.tiles_j), (unsigned)stacks, (unsigned)g.ksplit);
    hipLaunchKernelGGL((gemm_nt_q8w_kernel<BM, BN, LW>), grid, dim3(NT_THREADS + 64 * LW), lds, st, g);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return g.ksplit > 1 ? launch_splitk_reduce(g, stacks, st) : hipSuccess;
}

template <int BM, int BN, int WI>
static hipError_t launch_nt_q8r(const GemmNtArgs &g, int64_t stacks, hipStream_t st) {
    const size_t lds = (size_t)4 * (BM + BN) * NT_LDK * 2 + 2 * 256 * 16;
    if (const hipError_t e = ensure_lds_limit<&gemm_nt_q8r_kernel<BM, BN, WI>>(); e != hipSuccess) return e;
    dim3 grid((unsigned)((int64_t)g.tiles_i * g.tiles_j), (unsigned)stacks, (unsigned)g.ksplit);
    hipLaunchKernelGGL((gemm_nt_q8r_kernel<BM, BN, WI>), grid, dim3(2 * NT_THREADS), lds, st, g);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return g.ksplit > 1 ? launch_splitk_reduce(g, stacks, st) : hipSuccess;
}

// ---------------------------------------------------------------------------
// Short contractions (K <= 128: attention scores).  Such a product is a stream: the time
// goes into reading the operands once and writing the output.  A workgroup keeps a strip of
// 64 B rows (all of K) resident in LDS and walks the A row tiles of 128; the tile for step
// t+1 is prefetched into registers while step t is multiplied, and each wavefront stages and
// writes its own part of the output, so the stores of one step overlap the loads and MFMAs
// of the next.  K is padded with zeros to a multiple of 32 inside LDS only.
// PAIRS: output rows that start on 4 bytes and not on 16 (an even number of keys) leave as consecutive pairs (nt_epilogue_pairs).
// Scores of 32 heads x 300 x 300, 16 x 254 x 254, 6 x 964 x 964: 8.9 / 7.3 / 11.1 us on gemm_nt_kernel with its stores of
// sixteen values to each of four rows -> 6.9 / 5.6 / 10.3.  An odd number of keys stays there: single values in this kernel's order
// gain up to some 400 keys (401: 7.2 -> 6.2) and lose beyond (1027: 13.2 -> 16.1).
// ---------------------------------------------------------------------------
template <int KP, bool PAIRS>
__global__ __launch_bounds__(NT_THREADS, 2) void gemm_nt_shortk_kernel(GemmNtArgs g) {
    constexpr int BM = 128, BN = 64, WM = 64, WN = 32, TM = 4, TN = 2;
    constexpr int LDK = KP + 8;  // halfs per LDS row: an odd number of 16-byte slots, conflict-free fragment reads
    constexpr int KPV = KP / 8;  // 16-byte vectors per padded row
    constexpr int A_VEC = BM * KPV / NT_THREADS, B_VEC = BN * KPV / NT_THREADS;
    static_assert(KP % 32 == 0 && (BM * KPV) % NT_THREADS == 0 && (BN * KPV) % NT_THREADS == 0, "tile / thread split");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    half_t *Bs = (half_t *)smem;            // [BN][LDK]
    half_t *As = Bs + BN * LDK;             // [BM][LDK]
    uint8_t *Es = (uint8_t *)(As + BM * LDK); // per-wavefront output staging

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wi = wave >> 1, wj = wave & 1;
    const int fr = lane & 15, fg = lane >> 4;
    // Workgroups go to the eight XCDs round-robin by their linear number.  Taken as it comes, the strips of one stack
    // land on all eight and every L2 fetches that stack's operands (3 x the operand bytes at 32 x [512 x 80] . [512 x 80]^T);
    // when the grid divides by eight, XCD x takes the x-th eighth of the (stack, strip, part) items instead.
    uint32_t bx = blockIdx.x, by = blockIdx.y;
    if (const uint64_t total64 = (uint64_t)gridDim.x * gridDim.y; total64 < (1u << 31) && (total64 & 7u) == 0) {
        const uint32_t total = (uint32_t)total64;
        const uint32_t lin = blockIdx.x + gridDim.x * blockIdx.y, w = (lin & 7u) * (total >> 3) + (lin >> 3);
        by = w / gridDim.x, bx = w - by * gridDim.x;
    }
    // bx = strip * parts + part: the workgroups of a strip take its A tiles round-robin
    const int parts = g.tiles_i, part = (int)(bx % parts);
    const int64_t j0 = (int64_t)(bx / parts) * BN;
    const int64_t s = by;
    const int64_t a_el = (g.a_stack == 1 ? 0 : s) * g.a_bs, b_el = (g.b_stack == 1 ? 0 : s) * g.b_bs;
    const int kvecs = (int)(g.K >> 3);
    const uint4_t zero4 = {0u, 0u, 0u, 0u};

    // the B strip: global -> registers -> LDS, vectors past K zeroed
    {
        uint4_t rb[B_VEC];
#pragma unroll
        for (int e = 0; e < B_VEC; e++) {
            const int v = e * NT_THREADS + t, r = v / KPV, c = v - r * KPV;
            const int64_t gr = min(j0 + r, g.N - 1);
            rb[e] = *(const uint4_t *)(g.B + b_el + gr * g.b_js + 8 * min(c, kvecs - 1));
        }
#pragma unroll
        for (int e = 0; e < B_VEC; e++) {
            const int v = e * NT_THREADS + t, r = v / KPV, c = v - r * KPV;
            *(uint4_t *)(Bs + r * LDK + 8 * c) = c < kvecs ? rb[e] : zero4;
        }
    }
    uint4_t ra[A_VEC];
    auto load_a = [&](int64_t i0) {
#pragma unroll
        for (int e = 0; e < A_VEC; e++) {
            const int v = e * NT_THREADS + t, r = v / KPV, c = v - r * KPV;
            const int64_t gr = min(i0 + r, g.M - 1); // rows past the end duplicate the last one; never stored
            ra[e] = *(const uint4_t *)((const half_t *)g.A + a_el + gr * g.a_rs + 8 * min(c, kvecs - 1));
        }
    };
    auto store_a = [&]() {
#pragma unroll
        for (int e = 0; e < A_VEC; e++) {
            const int v = e * NT_THREADS + t, r = v / KPV, c = v - r * KPV;
            *(uint4_t *)(As + r * LDK + 8 * c) = c < kvecs ? ra[e] : zero4;
        }
    };
    const int64_t ntile = (g.M + BM - 1) / BM;
    load_a((int64_t)part * BM);
    for (int64_t it = part; it < ntile; it += parts) {
        store_a();
        __syncthreads();
        if (it + parts < ntile) load_a((it + parts) * BM); // in flight under the MFMAs and the output stage
        float4_t acc[TM][TN];
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
            for (int b = 0; b < TN; b++) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KP / 32; kk++) {
            half8_t fa[TM], fb[TN];
#pragma unroll
            for (int a = 0; a < TM; a++)
                fa[a] = __builtin_bit_cast(half8_t, *(const uint4_t *)(As + (wi * WM + a * 16 + fr) * LDK + kk * 32 + 8 * fg));
#pragma unroll
            for (int b = 0; b < TN; b++)
                fb[b] = __builtin_bit_cast(half8_t, *(const uint4_t *)(Bs + (wj * WN + b * 16 + fr) * LDK + kk * 32 + 8 * fg));
#pragma unroll
            for (int a = 0; a < TM; a++)
#pragma unroll
                for (int b = 0; b < TN; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[b], fa[a], acc[a][b], 0, 0, 0);
        }
        __syncthreads(); // every wavefront is done with As before the next tile overwrites it
        if constexpr (PAIRS) nt_epilogue_pairs<TM, TN, WM, WN>(g, acc, Es, s, it * BM, j0, wi, wj, wave, lane);
        else nt_epilogue<TM, TN, WM, WN>(g, acc, Es, s, it * BM, j0, wi, wj, wave, lane);
    }
}

// g.tiles_i carries the number of workgroups that share a strip.
template <int KP> static hipError_t launch_nt_shortk(const GemmNtArgs &g, int64_t stacks, hipStream_t st) {
    const size_t lds = (size_t)(64 + 128) * (KP + 8) * 2 + (size_t)4 * 32 * (64 + 8) * 2;
    dim3 grid((unsigned)((g.N + 63) / 64 * g.tiles_i), (unsigned)stacks);
    if (g.vec_epilogue) {
        if (const hipError_t e = ensure_lds_limit<&gemm_nt_shortk_kernel<KP, false>>(); e != hipSuccess) return e;
        hipLaunchKernelGGL((gemm_nt_shortk_kernel<KP, false>), grid, dim3(NT_THREADS), lds, st, g);
    } else {
        if (const hipError_t e = ensure_lds_limit<&gemm_nt_shortk_kernel<KP, true>>(); e != hipSuccess) return e;
        hipLaunchKernelGGL((gemm_nt_shortk_kernel<KP, true>), grid, dim3(NT_THREADS), lds, st, g);
    }
    return hipGetLastError();
}

template <int BM, int BN, int STAGES, int LW, bool TAIL>
static hipError_t launch_nt_dl_as(const GemmNtArgs &g, int64_t stacks, hipStream_t st) {
    const size_t lds = (size_t)STAGES * (BM + BN) * NT_LDK * 2;
    if (const hipError_t e = ensure_lds_limit<&gemm_nt_dl_kernel<BM, BN, STAGES, LW, TAIL>>(); e != hipSuccess) return e;
    dim3 grid((unsigned)((int64_t)g.tiles_i * g.tiles_j), (unsigned)stacks, (unsigned)g.ksplit);
    hipLaunchKernelGGL((gemm_nt_dl_kernel<BM, BN, STAGES, LW, TAIL>), grid, dim3(NT_THREADS + 64 * LW), lds, st, g);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return g.ksplit > 1 ? launch_splitk_reduce(g, stacks, st) : hipSuccess;
}

template <int BM, int BN, int STAGES, int LW>
static hipError_t launch_nt_dl(const GemmNtArgs &g, int64_t stacks, hipStream_t st) {
    return g.K % NT_BK ? launch_nt_dl_as<BM, BN, STAGES, LW, true>(g, stacks, st) : launch_nt_dl_as<BM, BN, STAGES, LW, false>(g, stacks, st);
}

static hipError_t launch_nt_wide(const GemmNtArgs &g, int64_t stacks, hipStream_t st) {
    constexpr int BM = 320, BN = 256;
    const size_t lds = (size_t)2 * (BM + BN) * NT_LDK * 2;
    if (const hipError_t e = ensure_lds_limit<&gemm_nt_wide_kernel<BM, BN, 2, 4>>(); e != hipSuccess) return e;
    dim3 grid((unsigned)((int64_t)g.tiles_i * g.tiles_j), (unsigned)stacks);
    hipLaunchKernelGGL((gemm_nt_wide_kernel<BM, BN, 2, 4>), grid, dim3(512), lds, st, g);
    return hipGetLastError();
}

// Tunable: non-zero keeps f16 problems on the register-staged kernel (for comparisons).
RT_TUNABLE(g_gemm_nt_no_direct, 0);
RT_TUNABLE(g_gemm_nt_wide, 0); // 1 / 2: never / always the 320 x 256 tiles (for comparisons)
RT_TUNABLE(g_gemm_nt_shortk_parts, 0); // workgroups per strip of the short-K kernel (0 = automatic)

template <int BM, int BN, bool KFULL>
static hipError_t launch_nt(const GemmNtArgs &g, int64_t stacks, hipStream_t st) {
    const size_t lds = (size_t)2 * (BM + BN) * NT_LDK * 2;
    if (const hipError_t e = ensure_lds_limit<&gemm_nt_kernel<BM, BN, KFULL>>(); e != hipSuccess) return e;
    dim3 grid((unsigned)((int64_t)g.tiles_i * g.tiles_j), (unsigned)stacks);
    hipLaunchKernelGGL((gemm_nt_kernel<BM, BN, KFULL>), grid, dim3(NT_THREADS), lds, st, g);
    return hipGetLastError();
}

// The grid of bm x bn tiles and the order its workgroups take them in.  An XCD's share of the tiles is either a block of
// (tiles_i / xi) x (tiles_j xi / 8) where the grid can be cut that way, or the x-th eighth of them in row-major order;
// of the possible ones, the one whose resident workgroups (up to 32) load the fewest bytes of operands per K step that
// their L2 does not hold already: for [2048 x 10240] . [2560 x 10240]^T (16 x 16 tiles) four row blocks and eight column
// blocks per XCD instead of two and sixteen; for 11008 x 4096 weights against 1000 rows (69 x 8 tiles) the
// plain eighths, nine row blocks by eight columns, where the only cut has 69 row blocks of one column (115.9 and
// 107.8 us; 8192 x 3072 against 200 rows, 52 x 2 tiles, K shared: 27.7 and 23.9).  a_bytes: of an element of A (the
// codes' one for Q8_0H).
static bool nt_set_tiles(GemmNtArgs &g, int bm, int bn, int a_bytes) {
    const int64_t ti = (g.M + bm - 1) / bm, tj = (g.N + bn - 1) / bn;
    if (ti * tj > 0x7fffffff) return false;
    g.tiles_i = (int)ti, g.tiles_j = (int)tj;
    g.xi = 0, g.pj = 1;
    const int64_t res = std::min<int64_t>(32, (ti * tj + 7) / 8); // workgroups resident on an XCD
    // the plain order: a share that is not whole rows of tiles begins in the middle of one
    int64_t least = ((res + tj - 1) / tj + ((ti * tj / 8) % tj ? 1 : 0)) * bm * a_bytes + std::min(tj, res) * bn * 2;
    for (int xi = 8; xi >= 1; xi /= 2) {
        const int xj = 8 / xi;
        if (ti % xi || tj % xj) continue;
        const int64_t rows = ti / xi, cols = tj / xj;
        // panels of four columns, wider when the block has too few rows to give 32 workgroups eight of them
        const int64_t pj = std::min(cols, std::max<int64_t>(4, 32 / rows));
        const int64_t cost = std::min<int64_t>(rows, (res + pj - 1) / pj) * bm * a_bytes + pj * bn * 2;
        if (cost < least) g.xi = xi, g.pj = (int)pj, least = cost;
    }
    if (g.xi) {
        g.xj_log2 = g.xi == 8 ? 0 : g.xi == 4 ? 1 : g.xi == 2 ? 2 : 3;
        g.rows = g.tiles_i / g.xi, g.cols = g.tiles_j >> g.xj_log2, g.panels = (g.cols + g.pj - 1) / g.pj;
    }
    return true;
}

// Tunable: 0 = automatic, 1 = never take this kernel (for comparisons).
RT_TUNABLE(g_gemm_nt_disable, 0);

// The tiles of the kernels that load global -> LDS and how K is shared among workgroups: the cheapest by an estimate in microseconds,
//   3 + rounds * (fixed - 3 + step * (1 + crowd * busy) * tiles of 64 k in a share) + the second kernel's time,
// busy the share of the compute units that has a workgroup.  The constants are a fit to the tiles and splits of 166 f16 and 176 Q8_0H
// products on the device (200 to 12000 x 9 to 1500, K from 96 to 14336), each with the weights in the caches and from HBM: the choice is 0.4 and 0.2 %
// above the best one on average, 16 and 7 % at worst.  (Fitted to few products with the weights in the caches, 128 x 128 tiles of f16 came out ahead of
// 96 x 128 ones that are faster either way: 9901 x 253 x 3840 45.7 and 41.3 us, 2229 x 943 x 3840 37.5 and 31.4.)  The largest tile alone, cut along K where
// it left half of the compute units idle, was the rule before: [512 x 2560] . [2560 x 2560]^T Q8_0H 30.2 -> 17.7 us (64 x 128 tiles,
// K whole), [512 x 2560] . [7680 x 2560]^T 43 -> 34.7 (128 x 128), 128 rows x 2560 x 2560 25.1 -> 12.7 (64 x 64, K in three),
// 1000 x 4096 x 4096 65.6 -> 52.8; f16 30 -> 15.9 of the first kind, [700 x 1280] . [5120 x 1280]^T 17.3 -> 14.9.
struct NtTile {
    int bm, bn;
    float fixed, step;
};
constexpr int kNtTiles = 5;
constexpr NtTile kTilesF16[kNtTiles] = {{160, 128, 8.6f, 0.415f}, {128, 128, 8.6f, 0.32f}, {96, 128, 7.2f, 0.285f}, {64, 128, 7.2f, 0.195f}, {64, 64, 4.5f, 0.137f}};
constexpr NtTile kTilesQ8w[kNtTiles] = {{160, 128, 8.6f, 0.69f}, {128, 128, 7.6f, 0.47f}, {96, 128, 7.5f, 0.417f}, {64, 128, 7.2f, 0.255f}, {64, 64, 5.7f, 0.185f}};
constexpr NtTile kTilesQ8r[kNtTiles] = {{160, 128, 8.2f, 0.70f}, {128, 128, 9.2f, 0.43f}, {96, 128, 7.7f, 0.427f}, {64, 128, 7.3f, 0.295f}, {64, 64, 6.7f, 0.222f}};
struct NtChoice {
    int bm = 160, bn = 128;
    int ks = 1;        // workgroups that share one tile's K
    int64_t k_len = 0; // of a share; the last may be shorter
};
// gemm_nt_q8w_kernel's shapes among those with Q8_0H weights
static bool nt_q8_whole(const Problem &p) { return p.K % 256 == 0 && p.a_bs % 512 == 0; }
static NtChoice nt_choose(const Problem &p, const DeviceInfo &dev, bool may_split) {
    const bool q8 = p.a_dt == RT_Q8_0H;
    const NtTile *tiles = !q8 ? kTilesF16 : nt_q8_whole(p) ? kTilesQ8w : kTilesQ8r;
    const float crowd = q8 ? 0.23f : 0.37f, pass = q8 ? 1.7f : 2.4f;
    const int64_t nk = (p.K + NT_BK - 1) / NT_BK;
    NtChoice best;
    best.k_len = p.K;
    float least = 3.4e38f;
    for (int i = 0; i < kNtTiles; i++) {
        const NtTile &t = tiles[i];
        const int64_t n = ((p.M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn) * p.stacks;
        if (t.bm < 128 && n > dev.num_cus) continue; // narrow tiles only where they all run at once
        for (int ks = 1; ks <= (may_split ? 16 : 1); ks++) {
            if (ks > 1 && n * ks > dev.num_cus) break; // the partial sums stay within 256 of the largest tiles on 256 compute units
            // Where K is whole units of 256 so are the shares (gemm_nt_q8w_kernel's have to be): equal ones of whole 512s or of at least 1024, and from
            // K = 2560 on of at least 1024 with a shorter last one (below, the smaller of two shares is hardly worth the second kernel).  Else
            // shares of at least 512, the last one shorter.  (Equal ones alone left a K of 17 or 43 units whole, and 56 of them on 70 tiles in two:
            // 4480 rows Q8_0H at 32, K = 4352 / 11008 / 14336 22.7 / 51 / 39.5 us and in three shares 15.3 / 26.4 / 31.2.)
            const bool whole = p.K % 256 == 0;
            const int64_t unit = whole ? 4 : 1, share = ((nk + ks - 1) / ks + unit - 1) / unit * unit;
            if (ks > 1 && (share < (whole && p.K % (512 * ks) != 0 ? 16 : 8) || (ks - 1) * share >= nk)) continue;
            if (ks > 1 && whole && p.K < 2560 && p.K % (256 * ks) != 0) continue;
            const int64_t rounds = (n * ks + dev.num_cus - 1) / dev.num_cus;
            const float busy = std::min(1.f, (float)(n * ks) / dev.num_cus);
            const float second = ks == 1 ? 0.f : pass + 0.1f * ks + (float)(p.stacks * ks * p.M * p.N) * (4.f / 4.5e6f);
            const float us = 3.f + rounds * (t.fixed - 3.f + t.step * (1.f + crowd * busy) * share) + second;
            if (us < least) least = us, best.bm = t.bm, best.bn = t.bn, best.ks = ks, best.k_len = ks == 1 ? p.K : share * NT_BK;
        }
    }
    return best;
}

// exchanges the operands' roles when that makes the output's contiguous axis the kernel's i axis
static bool nt_orient(Problem &p) {
    if (p.a_dt == RT_F16 && p.act_dt == RT_F16 && p.o_js == 1 && p.o_is != 1) {
        std::swap(p.M, p.N);
        std::swap(p.a_stack, p.b_stack);
        std::swap(p.a_bs, p.b_bs);
        std::swap(p.a_rs, p.b_js);
        std::swap(p.a_ks, p.b_ks);
        std::swap(p.o_is, p.o_js);
        p.bias_on_rows = !p.bias_on_rows;
        return true;
    }
    return false;
}

// bytes of workspace with which launch_gemm_nt splits this problem's K (0: it does not)
uint64_t gemm_nt_workspace_bytes(const Problem &p0, const DeviceInfo &dev) {
    Problem p = p0;
    nt_orient(p);
    if (p.a_ks != 1 || p.b_ks != 1 || p.M < 160 || p.N < 5) return 0;
    if ((p.a_dt != RT_F16 && p.a_dt != RT_Q8_0H) || p.K % 32 != 0 || p.K <= 256) return 0;
    const int ks = nt_choose(p, dev, true).ks;
    return ks > 1 ? (uint64_t)p.stacks * ks * p.M * p.N * sizeof(float) : 0;
}

// Whether rt_matmul_enqueue_static may share this product's K, on the one buffer that all its calls on a GPU have in common.  A program
// may have products in flight on several streams there that never touched it, so the products are those that it has always been for:
// K whole units of 256, at most half a compute unit per 160 x 128 tile, and equal shares of at least 1024.
bool gemm_nt_static_split(const Problem &p0, const DeviceInfo &dev) {
    Problem p = p0;
    nt_orient(p);
    if ((p.a_dt != RT_F16 && p.a_dt != RT_Q8_0H) || p.K % 256 != 0) return false;
    const int64_t tiles = ((p.M + 159) / 160) * ((p.N + 127) / 128) * p.stacks, units = p.K / 256;
    if (tiles <= 0 || tiles * 2 > dev.num_cus) return false;
    for (int ks = 2; ks <= 8 && tiles * ks <= dev.num_cus; ks++)
        if (units % ks == 0 && units / ks >= 4) return true;
    return false;
}

hipError_t launch_gemm_nt(const Problem &p0, const void *A, const void *B, const void *bias, void *out,
                          hipStream_t stream, const DeviceInfo &dev) {
    if (g_gemm_nt_disable) return hipErrorNotSupported;
    Problem p = p0;
    // Row-major output: compute the transposed product (operands exchanged), so that the
    // kernel's contiguous output axis, the one its 128-bit epilogue writes along, is this
    // problem's column axis.
    if (nt_orient(p)) std::swap(A, B);
    if (p.act_dt != RT_F16 || (p.a_dt != RT_F16 && p.a_dt != RT_Q8_0H)) return hipErrorNotSupported;
    if (p.a_ks != 1 || p.b_ks != 1 || p.K % 8 != 0 || p.K < 8) return hipErrorNotSupported;
    if (p.stacks > 65535 || p.M < 1 || p.N < 1) return hipErrorNotSupported;
    const bool q8 = p.a_dt == RT_Q8_0H;
    if (((uintptr_t)A & 15u) || ((uintptr_t)B & 15u) || (p.b_js * 2) % 16 || (p.b_bs * 2) % 16) return hipErrorNotSupported;
    if (q8 ? (p.K % 32 != 0) : ((p.a_rs * 2) % 16 != 0 || (p.a_bs * 2) % 16 != 0)) return hipErrorNotSupported;
    // small problems do not fill the tiles; the generic kernel handles them (at 10240 x 2560 f16 weights it takes
    // 19.7 us for 8 activation rows and 33 us for 16..48, the 64-row tiles here 17.4 us for any count up to 64)
    if (p.M < 160 || p.N < 5) return hipErrorNotSupported;
    if (!RT_NT_ABLATION && q8 && p.N <= 8 && p.K % 256 == 0 && !gemv_q8h_mfma_well(p, dev) && !gemv_q8h_few_leave(p, dev)) return hipErrorNotSupported; // launch_gemv's

    GemmNtArgs g{};
    g.A = A, g.B = (const half_t *)B, g.bias = (const half_t *)bias, g.out = (half_t *)out;
    if (q8) {
        const uint64_t n = (uint64_t)p.a_stack * p.M * p.K;
        g.scales = (const half_t *)((const uint8_t *)A + rt_q8_0_scale_offset(n));
        g.scale_dwords = (int64_t)((n / 32 * 2 + 255) / 256 * 64);
    }
    g.M = p.M, g.N = p.N, g.K = p.K;
    g.a_stack = p.a_stack, g.b_stack = p.b_stack;
    g.a_bs = p.a_bs, g.a_rs = p.a_rs;
    g.b_bs = p.b_bs, g.b_js = p.b_js;
    g.o_bs = p.o_bs, g.o_is = p.o_is, g.o_js = p.o_js;
    g.has_bias = p.has_bias, g.bias_on_rows = p.bias_on_rows, g.act = p.act;
    g.vec_epilogue = p.o_is == 1 && p.o_js % 8 == 0 && p.o_bs % 8 == 0 && ((uintptr_t)out & 15u) == 0;
    g.ksplit = 1, g.k_len = p.K, g.partial = nullptr;
    const bool kfull = p.K % NT_BK == 0;
    const bool pairs = p.o_is == 1 && p.o_js % 2 == 0 && p.o_bs % 2 == 0 && ((uintptr_t)out & 3u) == 0;
    if (!q8 && p.K <= 128 && (g.vec_epilogue || pairs) && !g_gemm_nt_no_direct && (p.N + 63) / 64 <= 0x7fffffff) {
        // resident-strip kernel, the output's i axis contiguous.  Strips are
        // split over several workgroups until the grid has a few workgroups per compute unit.
        const int64_t strips = (p.N + 63) / 64 * p.stacks, atiles = (p.M + 127) / 128;
        int parts = 1;
        while (parts < atiles && strips * parts < 2 * (int64_t)dev.num_cus) parts *= 2;
        if (g_gemm_nt_shortk_parts > 0) parts = g_gemm_nt_shortk_parts;
        g.tiles_i = (int)(parts < atiles ? parts : atiles);
        if (p.K <= 32) return launch_nt_shortk<32>(g, p.stacks, stream);
        if (p.K <= 64) return launch_nt_shortk<64>(g, p.stacks, stream);
        if (p.K <= 96) return launch_nt_shortk<96>(g, p.stacks, stream);
        return launch_nt_shortk<128>(g, p.stacks, stream);
    }
    if (!q8 && p.K <= 256) {
        // Short contractions (attention scores): the time goes into writing the output, not into
        // the K loop.  128 x 64 tiles need a third of the registers and LDS, so several
        // workgroups share a compute unit and one's epilogue overlaps another's loads.
        constexpr int SBM = 128, SBN = 64; // 128 outputs along the contiguous axis: whole cache lines per wavefront row
        if (!nt_set_tiles(g, SBM, SBN, 2)) return hipErrorNotSupported;
        return kfull ? launch_nt<SBM, SBN, true>(g, p.stacks, stream)
                     : launch_nt<SBM, SBN, false>(g, p.stacks, stream);
    }
    if (!q8 && (p.K % 32 != 0 || g_gemm_nt_no_direct)) {
        if (!nt_set_tiles(g, 160, 128, 2)) return hipErrorNotSupported;
        return kfull ? launch_nt<160, 128, true>(g, p.stacks, stream) : launch_nt<160, 128, false>(g, p.stacks, stream);
    }
    NtChoice c = nt_choose(p, dev, p.K > 256 && p.workspace && !((uintptr_t)p.workspace & 15u));
    if (c.ks > 1 && p.workspace_bytes < (uint64_t)p.stacks * c.ks * p.M * p.N * sizeof(float)) c = nt_choose(p, dev, false);
    if (!RT_NT_ABLATION && c.ks == 1 && gemv_chunks_unless_shared(p, dev)) // 17 to 32 rows of Q8_0H: faster in streaming launches (the timing-only builds have this file alone)
        if (const hipError_t e = gemv_chunks(p, A, B, bias, out, stream, dev); e != hipErrorNotSupported) return e;
    if (c.ks > 1) g.ksplit = c.ks, g.k_len = c.k_len, g.partial = (float *)p.workspace;
    if (!q8 && kfull && c.ks == 1 && g_gemm_nt_wide != 1 && p.a_rs >= 0 && p.b_js >= 0 && 2 * 320 * std::max(p.a_rs, p.b_js) < (int64_t(1) << 32)) {
        const int64_t tiles = ((p.M + 159) / 160) * ((p.N + 127) / 128), wide = ((p.M + 319) / 320) * ((p.N + 255) / 256) * p.stacks;
        const int64_t rounds = (tiles * p.stacks + dev.num_cus - 1) / dev.num_cus, rounds_wide = (wide + dev.num_cus - 1) / dev.num_cus;
        // A round of 320 x 256 tiles takes 12 + 0.030 K us on all compute units, one of 160 x 128 tiles 6.4 + 0.0080 K: four small
        // rounds are always longer (10240 x 2560 weights, 2048 activation rows: 108.5 us against 89.7), two never.  Three are
        // longer for a short K (1500 rows, K = 1024: 43.9 against 39.3), the same at K = 2560 and shorter beyond (1000 rows
        // x 11008 x 4096: 107.0 against 118.9; 1300 rows x 8192 x 4096: 101.5 against 102.6; two wide rounds against six small ones alike).
        const bool longer = 5 * rounds_wide < 2 * rounds && (3 * rounds_wide < rounds || p.K <= 2048);
        if ((g_gemm_nt_wide == 2 || longer) && nt_set_tiles(g, 320, 256, 2)) return launch_nt_wide(g, p.stacks, stream);
    }
    if (!nt_set_tiles(g, c.bm, c.bn, q8 ? 1 : 2)) return hipErrorNotSupported;
    if (!q8) {
        // two loading wavefronts: one and four measured the same within run-to-run spread.  The narrow tiles take as deep a ring as the
        // LDS holds: what a compute unit has in flight is what it can pull (10240 x 2560 f16 weights, 40 / 64 activation rows,
        // three stages of 64 x 128 -> six: 22.7 / 23.6 -> 20.0 / 22.1 us with the weights in HBM, 16.3 / 16.8 -> 14.8 / 15.7 from
        // the Infinity Cache; nine of 64 x 64: 18.3 / 20.5 and 12.6 / 13.6)
        if (c.bn == 64) return launch_nt_dl<64, 64, 9, 2>(g, p.stacks, stream);
        if (c.bm == 64) return launch_nt_dl<64, 128, 6, 2>(g, p.stacks, stream);
        if (c.bm == 96) return launch_nt_dl<96, 128, 5, 2>(g, p.stacks, stream);
        if (c.bm == 128) return launch_nt_dl<128, 128, 4, 2>(g, p.stacks, stream);
        return launch_nt_dl<160, 128, 3, 2>(g, p.stacks, stream);
    }
    if (nt_q8_whole(p)) {
        if (c.bn == 64) return launch_nt_q8w<64, 64, 4>(g, p.stacks, stream);
        if (c.bm == 64) return launch_nt_q8w<64, 128, 4>(g, p.stacks, stream);
        if (c.bm == 96) return launch_nt_q8w<96, 128, 4>(g, p.stacks, stream);
        if (c.bm == 128) return launch_nt_q8w<128, 128, 4>(g, p.stacks, stream);
        return launch_nt_q8w<160, 128, 4>(g, p.stacks, stream);
    }
    if (c.bn == 64) return launch_nt_q8r<64, 64, 2>(g, p.stacks, stream);
    if (c.bm == 64) return launch_nt_q8r<64, 128, 1>(g, p.stacks, stream);
    if (c.bm == 96) return launch_nt_q8r<96, 128, 1>(g, p.stacks, stream);
    if (c.bm == 128) return launch_nt_q8r<128, 128, 2>(g, p.stacks, stream);
    return launch_nt_q8r<160, 128, 1>(g, p.stacks, stream);
}

} // namespace rt

#if RT_NT_ABLATION
// Entry point of a timing-only build of this file (see RT_NT_ABLATION): the Linear form W[n x k] . X[m x k]^T + bias
// with f16 weights, output [m x n].  The measurement probes library holds one such build per variant.
extern "C" __attribute__((visibility("default"))) int RT_NT_ABL_ENTRY(const void *W, const void *X, const void *bias, void *out,
                                                                      int64_t n, int64_t m, int64_t k, void *stream) {
    rt::Problem p;
    p.a_dt = RT_F16, p.act_dt = RT_F16, p.M = n, p.N = m, p.K = k;
    p.a_rs = k, p.a_ks = 1, p.b_ks = 1, p.b_js = k, p.o_is = 1, p.o_js = n, p.has_bias = true, p.bias_on_rows = true;
    p.kernel = RT_KERNEL_GEMM_F16;
    return (int)rt::launch_gemm_nt(p, W, X, bias, out, (hipStream_t)stream, rt::DeviceInfo{});
}
#endif
