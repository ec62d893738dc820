// Q4_K weights x f16 activations for many activation rows (prefill), the weights never touching LDS:
// every multiplying wavefront decodes the raw blocks of its own 32 weight rows in registers, straight
// into the MFMA operand, and only the activation tile goes through LDS.  Where its 256 x 128 tiles fill
// the device a second kernel (gemm_q4k_wide_kernel, below) takes both through LDS, the blocks raw.
//
//   y[j, i] = sum_sb ( d_i,sb * sum_sub sum_{k in sub} x[j,k] (sc_i,sub q_i,k)  -  dmin_i,sb * sum_sub mn_i,sub S[j,sub] )
//   S[j, sub] = sum_{k in sub} x[j, k]
//
// The order of K inside an MFMA is free as long as both operands agree, so lane group g (lane / 16)
// of a weight fragment owns the 32 bytes g of a super-block's qs: the low nibbles are the values
// 64 g .. + 31 of the super-block (sub-block 2 g), the high nibbles the values 64 g + 32 .. + 63
// (sub-block 2 g + 1).  MFMA step t of a super-block takes from lane group g the values
// 64 g + 8 t .. + 7: bytes 8 (t % 4) .. + 7, low nibbles for t < 4, high for t >= 4.  A thread
// therefore reads a header and two 16-byte pieces per super-block and needs two of the eight scales
// and mins.  sc * q < 1024 is exact in f16 (fma(1024 + q, sc, -1024 sc) rounds once; the high
// nibbles stay in place as 1024 + 16 q against sc / 16), so a super-block chains through one MFMA
// accumulator and d is applied once per super-block in f32.  No weight is rounded.
//
// The sub-block sums of x fall out of the same layout: a lane of an activation fragment holds
// 8 values of sub-block 2 g (t < 4) or 2 g + 1 (t >= 4) of activation row lane % 16, so four dot
// products against ones per step give S for exactly the (row, sub-block pair) that the min-term MFMA
// wants from this lane.  Wavefront w sums the 16 activation rows of fragment w and shares them
// through LDS (two f16 parts, q4k_sum_parts); the min term of super-block sb is one MFMA per
// output tile, run under super-block sb + 1.
//
// A workgroup owns 128 weight rows x 64 activation rows: four multiplying wavefronts (32 weight rows
// x 64 activation rows each: 64 MFMAs per super-block, 8 for the min term).  The activation tiles come by
// LDS-DMA one super-block ahead in a ring of two stages.  With at most one workgroup per compute unit four more
// wavefronts issue those loads and nothing else (one per SIMD).  With more the multiplying wavefronts issue
// them: at 256 registers a SIMD holds two wavefronts, and a second workgroup's multiplying one is worth more there
// than a loading one, since the parts of a wavefront's step add up (below) and another's run beside them
// (8192 x 3072 at 300 / 512 / 1000 / 2048 activation rows 42.2 / 42.9 / 85.7 / 177.6 -> 37.9 / 40.3 / 78.3 / 161.5 us;
// 3072 x 8192 at 1000 rows 99.8 -> 91.9).  A staged row is 32 K-vectors
// and one of padding: the 16 rows of a fragment read start 4 banks apart and a read address is a
// base + 16 * step, an immediate.  One barrier per super-block.  The output tile leaves through LDS
// as 16-byte stores when the output is contiguous along the weight rows.  Also few rows against a K too long for the streaming kernels (gemm_q4k_few).
//
// What bounds it (measured by leaving parts out): the parts add up.  A wavefront's MFMAs (8 issue
// cycles each when vector instructions follow), its 339 vector instructions per super-block and the
// LDS pipe time of the compute unit's fragment reads (128 KB per super-block at 128 B/clk) each
// cost their full time whatever the order of instructions.  Two multiplying wavefronts per SIMD were
// measured: with 16 x 64 outputs each they double the fragment reads (27.7 against 26.7 us), with
// 32 x 32 each they decode every weight twice (32.3 us).
//
// The arithmetic is ggml's dequantize_row_q4_K (the reference holds only the block struct,
// crates/ratchet-loader/src/k_quants.rs:94-103); the caller convention is Linear's
// W.gemm(x, b, false, true, true) (crates/ratchet-nn/src/linear.rs:17-24).
#include "device_common.h"

#include <algorithm>

namespace rt {

struct GemmQ4kArgs {
    const uint8_t *blocks; // [stack][rows][K/256] super-blocks of 144 bytes
    const half_t *X;
    const half_t *bias;
    half_t *out;
    int64_t M, N; // weight rows, activation rows
    int64_t nsb;  // super-blocks per row
    int64_t a_stack, b_stack;
    int64_t b_bs, b_js;
    int64_t o_bs, o_is, o_js;
    int tiles_j, remap, vec_out;
    int has_bias, bias_on_rows, act;
    // K shared: blockIdx.z owns super-blocks [z * sb_len, (z + 1) * sb_len) and writes its f32 sums to partial [stack][share][N][M]; a
    // second kernel adds them up, then bias, activation, rounding
    int ksplit;
    int64_t sb_len;
    float *partial;
};

constexpr int QR_BN = 64; // activation rows per workgroup; weight rows: 16 per MFMA tile x TA tiles x MW multiplying wavefronts
// An activation stage holds one super-block of K for 64 rows: 32 K-vectors of 16 bytes per row and one of padding,
// so that the 16 rows of a fragment read start 4 banks apart and a read address is base + 16 * step.
constexpr int QR_ROWB = 33 * 16;       // bytes per staged row
constexpr int QR_XSB = QR_BN * QR_ROWB; // bytes per stage = 33 LDS-DMA instructions of 1 KB
// Activation stages: the tile of the next super-block is on its way while this one is multiplied.  A third stage (two
// tiles in flight) measured the same to 1 % at every grid size tried (alternating runs on one device), so the smaller
// footprint stays: two workgroups fit a compute unit's LDS.
constexpr int QR_XST = 2;
constexpr size_t QR_LDS = (size_t)QR_XST * QR_XSB + 2 * QR_BN * 4 * 8;

// Sums of x as MFMA operands.  32 f16 activations sum to up to 32 * 65504, so it is S / 32 that is held (dot products against 1 / 32, which are
// exact; dmin takes the 32): h = S / 32 rounded to f16, and l = (S / 32 - h) * 2^11 rounded, against mn and mn * 2^-11, both exact.  Neither part
// can overflow, and h + l * 2^-11 is S to 23 bits, one less than f32 (and S itself below 1 / 2).  Without the scales a sum beyond 2 * 65504 was cut
// off there.  Relative error of the f32 sums against float64, 2560 x 10240 at 16 rows, before and now: activations N(0, 1) 2.77e-7 and 2.71e-7, their
// absolute values 3.3e-6 and 2.6e-6, those times 4096 0.40 and 2.6e-6.
constexpr float kQ4kSumDiv = 32.0f, kQ4kSumLow = 2048.0f;
__device__ __forceinline__ uint2_t q4k_sum_parts(float s0, float s1) { // of two sums, divided by 32: (h, h), (l, l)
    const half2_t h = {(half_t)s0, (half_t)s1};
    const half2_t l = {(half_t)((s0 - (float)h[0]) * kQ4kSumLow), (half_t)((s1 - (float)h[1]) * kQ4kSumLow)};
    return uint2_t{__builtin_bit_cast(uint32_t, h), __builtin_bit_cast(uint32_t, l)};
}
__device__ __forceinline__ uint32_t q4k_low_mins(uint32_t mn) { // what the low parts are multiplied with
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, mn) * half2_t{(half_t)(1 / kQ4kSumLow), (half_t)(1 / kQ4kSumLow)});
}

// TA: MFMA tiles of weight rows per wavefront; MW: multiplying wavefronts (4: each sums the activation fragment of its number);
// LW: wavefronts that only issue the LDS-DMA (4, one per SIMD, or none: the multiplying ones issue it)
template <int TA, int MW, int LW>
__global__ __launch_bounds__(64 * (MW + LW), 2) void gemm_q4k_kernel(GemmQ4kArgs g) {
    constexpr int TB = 4;             // MFMA tiles per wavefront: TA of weight rows (second operand), TB of activation rows (first)
    constexpr int BM = 16 * TA * MW;  // weight rows per workgroup
    static_assert(MW == 4, "wavefront w sums the x of activation fragment w: four fragments, four wavefronts");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t *Xs = smem;                             // [QR_XST][64 rows][33 slots of 16 bytes]: K-vector v of row r in slot v
    uint2_t *Sx = (uint2_t *)(Xs + QR_XST * QR_XSB); // [2][64][4]: sums of x of super-block parity p, row, lane group: q4k_sum_parts

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int fr = lane & 15, fg = lane >> 4;
    const int64_t s = blockIdx.y;
    // the workgroups of one weight row block (one per block of activation rows) run on one XCD, whose L2 then
    // holds that block's raw weights for all of them
    uint32_t b = blockIdx.x;
    if (g.remap) b = (b & 7) * (gridDim.x >> 3) + (b >> 3);
    // (a division runs on the vector units: its result back into a scalar register, where it costs the main loop none of its own)
    const uint32_t ti = __builtin_amdgcn_readfirstlane(b / (uint32_t)g.tiles_j), tj = b - ti * (uint32_t)g.tiles_j;
    const int64_t i0 = (int64_t)ti * BM, j0 = (int64_t)tj * QR_BN;
    const int64_t sb0 = (int64_t)blockIdx.z * g.sb_len, nsb = min(g.sb_len, g.nsb - sb0); // this workgroup's share of K: > 0 (launcher)
    const uint8_t *blocks = g.blocks + ((g.a_stack == 1 ? 0 : s) * g.M * g.nsb + sb0) * 144;
    const half_t *X = g.X + (g.b_stack == 1 ? 0 : s) * g.b_bs + sb0 * 256;
    const int64_t last = nsb - 1;
    const bool vec_out = g.vec_out && g.ksplit == 1; // stored 16 bytes at a time

    if (LW > 0 && wave >= MW) {
        // ---- loading wavefront lw: LDS-DMA instruction i of a stage (i = lw, lw + 4, ...; 33 in all) fills the 1 KB
        // run of slots 64 i .. + 63; slot p is K-vector p % 33 of row p / 33 (the 33rd is padding and repeats the 32nd).
        // Each of the four issues nine: the ninth of wavefronts 1..3 repeats instruction 32.
        constexpr int NI = 9;
        const int lw = wave - MW;
        uint32_t xsrc[NI];
#pragma unroll
        for (int n = 0; n < NI; n++) {
            const uint32_t p = 64u * (uint32_t)min(4 * n + lw, 32) + (uint32_t)lane;
            const uint32_t row = p / 33u, v = min(p - 33u * row, 31u);
            xsrc[n] = (uint32_t)min(j0 + (int64_t)row, g.N - 1) * (uint32_t)g.b_js + 8u * v;
        }
        auto issue_x = [&](int stage, int64_t sb) {
            const half_t *xk = X + sb * 256;
#pragma unroll
            for (int n = 0; n < NI; n++)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(xk + xsrc[n]),
                                                 (__attribute__((address_space(3))) void *)(Xs + stage * QR_XSB + min(4 * n + lw, 32) * 1024), 16, 0, 0);
        };
        constexpr int kNewer = QR_XST == 3 ? NI : 0; // with three stages the newest tile may still be on its way
        constexpr int kOlder = 0x0F70 | (kNewer & 0xF) | (((kNewer >> 4) & 0x3) << 14);
        auto publish = [&]() {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(kOlder);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        issue_x(0, 0);
        if (QR_XST == 3) issue_x(1, min((int64_t)1, last));
        publish(); // super-block 0
        int fill = QR_XST - 1;
        for (int64_t sb = 0; sb < last; sb++) {
            // stage `fill` held super-block sb - 1, read for the last time before the barrier just passed
            issue_x(fill, min(sb + QR_XST - 1, last)); // past the end: the last one again, into a stage nobody reads
            publish();                                 // super-block sb + 1
            fill = fill == QR_XST - 1 ? 0 : fill + 1;
        }
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): nothing lands after the wavefront has ended
        __builtin_amdgcn_s_barrier();       // the multiplying wavefronts' last exchange of sums
        if (vec_out) __builtin_amdgcn_s_barrier(); // and their staged output tile
        return;
    }

    // ---- multiplying wavefront `wave`: weight rows i0 + 32 wave .. + 31.  Rows past the end repeat the last
    // valid one.  Offsets are 32-bit from wave-uniform bases (the launcher checks the ranges).
    struct Raw {
        uint4_t hdr, qa, qb;
    };
    uint32_t woff[TA];
#pragma unroll
    for (int a = 0; a < TA; a++) woff[a] = (uint32_t)min(i0 + wave * (16 * TA) + 16 * a + fr, g.M - 1) * (uint32_t)g.nsb * 144u;
    auto load_raw = [&](int64_t sb, Raw (&r)[TA]) {
        const uint8_t *bsb = blocks + sb * 144; // wave-uniform
#pragma unroll
        for (int a = 0; a < TA; a++) {
            r[a].hdr = *(const uint4_t *)(bsb + woff[a]);
            r[a].qa = *(const uint4_t *)(bsb + (woff[a] + 16u + 32u * (uint32_t)fg));
            r[a].qb = *(const uint4_t *)(bsb + (woff[a] + 32u + 32u * (uint32_t)fg));
        }
    };
    // what a thread keeps of a super-block's header: the scale pairs for its two sub-blocks as FMA operands,
    // and for the min term (a super-block late) d, dmin and the two mins as f16 integers
    struct Scl {
        half2_t s_lo, n_lo, s_hi, n_hi;
    };
    struct Fin {
        float d, dmin; // dmin * 32
        uint32_t mn;
    };
    const int sh = 16 * (fg & 1);
    const uint32_t upper = (fg & 2) ? ~0u : 0u; // sub-blocks 4..7: the scales and mins split over two bytes
    const half2_t k1024 = {(half_t)1024.0f, (half_t)1024.0f};
    auto header = [&](const Raw &r, Scl &sc, Fin &f) {
        // the 6-bit scales and mins (ggml get_scale_min_k4), four per dword; this thread's are 2 fg, 2 fg + 1
        const uint32_t S0 = r.hdr[1], S1 = r.hdr[2], S2 = r.hdr[3];
        const uint32_t sc47 = (S2 & 0x0F0F0F0Fu) | ((S0 >> 2) & 0x30303030u), mn47 = ((S2 >> 4) & 0x0F0F0F0Fu) | ((S1 >> 2) & 0x30303030u);
        const uint32_t scw = (sc47 & upper) | (S0 & 0x3F3F3F3Fu & ~upper); // no branch: a divergent one makes the compiler wait for every load
        const uint32_t mnw = (mn47 & upper) | (S1 & 0x3F3F3F3Fu & ~upper);
        const half2_t s2 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, scw >> sh, 0x04010400u)) - k1024;
        const half2_t m2 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, mnw >> sh, 0x04010400u)) - k1024;
        const half_t lo = s2[0], hi = s2[1] * (half_t)0.0625f;
        sc.s_lo = half2_t{lo, lo}, sc.s_hi = half2_t{hi, hi};
        sc.n_lo = sc.s_lo * (half_t)-1024.0f, sc.n_hi = sc.s_hi * (half_t)-1024.0f;
        const half2_t dm = __builtin_bit_cast(half2_t, r.hdr[0]);
        f.d = (float)dm[0], f.dmin = (float)dm[1] * kQ4kSumDiv, f.mn = __builtin_bit_cast(uint32_t, m2);
    };
    // weight fragment of step T: 8 values sc * q of this thread's row
    auto wfrag = [&](auto Tc, const Raw &r, const Scl &sc) {
        constexpr int T = decltype(Tc)::value;
        const uint4_t &q = (T & 2) ? r.qb : r.qa;
        const uint32_t mask = T < 4 ? 0x0F0F0F0Fu : 0xF0F0F0F0u;
        const uint32_t v0 = q[2 * (T & 1)] & mask, v1 = q[2 * (T & 1) + 1] & mask;
        const half2_t s2 = T < 4 ? sc.s_lo : sc.s_hi, n2 = T < 4 ? sc.n_lo : sc.n_hi;
        half2_t a = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v0, 0x04010400u));
        half2_t bb = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v0, 0x04030402u));
        half2_t c = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v1, 0x04010400u));
        half2_t d = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v1, 0x04030402u));
        a = __builtin_elementwise_fma(a, s2, n2), bb = __builtin_elementwise_fma(bb, s2, n2);
        c = __builtin_elementwise_fma(c, s2, n2), d = __builtin_elementwise_fma(d, s2, n2);
        return __builtin_bit_cast(half8_t, uint4_t{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, bb),
                                                   __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)});
    };
    // This wavefront's LDS stores (its sums of x) are done; past the barrier the next activation tile is whole,
    // the loading wavefront having waited for its slots, the stage of the tile before is free, and every
    // wavefront's sums of the super-block before are visible.
    auto tile_ready = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(LW == 0 ? 0x0070 : 0xC07F); // lgkmcnt(0); and, without loading wavefronts, vmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // LW == 0: this wavefront's share of the activation tile's LDS-DMA, the loading wavefronts' instructions.  As asm: behind the
    // builtin the compiler makes every fragment read wait for all loads in flight; no register is written by it, and
    // tile_ready waits for it.
    constexpr int NX = LW == 0 ? 9 : 1;
    uint32_t xoff[NX];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;
    if constexpr (LW == 0) {
#pragma unroll
        for (int n = 0; n < NX; n++) {
            const uint32_t p = 64u * (uint32_t)min(4 * n + wave, 32) + (uint32_t)lane, row = p / 33u, v = min(p - 33u * row, 31u);
            xoff[n] = 2u * ((uint32_t)min(j0 + (int64_t)row, g.N - 1) * (uint32_t)g.b_js + 8u * v);
        }
    }
    auto issue_x = [&](int stage, int64_t sb) __attribute__((always_inline)) {
        if constexpr (LW == 0) {
            const half_t *xk = X + sb * 256;
#pragma unroll
            for (int n = 0; n < NX; n++)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + (uint32_t)(stage * QR_XSB + min(4 * n + wave, 32) * 1024)),
                             "v"(xoff[n]), "s"(xk) : "m0", "memory");
        }
    };

    float4_t acc[TA][TB], P[2][TA][TB];
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
        for (int bq = 0; bq < TB; bq++) acc[a][bq] = zero, P[1][a][bq] = zero;
    Fin fin[2][TA];
#pragma unroll
    for (int a = 0; a < TA; a++) fin[1][a] = Fin{0.f, 0.f, 0u};
    // activation fragment bq of this wavefront is rows 16 ((bq + wave) % 4) .. + 15 of the tile, so that its
    // fragment 0, the one it sums, is fragment `wave`
    const uint32_t xlane = (uint32_t)(QR_ROWB * fr + 128 * fg);
    uint2_t *sx_mine = Sx + (16 * wave + fr) * 4 + fg;
    sx_mine[QR_BN * 4] = uint2_t{0u, 0u}; // parity 1 is read (against zero mins) under super-block 0
    const half2_t part32 = {(half_t)(1 / kQ4kSumDiv), (half_t)(1 / kQ4kSumDiv)};

    // The min term of the super-block before (parity Q) and its fold into the accumulators.
    auto read_sums = [&](int Q, uint2_t (&hl)[TB]) {
#pragma unroll
        for (int bq = 0; bq < TB; bq++) hl[bq] = Sx[Q * QR_BN * 4 + (16 * ((bq + wave) & 3) + fr) * 4 + fg];
    };
    auto finish = [&](auto Qc, const uint2_t (&hl)[TB]) {
        constexpr int Q = decltype(Qc)::value;
#pragma unroll
        for (int bq = 0; bq < TB; bq++) {
            const half8_t sf = __builtin_bit_cast(half8_t, uint4_t{hl[bq][0], hl[bq][1], 0u, 0u});
#pragma unroll
            for (int a = 0; a < TA; a++) {
                const half8_t mf = __builtin_bit_cast(half8_t, uint4_t{fin[Q][a].mn, q4k_low_mins(fin[Q][a].mn), 0u, 0u});
                const float4_t T = __builtin_amdgcn_mfma_f32_16x16x32_f16(sf, mf, zero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[a][bq][r] = fmaf(-fin[Q][a].dmin, T[r], fmaf(fin[Q][a].d, P[Q][a][bq][r], acc[a][bq][r]));
            }
        }
    };

    // One super-block of parity Pc: `cur` holds its raw blocks (loaded a super-block ago), `nxt` is the register
    // set that the super-block before has left.
    int xcur = 0;
    auto step = [&](auto Pc, int64_t sb, const Raw (&cur)[TA], Raw (&nxt)[TA]) {
        constexpr int PP = decltype(Pc)::value;
        tile_ready();
        issue_x(xcur ^ 1, min(sb + 1, last)); // past the end: the last one again, into a stage nobody reads
        load_raw(min(sb + 1, last), nxt);
        uint2_t hl[TB];
        read_sums(PP ^ 1, hl);
        __builtin_amdgcn_sched_barrier(0); // the loads stay here, a super-block ahead of their decoding
        Scl sc[TA];
#pragma unroll
        for (int a = 0; a < TA; a++) header(cur[a], sc[a], fin[PP][a]);
        finish(std::integral_constant<int, PP ^ 1>{}, hl);
        uint32_t xb[TB];
#pragma unroll
        for (int bq = 0; bq < TB; bq++) xb[bq] = xlane + (uint32_t)(xcur * QR_XSB + 16 * QR_ROWB * ((bq + wave) & 3));
        float S0 = 0.f, S1 = 0.f;
        auto xread = [&](int T, half8_t (&xf)[TB]) {
#pragma unroll
            for (int bq = 0; bq < TB; bq++) xf[bq] = __builtin_bit_cast(half8_t, *(const uint4_t *)(Xs + xb[bq] + 16 * T));
        };
        half8_t xf[2][TB];
        xread(0, xf[0]);
        // The order inside a super-block is the compiler's.  Pinned orders were measured: fragment reads a step ahead
        // of their MFMAs, one read in front of every second MFMA, one right behind every MFMA (where a bare loop of
        // MFMAs, packed FMAs and fragment reads issues them for 2 ns instead of 10: bench.py --issue-calibration);
        // with two weight tiles per wavefront all were the same or up to 4 % slower, with one tile the last was
        // 6 % faster.  Below two places are pinned where there are loading wavefronts, with which the compiler otherwise spreads a
        // super-block over more registers than there are (8192 x 3072 at 200 rows, two weight tiles, without / with 25.6 / 20.8 us, 6144 x 2048 at 240 19.0 /
        // 15.3; one tile, 8192 x 3072 at 128 rows, 14.8 / 14.4).
        auto mfma_step = [&](auto Tc) {
            constexpr int T = decltype(Tc)::value;
            if constexpr (T < 7) xread(T + 1, xf[(T + 1) & 1]);
            half8_t wf[TA];
#pragma unroll
            for (int a = 0; a < TA; a++) wf[a] = wfrag(Tc, cur[a], sc[a]);
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
                for (int bq = 0; bq < TB; bq++) // a super-block's first MFMA starts from zero: no clearing of P between super-blocks
                    P[PP][a][bq] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[T & 1][bq], wf[a], T == 0 ? zero : P[PP][a][bq], 0, 0, 0);
            const half8_t xs0 = xf[T & 1][0];
            float &S = T < 4 ? S0 : S1;
#pragma unroll
            for (int c = 0; c < 4; c++) S = __builtin_amdgcn_fdot2(half2_t{xs0[2 * c], xs0[2 * c + 1]}, part32, S, false);
        };
        mfma_step(std::integral_constant<int, 0>{});
        mfma_step(std::integral_constant<int, 1>{});
        mfma_step(std::integral_constant<int, 2>{});
        mfma_step(std::integral_constant<int, 3>{});
        if (TA == 2 && LW > 0) __builtin_amdgcn_sched_barrier(0);
        mfma_step(std::integral_constant<int, 4>{});
        mfma_step(std::integral_constant<int, 5>{});
        mfma_step(std::integral_constant<int, 6>{});
        mfma_step(std::integral_constant<int, 7>{});
        if (TA == 1) __builtin_amdgcn_sched_barrier(0);
        sx_mine[PP * QR_BN * 4] = q4k_sum_parts(S0, S1);
        xcur = xcur == QR_XST - 1 ? 0 : xcur + 1;
    };

    Raw r0[TA], r1[TA];
    issue_x(0, 0);
    load_raw(0, r0);
    // two super-blocks per trip, one straight run of instructions (a branch inside it makes the compiler wait
    // for every load in flight)
    int64_t sb = 0;
    for (; sb + 1 < nsb; sb += 2) {
        step(std::integral_constant<int, 0>{}, sb, r0, r1);
        step(std::integral_constant<int, 1>{}, sb + 1, r1, r0);
    }
    uint2_t hl[TB];
    if (sb < nsb) {
        step(std::integral_constant<int, 0>{}, sb, r0, r1);
        tile_ready();
        read_sums(0, hl);
        finish(std::integral_constant<int, 0>{}, hl);
    } else {
        tile_ready();
        read_sums(1, hl);
        finish(std::integral_constant<int, 1>{}, hl);
    }

    // acc[a][bq][r]: weight row i0 + 32 wave + 16 a + fr, activation row j0 + 16 ((bq + wave) % 4) + 4 fg + r
    if (g.ksplit > 1) {
        float *pt = g.partial + (s * g.ksplit + blockIdx.z) * g.N * g.M;
#pragma unroll
        for (int a = 0; a < TA; a++) {
            const int64_t i = i0 + wave * (16 * TA) + 16 * a + fr;
#pragma unroll
            for (int bq = 0; bq < TB; bq++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t j = j0 + 16 * ((bq + wave) & 3) + 4 * fg + r;
                    if (i < g.M && j < g.N) pt[j * g.M + i] = acc[a][bq][r];
                }
        }
        return;
    }
    // The bias before any store, since a load behind one is waited for by itself, and tiles past the last weight row through LDS too: with
    // both in the stores of an edge tile, whose outputs went one by one, the launch took 4 us longer wherever M % 128 was not 0
    // (M x K at activation rows, before and now, us: 1760 x 256 at 1683 12.9 and 8.6, 4288 x 256 at 206 9.2 and 5.4, 10848 x 2816 at 95 24.8 and
    // 20.7, 4192 x 768 at 318 12.9 and 8.4; 8192 x 3072 at 1000 75.0 and 75.2).
    if (g.has_bias) {
        if (g.bias_on_rows) {
#pragma unroll
            for (int a = 0; a < TA; a++) {
                const float bi = (float)(g.bias + i0)[min(wave * (16 * TA) + 16 * a + fr, (int)min<int64_t>(BM, g.M - i0) - 1)];
#pragma unroll
                for (int bq = 0; bq < TB; bq++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[a][bq][r] += bi;
            }
        } else {
#pragma unroll
            for (int bq = 0; bq < TB; bq++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float bj = (float)(g.bias + j0)[min(16 * ((bq + wave) & 3) + 4 * fg + r, (int)min<int64_t>(QR_BN, g.N - j0) - 1)];
#pragma unroll
                    for (int a = 0; a < TA; a++) acc[a][bq][r] += bj;
                }
        }
    }
    half_t *out = g.out + s * g.o_bs;
    if (vec_out) {
        // Output contiguous along the weight rows: the tile goes through LDS (the activation stages are free: every
        // wavefront's last fragment read and the last LDS-DMA lie before the barrier above) and leaves as 16-byte
        // stores, 256 bytes per activation row.
        constexpr int OLD = BM + 8; // halfs per staged row: rows 272 bytes apart spread the lane groups over the banks
        half_t *Os = (half_t *)smem;
        static_assert((size_t)QR_BN * OLD * 2 <= (size_t)QR_XST * QR_XSB, "the staged output tile fits the activation stages");
        rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
                for (int bq = 0; bq < TB; bq++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        Os[(16 * ((bq + wave) & 3) + 4 * fg + r) * OLD + wave * (16 * TA) + 16 * a + fr] = (half_t)rt_act_k<decltype(has_act)::value>(acc[a][bq][r]);
        });
        tile_ready();
#pragma unroll
        for (int k = 0; k < 2 * TA; k++) {
            constexpr int CPR = BM / 8; // 16-byte pieces per row
            const int idx = t + 64 * MW * k, row = idx / CPR, c = idx % CPR;
            if (j0 + row < g.N && i0 + 8 * c < g.M) *(uint4_t *)(out + (j0 + row) * g.o_js + i0 + 8 * c) = *(const uint4_t *)(Os + row * OLD + 8 * c);
        }
        return;
    }
    rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
        for (int a = 0; a < TA; a++) {
            const int64_t i = i0 + wave * (16 * TA) + 16 * a + fr;
            if (i >= g.M) continue;
#pragma unroll
            for (int bq = 0; bq < TB; bq++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t j = j0 + 16 * ((bq + wave) & 3) + 4 * fg + r;
                    if (j < g.N) out[i * g.o_is + j * g.o_js] = (half_t)rt_act_k<decltype(has_act)::value>(acc[a][bq][r]);
                }
        }
    });
}

// ---------------------------------------------------------------------------
// The same for many activation rows: 256 weight rows x 128 activation rows per workgroup, one workgroup per compute unit, eight
// wavefronts of 64 x 64 outputs on 32 x 32 x 16 MFMAs.
//
// Everything comes by LDS-DMA, the raw blocks too: a load that gives every lane 16 bytes of a row of its own is 64 lines to the
// compute unit's memory pipeline, and those loads were what the kernel above spends a third of its time on here; as runs of 144
// consecutive bytes they are a fifth of that.  Half the tile's activations per weight byte and half the fragment reads per MFMA are the
// larger tile's.  Measured, the kernel above and this: 8192 x 3072 against 1000 / 2048 activation rows 75.2 / 160 -> 60.2 / 122 us (0.84 PFLOP/s; with
// the MFMAs alone it is 41, and 36 without any of them).  What bounds it: MFMAs and what stands between them share a SIMD's issue (a step of a super-block
// is 4.4 us of which the MFMAs are 2.7 at the clock the chip then runs at), the LDS-DMA takes 0.5 of it, the sums of x 0.3.
//
// Lane half h = lane / 32 owns the 64 bytes h of a super-block's qs (sub-blocks 4 h .. + 3).  A super-block is two halves of eight
// steps: half H is chunk 2 h + H of 32 bytes, four steps of eight low nibbles and four of high ones.  A pair of nibbles stays where
// v_perm puts it, as the f16 subnormals q * 2^-24 (16 q * 2^-24), and one packed multiplication with sc * 2^10 (2^6) makes it
// sc * q * 2^-14 exactly; the 2^14 goes into d.
//
// A SIMD overlaps the vector instructions of one wavefront with the MFMAs of the other, and a wavefront's own with the MFMA before them:
// so the decoding of the step after, the header of the super-block after, the folds and the sums of x stand between the MFMAs, a few
// behind each.  Two stages of activations (a half super-block each), two of blocks; the barrier of a half stands
// before its last step, whose operands are in registers by then, so that the first reads of the next half run under that step.
// What is loaded there has a half's time to land.
//
// Sums of x: of the four wavefronts that share 64 activation rows, number w sums fragment w % 2 over the low (w < 2) or high nibbles'
// K; it takes its fragments and nibbles in an order that makes those its first ones, so that the code is the same for all.
//
// A chain here has 16 MFMAs of 16 k a super-block where the kernel above has 8 of 32; it is no less exact for that.  Relative error of the f32 sums
// against float64 in two shares, there and here, 300 activation rows x 2048 at K = 512 / 3072 / 8192: N(0, 1) 2.64e-7 / 2.65e-7 / 2.78e-7 and 2.55e-7 /
// 2.58e-7 / 2.72e-7, its absolute values 2.62e-6 / 2.64e-6 / 2.60e-6 and 2.58e-6 / 2.60e-6 / 2.56e-6.
// ---------------------------------------------------------------------------
constexpr int QW_BM = 256, QW_BN = 128;
constexpr int QW_ROWB = 17 * 16;          // bytes per staged activation row: 16 K-vectors and one of padding
constexpr int QW_XB = QW_BN * QW_ROWB;    // bytes per stage of activations = 34 LDS-DMA instructions
constexpr int QW_WB = QW_BM * 144;        // of blocks = 36 instructions; rows 144 bytes apart start 4 banks apart
constexpr int QW_SXB = QW_BN * 2 * 16;    // of the sums of x of a super-block: [row][lane half], the high parts of four, then their low parts (q4k_sum_parts)
constexpr size_t QW_LDS = 2 * (size_t)(QW_XB + QW_WB + QW_SXB) ;

__global__ __launch_bounds__(512, 2) void gemm_q4k_wide_kernel(GemmQ4kArgs g) {
    constexpr int TA = 2, TB = 2;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t *Xs = smem, *Ws = smem + 2 * QW_XB, *Sx = smem + 2 * (QW_XB + QW_WB);
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int fr = lane & 31, fh = lane >> 5;
    const int wi = wave >> 1, wj = wave & 1, wc = wi >> 1, wb = wi & 1;
    const int64_t s = blockIdx.y;
    uint32_t blk = blockIdx.x;
    if (g.remap) blk = (blk & 7) * (gridDim.x >> 3) + (blk >> 3); // as above
    const uint32_t ti = __builtin_amdgcn_readfirstlane(blk / (uint32_t)g.tiles_j), tj = blk - ti * (uint32_t)g.tiles_j;
    const int64_t i0 = (int64_t)ti * QW_BM, j0 = (int64_t)tj * QW_BN;
    const int64_t sb0 = (int64_t)blockIdx.z * g.sb_len, nsb = min(g.sb_len, g.nsb - sb0), last = nsb - 1; // this workgroup's share of K: > 0 (launcher)
    const uint8_t *blocks = g.blocks + ((g.a_stack == 1 ? 0 : s) * g.M * g.nsb + sb0) * 144;
    const half_t *X = g.X + (g.b_stack == 1 ? 0 : s) * g.b_bs + sb0 * 256;

    // LDS-DMA instruction i of a stage (wavefront i % 8) fills slots 64 i .. + 63 of 16 bytes.  Rows past the end repeat the last one.
    constexpr int ND = 5;
    const int ix = min(wave + 32, 33), iw5 = min(wave + 32, 35); // the fifth of a wavefront that has four repeats the stage's last
    const uint32_t x4 = 1024u * (uint32_t)(ix - wave), w4 = 1024u * (uint32_t)(iw5 - wave);
    uint32_t xoff[ND], woff[ND];
#pragma unroll
    for (int n = 0; n < ND; n++) {
        const uint32_t px = 64u * (uint32_t)min(wave + 8 * n, 33) + (uint32_t)lane, xr = px / 17u, xv = min(px - 17u * xr, 15u);
        const uint32_t pw = 64u * (uint32_t)min(wave + 8 * n, 35) + (uint32_t)lane, wr = pw / 9u, wv = pw - 9u * wr;
        xoff[n] = 2u * ((uint32_t)min(j0 + (int64_t)xr, g.N - 1) * (uint32_t)g.b_js + 128u * (xv >> 3) + 8u * (xv & 7u));
        woff[n] = (uint32_t)min(i0 + (int64_t)wr, g.M - 1) * (uint32_t)g.nsb * 144u + 16u * wv; // < 2^32: launcher
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem + 1024u * (uint32_t)wave;
    // as asm: see issue_x above
    auto dma = [&](uint32_t dst, uint32_t off, const void *base) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + dst), "v"(off), "s"(base) : "m0", "memory");
    };
    auto issue_x = [&](int half, int64_t sb) __attribute__((always_inline)) { // into stage `half`
        const half_t *xk = X + min(sb, last) * 256 + 64 * half; // past the end: the last one again, never used
#pragma unroll
        for (int n = 0; n < 4; n++) dma((uint32_t)(half * QW_XB + 8192 * n), xoff[n], xk);
        dma((uint32_t)(half * QW_XB) + x4, xoff[4], xk);
    };
    auto issue_w = [&](uint32_t stage, int64_t sb) __attribute__((always_inline)) { // stage in bytes
        const uint8_t *bsb = blocks + min(sb, last) * 144;
#pragma unroll
        for (int n = 0; n < 4; n++) dma(2 * QW_XB + stage + 8192u * n, woff[n], bsb);
        dma(2 * QW_XB + stage + w4, woff[4], bsb);
    };
    // This wavefront's loads have landed, its LDS stores are done and its reads have returned; past the barrier so have everyone's.
    auto meet = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    struct Scl {
        half2_t s[2]; // per half: of the sub-block taken first, second; sc * 2^10 for low nibbles, sc * 2^6 for high ones
    };
    struct Fin {
        float d, dmin; // d * 2^14, dmin * 32
        uint32_t mn[2];
    };
    const uint32_t upper = fh ? ~0u : 0u; // sub-blocks 4..7: the scales and mins split over two bytes
    const uint32_t order[2] = {wc ? 0x04000401u : 0x04010400u, wc ? 0x04020403u : 0x04030402u}; // v_perm's bytes of the two scales
    const half2_t k1024 = {(half_t)1024.0f, (half_t)1024.0f}, kup = {(half_t)(wc ? 64.0f : 1024.0f), (half_t)(wc ? 1024.0f : 64.0f)};
    const uint32_t mask[2] = {wc ? 0xF0F0F0F0u : 0x0F0F0F0Fu, wc ? 0x0F0F0F0Fu : 0xF0F0F0F0u};
    auto header = [&](const uint4_t &h, Scl &sc, Fin &f) __attribute__((always_inline)) {
        const uint32_t S0 = h[1], S1 = h[2], S2 = h[3];
        const uint32_t sc47 = (S2 & 0x0F0F0F0Fu) | ((S0 >> 2) & 0x30303030u), mn47 = ((S2 >> 4) & 0x0F0F0F0Fu) | ((S1 >> 2) & 0x30303030u);
        const uint32_t scw = (sc47 & upper) | (S0 & 0x3F3F3F3Fu & ~upper);
        const uint32_t mnw = (mn47 & upper) | (S1 & 0x3F3F3F3Fu & ~upper);
        sc.s[0] = (__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, scw, order[0])) - k1024) * kup;
        sc.s[1] = (__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, scw, order[1])) - k1024) * kup;
        f.mn[0] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, mnw, 0x04010400u)) - k1024);
        f.mn[1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, mnw, 0x04030402u)) - k1024);
        const half2_t dm = __builtin_bit_cast(half2_t, h[0]);
        f.d = (float)dm[0] * 16384.0f, f.dmin = (float)dm[1] * kQ4kSumDiv;
    };
    const float16_t zero = {};
    float16_t acc[TA][TB], P[TA][TB];
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
        for (int b = 0; b < TB; b++) acc[a][b] = zero, P[a][b] = zero;
    Scl sc[TA];
    Fin now[TA], fin[TA]; // of the super-block at hand, of the one before
    uint4_t hdr[TA], pc[TA][2], wf[2][TA]; // raw header; the half's two pieces; weight fragments of two steps
    half8_t xf[2][TB], sf[TB];
#pragma unroll
    for (int a = 0; a < TA; a++) fin[a] = Fin{0.f, 0.f, {0u, 0u}};
    // half `hf` of the weight fragment of step T of half H: four of its 8 values sc * q * 2^-14 of this lane's row
    auto wpart = [&](auto Hc, auto Tc, int a, int hf, uint4_t &w) __attribute__((always_inline)) {
        constexpr int H = decltype(Hc)::value, T = decltype(Tc)::value;
        const uint32_t v = pc[a][(T & 3) >> 1][2 * (T & 1) + hf] & mask[T >> 2];
        const half_t sv = sc[a].s[H][T >> 2];
        const half2_t s2 = {sv, sv};
        w[2 * hf] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, v, 0x04010400u)) * s2);
        w[2 * hf + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, v, 0x04030402u)) * s2);
    };
    uint32_t wat = (uint32_t)(144 * (64 * wi + fr)); // this lane's row of blocks in the current stage
    auto read_piece = [&](int half, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < TA; a++) pc[a][p] = *(const uint4_t *)(Ws + wat + 64 * fh + (16 + 32 * half + 16 * p + 32 * 144 * a));
    };
    auto read_header = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < TA; a++) hdr[a] = *(const uint4_t *)(Ws + wat + 32 * 144 * a);
    };
    uint32_t xat[TB][2], slane[TB]; // this lane's row of the activation fragments, the one it sums first: at the sub-block taken first, second; of their sums
#pragma unroll
    for (int b = 0; b < TB; b++) {
        const int row = 64 * wj + 32 * (b ^ wb) + fr;
        xat[b][0] = (uint32_t)(QW_ROWB * row + 128 * fh + 64 * wc), xat[b][1] = xat[b][0] + (wc ? -64 : 64), slane[b] = (uint32_t)(32 * row + 16 * fh);
    }
    auto xread = [&](int half, int T) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < TB; b++) xf[T & 1][b] = __builtin_bit_cast(half8_t, *(const uint4_t *)(Xs + xat[b][T >> 2] + (half * QW_XB + 16 * (T & 3))));
    };
    auto read_sums = [&](uint32_t q) __attribute__((always_inline)) { // of parity q, in bytes of Sx
#pragma unroll
        for (int b = 0; b < TB; b++) sf[b] = __builtin_bit_cast(half8_t, *(const uint4_t *)(Sx + q + slane[b]));
    };
    const half2_t part32 = {(half_t)(1 / kQ4kSumDiv), (half_t)(1 / kQ4kSumDiv)};
    // What is left of the super-block before, tile by tile: its sums times d, and its min term
    auto fold = [&](int a, int b) __attribute__((always_inline)) {
        const half8_t mf = __builtin_bit_cast(half8_t, uint4_t{fin[a].mn[0], fin[a].mn[1], q4k_low_mins(fin[a].mn[0]), q4k_low_mins(fin[a].mn[1])});
#pragma unroll
        for (int r = 0; r < 16; r++) acc[a][b][r] = fmaf(fin[a].d, P[a][b][r], acc[a][b][r]);
        P[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf[b], mf, zero, 0, 0, 0);
    };
    auto fold_min = [&](int a, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; r++) acc[a][b][r] = fmaf(-fin[a].dmin, P[a][b][r], acc[a][b][r]);
    };
    uint32_t wcur = 0, par = 0; // bytes: stage of this super-block's blocks, parity of its sums
    // Half H of a super-block.
    auto run_half = [&](auto Hc, int64_t sb) __attribute__((always_inline)) {
        constexpr int H = decltype(Hc)::value;
        float S = 0.f;
        auto sum_x = [&](int T, int c) __attribute__((always_inline)) {
            S = __builtin_amdgcn_fdot2(half2_t{xf[T & 1][0][2 * c], xf[T & 1][0][2 * c + 1]}, part32, S, false);
        };
        auto step = [&](auto Tc) __attribute__((always_inline)) {
            constexpr int T = decltype(Tc)::value;
            if constexpr (T < 7) xread(H, T + 1);
            if constexpr (T == 5) { // the registers' last values have been decoded
                if (H == 1) wat += QW_WB - 2 * wcur, read_header();
                read_piece(H ^ 1, 0);
            }
            if constexpr (T == 7) {
                meet();
                xread(H ^ 1, 0);
                read_piece(H ^ 1, 1);
                if (H == 1) read_sums(par);
                issue_x(H, sb + 1);
                if (H == 1) issue_w(wcur, sb + 2);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < TA * TB; m++) {
                const int a = m / TB, b = m % TB;
                if (H == 0 && T == 0) fold_min(a, b);
                P[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[T & 1][b], __builtin_bit_cast(half8_t, wf[T & 1][a]), H == 0 && T == 0 ? zero : P[a][b], 0, 0, 0);
                if constexpr (H == 1 && T == 7) {
                    if (b == 0) header(hdr[a], sc[a], now[a]);
                }
                wpart(std::integral_constant<int, T == 7 ? H ^ 1 : H>{}, std::integral_constant<int, (T + 1) % 8>{}, a, b, wf[(T + 1) & 1][a]);
                if (T < 4) sum_x(T, m);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (T == 4) {
                const uint2_t hl = q4k_sum_parts(S, 0.f);
                *(uint16_t *)(Sx + par + slane[0] + 4 * H + 2 * wc) = (uint16_t)hl[0];
                *(uint16_t *)(Sx + par + slane[0] + 8 + 4 * H + 2 * wc) = (uint16_t)hl[1];
            }
        };
        step(std::integral_constant<int, 0>{});
        if constexpr (H == 0)
#pragma unroll
            for (int a = 0; a < TA; a++) fin[a] = now[a];
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        step(std::integral_constant<int, 4>{});
        step(std::integral_constant<int, 5>{});
        step(std::integral_constant<int, 6>{});
        step(std::integral_constant<int, 7>{});
    };
    static_assert(TB == 2 && TA * TB == 4, "a step's MFMAs: half a weight fragment and a quarter of the sum of x behind each");

    issue_x(0, 0);
    issue_w(0, 0);
    issue_x(1, 0);
    issue_w(QW_WB, 1);
    asm volatile("s_waitcnt vmcnt(10)\n\ts_barrier" ::: "memory"); // the first two have landed
    read_header();
    read_piece(0, 0);
    read_piece(0, 1);
    xread(0, 0);
#pragma unroll
    for (int a = 0; a < TA; a++) {
        header(hdr[a], sc[a], now[a]);
#pragma unroll
        for (int hf = 0; hf < 2; hf++) wpart(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, a, hf, wf[0][a]);
    }
#pragma unroll
    for (int b = 0; b < TB; b++) sf[b] = half8_t{}; // nothing before the first super-block
    for (int64_t sb = 0; sb < nsb; sb++) {
#pragma unroll
        for (int m = 0; m < TA * TB; m++) {
            fold(m / TB, m % TB);
            __builtin_amdgcn_sched_barrier(0);
        }
        run_half(std::integral_constant<int, 0>{}, sb);
        run_half(std::integral_constant<int, 1>{}, sb);
        wcur = QW_WB - wcur, par ^= QW_SXB;
    }
#pragma unroll
    for (int m = 0; m < TA * TB; m++) fold(m / TB, m % TB);
#pragma unroll
    for (int m = 0; m < TA * TB; m++) fold_min(m / TB, m % TB);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // nothing lands once the output goes through LDS

    // acc[a][b][r]: weight row i0 + 64 wi + 32 a + fr, activation row j0 + 64 wj + 32 (b ^ wb) + 8 (r / 4) + 4 fh + r % 4
    const int iw = 64 * wi + fr;
    if (g.ksplit > 1) {
        float *pt = g.partial + (s * g.ksplit + blockIdx.z) * g.N * g.M;
#pragma unroll
        for (int a = 0; a < TA; a++) {
            const int64_t i = i0 + iw + 32 * a;
#pragma unroll
            for (int b = 0; b < TB; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int64_t j = j0 + 64 * wj + 32 * (b ^ wb) + 8 * (r >> 2) + 4 * fh + (r & 3);
                    if (i < g.M && j < g.N) pt[j * g.M + i] = acc[a][b][r];
                }
        }
        return;
    }
    // the bias before any store: behind one, every load would be waited for by itself
    if (g.has_bias) {
        if (g.bias_on_rows) {
#pragma unroll
            for (int a = 0; a < TA; a++) {
                const float bi = (float)(g.bias + i0)[min(iw + 32 * a, (int)min<int64_t>(QW_BM, g.M - i0) - 1)];
#pragma unroll
                for (int b = 0; b < TB; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[a][b][r] += bi;
            }
        } else {
#pragma unroll
            for (int b = 0; b < TB; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float bj = (float)(g.bias + j0)[min(64 * wj + 32 * (b ^ wb) + 8 * (r >> 2) + 4 * fh + (r & 3), (int)min<int64_t>(QW_BN, g.N - j0) - 1)];
#pragma unroll
                    for (int a = 0; a < TA; a++) acc[a][b][r] += bj;
                }
        }
    }
    half_t *out = g.out + s * g.o_bs;
    if (g.vec_out) { // through LDS, as above
        constexpr int OLD = QW_BM + 8, CPR = QW_BM / 8;
        half_t *Os = (half_t *)smem;
        static_assert((size_t)QW_BN * OLD * 2 <= QW_LDS, "the staged output tile fits");
        __syncthreads(); // every wavefront's LDS-DMA has landed
        rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
                for (int b = 0; b < TB; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        Os[(64 * wj + 32 * (b ^ wb) + 8 * (r >> 2) + 4 * fh + (r & 3)) * OLD + iw + 32 * a] = (half_t)rt_act_k<decltype(has_act)::value>(acc[a][b][r]);
        });
        __syncthreads();
#pragma unroll
        for (int k = 0; k < QW_BN * CPR / 512; k++) {
            const int idx = t + 512 * k, row = idx / CPR, c = idx % CPR;
            if (j0 + row < g.N && i0 + 8 * c < g.M) *(uint4_t *)(out + (j0 + row) * g.o_js + i0 + 8 * c) = *(const uint4_t *)(Os + row * OLD + 8 * c);
        }
        return;
    }
    rt_with_act(g.act, [&](auto has_act) {
#pragma unroll
        for (int a = 0; a < TA; a++) {
            const int64_t i = i0 + iw + 32 * a;
            if (i >= g.M) continue;
#pragma unroll
            for (int b = 0; b < TB; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int64_t j = j0 + 64 * wj + 32 * (b ^ wb) + 8 * (r >> 2) + 4 * fh + (r & 3);
                    if (j < g.N) out[i * g.o_is + j * g.o_js] = (half_t)rt_act_k<decltype(has_act)::value>(acc[a][b][r]);
                }
        }
    });
}

// Second pass of 3 to 8 rows: the shares' sums, bias, activation, rounding, a thread per output.  Infinite activations make the factored sums NaN (inf - inf
// of the two terms, 0 * inf of a nibble) where a weight times one is an infinity, as in the streaming kernel that takes these products without a
// workspace: a sum that is not finite is made again weight by weight (finite operands cannot give one: |d sc q x| < 2^42).
// 2560 x 10240 at 3 / 5 / 8 rows, both passes, with the other products' second pass and this: 13.7 / 13.4 / 13.4 and 12.7 / 12.5 / 12.5 us.
__global__ __launch_bounds__(256) void q4k_few_sums_kernel(GemmQ4kArgs g) {
    const int64_t s = blockIdx.y, n = g.M * g.N; // < 2^31: K is shared only where the tiles are no more than the compute units
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= n) return;
    const uint32_t j = idx / (uint32_t)g.M, i = idx - j * (uint32_t)g.M;
    const float *pt = g.partial + s * g.ksplit * n + idx;
    float v = 0.f;
#pragma unroll 4
    for (int z = 0; z < g.ksplit; z++) v += pt[z * n];
    if (!(fabsf(v) < INFINITY)) {
        const uint8_t *blk = g.blocks + ((g.a_stack == 1 ? 0 : s) * g.M + i) * g.nsb * 144;
        const half_t *x = g.X + (g.b_stack == 1 ? 0 : s) * g.b_bs + j * g.b_js;
        v = 0.f;
        for (int64_t b = 0; b < g.nsb; b++, blk += 144, x += 256) {
            const half2_t dm = *(const half2_t *)blk;
            for (int sub = 0; sub < 8; sub++) {
                int sc, mn;
                q4k_scale_min(sub, blk + 4, sc, mn);
                const float d = (float)dm[0] * (float)sc, m = (float)dm[1] * (float)mn;
                for (int e = 0; e < 32; e++) {
                    const float q = (float)(blk[16 + 32 * (sub >> 1) + e] >> (4 * (sub & 1)) & 15);
                    v += (d * q - m) * (float)x[32 * sub + e];
                }
            }
        }
    }
    if (g.has_bias) v += (float)g.bias[g.bias_on_rows ? i : j];
    g.out[s * g.o_bs + i * g.o_is + j * g.o_js] = (half_t)rt_act(v, g.act);
}

RT_TUNABLE(g_gemm_q4k_cfg, 0); // 14 / 24: always one / two weight tiles per wavefront (for comparisons)
RT_TUNABLE(g_gemm_q4k_disable, 0); // non-zero keeps Q4_K prefill on the generic kernel (for comparisons)

// Kernel and workgroups that share K, by an estimate in microseconds.  Of the first kernel: 5.5 + step * super-blocks of a share, 0.95 a
// step with one weight tile per wavefront, 1.6 with two, and the second kernel's time; more tiles of 128 rows than compute units run as
// many rounds, from four on they level out.  A wavefront's super-blocks are a chain, so with few tiles a long K
// took as long as with many; shared (M x K at activation rows, K whole and shared, us): 2560 x 10240 at 64 38.4 and 16.4, 3072 x 8192
// at 32 31.6 and 15.4, at 100 31.6 and 21.0, 3584 x 9472 at 148 38.1 and 30, 1024 x 4096 at 128 17.6 and 11.7, 2560 x 2560 at 40
// 12.3 and 10.2.  The margin of 0.3: 430 x 1280 at 228 took 10.1 whole and 10.9 in 5 shares, 828 x 1280 at 70 10.2 and 8.8.
// Without a workspace (and, of the first kernel, with more tiles of 128 rows than compute units) K stays whole.
// Of the 256 x 128 tiles: 7 + step * super-blocks of a workgroup, 3.4 a step while half the compute units rest, 4.5 (the clock falls) from 70 %
// of them on.  They are taken where that is less, by 3 % for what the estimate does not know (first kernel and this, us): 8192 x 3072 at
// 1000 75.2 and 60.2, 3072 x 8192 at 1000 91.6 and, in two shares, 75.3, 2560 x 10240 at 512 60.3 and, in six, 46.4, 6720 x 1024 at 939 31.2 and 24.2, 12864 x 7936 at
// 211 88.9 and 79.3; left to the first kernel: 13312 x 3840 at 569 (260 tiles) 94 and 128, 5376 x 1696 at 276 20 and 26, 4544 x 1536 at 775 23.6 and 29.4.
struct Q4kChoice {
    int ta = 2, ks = 1; // 16-row tiles per wavefront: 1, 2; 4: gemm_q4k_wide_kernel
};
static bool gemm_q4k_takes(const Problem &p) {
    return p.a_dt == RT_Q4_K && p.act_dt == RT_F16 && p.K % 256 == 0 && p.K >= 256 && p.b_ks == 1 && p.M >= 64 && p.N >= 3 && p.stacks <= 65535;
}
static Q4kChoice q4k_choose(const Problem &p, const DeviceInfo &dev, bool may_split) {
    // Four multiplying wavefronts of 32 weight rows x 64 activation rows each; when the grid of 16-row wavefronts
    // (64 weight rows per workgroup) still fits the compute units in one round, those: half the work per wavefront
    // (8192 x 3072 at 64 / 128 rows: 15.7 / 16.8 us against 22.6 / 23.6; 3072 x 8192 at 256 rows: 35 against 52 us).
    const int64_t tiles_j = (p.N + QR_BN - 1) / QR_BN, nsb = p.K / 256, cus = dev.num_cus;
    const int64_t wgs = ((p.M + 127) / 128) * tiles_j * p.stacks;
    auto sums = [&](int ks) { return 2.6f + 0.1f * ks + (float)(p.stacks * ks * p.M * p.N) * (4.f / 4.5e6f); }; // the second kernel
    Q4kChoice best;
    best.ta = ((p.M + 63) / 64) * tiles_j <= cus ? 1 : 2;
    float least = 5.2f + (best.ta == 1 ? 0.95f : 1.6f) * nsb;
    if (wgs > cus) {
        least = 5.2f + 1.6f * (float)nsb * (wgs <= 4 * cus ? (float)((wgs + cus - 1) / cus) : (float)wgs / (float)cus + 0.5f);
    } else if (may_split) {
        for (int ta = 1; ta <= 2; ta++) {
            const int64_t n = ((p.M + 64 * ta - 1) / (64 * ta)) * tiles_j * p.stacks;
            for (int ks = 2; ks <= 16 && n * ks <= cus; ks++) {
                const int64_t share = (nsb + ks - 1) / ks;
                if ((ks - 1) * share >= nsb) continue;
                const float us = 5.5f + (ta == 1 ? 0.95f : 1.6f) * share + sums(ks);
                if (us < least) least = us, best.ta = ta, best.ks = ks;
            }
        }
    }
    // the 256 x 128 tiles
    const int64_t n = ((p.M + QW_BM - 1) / QW_BM) * ((p.N + QW_BN - 1) / QW_BN) * p.stacks;
    for (int ks = 1; ks <= (may_split ? 16 : 1) && (ks == 1 || n * ks <= cus); ks++) {
        const int64_t share = (nsb + ks - 1) / ks;
        if ((ks - 1) * share >= nsb) continue;
        const float step = 3.4f + 1.1f * std::min(1.f, std::max(0.f, 5.f * (float)(n * ks) / (float)cus - 2.5f));
        const float us = 7.f + step * (float)((n * ks + cus - 1) / cus * share) + (ks > 1 ? sums(ks) : 0.f);
        if (1.03f * us < least) least = 1.03f * us, best.ta = 4, best.ks = ks;
    }
    return best;
}
// bytes of workspace with which launch_gemm_q4k shares this problem's K (0: it does not, or launch_gemv_chunked takes the problem first)
uint64_t gemm_q4k_workspace_bytes(const Problem &p, const DeviceInfo &dev) {
    if (!gemm_q4k_takes(p)) return 0;
    Problem chunk = p;
    chunk.N = std::min<int64_t>(p.N, 16);
    if (p.N <= 32 && gemv_q4k_mfma_fits(chunk, dev)) return 0;
    const int ks = q4k_choose(p, dev, true).ks;
    return ks > 1 ? (uint64_t)p.stacks * ks * p.M * p.N * sizeof(float) : 0;
}
// Whether 3 to 16 vectors are launch_gemm_q4k's: where the streaming matrix-core kernel's LDS ends (9 to 16 from K = 4352, 3 to 8 from 8448 on), up to
// 8, which the streaming kernel without matrix cores takes, only with K shared.  us, M x K, that or the generic kernel, here, here with K whole: 2560 x 4352 at 9
// / 16 vectors 71 / 72, 10.3, 18.3; x 10240 161 / 163, 13.5, 38; x 14336 224 / 227, 16, 52; 1280 x 8448 at 3 / 8 15.6 / 23.0, 9.7, 32; 2560 x 10240 at 3 / 5 / 8 16.8 / 21.9 / 32.2,
// 12.5, 38.
bool gemm_q4k_few(const Problem &p, const DeviceInfo &dev) {
    if (!gemm_q4k_takes(p) || p.N > 16 || gemv_q4k_mfma_fits(p, dev)) return false;
    if (p.N > 8) return true;
    const uint64_t need = gemm_q4k_workspace_bytes(p, dev);
    return need > 0 && p.workspace && !((uintptr_t)p.workspace & 15u) && p.workspace_bytes >= need;
}

// Q4_K weights x K-contiguous f16 activations: more rows than one streaming launch takes, and gemm_q4k_few.
// hipErrorNotSupported: another kernel must take the problem.
hipError_t launch_gemm_q4k(const Problem &p, const void *A, const void *B, const void *bias, void *out, hipStream_t stream,
                           const DeviceInfo &dev) {
    if (g_gemm_q4k_disable || !gemm_q4k_takes(p) || (p.N <= 16 && !gemm_q4k_few(p, dev))) return hipErrorNotSupported;
    if (((uintptr_t)A & 15u) || ((uintptr_t)B & 15u) || (p.b_js * 2) % 16 || (p.b_bs * 2) % 16) return hipErrorNotSupported;
    // 32-bit offsets within a stack, in bytes
    if (p.M * (p.K / 256) * 144 >= (int64_t(1) << 32) || p.N * p.b_js >= (int64_t(1) << 31)) return hipErrorNotSupported;
    GemmQ4kArgs g{};
    g.blocks = (const uint8_t *)A, g.X = (const half_t *)B, g.bias = (const half_t *)bias, g.out = (half_t *)out;
    g.M = p.M, g.N = p.N, g.nsb = p.K / 256;
    g.a_stack = p.a_stack, g.b_stack = p.b_stack;
    g.b_bs = p.b_bs, g.b_js = p.b_js;
    g.o_bs = p.o_bs, g.o_is = p.o_is, g.o_js = p.o_js;
    g.has_bias = p.has_bias, g.bias_on_rows = p.bias_on_rows, g.act = p.act;
    const int64_t tiles_j = (p.N + QR_BN - 1) / QR_BN;
    g.vec_out = p.o_is == 1 && p.M % 8 == 0 && p.o_js % 8 == 0 && p.o_bs % 8 == 0 && ((uintptr_t)out & 15u) == 0;
    Q4kChoice c = q4k_choose(p, dev, p.workspace && !((uintptr_t)p.workspace & 15u));
    if (c.ks > 1 && p.workspace_bytes < (uint64_t)p.stacks * c.ks * p.M * p.N * sizeof(float)) c = q4k_choose(p, dev, false);
    g.ksplit = c.ks, g.sb_len = (g.nsb + c.ks - 1) / c.ks, g.partial = (float *)p.workspace;
    if (g_gemm_q4k_cfg) c.ta = g_gemm_q4k_cfg == 14 ? 1 : 2;
    auto go = [&](auto kernel, int bm, int bn, int waves, size_t lds) -> hipError_t {
        const int64_t tiles_i = (p.M + bm - 1) / bm, tiles_j = (p.N + bn - 1) / bn;
        g.tiles_j = (int)tiles_j;
        if (tiles_i * tiles_j > 0x7fffffff) return hipErrorNotSupported;
        g.remap = (tiles_i * tiles_j) % 8 == 0;
        if (const hipError_t e = ensure_lds_limit<decltype(kernel)::value>(); e != hipSuccess) return e;
        hipLaunchKernelGGL(decltype(kernel)::value, dim3((unsigned)(tiles_i * tiles_j), (unsigned)p.stacks, (unsigned)c.ks), dim3(64 * waves), lds, stream, g);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        if (c.ks == 1) return hipSuccess;
        if (p.N > 8) return launch_splitk_sums(p, bias, out, g.partial, c.ks, stream);
        hipLaunchKernelGGL(q4k_few_sums_kernel, dim3((unsigned)((p.M * p.N + 255) / 256), (unsigned)p.stacks), dim3(256), 0, stream, g);
        return hipGetLastError();
    };
    if (c.ta == 4) return go(std::integral_constant<void (*)(GemmQ4kArgs), &gemm_q4k_wide_kernel>{}, QW_BM, QW_BN, 8, QW_LDS);
    if (c.ta == 1) return go(std::integral_constant<void (*)(GemmQ4kArgs), &gemm_q4k_kernel<1, 4, 4>>{}, 64, QR_BN, 8, QR_LDS);
    // more than one workgroup per compute unit: no loading wavefronts (see the file comment)
    if (((p.M + 127) / 128) * tiles_j * p.stacks > dev.num_cus) return go(std::integral_constant<void (*)(GemmQ4kArgs), &gemm_q4k_kernel<2, 4, 0>>{}, 128, QR_BN, 4, QR_LDS);
    return go(std::integral_constant<void (*)(GemmQ4kArgs), &gemm_q4k_kernel<2, 4, 4>>{}, 128, QR_BN, 8, QR_LDS);
}

} // namespace rt
