// Products with f32 activations on the bf16 matrix cores:
//   C[s, i, j] = sum_k X[s, i, k] * Y[s, j, k] (+ bias),  f32 out, f32 accumulate,
// X f32, Y f32 or a Q8_0F weight.  An f32 MFMA does 64 flops per cycle and SIMD, a bf16 MFMA 1024, and an f32 number is the
// exact sum of three bf16 ones ("limbs"): l0 = rn(x), l1 = rn(x - l0), l2 = x - l0 - l1, eight significant bits each and
// every difference exact.
//   f32 x f32    six MFMAs per tile and 16 k: l0.l0, l0.l1, l1.l0, l1.l1, l0.l2, l2.l0.  The three products left out are at
//                most 2^-26 of |x.y| together, a quarter of the rounding of a single f32 product.  The f32 MFMA rounds after every
//                product (K = 2 and 4: 0.77 and 0.62 of its results are correctly rounded, as of a chain of fused
//                multiply-adds); here sixteen products are added before the accumulator is rounded, six times per 16 k.
//                Relative errors against float64 at K = 3 / 64 / 384 / 2560 / 10240: 3.3e-8 / 1.1e-7 / 2.9e-7 / 2.8e-7 /
//                4.1e-7 (the last two with K shared), f32 MFMA 3.5e-8 / 1.4e-7 / 3.5e-7 / 9.1e-7 / 1.8e-6.  The sums are cut off, not
//                rounded to nearest: -1e-8 to -4e-7 on positive data for K = 100 to 10240, within the errors above.
//   f32 x Q8_0F  a code is an integer of at most eight bits, one exact limb: three MFMAs per tile and 16 k, from a zero
//                accumulator per block of 32, whose sums are folded into the accumulators with the block's scale in f32,
//                so no weight is rounded.
// bf16's smallest subnormal number is 2^-133 (the matrix cores take subnormal operands), f32's 2^-149: f32 operands are
// multiplied by 2^16 before they are split, so the sum of the limbs is exact for every f32 number, and the accumulator by
// 2^-32 (2^-16 against codes) as the bias is added.
// An operand whose limbs are not finite (infinities, NaNs, magnitudes from 2^112 on) makes its outputs NaN, a sum past 2^96
// (2^112) is infinite: a 32 x 32 tile with an output that is not finite is computed once more on the f32 matrix cores, so what the f32
// arithmetic gives for such inputs is what is stored.
//
// Wavefronts 4 and up load (global -> registers two stages ahead), split into limbs and store the limb planes to LDS;
// wavefronts 0..3 read fragments and multiply.  The split is six and a half vector instructions per value.  Beside a
// wavefront that issues 32x32x16 MFMAs back to back a SIMD still issues a vector instruction of its other wavefronts every
// 5.6 cycles (measured; 6.4 beside 16x16x32, whose MFMAs take 19 cycles for 16), so the splitting hides behind the MFMAs
// of a large tile, and two loading wavefronts per SIMD use those slots better than one.  Three LDS stages of 32 k: while
// stage s is multiplied, stage s + 1 is complete or about to be (its first fragments are read at the end of stage s) and
// stage s + 2 is being written; one barrier per stage, in the middle of the multiplication.  A workgroup walks its items
// (output tiles, or shares of one along K) as one sequence of stages, so the loads of the next tile run under the output of
// this one.
//
// LDS: per stage one plane per limb, rows of 64 bytes; row r holds its four 16-byte pieces at slots c ^ limb_swz(r), so
// that sixteen rows' pieces of one c cover all 64 banks, and so do the four-row groups of two neighbouring c that a 16-byte
// read of a wavefront takes together (no bank conflicts in either direction, by SQ_LDS_BANK_CONFLICT).
//
// Measured (device time, f32 MFMA kernels it replaces -> here): [1500 x 384] . [384 x 1536] + GELU 25.6 -> 17.9 us; the
// Whisper attention's [6 x 1500 x 64] . [6 x 64 x 1500] 31.5 -> 23.6, P . V 47.2 -> 22.0; Q8_0F weights against 200 rows,
// 10240 x 2560 163 -> 62 us, 2560 x 10240 (K shared) 299 -> 56.  What bounds it: the splitting and code conversion beside the
// MFMAs (a stage of 96 x 128 f32 takes 1650 cycles for 1190 of MFMAs), 2.7 us from launch to the first MFMA, and 1.7 us of
// output behind the last.  The f32 forms keep 20 to 50 scalar registers in lanes of vector registers; nothing goes to scratch.
#include "device_common.h"

#include <algorithm>

namespace rt {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_u __attribute__((ext_vector_type(4), aligned(4)));

// n / d for 0 <= n < 2^31 by a multiplication (round-up method of Granlund and Montgomery, 1994): an item is decoded on the way to
// the first load of a workgroup, and three scalar divisions there are a quarter of a microsecond.
struct LimbDiv {
    int d = 1;
    uint32_t m = 0, l = 0;
    LimbDiv() = default;
    explicit LimbDiv(int div) : d(div) {
        while ((1ull << l) < (uint64_t)d) l++;
        m = (uint32_t)(((1ull << 32) * ((1ull << l) - (uint64_t)d)) / (uint64_t)d + 1);
    }
    __device__ __forceinline__ int of(int n) const { return (int)((__umulhi(m, (uint32_t)n) + (uint32_t)n) >> l); }
};

struct GemmLimbArgs {
    const float *X;
    const void *Y;       // f32, or Q8_0F codes
    const float *scales; // Q8_0F scale stream of Y
    const float *bias;
    float *out;
    int64_t M, N, K;
    int64_t x_stack, y_stack;
    int64_t x_bs, x_is, x_ks;
    int64_t y_bs, y_js, y_ks;
    int64_t o_bs, o_is, o_js; // o_js is 1 for outputs written in whole lines
    int has_bias, bias_on_i, act;
    LimbDiv tiles_i, tiles_j, shares;
    int ksplit;
    int nk, stages;      // stages of 32 k: of one item, of all of K
    int items;           // stacks * shares * tiles_j * tiles_i; no more than the grid where ksplit > 1
    float *partial;      // split K: [stack][share][M][N]
};

__device__ __forceinline__ int limb_swz(int r) { // 0, 2, 3, 1 for r / 4 mod 4 = 0 .. 3
    const int i = (r >> 2) & 3;
    return (((i ^ (i >> 1)) & 1) << 1) | (i >> 1);
}

constexpr float kLimbScale = 65536.f;

// two f32 -> two bf16 in one register, and what is left of each
__device__ __forceinline__ uint32_t limb_take(float &x0, float &x1) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x0, x1}, bf16x2_t));
    x0 -= __builtin_bit_cast(float, h << 16);
    x1 -= __builtin_bit_cast(float, h & 0xffff0000u);
    return h;
}
// four int8 codes -> four bf16: a signed byte converted to f32 in one instruction has at most eight significant bits, all in
// its upper half
__device__ __forceinline__ uint2_t limb_codes(uint32_t v) {
    uint32_t a, b, c, d;
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(a) : "v"(v));
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(b) : "v"(v));
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(c) : "v"(v));
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(d) : "v"(v));
    return uint2_t{__builtin_amdgcn_perm(b, a, 0x07060302u), __builtin_amdgcn_perm(d, c, 0x07060302u)};
}

// One operand's part of a loading thread's work: R rows of a stage of 32 k, over PT threads.  Loads are a uniform
// pointer that advances along K plus 32-bit lane offsets that stay (the launcher checks that a tile's rows span less than
// 2 GiB).  A unit is W values of one row: k = 4c .. 4c + 3 and, with W = 8, k = 16 + 4c .. 16 + 4c + 3.  The order
// of k inside a stage is free as long as both operands agree; in this one four neighbouring lanes load 64 consecutive
// bytes, which the memory pipeline takes in one access (32 bytes apart it needs two), and a unit is a 16-byte piece of a limb row.
// KC: K is the contiguous axis (K >= 4).  Otherwise any strides, meant for contiguous rows: neighbouring lanes take
// neighbouring rows and a load is one value.
template <int R, bool KC, int PT> struct LimbFloat {
    static constexpr int W = R % (PT / 4) == 0 ? 8 : 4;    // values per unit: whole pieces where the threads deal out evenly
    static constexpr int UNITS = R * 32 / W, U = (UNITS + PT - 1) / PT, UPB = 32 / W, PLANES = 3; // units: of the stage, per thread, per row
    static constexpr int NO = KC ? U * W / 4 : U * W;             // load instructions
    static constexpr int BYTES = PLANES * R * 64;
    const uint8_t *base;
    uint32_t off[NO];
    float r[2][U * W];
    static __device__ __forceinline__ int unit(int u, int t) { return UNITS % PT == 0 ? u * PT + t : min(u * PT + t, UNITS - 1); }
    static __device__ __forceinline__ int row(int u, int t) { return KC ? unit(u, t) / UPB : unit(u, t) % R; }
    static __device__ __forceinline__ int piece(int u, int t) { return KC ? unit(u, t) % UPB : unit(u, t) / R; }
    // k of value e (a multiple of 4) of a unit within the stage
    static __device__ __forceinline__ int kin(int u, int t, int e) { return 4 * piece(u, t) + 4 * e; }
    // KC with fewer than four values left: the pointer goes back so that the last four are loaded
    __device__ __forceinline__ void back(int left) {
        if (KC && left < 4) base -= 4 * (4 - left);
    }
    // rows past the end repeat the last one (never stored); k past `left` values repeats the last ones (zeroed in store)
    __device__ __forceinline__ void aim(int64_t rows_left, int left, int64_t rs, int64_t ks, int t) {
        const int lim = max(left - (KC ? 4 : 1), 0), rl = (rows_left < R ? (int)rows_left : R) - 1;
#pragma unroll
        for (int i = 0; i < NO; i++) {
            const int u = i / (NO / U), e = (KC ? 4 : 1) * (i % (NO / U));
            const int rw = min(row(u, t), rl), k = min(kin(u, t, e & ~3) + (e & 3), lim);
            off[i] = 4u * ((uint32_t)rw * (uint32_t)rs + (uint32_t)k * (KC ? 1u : (uint32_t)ks));
        }
    }
    __device__ __forceinline__ void load(int set) {
#pragma unroll
        for (int i = 0; i < NO; i++) {
            if constexpr (KC) {
                const float4_t v = *(const float4_u *)(base + off[i]); // rows may start anywhere: dword-aligned 16-byte loads
#pragma unroll
                for (int e = 0; e < 4; e++) r[set][4 * i + e] = v[e];
            } else {
                r[set][i] = *(const float *)(base + off[i]);
            }
        }
    }
    // `left`: values of K in this stage
    __device__ __forceinline__ void store(int set, uint8_t *st, int left, int t) {
        if (left < 32) { // uniform: zeros past the end of K
#pragma unroll
            for (int i = 0; i < U * W / 4; i++) {
                const int n = left - kin(4 * i / W, t, 4 * i % W); // of these four, inside K
                float *v = r[set] + 4 * i;
                const float a = v[0], b = v[1], c = v[2], d = v[3];
                if constexpr (KC) { // four across the end were loaded as the last four
                    v[0] = n >= 4 ? a : n == 3 ? b : n == 2 ? c : n == 1 ? d : 0.f;
                    v[1] = n >= 4 ? b : n == 3 ? c : n == 2 ? d : 0.f;
                    v[2] = n >= 4 ? c : n == 3 ? d : 0.f;
                    v[3] = n >= 4 ? d : 0.f;
                } else {
                    v[0] = n > 0 ? a : 0.f, v[1] = n > 1 ? b : 0.f, v[2] = n > 2 ? c : 0.f, v[3] = n > 3 ? d : 0.f;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (UNITS % PT && u * PT + t >= UNITS) break;
            const int rw = row(u, t), q = piece(u, t); // with W = 4, q is half a piece: pieces q % 4, low half first
            uint8_t *d = st + rw * 64 + (((q & 3) ^ limb_swz(rw)) << 4) + ((q >> 2) << 3);
            float x[W];
#pragma unroll
            for (int e = 0; e < W; e++) x[e] = r[set][u * W + e] * kLimbScale;
#pragma unroll
            for (int l = 0; l < 3; l++) {
                uint32_t h[W / 2];
#pragma unroll
                for (int e = 0; e < W / 2; e++) h[e] = limb_take(x[2 * e], x[2 * e + 1]);
                if constexpr (W == 8) *(uint4_t *)(d + l * R * 64) = uint4_t{h[0], h[1], h[2], h[3]};
                else *(uint2_t *)(d + l * R * 64) = uint2_t{h[0], h[1]};
            }
        }
    }
};

// Q8_0F rows: a unit is 16 codes, half a block: half of each of a limb row's four pieces.  The stage's scales sit behind
// the plane.
template <int R, int PT> struct LimbCodes {
    static constexpr int UNITS = R * 2, U = (UNITS + PT - 1) / PT, PLANES = 1;
    static constexpr int BYTES = R * 64 + R * 4;
    static_assert(R <= PT, "a thread per scale");
    const uint8_t *base, *sbase;
    uint32_t off[U], soff;
    uint4_t r[2][U];
    float sc[2];
    static __device__ __forceinline__ int unit(int u, int t) { return UNITS % PT == 0 ? u * PT + t : min(u * PT + t, UNITS - 1); }
    __device__ __forceinline__ void aim(int64_t rows_left, int64_t rs, int t) {
        const int rl = (rows_left < R ? (int)rows_left : R) - 1;
#pragma unroll
        for (int u = 0; u < U; u++) off[u] = (uint32_t)min(unit(u, t) >> 1, rl) * (uint32_t)rs + 16u * (unit(u, t) & 1);
        soff = 4u * ((uint32_t)min(t, rl) * (uint32_t)(rs >> 5));
    }
    __device__ __forceinline__ void load(int set) {
#pragma unroll
        for (int u = 0; u < U; u++) r[set][u] = *(const uint4_t *)(base + off[u]);
        sc[set] = *(const float *)(sbase + soff);
    }
    __device__ __forceinline__ void store(int set, uint8_t *st, int t) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (UNITS % PT && u * PT + t >= UNITS) break;
            const int v = unit(u, t), rw = v >> 1, sw = limb_swz(rw);
            uint8_t *d = st + rw * 64 + ((v & 1) << 3);
#pragma unroll
            for (int c = 0; c < 4; c++) *(uint2_t *)(d + ((c ^ sw) << 4)) = limb_codes(r[set][u][c]);
        }
        if (t < R) *(float *)(st + R * 64 + t * 4) = sc[set];
    }
};

// BI x BJ outputs per item; WI x (4 / WI) multiplying wavefronts; PW loading wavefronts.
template <int BI, int BJ, int WI, int PW, bool Q8, bool XKC, bool YKC>
__global__ __launch_bounds__(256 + 64 * PW) void gemm_limb_kernel(GemmLimbArgs g) {
    constexpr int WJ = 4 / WI, TM = BI / WI / 32, TN = BJ / WJ / 32, PT = 64 * PW;
    constexpr int PY = Q8 ? 1 : 3;
    using LX = LimbFloat<BI, XKC, PT>;
    using LY = std::conditional_t<Q8, LimbCodes<BJ, PT>, LimbFloat<BJ, YKC, PT>>;
    constexpr int STAGE = LX::BYTES + LY::BYTES;
    static_assert(TM * WI * 32 == BI && TN * WJ * 32 == BJ && STAGE % 16 == 0, "tile must split into 32 x 32 MFMA tiles");

    extern __shared__ __attribute__((aligned(16))) uint8_t smem[]; // [3][STAGE]
    const int t = threadIdx.x - 256, lane = threadIdx.x & 63; // t: of the loading threads
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // Items of this workgroup: workgroups go round the 8 XCDs, each with an L2 of its own; XCD x takes the x-th eighth of
    // the items (in order: stack, share of K, column block, row block) and its workgroups deal them out among themselves.
    const int G = gridDim.x, w = blockIdx.x;
    int first, step, count;
    if ((G & 7) == 0) {
        const int lo = (int)((int64_t)g.items * (w & 7) / 8), hi = (int)((int64_t)g.items * ((w & 7) + 1) / 8);
        first = lo + (w >> 3), step = G >> 3;
        count = first < hi ? (hi - first + step - 1) / step : 0;
    } else {
        first = w, step = G, count = (g.items - w + G - 1) / G;
    }
    struct Item {
        int64_t s, i0, j0, k0;
        int z, nk; // share of K, stages
    };
    auto item = [&](int n) {
        const int it = first + n * step;
        Item r;
        const int a = g.tiles_i.of(it), b = g.tiles_j.of(a), c = g.shares.of(b);
        const int ti = it - a * g.tiles_i.d, tj = a - b * g.tiles_j.d;
        r.z = b - c * g.shares.d, r.s = c;
        r.i0 = (int64_t)ti * BI, r.j0 = (int64_t)tj * BJ, r.k0 = (int64_t)r.z * g.nk * 32;
        r.nk = min(g.nk, g.stages - r.z * g.nk); // the last share may be shorter
        return r;
    };
    if (count == 0) return;
    const int total = g.ksplit == 1 ? count * g.nk : item(0).nk; // stages, and barriers of every wavefront; a launch that shares K has one item per workgroup
    auto meet = [&]() __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): LDS stores are visible, fragment reads have returned
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    if (wave >= 4) {
        LX lx;
        LY ly;
        int n = 0, kt = 0, nk = 0;               // next stage to request
        int64_t k0 = 0, rows_x = 0, rows_y = 0;  // of that stage
        int left[2];                             // values of K in the stage each set holds
        auto request = [&](int set) __attribute__((always_inline)) {
            const bool fresh = kt == 0;
            if (fresh) {
                const Item it = item(min(n, count - 1));
                nk = it.nk, k0 = it.k0, rows_x = g.M - it.i0, rows_y = g.N - it.j0;
                lx.base = (const uint8_t *)(g.X + (g.x_stack == 1 ? 0 : it.s) * g.x_bs + it.i0 * g.x_is + k0 * g.x_ks);
                const int64_t y_el = (g.y_stack == 1 ? 0 : it.s) * g.y_bs + it.j0 * g.y_js;
                if constexpr (Q8) ly.base = (const uint8_t *)g.Y + y_el + k0, ly.sbase = (const uint8_t *)(g.scales + ((y_el + k0) >> 5));
                else ly.base = (const uint8_t *)((const float *)g.Y + y_el + k0 * g.y_ks);
            }
            left[set] = g.K - k0 < 32 ? (int)(g.K - k0) : 32;
            if (fresh || left[set] < 32) {
                lx.aim(rows_x, left[set], g.x_is, g.x_ks, t), lx.back(left[set]);
                if constexpr (Q8) ly.aim(rows_y, g.y_js, t); // K is whole blocks
                else ly.aim(rows_y, left[set], g.y_js, g.y_ks, t), ly.back(left[set]);
            }
            lx.load(set);
            ly.load(set);
            k0 += 32;
            lx.base += 128 * g.x_ks;
            if constexpr (Q8) ly.base += 32, ly.sbase += 4;
            else ly.base += 128 * g.y_ks;
            if (++kt == nk) kt = 0, n++;
        };
        auto deliver = [&](int set, uint8_t *st) __attribute__((always_inline)) {
            lx.store(set, st, left[set], t);
            if constexpr (Q8) ly.store(set, st + LX::BYTES, t);
            else ly.store(set, st + LX::BYTES, left[set], t);
        };
        request(0);
        request(1);
        int buf = 0;
        // two stages a turn, without a way out in between (the waits on the loads are counted exactly then); past an odd
        // number of stages the second one is stored where nobody reads any more
        for (int s = 0; s < total; s += 2) {
            deliver(0, smem + buf * STAGE);
            request(0);
            meet();
            buf = buf == 2 ? 0 : buf + 1;
            deliver(1, smem + buf * STAGE);
            request(1);
            if (s + 1 < total) meet();
            buf = buf == 2 ? 0 : buf + 1;
        }
        return;
    }

    // ---- multiplying wavefronts
    const int wi = wave / WJ, wj = wave % WJ;
    const int fr = lane & 31, fh = lane >> 5;
    // 16 k of a row (half h of the stage) are pieces 2h, 2h + 1: this lane's is 2h + fh
    const int l0 = fr * 64 + ((fh ^ limb_swz(fr)) << 4), flip = 32; // piece 2 + fh: slot ^ 2
    struct Spot { // a stage's addresses of this lane; what differs within the stage is a constant
        const uint8_t *x[2], *y[2], *s;
    };
    auto spot = [&](int buf) {
        const uint8_t *x = smem + buf * STAGE + wi * (BI / WI) * 64, *y = smem + buf * STAGE + LX::BYTES + wj * (BJ / WJ) * 64;
        return Spot{{x + l0, x + (l0 ^ flip)}, {y + l0, y + (l0 ^ flip)}, smem + buf * STAGE + LX::BYTES + BJ * 64 + (wj * (BJ / WJ) + fr) * 4};
    };
    auto frag_x = [&](const Spot &p, int h, int l, int a) { return __builtin_bit_cast(bf16x8_t, *(const uint4_t *)(p.x[h] + l * BI * 64 + a * 2048)); };
    auto frag_y = [&](const Spot &p, int h, int l, int b) { return __builtin_bit_cast(bf16x8_t, *(const uint4_t *)(p.y[h] + l * BJ * 64 + b * 2048)); };
    const float16_t zero = {};
    float16_t acc[TM][TN];
    auto clear = [&]() {
#pragma unroll
        for (int a = 0; a < TM; a++)
#pragma unroll
            for (int b = 0; b < TN; b++) acc[a][b] = zero;
    };
    float bj[TN]; // bias of this lane's columns, fetched when the item begins
    auto fetch_bias = [&](const Item &it) {
#pragma unroll
        for (int b = 0; b < TN; b++) {
            const int64_t j = it.j0 + wj * (BJ / WJ) + 32 * b + fr;
            bj[b] = g.has_bias && !g.bias_on_i && g.ksplit == 1 ? g.bias[min(j, g.N - 1)] : 0.f;
        }
    };
    uint64_t again = 0; // not zero once an output of this wavefront is not finite
    auto finish = [&](const Item &it) {
        const bool share = g.ksplit > 1;
        const int64_t iw = it.i0 + wi * (BI / WI), jw = it.j0 + wj * (BJ / WJ);
        const int64_t o_is = share ? g.N : g.o_is, o_js = share ? 1 : g.o_js;
        float *out = (share ? g.partial + (it.s * g.ksplit + it.z) * g.M * g.N : g.out + it.s * g.o_bs) + iw * o_is + jw * o_js;
        const bool row_bias = g.has_bias && g.bias_on_i && !share;
        const int act = share ? RT_ACT_NONE : g.act;
        constexpr float unscale = Q8 ? 1.f / kLimbScale : 1.f / (kLimbScale * kLimbScale);
        const int il = g.M - iw < BI ? (int)(g.M - iw) : BI, jl = g.N - jw < BJ ? (int)(g.N - jw) : BJ; // rows and columns inside
        float odd = 0.f; // NaN once an output of this lane is not finite
        // offsets inside the tile are 32-bit (the launcher checks)
        const uint32_t ois = (uint32_t)o_is, ojs = (uint32_t)o_js;
        if (ojs == 1 && !row_bias && (int)ois >= jl) {
            // Bounds are the buffer's: it ends with the tile's last element, and columns outside get an offset past any end.  Rows
            // outside lie past the end only where a row of the output is as long as the tile's part of it: an output of one
            // row may have any stride, a transposed one (one column of [N, 1]) has 1.
            const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(out, 0, il > 0 && jl > 0 ? (int)(4 * (((uint32_t)il - 1) * ois + (uint32_t)jl)) : 0, 0x00027000);
            rt_with_act(act, [&](auto has_act) {
#pragma unroll
                for (int b = 0; b < TN; b++) {
                    const int j = 32 * b + fr;
                    uint32_t off = j < jl ? 4u * ((uint32_t)(4 * fh) * ois + (uint32_t)j) : 0x80000000u;
#pragma unroll
                    for (int a = 0; a < TM; a++)
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            float v = acc[a][b][r];
                            odd = fmaf(v, 0.f, odd);
                            v = rt_act_k<decltype(has_act)::value>(fmaf(v, unscale, bj[b]));
                            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rsrc, off, 0, 0);
                            off += (r & 3) == 3 ? 20u * ois : 4u * ois;
                            if ((r & 7) == 7) __builtin_amdgcn_sched_barrier(0); // eight at a time: their chains of operations overlap
                        }
                }
            });
        } else { // outputs with a strided j axis, bias along i
#pragma unroll
            for (int b = 0; b < TN; b++)
#pragma unroll
                for (int a = 0; a < TM; a++) {
                    int i = 32 * a + 4 * fh, j = 32 * b + fr;
                    asm volatile("" : "+v"(i), "+v"(j)); // addresses and bounds tile by tile, not all at once
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        float v = acc[a][b][r];
                        odd = fmaf(v, 0.f, odd);
                        v = fmaf(v, unscale, bj[b]);
                        if (row_bias) v += g.bias[min(iw + i, g.M - 1)];
                        v = rt_act(v, act);
                        if (i < il && j < jl) out[(uint32_t)i * ois + (uint32_t)j * ojs] = v;
                        i += (r & 3) == 3 ? 5 : 1;
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
        }
        again |= __builtin_amdgcn_ballot_w64(odd != odd);
    };

    // Steps of a stage: f32, half h of the 32 k and row tile a, with X's fragments of the step and Y's of the half in two
    // sets each; Q8, row tile a, with X's fragments of both halves and Y's of the stage.  A step's fragments are requested a
    // step ahead.
    constexpr int LP[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}}; // limb pairs (of X, of Y), the small ones first
    constexpr int XS = Q8 && TM % 2 ? 3 : 2, XH = Q8 ? 2 : 1; // X: sets, halves per set
    static_assert(!Q8 || TM % XS == 0, "a stage starts with the set the one before it ended on");
    bf16x8_t fx[XS][XH][3], fy[2][TN][PY];
    int buf = 0, n = 0, kt = 0;
    Spot here = spot(0);
    const int nk = g.ksplit == 1 ? g.nk : total;
    fetch_bias(item(0));
    clear();
    meet(); // stage 0
#pragma unroll
    for (int l = 0; l < 3; l++)
#pragma unroll
        for (int h = 0; h < XH; h++) fx[0][h][l] = frag_x(here, h, l, 0);
#pragma unroll
    for (int b = 0; b < TN; b++)
#pragma unroll
        for (int l = 0; l < PY; l++) {
            fy[0][b][l] = frag_y(here, 0, l, b);
            if (Q8) fy[1][b][l] = frag_y(here, 1, l, b);
        }
    constexpr int PS = !Q8 ? 1 : TM * TN % 2 ? 3 : 2, PL = (TM * TN - 1) % PS; // sets of P, the last tile's
    static_assert(TM * TN % PS == 0, "a stage starts with the set after the one before it ended on");
    float16_t P[PS];           // Q8: a tile's sums from zero; folded while the next tile's MFMAs run
    float sc[Q8 ? 2 : 1][TN];  // scales of this stage and of the one before (of the tile still to fold)
    auto drop = [&]() {
        P[PL] = zero;
#pragma unroll
        for (int b = 0; b < TN; b++) sc[0][b] = sc[Q8 ? 1 : 0][b] = 0.f;
    };
    drop();
    for (int s = 0; s < total; s++) {
        buf = buf == 2 ? 0 : buf + 1;
        const Spot there = spot(buf);
        if constexpr (!Q8) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (h == 1 && s + 1 < total) meet(); // stage s + 1 is complete
#pragma unroll
                for (int a = 0; a < TM; a++) {
                    constexpr int kSteps = 2 * TM;
                    const int st = h * TM + a, cur = st & 1, nxt = cur ^ 1;
                    // the next step's X; Y of the other half: of this stage's second half during the first, of the next
                    // stage's first half during the second
#pragma unroll
                    for (int l = 0; l < 3; l++)
                        fx[nxt][0][l] = st + 1 == kSteps ? frag_x(there, 0, l, 0) : frag_x(here, (st + 1) / TM, l, (st + 1) % TM);
                    if (a == TM - 1)
#pragma unroll
                        for (int b = 0; b < TN; b++)
#pragma unroll
                            for (int l = 0; l < 3; l++) fy[h ^ 1][b][l] = h == 0 ? frag_y(here, 1, l, b) : frag_y(there, 0, l, b);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int p = 0; p < 6; p++)
#pragma unroll
                        for (int b = 0; b < TN; b++)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[cur][0][LP[p][0]], fy[h][b][LP[p][1]], acc[a][b], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        } else {
#pragma unroll
            for (int a = 0; a < TM; a++) {
                const int cur = a % XS, nxt = (a + 1) % XS;
                if (a == TM - 1 && s + 1 < total) meet(); // stage s + 1 is complete
#pragma unroll
                for (int l = 0; l < 3; l++)
#pragma unroll
                    for (int h = 0; h < 2; h++) fx[nxt][h][l] = a + 1 == TM ? frag_x(there, h, l, 0) : frag_x(here, h, l, a + 1);
                if (a == 0)
#pragma unroll
                    for (int b = 0; b < TN; b++) sc[1][b] = sc[0][b], sc[0][b] = *(const float *)(here.s + 128 * b);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < TN; b++) {
                    // tile (a, b) and, between its MFMAs, the fold of the tile before it
                    const int tl = a * TN + b, pc = tl % PS, pp = (tl + PS - 1) % PS;
                    const int fa = b > 0 ? a : (a + TM - 1) % TM, fb = (b + TN - 1) % TN;
                    const float d = sc[tl == 0 ? 1 : 0][fb];
#pragma unroll
                    for (int m = 0; m < 6; m++) {
                        const int h = m / 3, l = 2 - m % 3;
                        P[pc] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[cur][h][l], fy[h][b][0], m == 0 ? zero : P[pc], 0, 0, 0);
                        if (a == TM - 1 && m % 3 == 2) fy[h][b][0] = frag_y(there, h, 0, b); // read for the last time: the next stage's
#pragma unroll
                        for (int r = m * 16 / 6; r < (m + 1) * 16 / 6; r++) acc[fa][fb][r] = fmaf(d, P[pp][r], acc[fa][fb][r]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
        here = there;
        if (++kt == nk) {
            if constexpr (Q8) { // the last tile's sums
#pragma unroll
                for (int r = 0; r < 16; r++) acc[TM - 1][TN - 1][r] = fmaf(sc[0][TN - 1], P[PL][r], acc[TM - 1][TN - 1][r]);
                drop();
            }
            finish(item(n));
            kt = 0, n++; // with several items per workgroup every item has the same number of stages
            if (n < count) fetch_bias(item(n));
            clear();
        }
    }
    if (__builtin_expect_with_probability(again == 0, 1, 1.0)) return; // or the registers go to the loops below
    // The tiles with outputs that are not finite once more on the f32 matrix cores (see the file comment), after everything else: beside
    // the main loop's registers there is no room for it.  The arguments are read again through a pointer the compiler cannot
    // see through, or they would be kept, in spilled registers, from the kernel's start on.
    auto *ka = (const __attribute__((address_space(4))) GemmLimbArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka));
    const int64_t x_ks = XKC ? 1 : ka->x_ks, y_ks = YKC ? 1 : ka->y_ks;
    const bool share = ka->ksplit > 1, row_bias = ka->has_bias && ka->bias_on_i && !share;
    const int act = share ? RT_ACT_NONE : ka->act;
    const uint32_t ois = (uint32_t)(share ? ka->N : ka->o_is), ojs = share ? 1u : (uint32_t)ka->o_js;
#pragma unroll 1
    for (n = 0; n < count; n++) {
        const Item it = item(n);
        const int64_t iw = it.i0 + wi * (BI / WI), jw = it.j0 + wj * (BJ / WJ);
        float *out = (share ? ka->partial + (it.s * ka->ksplit + it.z) * ka->M * ka->N : ka->out + it.s * ka->o_bs) + iw * ois + jw * ojs;
        const int il = ka->M - iw < BI ? (int)(ka->M - iw) : BI, jl = ka->N - jw < BJ ? (int)(ka->N - jw) : BJ;
        const int64_t kend = min(ka->K, it.k0 + (int64_t)ka->nk * 32);
        const float *X = ka->X + (ka->x_stack == 1 ? 0 : it.s) * ka->x_bs;
        const int64_t y_el = (ka->y_stack == 1 ? 0 : it.s) * ka->y_bs;
#pragma unroll 1
        for (int ab = 0; ab < TM * TN; ab++) {
            const int a = ab / TN, b = ab - a * TN, ir = 32 * a + 4 * fh, j = 32 * b + fr; // this lane's outputs: rows ir + 8 (r / 4) + r % 4
            const uint32_t at0 = (uint32_t)ir * ois + (uint32_t)j * ojs;
            uint32_t bad = 0, at = at0; // bit r: output r
#pragma unroll 1
            for (int r = 0; r < 16; r++) {
                if (ir + 8 * (r >> 2) + (r & 3) < il && j < jl && !(__builtin_fabsf(out[at]) <= 3.4028234e38f)) bad |= 1u << r;
                at += (r & 3) == 3 ? 5 * ois : ois;
            }
            if (!__any(bad != 0)) continue;
            // lane half h supplies k + 4 h .. + 3 of eight, one of them to each MFMA
            const float *xp = X + min(iw + 32 * a + fr, ka->M - 1) * ka->x_is + (it.k0 + 4 * fh) * x_ks;
            const int64_t ye = y_el + min(jw + j, ka->N - 1) * ka->y_js + (it.k0 + 4 * fh) * y_ks;
            const float *yp = (const float *)ka->Y + ye;           // f32
            const int8_t *cp = (const int8_t *)ka->Y + ye;         // Q8_0F
            const float *sp = ka->scales + (ye >> 5);
            float16_t P = zero;
            auto four = [&](auto last, int64_t n) __attribute__((always_inline)) { // n: of this lane's four, inside K
                constexpr bool LAST = decltype(last)::value;
                float xv[4], yv[4];
#pragma unroll
                for (int e = 0; e < 4; e++) xv[e] = !LAST || e < n ? *xp : 0.f, xp += x_ks;
                if constexpr (Q8) { // K is whole blocks of 32
                    const uint32_t c = *(const uint32_t *)cp;
#pragma unroll
                    for (int e = 0; e < 4; e++) yv[e] = (float)(int8_t)(c >> (8 * e)) * *sp;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) yv[e] = !LAST || e < n ? *yp : 0.f, yp += y_ks;
                }
                xp += 4 * x_ks, yp += 4 * y_ks, cp += 8;
#pragma unroll
                for (int e = 0; e < 4; e++) P = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[e], yv[e], P, 0, 0, 0);
            };
            int64_t left = kend - it.k0;
            // eights at a time: more only where a load's address costs no registers of its own
            constexpr int CH = XKC && (Q8 || YKC) ? 4 : 1;
#pragma unroll 1
            for (; left >= 8 * CH; left -= 8 * CH) {
#pragma unroll
                for (int u = 0; u < CH; u++) four(std::false_type{}, 4);
                if constexpr (Q8) sp += CH == 4 || (left & 31) == 8; // at the end of a block
            }
            if constexpr (!Q8) {
#pragma unroll 1
                for (; left > 0; left -= 8) four(std::true_type{}, left - 4 * fh);
            }
            const float bias_j = ka->has_bias && !ka->bias_on_i && !share ? ka->bias[min(jw + j, ka->N - 1)] : 0.f;
            at = at0;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                if (bad >> r & 1) out[at] = rt_act(P[r] + (row_bias ? ka->bias[iw + ir + 8 * (r >> 2) + (r & 3)] : bias_j), act);
                at += (r & 3) == 3 ? 5 * ois : ois;
            }
        }
    }
}

// Second pass of a launch that shares K: out = act(sum over the shares + bias), in the shares' order.
__global__ __launch_bounds__(256) void limb_reduce_kernel(GemmLimbArgs g) {
    const int64_t s = blockIdx.y, nq = (g.N + 3) >> 2, total = nq * g.M, sstride = g.N * g.M;
    const float *pt = g.partial + s * g.ksplit * sstride;
    float *out = g.out + s * g.o_bs;
    for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
        const int64_t i = idx / nq, j = (idx - i * nq) << 2;
        const int n = (int)min<int64_t>(4, g.N - j);
        const float *src = pt + i * g.N + j;
        float4_t v = {0.f, 0.f, 0.f, 0.f};
        if ((g.N & 3) == 0) {
            for (int z = 0; z < g.ksplit; z++) v += *(const float4_t *)(src + z * sstride);
        } else {
            for (int z = 0; z < g.ksplit; z++)
                for (int e = 0; e < n; e++) v[e] += src[z * sstride + e];
        }
        for (int e = 0; e < n; e++) v[e] = rt_act(v[e] + (g.has_bias ? g.bias[g.bias_on_i ? i : j + e] : 0.f), g.act);
        float *o = out + i * g.o_is + j * g.o_js;
        if (n == 4 && g.o_js == 1 && ((uintptr_t)o & 15u) == 0) {
            *(float4_t *)o = v;
        } else {
            for (int e = 0; e < n; e++) o[e * g.o_js] = v[e];
        }
    }
}

namespace {

// Tile and shares of K for one problem.  The estimate is in cycles of a compute unit: a stage costs what its MFMAs take or
// what its vector instructions and loads take beside them, whichever is more; a workgroup does ceil(items / CUs) items.
struct LimbPlan {
    int bi = 0, bj = 0, ksplit = 1, nk = 0;
    double cost = 1e300;
};
struct LimbTile {
    int bi, bj;
};
constexpr LimbTile kFloatTiles[] = {{128, 128}, {96, 128}, {64, 128}, {128, 64}, {64, 64}};
constexpr LimbTile kCodeTiles[] = {{128, 128}, {96, 128}, {64, 128}};

LimbPlan limb_plan(const Problem &p, const DeviceInfo &dev, bool share) {
    const bool q8 = p.a_dt == RT_Q8_0F;
    const int64_t I = q8 ? p.N : p.M, J = q8 ? p.M : p.N; // limb_orient has run
    const int64_t stages = (p.K + 31) / 32;
    LimbPlan best;
    auto offer = [&](LimbTile t) {
        const double tiles32 = (t.bi / 32) * (t.bj / 32) / 4.0; // per SIMD
        const double mul = tiles32 * (q8 ? 6 : 12) * 33 + 100;
        const double vec = 5.8 * ((t.bi + (q8 ? 0 : t.bj)) * 32 / 256 * 6.0 + (q8 ? t.bj * 32 / 256 * 2.0 + tiles32 * 16 : 0.0) + 50);
        const double fill = (t.bi * 128.0 + t.bj * (q8 ? 64.0 + 128.0 : 128.0)) / 28;
        const double stage = std::max(mul, std::max(vec, fill)) + 60;
        const int64_t tiles = ((I + t.bi - 1) / t.bi) * ((J + t.bj - 1) / t.bj) * p.stacks;
        for (int ks = 1; ks <= (share ? 16 : 1); ks++) {
            const int64_t nk = (stages + ks - 1) / ks;
            if (ks > 1 && (nk < 8 || (int64_t)(ks - 1) * nk >= stages || tiles * ks > dev.num_cus)) continue;
            const double bytes = (double)p.stacks * p.M * p.N * 4;
            if (ks > 1 && bytes * ks > (double)RT_STATIC_SCRATCH_BYTES) continue;
            const int64_t rounds = (tiles * ks + dev.num_cus - 1) / dev.num_cus;
            double cost = (double)rounds * (nk * stage + 1000 + t.bi * t.bj * 0.15) + 5000;
            if (ks > 1) cost += 6000 + bytes * (ks + 1) / 1500; // the second kernel
            if (cost < best.cost) best.cost = cost, best.bi = t.bi, best.bj = t.bj, best.ksplit = ks, best.nk = (int)nk;
        }
    };
    if (q8)
        for (LimbTile t : kCodeTiles) offer(t);
    else
        for (LimbTile t : kFloatTiles) offer(t);
    return best;
}

// exchanges the operands' roles when that makes the output's contiguous axis the kernel's j axis
bool limb_orient(Problem &p) {
    if (p.a_dt != RT_F32 || p.o_is != 1 || p.o_js == 1) return false;
    std::swap(p.M, p.N);
    std::swap(p.a_stack, p.b_stack);
    std::swap(p.a_bs, p.b_bs);
    std::swap(p.a_rs, p.b_js);
    std::swap(p.a_ks, p.b_ks);
    std::swap(p.o_is, p.o_js);
    p.bias_on_rows = !p.bias_on_rows;
    return true;
}

// Everything with f32 activations but small f32 products.  Those launch_gemm_f32_small has taken before; of what it
// cannot (operands not aligned to 16 bytes, few rows), with two stages and less than a tile of 64 x 64 per compute unit, or
// one stage and less than two, there is nothing to pipeline (8 heads x 22 positions, the attention's three operators: 12.8 us here,
// 12.0 on the generic kernel; 20 x [300 x 31] . [31 x 300] 7.7 and 6.7, 32 x [512 x 31] . [31 x 512] 13.5 and 17.0).
// K of 1 and 2 go to the generic kernel: the f32 MFMA rounds once per product, so it gives an outer product correctly rounded,
// and the limbs cannot (relative error against float64 2.5e-8 and 3.1e-8 there, 3.5e-8 and 3.3e-8 here; from K = 3 on it is smaller
// here, 3.3e-8 to 3.5e-8).
bool limb_takes(const Problem &p, const DeviceInfo &dev) {
    if (p.act_dt != RT_F32 || (p.a_dt != RT_F32 && p.a_dt != RT_Q8_0F) || p.M <= 0 || p.N <= 0 || p.K <= 0 || p.stacks <= 0) return false;
    return p.a_dt == RT_Q8_0F || p.K > 64 || (p.K > 2 && ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.stacks > (p.K <= 32 ? 2 : 1) * (int64_t)dev.num_cus);
}

template <int BI, int BJ, int WI, int PW, bool Q8, bool XKC, bool YKC> hipError_t launch_limb_k(const GemmLimbArgs &g, unsigned grid, hipStream_t st) {
    constexpr int Y = Q8 ? LimbCodes<BJ, 64 * PW>::BYTES : LimbFloat<BJ, YKC, 64 * PW>::BYTES;
    constexpr size_t lds = 3 * (size_t)(LimbFloat<BI, XKC, 64 * PW>::BYTES + Y);
    static_assert(lds <= 160 * 1024, "three stages");
    if (const hipError_t e = ensure_lds_limit<&gemm_limb_kernel<BI, BJ, WI, PW, Q8, XKC, YKC>>(); e != hipSuccess) return e;
    hipLaunchKernelGGL((gemm_limb_kernel<BI, BJ, WI, PW, Q8, XKC, YKC>), dim3(grid), dim3(256 + 64 * PW), lds, st, g);
    return hipGetLastError();
}
template <int BI, int BJ, int WI> hipError_t launch_limb_f32(const GemmLimbArgs &g, bool xkc, bool ykc, unsigned grid, hipStream_t st) {
    if (xkc) return ykc ? launch_limb_k<BI, BJ, WI, 8, false, true, true>(g, grid, st) : launch_limb_k<BI, BJ, WI, 8, false, true, false>(g, grid, st);
    return ykc ? launch_limb_k<BI, BJ, WI, 8, false, false, true>(g, grid, st) : launch_limb_k<BI, BJ, WI, 8, false, false, false>(g, grid, st);
}
template <int BI, int BJ, int WI, int PW> hipError_t launch_limb_q8(const GemmLimbArgs &g, bool xkc, unsigned grid, hipStream_t st) {
    return xkc ? launch_limb_k<BI, BJ, WI, PW, true, true, true>(g, grid, st) : launch_limb_k<BI, BJ, WI, PW, true, false, true>(g, grid, st);
}

} // namespace

// bytes of workspace with which launch_gemm_limb shares this problem's K (0: it does not)
uint64_t gemm_limb_workspace_bytes(const Problem &p0, const DeviceInfo &dev) {
    Problem p = p0;
    limb_orient(p);
    if (!limb_takes(p, dev)) return 0;
    const LimbPlan pl = limb_plan(p, dev, true);
    return pl.ksplit > 1 ? (uint64_t)p.stacks * pl.ksplit * p.M * p.N * sizeof(float) : 0;
}

// Any strides; quantized rows 16-byte aligned.  hipErrorNotSupported: another kernel must take the problem.
hipError_t launch_gemm_limb(const Problem &p0, const void *A0, const void *B0, const void *bias, void *out, hipStream_t stream,
                            const DeviceInfo &dev) {
    Problem p = p0;
    const void *A = A0, *B = B0;
    if (limb_orient(p)) std::swap(A, B);
    if (!limb_takes(p, dev)) return hipErrorNotSupported;
    const bool q8 = p.a_dt == RT_Q8_0F;
    if (q8 && ((uintptr_t)A & 15u)) return hipErrorNotSupported;
    LimbPlan pl = limb_plan(p, dev, p.workspace != nullptr && !((uintptr_t)p.workspace & 15u));
    if (pl.ksplit > 1 && p.workspace_bytes < (uint64_t)p.stacks * pl.ksplit * p.M * p.N * sizeof(float)) pl = limb_plan(p, dev, false);
    // A long K that is not shared, in few tiles: a workgroup's own chain of stages is all there is, and with 48 to 64 columns, both
    // operands K-contiguous, the f32 kernel's is the shorter (48 rows x 384 x 1536: 23.4 us, 25.2 here; x 2560 x 2560 37.2, 40.1).
    // From here, not as a family of its own: a plan keeps the family, and the workspace may come and go.
    if (!q8 && pl.ksplit == 1 && p0.N <= 64 && p0.b_ks == 1 && gemm_f32_few_tiles(p0, dev)) {
        if (const hipError_t e = launch_gemm_f32(p0, A0, B0, bias, out, stream, dev); e != hipErrorNotSupported) return e;
    }
    GemmLimbArgs g{};
    g.bias = (const float *)bias, g.out = (float *)out;
    g.K = p.K, g.o_bs = p.o_bs, g.has_bias = p.has_bias, g.act = p.act;
    if (q8) { // the weight's rows are the kernel's j axis
        g.X = (const float *)B, g.Y = A;
        g.scales = (const float *)((const uint8_t *)A + rt_q8_0_scale_offset((uint64_t)p.a_stack * p.M * p.K));
        g.M = p.N, g.N = p.M;
        g.x_stack = p.b_stack, g.y_stack = p.a_stack;
        g.x_bs = p.b_bs, g.x_is = p.b_js, g.x_ks = p.b_ks;
        g.y_bs = p.a_bs, g.y_js = p.a_rs, g.y_ks = p.a_ks;
        g.o_is = p.o_js, g.o_js = p.o_is, g.bias_on_i = !p.bias_on_rows;
    } else {
        g.X = (const float *)A, g.Y = B;
        g.M = p.M, g.N = p.N;
        g.x_stack = p.a_stack, g.y_stack = p.b_stack;
        g.x_bs = p.a_bs, g.x_is = p.a_rs, g.x_ks = p.a_ks;
        g.y_bs = p.b_bs, g.y_js = p.b_js, g.y_ks = p.b_ks;
        g.o_is = p.o_is, g.o_js = p.o_js, g.bias_on_i = p.bias_on_rows;
    }
    g.ksplit = pl.ksplit, g.nk = pl.nk, g.partial = (float *)p.workspace;
    const int64_t ti = (g.M + pl.bi - 1) / pl.bi, tj = (g.N + pl.bj - 1) / pl.bj;
    const double items = (double)ti * tj * p.stacks * pl.ksplit;
    // offsets inside a tile and a stage are 32-bit, and so are the counts of items and stages
    const double span = std::max(128.0 * 4 * (g.x_is + g.x_ks), std::max(128.0 * 4 * (g.y_js + g.y_ks), 128.0 * 4 * (g.o_is + g.o_js)));
    if (span > 2e9 || items > 1e9 || g.K > (int64_t)1 << 34) return hipErrorNotSupported;
    g.stages = (int)((p.K + 31) / 32);
    g.tiles_i = LimbDiv((int)ti), g.tiles_j = LimbDiv((int)tj), g.shares = LimbDiv(pl.ksplit), g.items = (int)items;
    const unsigned grid = (unsigned)(g.items < dev.num_cus ? g.items : dev.num_cus);
    if (items / grid * pl.nk > 1e9) return hipErrorNotSupported;
    const bool xkc = g.x_ks == 1 && p.K >= 4, ykc = g.y_ks == 1 && p.K >= 4;
    hipError_t e;
    if (q8)
        e = pl.bi == 128 ? launch_limb_q8<128, 128, 2, 4>(g, xkc, grid, stream) : pl.bi == 96 ? launch_limb_q8<96, 128, 1, 4>(g, xkc, grid, stream)
                                                                                            : launch_limb_q8<64, 128, 1, 8>(g, xkc, grid, stream);
    else if (pl.bi == 128)
        e = pl.bj == 128 ? launch_limb_f32<128, 128, 2>(g, xkc, ykc, grid, stream) : launch_limb_f32<128, 64, 2>(g, xkc, ykc, grid, stream);
    else if (pl.bi == 96)
        e = launch_limb_f32<96, 128, 1>(g, xkc, ykc, grid, stream);
    else
        e = pl.bj == 128 ? launch_limb_f32<64, 128, 2>(g, xkc, ykc, grid, stream) : launch_limb_f32<64, 64, 2>(g, xkc, ykc, grid, stream);
    if (e != hipSuccess || g.ksplit == 1) return e;
    const int64_t total = ((g.N + 3) >> 2) * g.M;
    hipLaunchKernelGGL(limb_reduce_kernel, dim3((unsigned)((total + 255) / 256 > 8192 ? 8192 : (total + 255) / 256), (unsigned)p.stacks), dim3(256), 0, stream, g);
    return hipGetLastError();
}

} // namespace rt
