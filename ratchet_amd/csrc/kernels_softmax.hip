// In-place softmax over the last dimension:  x[r, :] <- exp(x[r, :] - max_r) / sum_r.
// The step between the two attention matmuls (scores -> probabilities).  HBM-bound: one read
// and one write of the tensor.
//
// Fast path: one wavefront per row, the whole row in registers (up to 8 x 16 bytes per lane),
// so the tensor is read exactly once; maximum, exponentials and sum are f32 whatever the
// storage type, reduced across the wavefront with DPP shuffles; the result is rounded once.
// Rows that do not begin and end on 16 bytes (EDGES) are taken as the aligned vectors they touch; a vector shared with a neighbour is
// read whole (the neighbour's values, which may be changing, are dropped; at the tensor's ends it is read value by value) and its own values
// are written one by one: 6 x 964 x 964 in f16 15.2 us on the
// kernel below, which re-reads a row (from L2) for each of its three passes, -> 8.1; 8 x 874 x 874 in f32 17.2 -> 11.3.  It keeps the rows too
// long for registers and, where they are few (launch_softmax_t) or have fewer than 128 values, those for which it has more wavefronts
// (6 x 62 x 62 in f16: 2.9 and 3.8).
//
// Role in the reference: ops/softmax.rs:52-183 (one 128-thread workgroup per row, reductions
// through workgroup memory, arithmetic in the tensor's own type).  Differences, both tighter:
// f16 tensors are reduced in f32, and the running maximum starts from the data rather than
// from a finite floor, so rows made only of very negative values still normalise.
#include <limits>

#include "device_common.h"

namespace rt {


template <typename T> struct SoftmaxVec;
template <> struct SoftmaxVec<float> {
    static constexpr int EV = 4;
    __device__ __forceinline__ static float get(const uint4_t &v, int e) { return __builtin_bit_cast(float4_t, v)[e]; }
    template <typename F> __device__ __forceinline__ static uint4_t make(F f) {
        return __builtin_bit_cast(uint4_t, float4_t{f(0), f(1), f(2), f(3)});
    }
};
template <> struct SoftmaxVec<half_t> {
    static constexpr int EV = 8;
    __device__ __forceinline__ static float get(const uint4_t &v, int e) { return (float)__builtin_bit_cast(half8_t, v)[e]; }
    template <typename F> __device__ __forceinline__ static uint4_t make(F f) {
        return __builtin_bit_cast(uint4_t, half8_t{(half_t)f(0), (half_t)f(1), (half_t)f(2), (half_t)f(3), (half_t)f(4),
                                                   (half_t)f(5), (half_t)f(6), (half_t)f(7)});
    }
};

// VPL: 16-byte vectors per lane; a row of n values has, or touches, at most 64 * VPL vectors.
template <typename T, int VPL, bool EDGES>
__global__ __launch_bounds__(256) void softmax_rows_kernel(T *x, int64_t rows, int n) {
    constexpr int EV = SoftmaxVec<T>::EV;
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return; // whole wavefronts leave together
    T *const first = x + row * n;
    const int head = EDGES ? (int)((uintptr_t)first & 15u) / (int)sizeof(T) : 0; // values of the first vector in front of the row
    uint4_t *p = (uint4_t *)(first - head);
    const int nvec = EDGES ? (head + n + EV - 1) / EV : n / EV;
    // a vector that is not the row's alone: its values lo .. hi - 1 are
    auto shared = [&](int v, int &lo, int &hi) {
        lo = v == 0 ? head : 0, hi = min(EV, head + n - v * EV);
        return EDGES && hi - lo < EV;
    };
    float f[VPL][EV];
    const float ninf = -std::numeric_limits<float>::infinity();
    float m = ninf;
#pragma unroll
    for (int i = 0; i < VPL; i++) {
        const int v = lane + 64 * i;
        uint4_t raw = {0u, 0u, 0u, 0u};
        int lo, hi;
        const bool part = shared(v, lo, hi), outside = EDGES && ((T *)(p + v) < x || (T *)(p + v) + EV > x + rows * n);
        if (v < nvec && !outside) raw = __builtin_nontemporal_load(p + v); // read once, written once: nothing to keep in the caches
#pragma unroll
        for (int e = 0; e < EV; e++) f[i][e] = v < nvec && !(part && (e < lo || e >= hi)) ? SoftmaxVec<T>::get(raw, e) : ninf;
        if (EDGES && v < nvec && outside) {
#pragma unroll
            for (int e = 0; e < EV; e++)
                if (e >= lo && e < hi) f[i][e] = to_f32(((const T *)(p + v))[e]);
        }
#pragma unroll
        for (int e = 0; e < EV; e++) m = fmaxf(m, f[i][e]);
    }
    m = wave_max(m);
    if (m == ninf) m = 0.f; // a row of -inf: exp(-inf - 0) = 0 everywhere, 0 / 0 = NaN as the formula says
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; i++)
#pragma unroll
        for (int e = 0; e < EV; e++) {
            f[i][e] = expf(f[i][e] - m);
            s += f[i][e];
        }
    s = wave_sum(s);
    // f16 rows are bound by instructions, not memory: f / s as f * rn(1 / s) and one correction by its remainder, three
    // instructions per value for the eleven of a division and the correctly rounded quotient all the same (Markstein, 1990;
    // s = 0 and NaN give NaN as they should).  32 x 512 x 512 in f16: Q.K^T, softmax and P.V together 26.9 -> 25.6 us.  f32 rows
    // move twice the bytes per value and keep the division: no gain beyond the spread between cards (6 x 1500 x 1500, the three
    // operators: 67.6 and 69.7 us with the division, 68.4 without).
    const float rs = 1.f / s;
    auto quotient = [&](float a) {
        if constexpr (sizeof(T) == 4) return a / s;
        const float q = a * rs;
        return fmaf(fmaf(-q, s, a), rs, q);
    };
#pragma unroll
    for (int i = 0; i < VPL; i++) {
        const int v = lane + 64 * i;
        int lo, hi;
        const bool part = shared(v, lo, hi);
        if (v < nvec && !part) __builtin_nontemporal_store(SoftmaxVec<T>::make([&](int e) { return quotient(f[i][e]); }), p + v);
        if (EDGES && v < nvec && part) {
#pragma unroll
            for (int e = 0; e < EV; e++)
                if (e >= lo && e < hi) ((T *)(p + v))[e] = from_f32<T>(quotient(f[i][e]));
        }
    }
}

// One 256-thread workgroup per row, any length.
template <typename T>
__global__ __launch_bounds__(256) void softmax_generic_kernel(T *x, int64_t n) {
    __shared__ float red[4];
    T *p = x + (int64_t)blockIdx.x * n;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const float ninf = -std::numeric_limits<float>::infinity();
    float m = ninf;
    for (int64_t i = t; i < n; i += 256) m = fmaxf(m, to_f32(p[i]));
    m = wave_max(m);
    if (lane == 0) red[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    if (m == ninf) m = 0.f;
    __syncthreads();
    float s = 0.f;
    for (int64_t i = t; i < n; i += 256) s += expf(to_f32(p[i]) - m);
    s = wave_sum(s);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    s = (red[0] + red[1]) + (red[2] + red[3]);
    for (int64_t i = t; i < n; i += 256) p[i] = from_f32<T>(expf(to_f32(p[i]) - m) / s);
}

template <typename T> static hipError_t launch_softmax_t(void *x, int64_t rows, int64_t n, hipStream_t st) {
    constexpr int EV = SoftmaxVec<T>::EV;
    if (rows == 0 || n == 0) return hipSuccess;
    const bool whole = n % EV == 0 && ((uintptr_t)x & 15u) == 0;
    const int64_t nvec = whole ? n / EV : (n + 2 * EV - 2) / EV; // vectors a row touches at the most
    // Rows that do not begin on 16 bytes: a wavefront per row pays its edges where rows are few, and the workgroup per row of the other kernel
    // then has them all in flight at once.  us, f32 there and here: 512 x 333 3.75 / 4.34, 1024 x 333 4.10 / 4.44, 1024 x 1001 5.95 / 5.72, 1800 x 333
    // 4.81 / 4.95, 2200 x 133 / 333 4.24 / 4.12 and 5.71 / 5.35; f16: 512 x 133 3.24 / 4.02, 768 x 701 4.56 / 5.03, 1024 x 133 / 333 / 1001 3.41 / 4.07,
    // 4.22 / 4.13 and 5.68 / 5.05, 2200 x 203 4.59 / 4.78, 3000 x 133 4.84 / 4.81.
    const bool many = n >= 128 && rows >= (n >= (EV == 8 ? 320 : 1000) ? 1024 : EV == 8 ? 3000 : 2048);
    if (nvec <= 64 * 8 && (whole || many)) {
        const int64_t blocks = (rows + 3) / 4;
        if (blocks > 0x7fffffff) return hipErrorInvalidValue;
        auto rows_of = [&](auto VPL) {
            constexpr int vpl = decltype(VPL)::value;
            if (whole) hipLaunchKernelGGL((softmax_rows_kernel<T, vpl, false>), dim3((unsigned)blocks), dim3(256), 0, st, (T *)x, rows, (int)n);
            else hipLaunchKernelGGL((softmax_rows_kernel<T, vpl, true>), dim3((unsigned)blocks), dim3(256), 0, st, (T *)x, rows, (int)n);
        };
        if (nvec <= 64) rows_of(std::integral_constant<int, 1>{});
        else if (nvec <= 128) rows_of(std::integral_constant<int, 2>{});
        else if (nvec <= 256) rows_of(std::integral_constant<int, 4>{});
        else rows_of(std::integral_constant<int, 8>{});
        return hipGetLastError();
    }
    if (rows > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((softmax_generic_kernel<T>), dim3((unsigned)rows), dim3(256), 0, st, (T *)x, n);
    return hipGetLastError();
}

hipError_t launch_softmax(int dtype, void *x, int64_t rows, int64_t n, hipStream_t stream) {
    return dtype == RT_F16 ? launch_softmax_t<half_t>(x, rows, n, stream) : launch_softmax_t<float>(x, rows, n, stream);
}

} // namespace rt
