// Single-pass reductions: min/max (FL bit width, scale, patch thresholds)
// and the fused statistics pass the planner reads.
//
// Every workgroup reduces a grid-stride share with 16-byte loads and writes a
// partial; the last workgroup to finish (tickets that it resets) folds the
// partials and hands the result to the host itself where the host asked for
// it.  A launch of its own for the fold and one for the read-back cost 6 us on
// the device and 7 us of launching for a few kilobytes.
#include <algorithm>
#include <cstddef>
#include <vector>
#include <limits>

#include "dispatch.h"
#include "k_common.h"
#include "kernels.h"

namespace ddj {

namespace {

__device__ __forceinline__ uint64_t block_reduce_min(uint64_t v, uint64_t* sm) {
    v = wave_min(v);
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    if (lane == 0) sm[wid] = v;
    __syncthreads();
    uint64_t r = sm[0];
    for (int w = 1; w < kBlock / kWave; w++) r = sm[w] < r ? sm[w] : r;
    __syncthreads();
    return r;
}
__device__ __forceinline__ uint64_t block_reduce_max(uint64_t v, uint64_t* sm) {
    v = wave_max(v);
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    if (lane == 0) sm[wid] = v;
    __syncthreads();
    uint64_t r = sm[0];
    for (int w = 1; w < kBlock / kWave; w++) r = sm[w] > r ? sm[w] : r;
    __syncthreads();
    return r;
}
__device__ __forceinline__ uint64_t rd(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t rd32(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ------------------------------------------------------------------ minmax
// Keys of the reference's minimum and maximum: thrust::minmax_element
// (util/statistics/cuda_array_statistics.cu:20-28) under operator<, taken as
// the sequential fold m = x[0]; m = x[i] < m ? x[i] : m.  For floats that
// means: NaN rows never win, so a NaN in row 0 is both the minimum and the
// maximum; -0.0 and +0.0 tie, and the first zero in row order gives the sign.
// Rows feed add(); `zf` keeps (row << 1 | sign) of the first zero.
template <typename T, bool FLOAT = std::is_floating_point<T>::value> struct FoldKeys {
    uint64_t zf = ~0ull;
    uint64_t kmn = ~0ull, kmx = 0;
    __device__ __forceinline__ void add(T v, size_t row) {
        if (v != v) return;
        if (v == T(0)) {
            const uint64_t z = ((uint64_t)row << 1) | (__builtin_signbit(v) ? 1ull : 0ull);
            zf = z < zf ? z : zf;
            v = T(0);
        }
        const uint64_t key = order_key(v);
        kmn = key < kmn ? key : kmn;
        kmx = key > kmx ? key : kmx;
    }
    __device__ __forceinline__ uint64_t min_key() const { return kmn; }
    __device__ __forceinline__ uint64_t max_key() const { return kmx; }
};
// Integers: native compares per row (order keys are monotone in the value),
// keys only for the result; with no rows the keys are ~0 / 0 as above.
template <typename T> struct FoldKeys<T, false> {
    uint64_t zf = ~0ull;
    T mn = std::numeric_limits<T>::max(), mx = std::numeric_limits<T>::min();
    bool any = false;
    __device__ __forceinline__ void add(T v, size_t) {
        mn = v < mn ? v : mn;
        mx = v > mx ? v : mx;
        any = true;
    }
    __device__ __forceinline__ uint64_t min_key() const { return any ? order_key(mn) : ~0ull; }
    __device__ __forceinline__ uint64_t max_key() const { return any ? order_key(mx) : 0ull; }
};

// Final keys from the reduced ones and row 0.
template <typename T> __device__ __forceinline__ void fold_fixup(const T* x, uint64_t& mn, uint64_t& mx, uint64_t zf) {
    if constexpr (std::is_floating_point<T>::value) {
        const T x0 = x[0];
        if (x0 != x0) {
            mn = mx = order_key(x0);
            return;
        }
        if (zf != ~0ull && (zf & 1)) {
            const uint64_t kz = order_key(T(0)), knz = order_key(-T(0));
            if (mn == kz) mn = knz;
            if (mx == kz) mx = knz;
        }
    }
}

// What the last workgroup of a min/max pass does with the partials (STRIDE
// keys each: min, max, then the first zero and the precision where kept).
struct FoldTail {
    uint32_t* tickets = nullptr;
    MinMaxResult* out = nullptr;  // device result, or null
    HostOut host;                 // {min key, max key, precision}
};

template <typename T, int STRIDE>
__device__ __forceinline__ void fold_partials(const FoldTail& ft, const uint64_t* partials, const T* x, uint64_t* sm,
                                              bool* flag) {
    if (!last_of_grid(ft.tickets, flag)) return;
    uint64_t mn = ~0ull, mx = 0, zf = ~0ull, pr = 0;
    for (uint32_t b = threadIdx.x; b < gridDim.x; b += kBlock) {
        const uint64_t a = rd(partials + STRIDE * b), z = rd(partials + STRIDE * b + 1);
        const uint64_t q = STRIDE >= 3 ? rd(partials + STRIDE * b + 2) : ~0ull;
        const uint64_t p = STRIDE == 4 ? rd(partials + STRIDE * b + 3) : 0ull;
        mn = a < mn ? a : mn;
        mx = z > mx ? z : mx;
        zf = q < zf ? q : zf;
        pr = p > pr ? p : pr;
    }
    mn = block_reduce_min(mn, sm);
    mx = block_reduce_max(mx, sm);
    if (STRIDE >= 3 && std::is_floating_point<T>::value) zf = block_reduce_min(zf, sm);
    if (STRIDE == 4) pr = block_reduce_max(pr, sm);
    if (threadIdx.x == 0) {
        if (STRIDE >= 3) fold_fixup(x, mn, mx, zf);
        if (ft.out) {
            ft.out->min_key = mn;
            ft.out->max_key = mx;
        }
        if (ft.host.dst) {
            uint64_t* h = reinterpret_cast<uint64_t*>(ft.host.dst);
            h[0] = mn;
            h[1] = mx;
            h[2] = pr;
        }
    }
    if (ft.host.dst) host_out_done(ft.host);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_minmax(const T* __restrict__ x, size_t n, uint64_t* __restrict__ partials,
                                                   FoldTail ft) {
    __shared__ uint64_t sm[kBlock / kWave];
    __shared__ bool last;
    FoldKeys<T> f;
    const size_t tid = (size_t)blockIdx.x * kBlock + threadIdx.x, stride = (size_t)gridDim.x * kBlock;
    constexpr int V = 16 / sizeof(T);
    size_t done = 0;
    if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
        const u32x4* xv = reinterpret_cast<const u32x4*>(x);
        const size_t nv = n / V;
        constexpr int U = 4;  // loads in flight per thread
        for (size_t i0 = tid; i0 < nv; i0 += U * stride) {
            u32x4 v[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const size_t i = i0 + u * stride;
                if (i < nv) v[u] = xv[i];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const size_t i = i0 + u * stride;
                if (i >= nv) break;
                T vals[V];
                __builtin_memcpy(vals, &v[u], 16);
#pragma unroll
                for (int k = 0; k < V; k++) f.add(vals[k], i * V + k);
            }
        }
        done = nv * V;
    }
    for (size_t i = done + tid; i < n; i += stride) f.add(x[i], i);
    uint64_t mn = block_reduce_min(f.min_key(), sm);
    uint64_t mx = block_reduce_max(f.max_key(), sm);
    uint64_t zf = block_reduce_min(f.zf, sm);
    if (threadIdx.x == 0) {
        st_agent(partials + 3 * blockIdx.x, mn);
        st_agent(partials + 3 * blockIdx.x + 1, mx);
        st_agent(partials + 3 * blockIdx.x + 2, zf);
    }
    fold_partials<T, 3>(ft, partials, x, sm, &last);
}

// Min/max of the wrapping differences d[i] = x[i+1] - x[i], i < n - 1, read
// straight from x (the delta encoder's output is never written when an FL
// node consumes it).  Integer types only.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_minmax_delta(const T* __restrict__ x, size_t n, uint64_t* __restrict__ partials,
                                                         FoldTail ft) {
    __shared__ uint64_t sm[kBlock / kWave];
    __shared__ bool last;
    using U = typename UnsignedOf<T>::type;
    T dmn = std::numeric_limits<T>::max(), dmx = std::numeric_limits<T>::min();
    bool any = false;
    auto add = [&](T a, T b) {  // d = b - a, wrapping in T
        const T d = (T)(U)((U)b - (U)a);
        dmn = d < dmn ? d : dmn;
        dmx = d > dmx ? d : dmx;
        any = true;
    };
    const size_t m = n - 1;
    const size_t tid = (size_t)blockIdx.x * kBlock + threadIdx.x, stride = (size_t)gridDim.x * kBlock;
    constexpr int V = 16 / sizeof(T);
    size_t done = 0;
    if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
        const u32x4* xv = reinterpret_cast<const u32x4*>(x);
        const size_t nv = m / V;  // vectors whose V deltas are all in range (x[i*V+V] exists)
        constexpr int Uf = 4;
        const int lane = threadIdx.x & (kWave - 1);
        for (size_t i0 = tid; i0 < nv; i0 += Uf * stride) {
            u32x4 v[Uf];
            T nx[Uf];
            // The row after vector i starts vector i + 1, which the next lane
            // holds (lanes take consecutive vectors); the last lane of the
            // wave, and the thread with the last vector, load it with the
            // vectors so that the loop waits on memory once.
#pragma unroll
            for (int u = 0; u < Uf; u++) {
                const size_t i = i0 + u * stride;
                if (i < nv) {
                    v[u] = xv[i];
                    if (lane == kWave - 1 || i + 1 >= nv) nx[u] = x[(i + 1) * V];  // (i + 1) * V <= m < n
                }
            }
#pragma unroll
            for (int u = 0; u < Uf; u++) {
                const size_t i = i0 + u * stride;
                // first 8 bytes of the next lane's vector (all lanes take part)
                const uint32_t nb0 = (uint32_t)__shfl_down((int)v[u].x, 1, kWave);
                const uint32_t nb1 = (uint32_t)__shfl_down((int)v[u].y, 1, kWave);
                if (i >= nv) continue;
                T vals[V + 1];
                __builtin_memcpy(vals, &v[u], 16);
                if (lane == kWave - 1 || i + 1 >= nv) {
                    vals[V] = nx[u];
                } else {
                    const uint64_t nb = ((uint64_t)nb1 << 32) | nb0;
                    __builtin_memcpy(&vals[V], &nb, sizeof(T));
                }
#pragma unroll
                for (int k = 0; k < V; k++) add(vals[k], vals[k + 1]);
            }
        }
        done = nv * V;
    }
    for (size_t i = done + tid; i < m; i += stride) add(x[i], x[i + 1]);
    uint64_t mn = block_reduce_min(any ? order_key(dmn) : ~0ull, sm);
    uint64_t mx = block_reduce_max(any ? order_key(dmx) : 0ull, sm);
    if (threadIdx.x == 0) {
        st_agent(partials + 2 * blockIdx.x, mn);
        st_agent(partials + 2 * blockIdx.x + 1, mx);
    }
    fold_partials<T, 2>(ft, partials, x, sm, &last);
}

// ------------------------------------------------------------------- stats
// _getFloatPrecision (reference util/statistics/cuda_array_statistics.cu:37-44)
// as the loop count k of round(x*10^k)/10^k != x in float arithmetic.
__device__ __forceinline__ uint32_t float_precision(float number) {
    float e = 1.0f;
    uint32_t k = 0;
    while (k < 10) {
        float r = roundf(number * e);
        if (__fdiv_rn(r, e) == number) break;
        e *= 10.0f;
        k++;
    }
    return k;
}
// The maximum of float_precision over the rows seen: a row that k = prec
// decimals represent has a precision of at most prec, so only a row that fails
// that one test (whose power of ten, exact in float up to 10^10, is kept with
// prec) runs the loop.  One division a row in place of one per decimal.
struct MaxPrecision {
    uint32_t prec = 0;
    float e = 1.0f;
    __device__ __forceinline__ void add(float number) {
        if (prec >= 10 || __fdiv_rn(roundf(number * e), e) == number) return;
        const uint32_t p = float_precision(number);
        while (prec < p) {
            prec++;
            e *= 10.0f;
        }
    }
};

// Min/max keys and the float precision (the maximum of float_precision
// over the rows, as the statistics pass computes it) in one pass: the two
// inputs of the floatToInt encoder (float_to_int_encoding.cu).  Partials:
// {min, max, first zero, precision} per workgroup.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_minmax_prec(const T* __restrict__ x, size_t n,
                                                        uint64_t* __restrict__ partials, FoldTail ft) {
    __shared__ uint64_t sm[kBlock / kWave];
    __shared__ bool last;
    FoldKeys<T> f;
    MaxPrecision pm;
    auto add = [&](T v, size_t row) {
        f.add(v, row);
        pm.add((float)v);
    };
    const size_t tid = (size_t)blockIdx.x * kBlock + threadIdx.x, stride = (size_t)gridDim.x * kBlock;
    constexpr int V = 16 / sizeof(T);
    size_t done = 0;
    if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
        const u32x4* xv = reinterpret_cast<const u32x4*>(x);
        const size_t nv = n / V;
        constexpr int U = 4;  // loads in flight per thread
        for (size_t i0 = tid; i0 < nv; i0 += U * stride) {
            u32x4 v[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const size_t i = i0 + u * stride;
                if (i < nv) v[u] = xv[i];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const size_t i = i0 + u * stride;
                if (i >= nv) break;
                T vals[V];
                __builtin_memcpy(vals, &v[u], 16);
#pragma unroll
                for (int k = 0; k < V; k++) add(vals[k], i * V + k);
            }
        }
        done = nv * V;
    }
    for (size_t i = done + tid; i < n; i += stride) add(x[i], i);
    const uint64_t mn = block_reduce_min(f.min_key(), sm);
    const uint64_t mx = block_reduce_max(f.max_key(), sm);
    const uint64_t zf = block_reduce_min(f.zf, sm);
    const uint64_t pr = block_reduce_max((uint64_t)pm.prec, sm);
    if (threadIdx.x == 0) {
        st_agent(partials + 4 * blockIdx.x, mn);
        st_agent(partials + 4 * blockIdx.x + 1, mx);
        st_agent(partials + 4 * blockIdx.x + 2, zf);
        st_agent(partials + 4 * blockIdx.x + 3, pr);
    }
    fold_partials<T, 4>(ft, partials, x, sm, &last);
}

template <typename T> __device__ __forceinline__ int32_t to_int32_sat(T v) {
    if constexpr (std::is_floating_point<T>::value) {
        double d = (double)v;
        if (d != d) return 0;
        if (d >= 2147483647.0) return 2147483647;
        if (d <= -2147483648.0) return (-2147483647 - 1);
        return (int32_t)d;
    } else {
        return (int32_t)(int64_t)v;
    }
}

template <typename T> __device__ __forceinline__ bool rl_equal(T a, T b) {
    // _rlMetricKernel (cuda_array_statistics.cu:97-115): int value = data[idx]; value == data[idx+1]
    int32_t v = to_int32_sat(a);
    if constexpr (std::is_floating_point<T>::value)
        return (T)v == b;
    else
        return (int64_t)v == (int64_t)b;
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

template <typename T> __device__ __forceinline__ uint64_t zigzag_bits(T v) {
    if constexpr (std::is_floating_point<T>::value) {
        return ubits(v);
    } else {
        int64_t s = (int64_t)v;
        return ((uint64_t)s << 1) ^ (uint64_t)(s >> 63);
    }
}
__device__ __forceinline__ uint32_t bitwidth64(uint64_t v) { return v ? 64 - __clzll(v) : 0; }

struct StatsAcc {
    uint64_t mn, mx, zf, unsorted, rl_eq, runs, sum_bits;
    double sum_f;
    uint32_t prec, dmax;
};

// LDS copies of the bit-width histogram: lane l counts in copy l % 32, so the
// rows of a wave, which mostly share a width, never meet in a bank (two lanes
// of the wave share a copy).
constexpr int kHistCopies = 32;

template <typename T>
__device__ __forceinline__ void stats_elem(StatsAcc& a, T v, T next, bool has_next, bool has_next2, size_t row,
                                           uint32_t* sm_hist, volatile uint32_t* sm_hll) {
    if constexpr (std::is_floating_point<T>::value) {
        FoldKeys<T> fk;
        fk.kmn = a.mn;
        fk.kmx = a.mx;
        fk.zf = a.zf;
        fk.add(v, row);
        a.mn = fk.kmn;
        a.mx = fk.kmx;
        a.zf = fk.zf;
    } else {
        const uint64_t key = order_key(v);
        a.mn = key < a.mn ? key : a.mn;
        a.mx = key > a.mx ? key : a.mx;
    }
    if constexpr (std::is_floating_point<T>::value) {
        a.sum_f += (double)v;
        uint32_t p = float_precision((float)v);
        a.prec = p > a.prec ? p : a.prec;
    } else {
        a.sum_bits += (uint64_t)(int64_t)v;
    }
    if (has_next) {
        if (v > next) a.unsorted = 1;
        if (!(next == v)) a.runs++;
        if constexpr (!std::is_floating_point<T>::value) {
            constexpr int W = 8 * sizeof(T);
            const uint64_t d = ubits(next) - ubits(v);
            const int64_t sd = (int64_t)(d << (64 - W)) >> (64 - W);  // wrap to W bits, sign-extend
            const uint64_t z = ((uint64_t)sd << 1) ^ (uint64_t)(sd >> 63);
            const uint32_t bw = bitwidth64(z);
            a.dmax = bw > a.dmax ? bw : a.dmax;
        }
    }
    if (has_next2 && rl_equal(v, next)) a.rl_eq++;
    atomicAdd(&sm_hist[bitwidth64(zigzag_bits(v)) * kHistCopies + (threadIdx.x & (kHistCopies - 1))], 1u);
    const uint64_t h = mix64(ubits(v) + 0x9e3779b97f4a7c15ull);
    const uint32_t reg = (uint32_t)(h >> 58);
    const uint32_t rank = (uint32_t)__clzll((h << 6) | (1ull << 5)) + 1;
    // registers only grow: after a few rows nearly every row reads a register
    // at or above its rank and skips the atomic
    if (rank > sm_hll[reg]) atomicMax(const_cast<uint32_t*>(&sm_hll[reg]), rank);
}

// The scalar fields of the threads' accumulators reduced over the workgroup
// (one barrier for all of them); every thread gets the result.
__device__ __forceinline__ StatsAcc block_fold(StatsAcc a, StatsAcc* sm /* kBlock / kWave */) {
    a.mn = wave_min(a.mn);
    a.mx = wave_max(a.mx);
    a.zf = wave_min(a.zf);
    a.unsorted = __ballot(a.unsorted != 0) != 0;
    a.rl_eq = wave_sum(a.rl_eq);
    a.runs = wave_sum(a.runs);
    a.sum_bits = wave_sum(a.sum_bits);
    a.sum_f = wave_sum(a.sum_f);
    a.prec = wave_max(a.prec);
    a.dmax = wave_max(a.dmax);
    if ((threadIdx.x & (kWave - 1)) == 0) sm[threadIdx.x / kWave] = a;
    __syncthreads();
    StatsAcc r{~0ull, 0, ~0ull, 0, 0, 0, 0, 0.0, 0, 0};
#pragma unroll
    for (int w = 0; w < kBlock / kWave; w++) {
        const StatsAcc q = sm[w];
        r.mn = q.mn < r.mn ? q.mn : r.mn;
        r.mx = q.mx > r.mx ? q.mx : r.mx;
        r.zf = q.zf < r.zf ? q.zf : r.zf;
        r.unsorted |= q.unsorted;
        r.rl_eq += q.rl_eq;
        r.runs += q.runs;
        r.sum_bits += q.sum_bits;
        r.sum_f += q.sum_f;
        r.prec = q.prec > r.prec ? q.prec : r.prec;
        r.dmax = q.dmax > r.dmax ? q.dmax : r.dmax;
    }
    __syncthreads();  // sm may be rewritten
    return r;
}

// Bound by latency on the planner's blocks of 10^4..10^5 rows.  The last
// workgroup folds the others' 129 histogram and HyperLogLog words with all
// its threads, consecutive lanes on consecutive words and kFold loads in
// flight each (one thread per workgroup, walking that workgroup's 129 words
// one atomic load at a time, took 112 us on 65,537 int32 rows, now 13, and
// 34 us on 10,000 rows, now 10).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_stats(const T* __restrict__ x, size_t n, DevStats* __restrict__ partials,
                                                  uint32_t* tickets, HostOut host) {
    constexpr int kBins = 65, kRegs = 64;
    __shared__ StatsAcc sm[kBlock / kWave];
    __shared__ uint32_t sm_hist[kBins * kHistCopies];
    __shared__ uint32_t sm_hll[kRegs];
    __shared__ uint32_t fin[kBins + kRegs];  // the folded bins, then the registers
    __shared__ bool last;
    for (int i = threadIdx.x; i < kBins * kHistCopies; i += kBlock) sm_hist[i] = 0;
    for (int i = threadIdx.x; i < kRegs; i += kBlock) sm_hll[i] = 0;
    for (int i = threadIdx.x; i < kBins + kRegs; i += kBlock) fin[i] = 0;
    __syncthreads();
    StatsAcc a{~0ull, 0, ~0ull, 0, 0, 0, 0, 0.0, 0, 0};
    const size_t tid = (size_t)blockIdx.x * kBlock + threadIdx.x, stride = (size_t)gridDim.x * kBlock;
    constexpr int V = 16 / sizeof(T);
    size_t done = 0;
    if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {
        const u32x4* xv = reinterpret_cast<const u32x4*>(x);
        const size_t nv = n / V;
        for (size_t i = tid; i < nv; i += stride) {
            u32x4 v = xv[i];
            T vals[V + 1];
            __builtin_memcpy(vals, &v, 16);
            const size_t base = i * V;
            vals[V] = (base + V < n) ? x[base + V] : T(0);
#pragma unroll
            for (int k = 0; k < V; k++)
                stats_elem(a, vals[k], vals[k + 1], base + k + 1 < n, base + k + 2 < n, base + k, sm_hist, sm_hll);
        }
        done = nv * V;
    }
    for (size_t i = done + tid; i < n; i += stride) {
        T v = x[i];
        T nx = (i + 1 < n) ? x[i + 1] : T(0);
        stats_elem(a, v, nx, i + 1 < n, i + 2 < n, i, sm_hist, sm_hll);
    }
    a = block_fold(a, sm);  // its barriers also complete sm_hist and sm_hll
    DevStats* p = partials + blockIdx.x;
    static_assert(offsetof(DevStats, hll) == offsetof(DevStats, bit_hist) + 4 * kBins, "bins and registers adjoin");
    if (threadIdx.x == 0) {
        st_agent(&p->min_key, a.mn);
        st_agent(&p->max_key, a.mx);
        st_agent(&p->first_zero, a.zf);
        st_agent(&p->unsorted, a.unsorted);
        st_agent(&p->rl_eq, a.rl_eq);
        st_agent(&p->runs, a.runs);
        st_agent(&p->sum_bits, a.sum_bits);
        uint64_t sfb;
        __builtin_memcpy(&sfb, &a.sum_f, 8);
        st_agent(reinterpret_cast<uint64_t*>(&p->sum_f), sfb);
        st_agent(&p->precision, a.prec);
        st_agent(&p->delta_bits_max, a.dmax);
    }
    for (int i = threadIdx.x; i < kBins + kRegs; i += kBlock) {
        uint32_t v = 0;
        if (i < kBins) {  // rotated, so that the lanes' reads spread over the banks
            for (int k = 0; k < kHistCopies; k++) v += sm_hist[i * kHistCopies + ((i + k) & (kHistCopies - 1))];
        } else {
            v = sm_hll[i - kBins];
        }
        st_agent(&p->bit_hist[0] + i, v);
    }
    if (!last_of_grid(tickets, &last)) return;
    StatsAcc f{~0ull, 0, ~0ull, 0, 0, 0, 0, 0.0, 0, 0};
    for (uint32_t b = threadIdx.x; b < gridDim.x; b += kBlock) {
        const DevStats* q = partials + b;
        const uint64_t v0 = rd(&q->min_key), v1 = rd(&q->max_key);
        f.mn = v0 < f.mn ? v0 : f.mn;
        f.mx = v1 > f.mx ? v1 : f.mx;
        const uint64_t z1 = rd(&q->first_zero);
        f.zf = z1 < f.zf ? z1 : f.zf;
        f.unsorted |= rd(&q->unsorted);
        f.rl_eq += rd(&q->rl_eq);
        f.runs += rd(&q->runs);
        f.sum_bits += rd(&q->sum_bits);
        const uint64_t sfb = rd(reinterpret_cast<const uint64_t*>(&q->sum_f));
        double sfd;
        __builtin_memcpy(&sfd, &sfb, 8);
        f.sum_f += sfd;
        const uint32_t pp = rd32(&q->precision), dd = rd32(&q->delta_bits_max);
        f.prec = pp > f.prec ? pp : f.prec;
        f.dmax = dd > f.dmax ? dd : f.dmax;
    }
    constexpr int kFold = 8;
    const uint32_t words = gridDim.x * (kBins + kRegs);
    for (uint32_t i0 = threadIdx.x; i0 < words; i0 += kFold * kBlock) {
        uint32_t v[kFold];
#pragma unroll
        for (int u = 0; u < kFold; u++) {
            const uint32_t i = i0 + u * kBlock, b = i / (kBins + kRegs), e = i - b * (kBins + kRegs);
            v[u] = i < words ? rd32(&partials[b].bit_hist[0] + e) : 0u;
        }
#pragma unroll
        for (int u = 0; u < kFold; u++) {
            const uint32_t i = i0 + u * kBlock, e = i % (kBins + kRegs);
            if (i >= words) break;
            if (e < (uint32_t)kBins)
                atomicAdd(&fin[e], v[u]);
            else
                atomicMax(&fin[e], v[u]);
        }
    }
    f = block_fold(f, sm);  // its barriers also complete fin
    DevStats* out = reinterpret_cast<DevStats*>(host.dst);
    for (int i = threadIdx.x; i < kBins; i += kBlock) out->bit_hist[i] = fin[i];
    for (int i = threadIdx.x; i < kRegs; i += kBlock) out->hll[i] = fin[kBins + i];
    if (threadIdx.x == 0) {
        fold_fixup(x, f.mn, f.mx, f.zf);
        out->min_key = f.mn;
        out->max_key = f.mx;
        out->first_zero = f.zf;
        out->unsorted = f.unsorted;
        out->rl_eq = f.rl_eq;
        out->runs = f.runs + (n > 0 ? 1 : 0);
        out->sum_bits = f.sum_bits;
        out->sum_f = f.sum_f;
        out->precision = f.prec;
        out->delta_bits_max = f.dmax;
    }
    host_out_done(host);
}

// Workgroups of a reduction: two a CU, unless the rows are fewer.  Min/max of 64M
// int32 rows 47.2 us (four a CU: 48.2), of their deltas 47.5 (50.3); the statistics
// of 4M int32 rows 67 us (96), of 8M 86 (113), of 33.5M 207 (204), of 33.5M floats
// 144 (164), and at 1M rows or fewer the same.
int reduce_grid(Ctx* c, size_t n, int elem, int per_cu = 2) {
    const size_t per_block = (size_t)kBlock * (16 / elem) * 4;
    const size_t g = (n + per_block - 1) / per_block;
    const size_t cap = (size_t)c->cu_count * per_cu;
    return (int)std::max<size_t>(1, std::min(g, cap));
}

}  // namespace

HostOut launch_minmax(Ctx* c, int dtype, const void* x, size_t n, bool delta, MinMaxResult* d_result) {
    if (n == 0 || (delta && n < 2)) fail(DDJ_EINVAL, "min/max of too few rows");
    FoldTail ft;
    ft.tickets = c->control->tickets;
    ft.out = d_result;
    ft.host = host_out(c);
    dispatch_native(dtype, [&](auto tag) {
        using T = decltype(tag);
        const int grid = reduce_grid(c, n, sizeof(T));
        DevBuf partials(c, 24 * (size_t)grid);
        KernelTimer kt_(c, delta ? "k_minmax_delta" : "k_minmax");
        if (!delta) {
            hipLaunchKernelGGL(k_minmax<T>, dim3(grid), dim3(kBlock), 0, c->stream, static_cast<const T*>(x), n,
                               partials.get<uint64_t>(), ft);
        } else {
            if constexpr (std::is_floating_point<T>::value)
                fail(DDJ_EINVAL, "delta min/max: integer columns only");
            else
                hipLaunchKernelGGL(k_minmax_delta<T>, dim3(grid), dim3(kBlock), 0, c->stream, static_cast<const T*>(x),
                                   n, partials.get<uint64_t>(), ft);
        }
        HIPC(hipGetLastError());
    });
    return ft.host;
}

MinMaxResult wait_minmax(Ctx* c, const HostOut& h) {
    MinMaxResult r;
    memcpy(&r, wait_host_out(c, h), sizeof r);
    return r;
}

MinMaxResult minmax_to_host(Ctx* c, int dtype, const void* x, size_t n, bool delta) {
    return wait_minmax(c, launch_minmax(c, dtype, x, n, delta, nullptr));
}

FloatScanResult float_scan(Ctx* c, int dtype, const void* x, size_t n) {
    if (n == 0) fail(DDJ_EINVAL, "float scan of an empty array");
    FoldTail ft;
    ft.tickets = c->control->tickets;
    ft.host = host_out(c);
    dispatch_native(dtype, [&](auto tag) {
        using T = decltype(tag);
        if constexpr (std::is_floating_point<T>::value) {
            // the precision's divisions need more waves than a plain pass
            const int grid = reduce_grid(c, n, sizeof(T), 8);
            DevBuf partials(c, 32 * (size_t)grid);
            kernel_bytes(c, "k_minmax_prec", (double)n * sizeof(T));
            KernelTimer kt_(c, "k_minmax_prec");
            hipLaunchKernelGGL(k_minmax_prec<T>, dim3(grid), dim3(kBlock), 0, c->stream, static_cast<const T*>(x), n,
                               partials.get<uint64_t>(), ft);
            HIPC(hipGetLastError());
        } else {
            fail(DDJ_EINVAL, "float scan of an integer column");
        }
    });
    FloatScanResult r;
    memcpy(&r, wait_host_out(c, ft.host), sizeof r);
    return r;
}

void decode_minmax(int dtype, const MinMaxResult& r, void* mn, void* mx) {
    dispatch_native(dtype, [&](auto tag) {
        using T = decltype(tag);
        T a = from_order_key<T>(r.min_key), b = from_order_key<T>(r.max_key);
        memcpy(mn, &a, sizeof(T));
        memcpy(mx, &b, sizeof(T));
    });
}

DevStats device_stats(Ctx* c, int dtype, const void* x, size_t n) {
    if (n == 0) fail(DDJ_EINVAL, "stats of an empty array");
    static_assert(sizeof(DevStats) <= kHostOutBytes, "the record fits the result slot");
    const HostOut h = host_out(c);
    dispatch_native(dtype, [&](auto tag) {
        using T = decltype(tag);
        const int grid = reduce_grid(c, n, sizeof(T));
        DevBuf partials(c, sizeof(DevStats) * (size_t)grid);
        KernelTimer kt_(c, "k_stats");
        hipLaunchKernelGGL(k_stats<T>, dim3(grid), dim3(kBlock), 0, c->stream, static_cast<const T*>(x), n,
                           partials.get<DevStats>(), c->control->tickets, h);
        HIPC(hipGetLastError());
    });
    DevStats r;
    memcpy(&r, wait_host_out(c, h), sizeof r);
    return r;
}

}  // namespace ddj
