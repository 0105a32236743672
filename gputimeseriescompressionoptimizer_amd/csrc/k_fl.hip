// FL bit-packing (the reference's AFL encoding as it is actually called,
// run_afl_compress_gpu<T,1> / run_afl_decompress_gpu<T,1>,
// compression/afl/afl_gpu.cu:67-195).
//
// The reference stream is a contiguous LSB-first bit stream in words of T:
// value i occupies stream bits [i*b, (i+1)*b), stream bit p being bit p%W of
// word p/W.  On a little-endian machine that stream is the same byte sequence
// for every word width, so both kernels work on 32-bit words whatever T is;
// only the total length is rounded to whole T words.
//
// Pack: a workgroup owns a tile of 4096 values (a whole number of output
// words for any b), stages the values in LDS with 16-byte loads and emits
// the tile's 128*b output words, one word per thread-iteration, each word
// OR-ing the <= ceil(32/b)+1 values that overlap it.  Loads and stores are
// both fully coalesced.
//
// Unpack: a workgroup stages the tile's input in LDS from the aligned
// 16-byte chunks that hold it (an aligned chunk containing a valid byte never
// crosses a page, so the stream may start at any byte address) and every
// thread extracts values with a 64/96-bit funnel shift.
#include <type_traits>

#include "dispatch.h"
#include "k_common.h"
#include "kernels.h"
#include "k_fl_tile.h"

namespace ddj {

namespace {

template <typename T, bool DELTA = false>
__global__ __launch_bounds__(kBlock) void k_fl_pack(const T* __restrict__ x, size_t n, const MinMaxResult* mm,
                                                    int fixed_bits, uint8_t* __restrict__ out, size_t out_bytes,
                                                    SmallPieces sp) {
    __shared__ __attribute__((aligned(16))) T vals[kFlLdsVals];
    if ((size_t)blockIdx.x * kFlTile >= n) {  // one past the tiles
        write_small(sp);
        return;
    }
    int b = fixed_bits;
    if (mm) b = bitlen_of<T>(from_order_key<T>(mm->min_key), from_order_key<T>(mm->max_key));
    fl_pack_tile<T, DELTA>(x, n, b, out, out_bytes, blockIdx.x, vals);
}

template <typename T, int MAXB>
__global__ __launch_bounds__(kBlock) void k_fl_unpack(const uint8_t* __restrict__ in, size_t in_bytes, size_t n,
                                                      int b, T* __restrict__ out, size_t vbase) {
    // rows [vbase, vbase + n) of the stream into out[0, n)
    __shared__ __attribute__((aligned(16))) uint32_t w[fl_stage_words<MAXB>()];
    const size_t v0 = (size_t)blockIdx.x * kFlTile;
    const int nv = (int)((n - v0) < (size_t)kFlTile ? (n - v0) : (size_t)kFlTile);
    const int a = stage_fl_words(in, in_bytes, vbase + v0, nv, b, w);
    __syncthreads();
    const uint64_t mask = lowmask64(b);
    constexpr int V = 16 / (int)sizeof(T);
    if (nv == kFlTile && (reinterpret_cast<uintptr_t>(out + v0) & 15) == 0) {
        // whole tile: each lane unpacks V consecutive values into one 16-byte
        // store (a cached store: RLE's values and lengths are read next)
        u32x4* o4 = reinterpret_cast<u32x4*>(out + v0);
        for (int i = threadIdx.x; i < kFlTile / V; i += kBlock) {
            T vals[V];
#pragma unroll
            for (int k = 0; k < V; k++) vals[k] = (T)fl_value(w, V * i + k, b, a, mask);
            u32x4 q;
            __builtin_memcpy(&q, vals, 16);
            o4[i] = q;
        }
    } else {
        // consecutive lanes take consecutive values: their LDS reads spread over the banks
        for (int k = threadIdx.x; k < nv; k += kBlock) out[v0 + k] = (T)fl_value(w, k, b, a, mask);
    }
}

// DeltaEncoding::Decode over AflEncoding::Decode without writing the deltas
// (delta_encoding.cu:74-102 on afl_encoding.cu:74-113): k_fl_delta_sums
// unpacks each tile of 4096 b-bit deltas and writes their sum, k_scan_tiles
// turns the sums into tile prefixes, and k_fl_unpack_delta_scan unpacks the
// tile again and prefix-sums it (wrapping in T) on top of the first row and
// its prefix.  The packed stream is b/8 bytes a row, so reading it twice
// costs far less than writing and re-reading the deltas.  out has m + 1 rows.
template <int MAXB>
__global__ __launch_bounds__(kBlock) void k_fl_delta_sums(const uint8_t* __restrict__ in, size_t in_bytes, size_t m,
                                                          int b, uint64_t* __restrict__ vals, size_t split,
                                                          size_t m2, ScanTail st) {
    // sums of the deltas [0, m), one per tile of 4096; with split > 0, of
    // [0, split) in the first ceil(split / 4096) tiles and of [split, split +
    // m2) in the others (a row range: the deltas before it and its own)
    __shared__ __attribute__((aligned(16))) uint32_t w[fl_stage_words<MAXB>()];
    __shared__ uint64_t red[kBlock / kWave];
    size_t tile = blockIdx.x, vbase = 0;
    if (split) {  // uniform
        const size_t before = (split + kFlTile - 1) / kFlTile;
        if (tile >= before) {
            tile -= before;
            vbase = split;
            m = m2;
        } else {
            m = split;
        }
    }
    const size_t v0 = tile * kFlTile;
    const int nv = v0 < m ? (int)((m - v0) < (size_t)kFlTile ? (m - v0) : (size_t)kFlTile) : 0;
    uint64_t sum = 0;
    if (MAXB == 32 && b == 32 && nv == kFlTile && 4 * (vbase + v0 + kFlTile) + 4 <= in_bytes) {  // uniform
        // 32-bit deltas are the stream's own words: no staging.  The word after
        // a load's four (a stream at any byte address) is the next lane's first.
        const uintptr_t at = reinterpret_cast<uintptr_t>(in) + 4 * (vbase + v0);
        const uint32_t r = (uint32_t)(at & 3);
        const uint32_t* p = reinterpret_cast<const uint32_t*>(at & ~(uintptr_t)3);
#pragma unroll
        for (int q = 0; q < kFlTile / 4 / kBlock; q++) {
            const int i = 4 * (threadIdx.x + q * kBlock);
            const uint32_t w0 = p[i], w1 = p[i + 1], w2 = p[i + 2], w3 = p[i + 3], w4 = r ? p[i + 4] : 0u;
            sum += (uint64_t)__builtin_amdgcn_alignbyte(w1, w0, r) + __builtin_amdgcn_alignbyte(w2, w1, r) +
                   __builtin_amdgcn_alignbyte(w3, w2, r) + __builtin_amdgcn_alignbyte(w4, w3, r);
        }
    } else {
        const int a = stage_fl_words(in, in_bytes, vbase + v0, nv, b, w);
        __syncthreads();
        const uint64_t mask = lowmask64(b);
        for (int k = threadIdx.x; k < nv; k += kBlock) sum += fl_value(w, k, b, a, mask);
    }
    uint64_t total;
    block_exclusive_scan<uint64_t>(sum, &total, red);
    if (threadIdx.x == 0) put_tile(st, vals, blockIdx.x, total);
    scan_tail(st, vals);
}

// OUT: the row type written: T, or with T = int32 the float or double that a
// floatToInt node above decodes to (row / 10^p in double, as
// k_int_to_float).  `bias` is added to every row (a scale node above): it joins
// the first row.  The nodes above then need no pass of their own: a float64
// column of 33.5M rows decodes in 66 us instead of 78 + 74, a float32 one
// through scale in 42 instead of 78 + 58 + 45.
template <typename T, int MAXB, typename OUT>
__global__ __launch_bounds__(kBlock) void k_fl_unpack_delta_scan(const uint8_t* first_bytes, const uint8_t* __restrict__ in,
                                                                 size_t in_bytes, size_t m, int b, OUT* __restrict__ out,
                                                                 const uint64_t* __restrict__ prefix, size_t vbase,
                                                                 uint64_t bias, double pow10) {
    // rows r[0] = first + bias + prefix[0]; r[i + 1] = r[i] + d[vbase + i] for i < m
    // the staged words, then the tile's rows (one pad slot per 16, which spreads
    // the 16 consecutive rows of every thread over the banks)
    constexpr int kPer = kFlTile / kBlock;  // 16 consecutive values per thread
    auto slot = [](int i) { return i + (i >> 4); };
    __shared__ __attribute__((aligned(16))) uint32_t w[cmax(fl_stage_words<MAXB>(), (kFlTile + kFlTile / 16) * (int)sizeof(T) / 4)];
    __shared__ uint64_t red[kBlock / kWave];
    auto conv = [&](T v) -> OUT {
        if constexpr (std::is_same<T, OUT>::value)
            return v;
        else
            return (OUT)__ddiv_rn((double)(OUT)v, pow10);
    };
    T first;
    __builtin_memcpy(&first, first_bytes, sizeof(T));
    const uint32_t tile = blockIdx.x;
    const size_t v0 = (size_t)tile * kFlTile;
    const int nv = (int)((m - v0) < (size_t)kFlTile ? (m - v0) : (size_t)kFlTile);
    uint64_t d[kPer], sum = 0;
    if (MAXB == 32 && sizeof(T) == 4 && b == 32 && nv == kFlTile && 4 * (vbase + v0 + kFlTile) + 4 <= in_bytes) {
        // uniform: 32-bit deltas are the stream's own words, each thread's 16 of
        // them (at any byte address) straight into registers
        const uintptr_t at = reinterpret_cast<uintptr_t>(in) + 4 * (vbase + v0 + (size_t)threadIdx.x * kPer);
        const uint32_t r = (uint32_t)(at & 3);
        const uint32_t* p = reinterpret_cast<const uint32_t*>(at & ~(uintptr_t)3);
        uint32_t x[kPer + 1];
#pragma unroll
        for (int k = 0; k < kPer; k++) x[k] = p[k];
        x[kPer] = r ? p[kPer] : 0u;
#pragma unroll
        for (int k = 0; k < kPer; k++) d[k] = __builtin_amdgcn_alignbyte(x[k + 1], x[k], r);
    } else {
        const int a = stage_fl_words(in, in_bytes, vbase + v0, nv, b, w);
        __syncthreads();
        const uint64_t mask = lowmask64(b);
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = threadIdx.x * kPer + k;
            d[k] = i < nv ? fl_value(w, i, b, a, mask) : 0;
        }
    }
#pragma unroll
    for (int k = 0; k < kPer; k++) sum += d[k];
    uint64_t total;
    const uint64_t excl = block_exclusive_scan<uint64_t>(sum, &total, red);  // a barrier: w is free again
    T* res = reinterpret_cast<T*>(w);
    uint64_t run = ubits(first) + bias + prefix[tile] + excl;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        run += d[k];
        res[slot(threadIdx.x * kPer + k)] = (T)run;
    }
    __syncthreads();
    // out[v0 + 1 ..]: single rows up to a 16-byte boundary, then 16-byte
    // stores from consecutive lanes, then single rows
    OUT* dst = out + v0 + 1;
    constexpr int V = 16 / (int)sizeof(OUT);
    int head = (int)(((16 - (reinterpret_cast<uintptr_t>(dst) & 15)) & 15) / sizeof(OUT));
    head = head < nv ? head : nv;
    int nq = (nv - head) / V;
    if ((reinterpret_cast<uintptr_t>(dst) % sizeof(OUT)) != 0) {  // not on a row boundary: rows only
        head = 0;
        nq = 0;
    }
    if ((int)threadIdx.x < head) dst[threadIdx.x] = conv(res[slot(threadIdx.x)]);
    u32x4* d4 = reinterpret_cast<u32x4*>(dst + head);
    for (int i = threadIdx.x; i < nq; i += kBlock) {
        OUT vals[V];
#pragma unroll
        for (int k = 0; k < V; k++) vals[k] = conv(res[slot(head + V * i + k)]);
        u32x4 q;
        __builtin_memcpy(&q, vals, 16);
        __builtin_nontemporal_store(q, d4 + i);
    }
    for (int i = head + V * nq + threadIdx.x; i < nv; i += kBlock) dst[i] = conv(res[slot(i)]);
    if (tile == 0 && threadIdx.x == 0) out[0] = conv((T)(ubits(first) + bias + prefix[0]));
}

}  // namespace

namespace {
// Calls f(std::integral_constant<int, MAXB>) with the narrowest staging class
// (16, 32 or 64 bits) that holds b.
template <typename F> void with_maxb(int b, F&& f) {
    if (b <= 16)
        f(std::integral_constant<int, 16>{});
    else if (b <= 32)
        f(std::integral_constant<int, 32>{});
    else
        f(std::integral_constant<int, 64>{});
}
}  // namespace

void launch_fl_pack(Ctx* c, int dtype, const void* x, size_t n, const MinMaxResult* mm, int bits, void* out,
                    size_t out_bytes, const SmallPieces& sp) {
    if (n == 0) return;
    const int esize = (int)dtype_size(dtype);
    dispatch_int(esize, [&](auto tag) {
        using T = decltype(tag);
        if (out_bytes == 0) {  // the widest b, rounded up to whole words
            const int maxb = mm ? 8 * (int)sizeof(T) : bits;
            const uint64_t W = 8 * sizeof(T);
            out_bytes = ((size_t)((maxb * (uint64_t)n + W - 1) / W) * sizeof(T) + 3) & ~size_t(3);
        }
        const size_t tiles = (n + kFlTile - 1) / kFlTile;
        { KernelTimer kt_(c, "k_fl_pack"); hipLaunchKernelGGL(k_fl_pack<T>, dim3((unsigned)(tiles + (sp.count ? 1 : 0))), dim3(kBlock), 0, c->stream,
                           static_cast<const T*>(x), n, mm, bits, static_cast<uint8_t*>(out), out_bytes, sp); }
        HIPC(hipGetLastError());
    });
}

void launch_fl_pack_delta(Ctx* c, int elem_size, const void* x, size_t m, const MinMaxResult* mm, void* out, int bits,
                          size_t out_bytes, const SmallPieces& sp) {
    if (m == 0) return;
    dispatch_int(elem_size, [&](auto tag) {
        using T = decltype(tag);
        if (out_bytes == 0) {  // the widest b, rounded up to whole words
            const uint64_t W = 8 * sizeof(T);
            out_bytes = ((size_t)((W * m + W - 1) / W) * sizeof(T) + 3) & ~size_t(3);
        }
        const size_t tiles = (m + kFlTile - 1) / kFlTile;
        { KernelTimer kt_(c, "k_fl_pack"); hipLaunchKernelGGL((k_fl_pack<T, true>), dim3((unsigned)(tiles + (sp.count ? 1 : 0))), dim3(kBlock), 0, c->stream,
                           static_cast<const T*>(x), m, mm, bits, static_cast<uint8_t*>(out), out_bytes, sp); }
        HIPC(hipGetLastError());
    });
}

size_t fl_unpack_delta_scratch_words(size_t m) { return 2 * ((m + kFlTile - 1) / kFlTile) + 1; }

void launch_fl_unpack_delta(Ctx* c, int elem_size, const uint8_t* first, const uint8_t* in, size_t in_bytes, size_t m,
                           int bits, void* out, uint64_t* tile_scratch, const FlDeltaOut& o) {
    dispatch_int(elem_size, [&](auto tag) {
        using T = decltype(tag);
        if (bits <= 0 || bits > 8 * (int)sizeof(T)) fail(DDJ_ECORRUPT, "FL bit width out of range");
        if (o.dtype >= 0 && sizeof(T) != 4) fail(DDJ_EINVAL, "converted rows come from int32 deltas");
        const bool plain = o.dtype < 0 && o.bias == 0;
        if (m == 0 && plain) {
            d2d(c, out, first, sizeof(T));
            return;
        }
        const size_t tiles = m ? (m + kFlTile - 1) / kFlTile : 1;
        std::unique_ptr<TileScan> own_scan;
        uint64_t* vals = tile_scratch;
        if (!vals) {
            own_scan = std::make_unique<TileScan>(c, tiles);
            vals = own_scan->vals;
        }
        uint64_t* prefix = vals + tiles;
        // caller's scratch: a scan launch of its own, which touches nothing
        // that other calls of the context share
        const ScanTail st = own_scan ? own_scan->tail(c, false) : ScanTail{};
        kernel_bytes(c, "k_fl_delta_sums", (double)((m * (uint64_t)bits + 7) / 8));
        with_maxb(bits, [&](auto mb) {
            constexpr int MAXB = decltype(mb)::value;
            { KernelTimer kt_(c, "k_fl_delta_sums"); hipLaunchKernelGGL(k_fl_delta_sums<MAXB>, dim3((unsigned)tiles), dim3(kBlock), 0, c->stream,
                               in, in_bytes, m, bits, vals, (size_t)0, (size_t)0, st); }
            HIPC(hipGetLastError());
            if (own_scan)
                own_scan->finish(c, st);
            else
                launch_scan_tiles(c, vals, tiles, prefix);
            KernelTimer kt_(c, "k_fl_unpack_delta_scan");
            auto run = [&](auto out_tag) {
                using OUT = decltype(out_tag);
                hipLaunchKernelGGL((k_fl_unpack_delta_scan<T, MAXB, OUT>), dim3((unsigned)tiles), dim3(kBlock), 0, c->stream,
                                   first, in, in_bytes, m, bits, static_cast<OUT*>(out), (const uint64_t*)prefix, (size_t)0,
                                   o.bias, o.pow10);
            };
            if constexpr (sizeof(T) == 4) {
                if (o.dtype == DDJ_D_FLOAT) return run(float());
                if (o.dtype == DDJ_D_DOUBLE) return run(double());
            }
            run(T());
        });
        HIPC(hipGetLastError());
    });
}

void launch_fl_unpack(Ctx* c, int dtype, const uint8_t* in, size_t in_bytes, size_t n, int bits, void* out,
                      size_t first_row) {
    if (n == 0) return;
    const int esize = (int)dtype_size(dtype);
    dispatch_int(esize, [&](auto tag) {
        using T = decltype(tag);
        if (bits <= 0 || bits > 8 * (int)sizeof(T)) fail(DDJ_ECORRUPT, "FL bit width out of range");
        const size_t tiles = (n + kFlTile - 1) / kFlTile;
        with_maxb(bits, [&](auto mb) {
            constexpr int MAXB = decltype(mb)::value;
            KernelTimer kt_(c, "k_fl_unpack");
            hipLaunchKernelGGL((k_fl_unpack<T, MAXB>), dim3((unsigned)tiles), dim3(kBlock), 0, c->stream, in, in_bytes, n,
                               bits, static_cast<T*>(out), first_row);
        });
        HIPC(hipGetLastError());
    });
}

void launch_fl_unpack_delta_rows(Ctx* c, int elem_size, const uint8_t* first, const uint8_t* in, size_t in_bytes,
                                 int bits, size_t begin, size_t count, void* out) {
    if (count == 0) return;
    dispatch_int(elem_size, [&](auto tag) {
        using T = decltype(tag);
        if (bits <= 0 || bits > 8 * (int)sizeof(T)) fail(DDJ_ECORRUPT, "FL bit width out of range");
        // tile sums of the deltas before the range (part A) and inside it
        // (part B) in one array: one scan gives part B's prefixes on top of
        // the sum of everything before the range
        const size_t mb = count - 1;
        const size_t ta = (begin + kFlTile - 1) / kFlTile;
        const size_t tb = mb ? (mb + kFlTile - 1) / kFlTile : 1;
        TileScan ts(c, ta + tb);
        kernel_bytes(c, "k_fl_delta_sums", (double)(((begin + mb) * (uint64_t)bits + 7) / 8));
        with_maxb(bits, [&](auto mbits) {
            constexpr int MAXB = decltype(mbits)::value;
            const ScanTail st = ts.tail(c, false);
            {
                KernelTimer kt_(c, "k_fl_delta_sums");
                hipLaunchKernelGGL(k_fl_delta_sums<MAXB>, dim3((unsigned)(ta + tb)), dim3(kBlock), 0, c->stream, in,
                                   in_bytes, mb, bits, ts.vals, begin, mb, st);
            }
            HIPC(hipGetLastError());
            ts.finish(c, st);
            KernelTimer kt_(c, "k_fl_unpack_delta_scan");
            hipLaunchKernelGGL((k_fl_unpack_delta_scan<T, MAXB, T>), dim3((unsigned)tb), dim3(kBlock), 0, c->stream, first,
                               in, in_bytes, mb, bits, static_cast<T*>(out), (const uint64_t*)(ts.prefix + ta), begin,
                               (uint64_t)0, 1.0);
        });
        HIPC(hipGetLastError());
    });
}

}  // namespace ddj
