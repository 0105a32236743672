// Most-frequent values (Histogram::GetMostFrequent, reference
// util/histogram/histogram.cpp:29-41 -> thrust_sparse_histogram.cu:20-69 and
// most_frequent.cu:10-26): exact counts of every distinct value, then the K
// largest counts, equal counts ordered by the smaller value (what the
// reference's stable sort of key-sorted bins yields).
//
// Counting: each workgroup aggregates its rows in LDS (plain LDS atomics; the
// up to 16 rows a thread loads at once keep HBM busy while they wait): integers
// near the first row by offset, other keys in a hash table of kHistParts
// partitions, each key's partition fixed by its hash.  The workgroups write
// their keys and counts out; the last of them adds them up in LDS if they are
// few, else k_hist_merge does, one workgroup per partition, so that no key is
// counted through device-scope atomics.  A column with more distinct keys than
// these tables hold is counted again by more workgroups of fewer rows each,
// and, past what those or the merge's tables hold, into a global
// open-addressing table (64-bit keys, ~0 = empty).  A value equal to a table's empty marker is counted on the side.
// Floats count -0.0 with +0.0 (operator==), reporting -0.0 when one was seen
// (it sorts first in the reference).  A NaN equals nothing, so each NaN row is
// a bin of count 1: they stay out of the tables, and every workgroup keeps the
// four smallest (radix order) NaN rows, which is all the top-K can ever take
// from them.  Columns of a few thousand rows are counted whole in one
// workgroup's LDS (k_hist_small).  The global table starts at 2n slots (at
// least 1024, at most 64K, or what k_hist_merge's tables found too many keys
// for); if it ends up more than 70% full the host retries
// once with a table of twice the keys seen (the exact count, and with a full
// table the HyperLogLog estimate of the keys that it turned away), and a second
// retry, never needed in practice, sizes it for every row distinct.
#include <cmath>
#include <type_traits>

#include "dispatch.h"
#include "k_common.h"
#include "kernels.h"

namespace ddj {

namespace {

constexpr uint64_t kEmpty = ~0ull;
constexpr int kMaxK = 4;

constexpr uint32_t kTooSmall = 1, kNeedMerge = 2;  // HistCtl::overflow
struct HistCtl {
    unsigned long long distinct;
    unsigned long long special;  // rows whose bit pattern (4- and 8-byte types) marks an empty slot
    unsigned long long nans;     // NaN rows (floats)
    uint32_t overflow;           // kTooSmall: a table was; kNeedMerge
    uint32_t negzero;
};

__device__ __forceinline__ uint64_t hmix(uint64_t z) {
    z ^= z >> 33;
    z *= 0xff51afd7ed558ccdull;
    z ^= z >> 33;
    z *= 0xc4ceb9fe1a85ec53ull;
    z ^= z >> 33;
    return z;
}

template <typename T> __device__ __forceinline__ uint64_t hist_key(T v, bool& negzero) {
    if constexpr (std::is_floating_point<T>::value) {
        if (v == T(0)) {
            if (__builtin_signbit(v)) negzero = true;
            return 0;
        }
    }
    return ubits(v);
}

// The global table.  New keys are counted per thread and summed (a counter
// bumped once per new key serializes every workgroup on one address, which for
// a column of 10^4 distinct rows was most of the count's time).  A table that
// fills is dropped and counted again in a larger one, so a thread that once
// found no slot (no free one within kProbes: far past what a table 70% full
// needs) adds no more keys and only notes them for the estimate that sizes the
// next table.  Sized by the rows turned away, every one of them possibly a new
// key, 64M rows of 65,536 values took tables of 2 GiB and 23.5 ms; by the
// estimate 4 MiB and 21.2 ms.
constexpr uint64_t kProbes = 512;
constexpr int kHllBits = 10, kHllRegs = 1 << kHllBits;  // within 3% (one sigma)
// Notes a key in a workgroup's registers (LDS).  By the high bits of its hash:
// the keys that meet a full stretch of a table share low ones.
__device__ __forceinline__ void hll_note(uint64_t key, volatile uint32_t* regs) {
    const uint64_t h = hmix(key);
    const uint32_t r = (uint32_t)(h >> (64 - kHllBits));
    const uint32_t rank = (uint32_t)__clzll((h << kHllBits) | (1ull << (kHllBits - 1))) + 1;
    if (rank > regs[r]) atomicMax(const_cast<uint32_t*>(&regs[r]), rank);
}
// A workgroup's register into the column's.
__device__ __forceinline__ void hll_merge(uint32_t* hll, int r, uint32_t rank) {
    if (rank > __hip_atomic_load(&hll[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&hll[r], rank);
}

struct GlobalTable {
    unsigned long long* keys = nullptr;
    unsigned long long* counts = nullptr;
    uint64_t mask = 0;
    HistCtl* ctl = nullptr;
    uint32_t* hll = nullptr;  // kHllRegs registers: the keys turned away
    uint32_t fresh = 0;       // keys this thread brought in
    bool full = false;        // it found no slot for one
    __device__ __forceinline__ uint64_t home(uint64_t key) const { return hmix(key) & mask; }
    __device__ __forceinline__ unsigned long long peek(uint64_t s) const {
        return __hip_atomic_load(&keys[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // regs: the workgroup's registers (LDS)
    __device__ __forceinline__ void add(uint64_t key, unsigned long long cnt, volatile uint32_t* regs) {
        if (!full) {
            uint64_t s = home(key);
            for (uint64_t p = 0; p <= mask && p < kProbes; p++) {
                unsigned long long seen = peek(s);
                if (seen == kEmpty) {
                    const unsigned long long prev = atomicCAS(&keys[s], kEmpty, (unsigned long long)key);
                    if (prev == kEmpty) fresh++;
                    seen = prev == kEmpty ? key : prev;
                }
                if (seen == key) {
                    atomicAdd(&counts[s], cnt);
                    return;
                }
                s = (s + 1) & mask;
            }
            full = true;
        }
        hll_note(key, regs);
    }
};

// How many keys the registers have seen.
double hll_estimate(const uint32_t* regs) {
    const double m = kHllRegs;
    double sum = 0;
    int zeros = 0;
    for (int i = 0; i < kHllRegs; i++) {
        sum += std::ldexp(1.0, -(int)regs[i]);
        zeros += regs[i] == 0;
    }
    const double e = 0.7213 / (1.0 + 1.079 / m) * m * m / sum;
    return e <= 2.5 * m && zeros ? m * std::log(m / zeros) : e;
}

// Ascending list of the (up to) four smallest keys seen, with multiplicity.
struct Small4 {
    uint64_t l[kMaxK];
    int c = 0;
    __device__ __forceinline__ void insert(uint64_t k) {
#pragma unroll
        for (int j = 0; j < kMaxK; j++) {
            if (j < c) {
                if (k < l[j]) {
                    const uint64_t t = l[j];
                    l[j] = k;
                    k = t;
                }
            } else if (j == c) {
                l[j] = k;
            }
        }
        c = c < kMaxK ? c + 1 : kMaxK;
    }
    __device__ __forceinline__ void pop() {
#pragma unroll
        for (int j = 0; j + 1 < kMaxK; j++) l[j] = l[j + 1];
        c--;
    }
};

// Four smallest keys of the workgroup (each thread holds a Small4) into
// out_keys[0..*out_n).  Wave rounds take the smallest head, then thread 0
// merges the waves' lists.
template <int NT>
__device__ void block_small4(Small4& s, uint64_t* sm_keys /* NT/kWave * kMaxK */, int* sm_cnt /* NT/kWave */,
                             uint64_t* out_keys, uint32_t* out_n) {
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    int got = 0;
    for (int r = 0; r < kMaxK; r++) {
        const bool has = s.c > 0;
        const uint64_t h = has ? s.l[0] : ~0ull;
        const uint64_t m = wave_min(h);
        const uint64_t who = __ballot(has && h == m);
        if (who == 0) break;
        if (lane == __builtin_ctzll(who)) s.pop();
        if (lane == 0) sm_keys[wid * kMaxK + r] = m;
        got++;
    }
    if (lane == 0) sm_cnt[wid] = got;
    __syncthreads();
    if (threadIdx.x == 0) {
        Small4 b;
        for (int w = 0; w < NT / kWave; w++)
            for (int r = 0; r < sm_cnt[w]; r++) b.insert(sm_keys[w * kMaxK + r]);
#pragma unroll
        for (int r = 0; r < kMaxK; r++)
            if (r < b.c) out_keys[r] = b.l[r];
        *out_n = (uint32_t)b.c;
    }
}

// The counting workgroup's hash table: kHistParts partitions of 192 slots of
// 4-byte keys (narrower types widened) or 128 of 8-byte keys.  A hash of the
// key's folded halves in 32 bits (cheaper than hmix's 64-bit multiplies, which
// the other tables keep) gives the partition and the slot to start from; probing
// stays inside the partition.
//
// SPREAD: one multiplication, which lays whole numbers in a row (codes, ids)
// out evenly, so that 10,000 of them fill the table without long probes (16M
// rows of them 57 us, with the mix 332).  But it packs the rows of some arithmetic
// progressions (strides 10946, 50549, ...; sampled times are such columns) into
// one end of a table: 10,000 of them took 3000-4700 probes a row.  Where nothing
// comes after it that would count such columns, the hash is a mix.
template <typename T> using HistKey = typename std::conditional<sizeof(T) == 8, unsigned long long, uint32_t>::type;
constexpr int kHistParts = 64;
template <typename T> constexpr int part_slots() { return sizeof(T) == 8 ? 128 : 192; }
// A partition written out: the keys in use with their counts, in any order.
template <typename KT> struct HistEntry {
    KT key;
    uint32_t count;
};
template <bool SPREAD> __device__ __forceinline__ uint32_t lds_hash(uint64_t key) {
    uint32_t a = (uint32_t)key ^ ((uint32_t)(key >> 32) * 0x85ebca6bu);
    if (SPREAD) return a * 0x9E3779B1u;
    a = (a ^ (a >> 16)) * 0x85ebca6bu;
    a = (a ^ (a >> 13)) * 0xc2b2ae35u;
    return a ^ (a >> 16);
}

// What a counting workgroup saw outside its tables.
struct HistInfo {
    unsigned long long special, nans;
    uint32_t negzero, overflow;
    uint32_t nan_n, pad;
    uint64_t nan_keys[kMaxK];
};

// Workgroups of 1024 threads, one per CU, stride over tiles of 16 rows a
// thread, whose loads are issued together.
//
// Columns that leave a workgroup no more than few_rows a thread are counted in
// tiles of that many, one a workgroup: distinct or not, their keys fit its table
// (two thirds and half of its slots), so that only the merge's tables can be
// too small.  With 16 rows a thread every column of more than 5,500 random keys
// (3,500 of 8 bytes) was counted in vain and then again in the global table.  A
// dictionary encode of 100,000 int32 rows with 16,000 keys 231 us, of int64 rows
// 251, now 86 and 82 (in the global table alone 184 and 185); of 1M rows with
// 60,000 keys 1187 and 1247, now 125 and 106; of 100,000 rows with 50 keys 55 and
// 56, now 53 and 52.
constexpr int kHistThreads = 1024, kMergeThreads = 1024, kMergeSlots = 4096;
template <typename T> constexpr int few_rows() { return sizeof(T) == 8 ? 4 : sizeof(T) == 1 ? 16 : 8; }
// Entries a workgroup may write out.
template <typename T, int PER> constexpr int seg_slots() {
    return PER < 16 ? PER * kHistThreads : kHistParts * part_slots<T>();
}

// Integer columns: keys within kWindow / 2 of the first row's (dictionary
// codes, categories, most small integers) are counted by their offset, in
// kCopies copies of the window, lane l in copy l % kCopies: no key compare, no
// probing, and few lanes of a wave on one bank.  The count of the 64M-row
// Zipf(1.2)/50 column was bound by the probe loop's instructions and the LDS
// atomics' same-address conflicts (92 us); with the window it takes 53, against
// 42 for a plain pass over the column.
constexpr int kWindow = 1024, kCopies = 8;

struct Cand {
    unsigned long long count;
    uint64_t key;
};

// What the host gets: the table's state and the best K (the rest empty).
struct HistResult {
    HistCtl ctl;
    Cand top[kMaxK];
};

template <typename T> __device__ __forceinline__ bool better(const Cand& a, const Cand& b) {
    if (a.count != b.count) return a.count > b.count;
    T va, vb;
    using U = typename UnsignedOf<T>::type;
    U ua = (U)a.key, ub = (U)b.key;
    __builtin_memcpy(&va, &ua, sizeof(T));
    __builtin_memcpy(&vb, &ub, sizeof(T));
    return order_key(va) < order_key(vb);
}

// Inserts c into the sorted list top[0..K) (K <= kMaxK).  Loops run to
// kMaxK with guards so that a register-resident list keeps constant indices.
template <typename T> __device__ __forceinline__ void push(Cand* top, int K, Cand c) {
    if (c.count == 0) return;
    int pos = 0;  // entries that stay ahead of c
#pragma unroll
    for (int i = 0; i < kMaxK; i++)
        if (i < K && top[i].count != 0 && !better<T>(c, top[i])) pos = i + 1;
    if (pos >= K) return;
#pragma unroll
    for (int j = kMaxK - 1; j > 0; j--)
        if (j < K && j > pos) top[j] = top[j - 1];
#pragma unroll
    for (int i = 0; i < kMaxK; i++)
        if (i == pos) top[i] = c;
}

// The best K candidates of a wave whose lanes hold sorted lists of K: K
// rounds, each taking the largest head (by count; the heads that tie by the
// smaller order key) off its lane's list.  Lane 0 writes round r's to out[r]
// (count 0 when the lists are empty).  One wave maximum and one ballot a
// round: a pairwise merge of the lists through LDS, with its lists indexed by
// data, took 13-18 us a launch, this 5.
template <typename T> __device__ __forceinline__ void wave_best(Cand* top, int K, Cand* out) {
    const int lane = threadIdx.x & (kWave - 1);
    for (int r = 0; r < K; r++) {  // uniform
        const unsigned long long m = wave_max(top[0].count);
        uint64_t who = __ballot(top[0].count == m);
        if (m != 0 && (who & (who - 1)) != 0) {  // a tie (uniform)
            T v;
            using U = typename UnsignedOf<T>::type;
            const U u = (U)top[0].key;
            __builtin_memcpy(&v, &u, sizeof(T));
            const bool mine = top[0].count == m;
            const uint64_t ok = mine ? order_key(v) : ~0ull;
            const uint64_t k = wave_min(ok);
            who = __ballot(mine && ok == k);
        }
        if (lane == __builtin_ctzll(who)) {
            out[r] = m ? top[0] : Cand{0, 0};
#pragma unroll
            for (int i = 0; i + 1 < kMaxK; i++) top[i] = top[i + 1];
            top[kMaxK - 1] = Cand{0, 0};
        }
    }
}

// The best K of the workgroup's sorted lists into out[0..K), by wave 0 (sc:
// LDS for kMaxK candidates per wave); the other waves only contribute.
template <typename T, int NT = kBlock> __device__ void block_best(Cand* top, int K, Cand* sc, Cand* out) {
    const int wid = threadIdx.x / kWave;
    wave_best<T>(top, K, sc + wid * kMaxK);
    __syncthreads();
    if (wid == 0) {
        Cand one[kMaxK];
#pragma unroll
        for (int i = 0; i < kMaxK; i++) one[i] = Cand{0, 0};
        const int t = threadIdx.x;
        static_assert(NT / kWave * kMaxK <= kWave, "a candidate a lane");
        if (t < NT / kWave * kMaxK && (t & (kMaxK - 1)) < K) one[0] = sc[t];
        wave_best<T>(one, K, out);
    }
    __syncthreads();
}

// The host's result from the best K of the tables (thread 0 of the last
// workgroup) and the counting workgroups' records: rows of the empty markers'
// bit pattern (all ones), and every NaN row as a bin of count 1.
template <typename T>
__device__ void finish_topk(const Cand* best, int K, HistCtl ctl, const HistInfo* info, uint32_t blocks,
                            HistResult* out) {
    Cand b[kMaxK];
#pragma unroll
    for (int i = 0; i < kMaxK; i++) b[i] = i < K ? best[i] : Cand{0, 0};
    if (ctl.special) push<T>(b, K, Cand{ctl.special, (uint64_t)(HistKey<T>)~(HistKey<T>)0});
    if (std::is_floating_point<T>::value && ctl.nans)
        for (uint32_t g = 0; g < blocks; g++)
            for (uint32_t r = 0, nr = ld_agent(&info[g].nan_n); r < nr; r++)
                push<T>(b, K, Cand{1ull, ubits(from_order_key<T>(ld_agent(&info[g].nan_keys[r])))});
    out->ctl = ctl;
#pragma unroll
    for (int i = 0; i < kMaxK; i++) out->top[i] = b[i];
}

// The counting workgroups' records summed into ctl (LDS), by one workgroup.
template <int NT> __device__ __forceinline__ void fold_info(const HistInfo* info, uint32_t blocks, HistCtl* ctl) {
    for (uint32_t g = threadIdx.x; g < blocks; g += NT) {
        const unsigned long long special = ld_agent(&info[g].special), nans = ld_agent(&info[g].nans);
        const uint32_t negzero = ld_agent(&info[g].negzero), over = ld_agent(&info[g].overflow);
        if (special) atomicAdd(&ctl->special, special);
        if (nans) atomicAdd(&ctl->nans, nans);
        if (negzero) atomicOr(&ctl->negzero, 1u);
        if (over) atomicOr(&ctl->overflow, kTooSmall);
    }
}

// A table's entries into sorted lists of K, a list a thread, and the keys
// counted into *distinct.
template <typename T, int SLOTS, int NT, typename KT, typename CT>
__device__ __forceinline__ void take_table(const KT* skey, const CT* scnt, Cand* top, int K, uint32_t* distinct) {
#pragma unroll
    for (int i = 0; i < kMaxK; i++) top[i] = Cand{0, 0};
    uint32_t d = 0;
    for (int s = threadIdx.x; s < SLOTS; s += NT)
        if (scnt[s]) {
            d++;
            push<T>(top, K, Cand{scnt[s], (uint64_t)skey[s]});
        }
    d = wave_sum(d);
    if ((threadIdx.x & (kWave - 1)) == 0 && d) atomicAdd(distinct, d);
}

// The segment that entry e lies in: first[s] <= e < first[s + 1].
__device__ __forceinline__ uint32_t segment_of(const uint32_t* first, uint32_t segments, uint32_t e) {
    uint32_t lo = 0, hi = segments;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (first[mid] <= e)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// GLOBAL: the tables are flushed into, and keys without a slot added to, the
// global table, which k_hist_topk searches.  Else the workgroup's used slots
// go to segs (its seg_slots entries from blockIdx.x on, partition
// by partition, partition p from off[p * grid + workgroup] on), and a key
// without a slot ends the count (info[].overflow: the host counts again with
// GLOBAL).  With a tail, the last workgroup adds all workgroups' entries up itself
// and hands the best K to the host, if its table has a slot for each or, up to
// kTailEntries, no workgroup has more than kTailKeys (columns of few distinct
// values); else (kNeedMerge), or if too many turn out distinct, k_hist_merge does.
// 300,000 int64 rows of 130 values, 9,600 entries: 62 us encoded, through the merge
// 71.  13,000 distinct rows, all of them entries: 47 us counted in two launches, and
// after a tail that took 256 probes to find its table full 401.
constexpr uint32_t kTailEntries = 16384, kTailKeys = 512;
struct HistTail {
    uint32_t* tickets = nullptr;
    int K = 0;
    HostOut host;
};
template <typename T, int PER, bool GLOBAL>
__global__ __launch_bounds__(kHistThreads) void k_hist_count(const T* __restrict__ x, size_t n, GlobalTable table,
                                                             HistEntry<HistKey<T>>* __restrict__ segs,
                                                             uint32_t* __restrict__ off, HistInfo* __restrict__ info,
                                                             uint32_t* __restrict__ hll, HistTail tail) {
    using KT = HistKey<T>;
    constexpr KT kFree = (KT)~(KT)0;  // an empty slot; rows of that bit pattern are counted on the side
    constexpr int PS = part_slots<T>(), kLdsSlots = kHistParts * PS;
    __shared__ __attribute__((aligned(16))) KT skey[kLdsSlots];
    __shared__ __attribute__((aligned(16))) uint32_t scnt[kLdsSlots];
    __shared__ uint64_t s_nk[kHistThreads / kWave * kMaxK];
    __shared__ int s_nc[kHistThreads / kWave];
    __shared__ uint32_t s_new;   // keys this workgroup brought into the global table
    __shared__ uint32_t s_over;  // a key found no slot
    __shared__ uint32_t s_hll[GLOBAL ? kHllRegs : 1];  // keys that the global table turned away
    __shared__ unsigned long long s_special, s_nans;
    __shared__ uint32_t s_negzero;
    constexpr bool kInt = !std::is_floating_point<T>::value;
    using U = typename UnsignedOf<T>::type;
    __shared__ __attribute__((aligned(16))) uint32_t win[kInt ? kWindow * kCopies : 4];
    const U wbase = kInt ? (U)(ubits(x[0]) - kWindow / 2) : U(0);  // wraps in the type
    auto fill = [](void* p, int bytes, uint32_t v) {
        u32x4* q = reinterpret_cast<u32x4*>(p);
        for (int i = threadIdx.x; i < bytes / 16; i += kHistThreads) q[i] = u32x4{v, v, v, v};
    };
    if (kInt) fill(win, sizeof win, 0u);
    fill(skey, sizeof skey, ~0u);
    fill(scnt, sizeof scnt, 0u);
    static_assert(kHllRegs == kHistThreads && kHllRegs == kMergeThreads, "a register a thread");
    if (GLOBAL)
        s_hll[threadIdx.x] = 0;
    else if (blockIdx.x == 0)
        hll[threadIdx.x] = 0;  // k_hist_merge's
    if (threadIdx.x == 0) {
        s_new = s_over = s_negzero = 0;
        s_special = s_nans = 0;
    }
    __syncthreads();
    Small4 nan4;
    unsigned long long special = 0, nans = 0;
    bool negzero = false;
    // Probes for a slot: with few rows, whose keys all have one, the whole
    // partition; 24 let 5,500 random keys of 4 bytes and 3,500 of 8 find one (48:
    // 7,500 and 5,000, but twice the loop unrolled into every row's place: 20M
    // int16 rows of 60 values 28 us for 19); before the global table, which most
    // rows of a column with that many keys end up in anyway, 8.
    constexpr int probes = GLOBAL ? 8 : PER < 16 ? PS : 24;
    // Adds `add` rows of `key` to its partition; a key without a slot goes to
    // the global table, or ends the count.
    auto lds_add = [&](KT key, uint32_t add) {
        const uint64_t at = (uint64_t)lds_hash<(PER == 16 && !GLOBAL)>((uint64_t)key) * kHistParts;
        const uint32_t base = (uint32_t)(at >> 32) * PS;
        uint32_t h = (uint32_t)(((uint64_t)(uint32_t)at * PS) >> 32);
        for (int p = 0; p < probes; p++) {
            const uint32_t s = base + h;
            h = h + 1 < (uint32_t)PS ? h + 1 : 0;
            KT k = skey[s];
            if (k == kFree) k = atomicCAS(&skey[s], kFree, key);
            if (k == kFree || k == key) {
                atomicAdd(&scnt[s], add);
                return;
            }
        }
        if (GLOBAL)
            table.add((uint64_t)key, add, s_hll);
        else
            s_over = 1;
    };
    // Two keys per thread counted in registers (the first two distinct keys
    // the thread meets): on skewed columns most rows hit them and skip the
    // LDS atomics, whose same-address conflicts are the cost.
    KT rk0 = kFree, rk1 = kFree;
    uint32_t rc0 = 0, rc1 = 0;
    auto count = [&](T v) {
        if constexpr (std::is_floating_point<T>::value) {
            if (v != v) {
                nan4.insert(order_key(v));
                nans++;
                return;
            }
        }
        if constexpr (kInt) {
            const U off = (U)((U)ubits(v) - wbase);
            if (sizeof(U) == 1 || (uint64_t)off < (uint64_t)kWindow) {
                atomicAdd(&win[(uint32_t)off * kCopies + (threadIdx.x & (kCopies - 1))], 1u);
                return;
            }
        }
        const KT key = (KT)hist_key(v, negzero);
        if (key == kFree) {
            special++;
            return;
        }
        if (key == rk0) {
            rc0++;
        } else if (key == rk1) {
            rc1++;
        } else if (rk0 == kFree) {
            rk0 = key;
            rc0 = 1;
        } else if (rk1 == kFree) {
            rk1 = key;
            rc1 = 1;
        } else {
            lds_add(key, 1u);
        }
    };
    auto gave_up = [&] { return !GLOBAL && *(volatile uint32_t*)&s_over != 0; };
    constexpr int kPer = PER, kRows = kPer * kHistThreads;
    constexpr int V = 16 / sizeof(T);
    constexpr int Q = kRows / V / kHistThreads;  // 16-byte loads per thread and tile
    const size_t tiles = (n + kRows - 1) / kRows;
    const bool aligned = (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    for (size_t t = blockIdx.x; t < tiles; t += gridDim.x) {  // uniform per workgroup
        if (gave_up()) break;  // (each wave by itself: the count is dropped)
        const size_t base = t * kRows;
        if (aligned && base + kRows <= n) {
            const u32x4* s4 = reinterpret_cast<const u32x4*>(x + base);
            u32x4 w[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) w[q] = s4[threadIdx.x + kHistThreads * q];
#pragma unroll
            for (int q = 0; q < Q; q++) {
                if (Q >= 4 && q == Q / 2 && gave_up()) break;
                T v[V];
                __builtin_memcpy(v, &w[q], 16);
#pragma unroll
                for (int k = 0; k < V; k++) count(v[k]);
            }
        } else {
            const int cnt = (int)((n - base) < (size_t)kRows ? (n - base) : (size_t)kRows);
            T v[kPer];
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                const int i = threadIdx.x + k * kHistThreads;
                if (i < cnt) v[k] = x[base + i];
            }
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                if (k == kPer / 2 && gave_up()) break;
                if ((int)threadIdx.x + k * kHistThreads < cnt) count(v[k]);
            }
        }
    }
    if (rk0 != kFree) lds_add(rk0, rc0);
    if (rk1 != kFree) lds_add(rk1, rc1);
    __syncthreads();
    if constexpr (kInt) {
        // a thread sums one offset's copies and adds its key to the table
        static_assert(kWindow == kHistThreads, "one offset a thread");
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < kCopies; k++) c += win[threadIdx.x * kCopies + ((threadIdx.x + k) & (kCopies - 1))];
        if (c) {
            const KT key = (KT)(U)(wbase + (U)threadIdx.x);
            if (key == kFree)
                special += c;
            else
                lds_add(key, c);
        }
        __syncthreads();
    }
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    if (GLOBAL) {
        for (int s = threadIdx.x; s < kLdsSlots; s += kHistThreads)
            if (skey[s] != kFree) table.add((uint64_t)skey[s], scnt[s], s_hll);
        const uint32_t fresh = wave_sum(table.fresh);
        if (lane == 0 && fresh) atomicAdd(&s_new, fresh);
        if (__syncthreads_or(table.full)) {
            if (threadIdx.x == 0) atomicOr(&table.ctl->overflow, kTooSmall);
            hll_merge(table.hll, threadIdx.x, s_hll[threadIdx.x]);
        }
        if (threadIdx.x == 0 && s_new) atomicAdd(&table.ctl->distinct, (unsigned long long)s_new);
    } else {
        // partitions' used slots, where each begins, then the entries
        __shared__ uint32_t s_off[kHistParts + 1];
        static_assert(kHistParts == kWave && PS % kWave == 0, "a partition a lane, whole waves of slots");
        constexpr int C = PS / kWave;  // slots a lane
        for (int p = wid; p < kHistParts; p += kHistThreads / kWave) {
            uint32_t used = 0;
#pragma unroll
            for (int q = 0; q < C; q++) used += __popcll(__ballot(scnt[p * PS + lane + q * kWave] != 0));
            if (lane == 0) s_off[p] = used;
        }
        __syncthreads();
        if (wid == 0) {
            const uint32_t used = s_off[lane], upto = wave_inclusive_scan(used);
            s_off[lane] = upto - used;
            if (lane == kWave - 1) s_off[kHistParts] = upto;
        }
        __syncthreads();
        HistEntry<KT>* mine = segs + (size_t)blockIdx.x * seg_slots<T, PER>();
        for (int p = wid; p < kHistParts; p += kHistThreads / kWave) {
            uint32_t at = s_off[p];
#pragma unroll
            for (int q = 0; q < C; q++) {
                const KT k = skey[p * PS + lane + q * kWave];
                const uint32_t c = scnt[p * PS + lane + q * kWave];
                const uint64_t has = __ballot(c != 0);
                if (c) {
                    HistEntry<KT>* e = mine + at + __popcll(has & ((1ull << lane) - 1));
                    st_agent(&e->key, k);
                    st_agent(&e->count, c);
                }
                at += __popcll(has);
            }
        }
        for (int p = threadIdx.x; p <= kHistParts; p += kHistThreads) st_agent(&off[(size_t)p * gridDim.x + blockIdx.x], s_off[p]);
    }
    const bool nz = __ballot(negzero) != 0;
    special = wave_sum(special);
    nans = wave_sum(nans);
    if (lane == 0) {
        if (nz) atomicOr(&s_negzero, 1u);
        if (special) atomicAdd(&s_special, special);
        if (nans) atomicAdd(&s_nans, nans);
    }
    HistInfo* me = info + blockIdx.x;
    __shared__ uint64_t nan_keys[kMaxK];
    __shared__ uint32_t nan_n;
    if (threadIdx.x == 0) nan_n = 0;
    __syncthreads();
    if constexpr (std::is_floating_point<T>::value) block_small4<kHistThreads>(nan4, s_nk, s_nc, nan_keys, &nan_n);
    __syncthreads();
    if (threadIdx.x == 0) {
        st_agent(&me->special, s_special);
        st_agent(&me->nans, s_nans);
        st_agent(&me->negzero, s_negzero);
        st_agent(&me->overflow, s_over);
        st_agent(&me->nan_n, nan_n);
        for (uint32_t r = 0; r < nan_n; r++) st_agent(&me->nan_keys[r], nan_keys[r]);
    }
    if constexpr (!GLOBAL) {
        __shared__ bool last;
        if (!tail.tickets || !last_of_grid(tail.tickets, &last)) return;
        // every workgroup's entries: how many, and where they begin
        __shared__ uint32_t first[kHistThreads + 1];
        __shared__ uint32_t red[kHistThreads / kWave];
        __shared__ HistCtl ctl;
        __shared__ uint32_t s_distinct, s_most;
        __shared__ Cand sc[kHistThreads / kWave * kMaxK];
        __shared__ Cand best[kMaxK];
        const uint32_t blocks = gridDim.x;  // <= kHistThreads
        const uint32_t have = threadIdx.x < blocks ? ld_agent(&off[(size_t)kHistParts * blocks + threadIdx.x]) : 0u;
        if (threadIdx.x == 0) {
            ctl = HistCtl{};
            s_distinct = s_most = 0;
        }
        fill(skey, sizeof skey, ~0u);
        fill(scnt, sizeof scnt, 0u);
        uint32_t total;
        first[threadIdx.x] = block_exclusive_scan<uint32_t, kHistThreads>(have, &total, red);
        const uint32_t most = wave_max(have);
        if (lane == 0) atomicMax(&s_most, most);
        __syncthreads();
        fold_info<kHistThreads>(info, blocks, &ctl);
        HistResult* out = reinterpret_cast<HistResult*>(tail.host.dst);
        const bool few = (total <= (uint32_t)kLdsSlots || (total <= kTailEntries && s_most <= kTailKeys)) && n < (1ull << 32);
        constexpr int F = 4;  // entries in flight a thread
        for (uint32_t e0 = threadIdx.x; few && e0 < total; e0 += F * kHistThreads) {
            KT key[F];
            uint32_t cnt[F];
#pragma unroll
            for (int f = 0; f < F; f++) {
                const uint32_t e = e0 + f * kHistThreads;
                cnt[f] = 0;
                if (e < total) {
                    const uint32_t w = segment_of(first, blocks, e);
                    const HistEntry<KT>* en = segs + (size_t)w * seg_slots<T, PER>() + (e - first[w]);
                    key[f] = ld_agent(&en->key);
                    cnt[f] = ld_agent(&en->count);
                }
            }
#pragma unroll
            for (int f = 0; f < F; f++) {
                if (!cnt[f]) continue;
                const uint32_t h = lds_hash<false>((uint64_t)key[f]), step = 6 * (h & 255) + 1;  // as k_hist_small's
                uint32_t s = (uint32_t)(((uint64_t)h * kLdsSlots) >> 32);
                int left = 32;
                for (; left > 0; left--) {
                    KT k = skey[s];
                    if (k == kFree) k = atomicCAS(&skey[s], kFree, key[f]);
                    if (k == kFree || k == key[f]) {
                        atomicAdd(&scnt[s], cnt[f]);
                        break;
                    }
                    s = s + step < (uint32_t)kLdsSlots ? s + step : s + step - kLdsSlots;
                }
                if (left == 0) atomicOr(&ctl.overflow, kNeedMerge);
            }
            if (*(volatile uint32_t*)&ctl.overflow) break;  // (each wave by itself: the sums are dropped)
        }
        if (!few && threadIdx.x == 0) atomicOr(&ctl.overflow, kNeedMerge);
        __syncthreads();
        if (ctl.overflow) {  // uniform
            if (threadIdx.x == 0) out->ctl = ctl;
        } else {
            Cand top[kMaxK];
            take_table<T, kLdsSlots, kHistThreads>(skey, scnt, top, tail.K, &s_distinct);
            block_best<T, kHistThreads>(top, tail.K, sc, best);  // its barriers complete s_distinct
            if (threadIdx.x == 0) {
                ctl.distinct = s_distinct;
                finish_topk<T>(best, tail.K, ctl, info, blocks, out);
            }
        }
        host_out_done(tail.host);
    }
}

// The best K over all workgroups, from the K each has in best: partials by
// tickets, and the last workgroup takes the best of them into best.  Whether
// this is that workgroup.
template <typename T, int NT>
__device__ __forceinline__ bool best_of_grid(Cand* top, int K, Cand* sc, Cand* best, Cand* partials, uint32_t* tickets,
                                             bool* last) {
    if (threadIdx.x < K) {
        st_agent(reinterpret_cast<uint64_t*>(&partials[blockIdx.x * K + threadIdx.x].count),
                 (uint64_t)best[threadIdx.x].count);
        st_agent(&partials[blockIdx.x * K + threadIdx.x].key, best[threadIdx.x].key);
    }
    if (!last_of_grid(tickets, last)) return false;
#pragma unroll
    for (int i = 0; i < kMaxK; i++) top[i] = Cand{0, 0};
    for (uint32_t i = threadIdx.x; i < gridDim.x * (uint32_t)K; i += NT) {
        Cand c;
        c.count = __hip_atomic_load(&partials[i].count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        c.key = __hip_atomic_load(&partials[i].key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        push<T>(top, K, c);
    }
    block_best<T, NT>(top, K, sc, best);
    return true;
}

// One workgroup per partition: the counting workgroups' entries added up in an
// LDS table (an entry a thread, several in flight), then the best K.  Replaces
// a global table that every workgroup flushed its keys into with device-scope
// atomics, the launch that cleared it and the one that searched its 64K slots:
// 5M rows of long-tailed volumes 2 + 72 + 11 us, now 20 + 22; 16M rows, whose
// table overflowed and was counted again, 2.5 ms, now 38 + 32 us.
template <typename T>
__global__ __launch_bounds__(kMergeThreads) void k_hist_merge(const HistEntry<HistKey<T>>* __restrict__ segs,
                                                              const uint32_t* __restrict__ off,
                                                              const HistInfo* __restrict__ info, uint32_t blocks,
                                                              uint32_t slots /* entries a workgroup */, int K,
                                                              Cand* partials, uint32_t* part_ctl, uint32_t* hll,
                                                              uint32_t* tickets, HostOut host) {
    using KT = HistKey<T>;
    constexpr KT kFree = (KT)~(KT)0;
    constexpr int W = kMergeThreads / kWave;
    __shared__ __attribute__((aligned(16))) KT skey[kMergeSlots];
    __shared__ unsigned long long scnt[kMergeSlots];
    __shared__ Cand sc[W * kMaxK];
    __shared__ Cand best[kMaxK];
    __shared__ HistCtl ctl;
    __shared__ uint32_t s_distinct, s_over;
    __shared__ uint32_t s_hll[kHllRegs];  // keys turned away
    __shared__ uint32_t first[kMergeThreads];  // of the partition's entries, where each workgroup's begin
    __shared__ uint32_t begin[kMergeThreads];  // and where they are among the workgroup's
    __shared__ uint32_t red[W];
    __shared__ bool last;
    const uint32_t* row = off + (size_t)blockIdx.x * blocks;  // blocks <= kMergeThreads
    // a counting workgroup's table was too small (the same in every workgroup
    // here): nothing to add up, and no tickets are taken
    if (__syncthreads_or(threadIdx.x < blocks && info[threadIdx.x].overflow)) {
        if (blockIdx.x != 0) return;
        if (threadIdx.x == 0) {
            ctl = HistCtl{};
            ctl.overflow = kTooSmall;
            reinterpret_cast<HistResult*>(host.dst)->ctl = ctl;
        }
        host_out_done(host);
        return;
    }
    const uint32_t at = threadIdx.x < blocks ? row[threadIdx.x] : 0u;
    const uint32_t mine = threadIdx.x < blocks ? row[blocks + threadIdx.x] - at : 0u;
    for (int i = threadIdx.x; i < kMergeSlots; i += kMergeThreads) {
        skey[i] = kFree;
        scnt[i] = 0;
    }
    s_hll[threadIdx.x] = 0;
    if (threadIdx.x == 0) {
        s_distinct = s_over = 0;
        ctl = HistCtl{};
    }
    uint32_t total;
    first[threadIdx.x] = block_exclusive_scan<uint32_t, kMergeThreads>(mine, &total, red);
    begin[threadIdx.x] = at;
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    constexpr int F = 4;  // entries in flight a thread
    for (uint32_t e0 = threadIdx.x; e0 < total; e0 += F * kMergeThreads) {
        HistEntry<KT> en[F];
#pragma unroll
        for (int f = 0; f < F; f++) {
            const uint32_t e = e0 + f * kMergeThreads;
            en[f].count = 0;
            if (e < total) {
                const uint32_t w = segment_of(first, blocks, e);
                en[f] = segs[(size_t)w * slots + begin[w] + (e - first[w])];
            }
        }
#pragma unroll
        for (int f = 0; f < F; f++) {
            if (!en[f].count) continue;
            const uint64_t h = hmix((uint64_t)en[f].key);
            const uint32_t step = (uint32_t)(h >> 32) | 1;  // odd: visits every slot
            uint32_t s = (uint32_t)h & (kMergeSlots - 1);
            // past 85% full the count runs again with the global table, and the
            // keys left over only go into the estimate that sizes it
            int left = *(volatile uint32_t*)&s_over ? 0 : 64;
            for (; left > 0; left--) {
                KT have = skey[s];
                if (have == kFree) have = atomicCAS(&skey[s], kFree, en[f].key);
                if (have == kFree || have == en[f].key) {
                    atomicAdd(&scnt[s], (unsigned long long)en[f].count);
                    break;
                }
                s = (s + step) & (kMergeSlots - 1);
            }
            if (left == 0) {
                s_over = 1;
                hll_note((uint64_t)en[f].key, s_hll);
            }
        }
    }
    __syncthreads();
    if (s_over) hll_merge(hll, threadIdx.x, s_hll[threadIdx.x]);
    Cand top[kMaxK];
    take_table<T, kMergeSlots, kMergeThreads>(skey, scnt, top, K, &s_distinct);
    block_best<T, kMergeThreads>(top, K, sc, best);  // its barriers complete s_distinct
    if (threadIdx.x == 0) {
        st_agent(&part_ctl[2 * blockIdx.x], s_distinct);
        st_agent(&part_ctl[2 * blockIdx.x + 1], s_over);
    }
    if (!best_of_grid<T, kMergeThreads>(top, K, sc, best, partials, tickets, &last)) return;
    for (uint32_t i = threadIdx.x; i < gridDim.x; i += kMergeThreads) {
        atomicAdd(&ctl.distinct, (unsigned long long)ld_agent(&part_ctl[2 * i]));
        if (ld_agent(&part_ctl[2 * i + 1])) atomicOr(&ctl.overflow, kTooSmall);
    }
    fold_info<kMergeThreads>(info, blocks, &ctl);
    __syncthreads();
    if (threadIdx.x == 0) finish_topk<T>(best, K, ctl, info, blocks, reinterpret_cast<HistResult*>(host.dst));
    host_out_done(host);
}

// The best K of the global table.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_hist_topk(GlobalTable table, int K, Cand* partials, uint32_t* tickets,
                                                      const HistInfo* info, uint32_t blocks, HostOut host) {
    __shared__ Cand sc[kBlock / kWave * kMaxK];
    __shared__ Cand best[kMaxK];
    __shared__ HistCtl ctl;
    __shared__ bool last;
    Cand top[kMaxK];
#pragma unroll
    for (int i = 0; i < kMaxK; i++) top[i] = Cand{0, 0};
    const size_t stride = (size_t)gridDim.x * kBlock;
    for (size_t s = (size_t)blockIdx.x * kBlock + threadIdx.x; s <= table.mask; s += stride) {
        const uint64_t k = table.keys[s];
        if (k != kEmpty) push<T>(top, K, Cand{table.counts[s], k});
    }
    block_best<T>(top, K, sc, best);
    if (!best_of_grid<T, kBlock>(top, K, sc, best, partials, tickets, &last)) return;
    if (threadIdx.x == 0) ctl = *table.ctl;
    __syncthreads();
    fold_info<kBlock>(info, blocks, &ctl);
    __syncthreads();
    if (threadIdx.x == 0) finish_topk<T>(best, K, ctl, info, blocks, reinterpret_cast<HistResult*>(host.dst));
    host_out_done(host);
}

// Columns of a few thousand rows (the planner's samples): one workgroup
// counts every row in an LDS table that can hold them all distinct, takes the
// best K and hands them to the host: one launch for four (table fill, count,
// top-K, read-back), and no device-scope atomics (10,000 distinct int32 rows by
// HIP events: 7 + 90 + 24 us in three launches, now 34).  The limits keep the table at
// most 2/3 full (8-byte keys 5/6, which is what LDS allows a 10,000-row
// sample).  The probes' step is the key's own (6 k + 1, which has no factor in
// common with the 2^a 3^b slots, so that it visits all of them); a key without a
// slot after kSmallProbes of them, which takes keys made for it, has the
// column counted by the other kernels.
constexpr int kSmallProbes = 512;
template <typename T> constexpr int small_slots() { return sizeof(T) == 8 ? 12288 : 18432; }
template <typename T> constexpr size_t small_rows() { return sizeof(T) == 8 ? 10240 : 12288; }

template <typename T>
__global__ __launch_bounds__(kHistThreads) void k_hist_small(const T* __restrict__ x, uint32_t n, int K, HostOut host) {
    using KT = HistKey<T>;
    constexpr KT kFree = (KT)~(KT)0;  // an empty slot; rows of that bit pattern are counted on the side
    constexpr int S = small_slots<T>(), W = kHistThreads / kWave;
    static_assert(S == 12288 || S == 18432, "no prime factors but 2 and 3; steps are shorter");
    __shared__ KT skey[S];
    __shared__ uint32_t scnt[S];
    __shared__ Cand sc[W * kMaxK];
    __shared__ Cand best[kMaxK];
    __shared__ uint64_t s_nk[W * kMaxK], nan_keys[kMaxK];
    __shared__ int s_nc[W];
    __shared__ uint32_t nan_n, s_distinct, s_special, s_nans, s_negzero, s_over;
    for (int i = threadIdx.x; i < S; i += kHistThreads) {
        skey[i] = kFree;
        scnt[i] = 0;
    }
    if (threadIdx.x == 0) s_distinct = s_special = s_nans = s_negzero = s_over = nan_n = 0;
    __syncthreads();
    bool negzero = false;
    uint32_t special = 0, nans = 0, distinct = 0;
    Small4 nan4;
    constexpr int R = (int)((small_rows<T>() + kHistThreads - 1) / kHistThreads);
    T v[R];
#pragma unroll
    for (int r = 0; r < R; r++) {  // every load in flight at once
        const uint32_t i = threadIdx.x + r * kHistThreads;
        if (i < n) v[r] = x[i];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (threadIdx.x + r * kHistThreads >= n) break;
        if constexpr (std::is_floating_point<T>::value) {
            if (v[r] != v[r]) {
                nan4.insert(order_key(v[r]));
                nans++;
                continue;
            }
        }
        const KT key = (KT)hist_key(v[r], negzero);
        if (key == kFree) {
            special++;
            continue;
        }
        const uint32_t h = lds_hash<false>((uint64_t)key), step = 6 * (h & 255) + 1;
        uint32_t s = (uint32_t)(((uint64_t)h * S) >> 32);
        int left = kSmallProbes;
        for (; left > 0; left--) {
            KT k = skey[s];
            if (k == kFree) k = atomicCAS(&skey[s], kFree, key);
            if (k == kFree || k == key) {
                atomicAdd(&scnt[s], 1u);
                break;
            }
            s = s + step < (uint32_t)S ? s + step : s + step - S;
        }
        if (left == 0) s_over = 1;
    }
    __syncthreads();
    Cand top[kMaxK];
#pragma unroll
    for (int i = 0; i < kMaxK; i++) top[i] = Cand{0, 0};
    for (int s = threadIdx.x; s < S; s += kHistThreads) {
        const uint32_t c = scnt[s];
        if (c) {
            distinct++;
            push<T>(top, K, Cand{c, (uint64_t)skey[s]});
        }
    }
    distinct = wave_sum(distinct);
    special = wave_sum(special);
    nans = wave_sum(nans);
    const bool nz = __ballot(negzero) != 0;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        atomicAdd(&s_distinct, distinct);
        if (special) atomicAdd(&s_special, special);
        if (nans) atomicAdd(&s_nans, nans);
        if (nz) atomicOr(&s_negzero, 1u);
    }
    if constexpr (std::is_floating_point<T>::value)
        block_small4<kHistThreads>(nan4, s_nk, s_nc, nan_keys, &nan_n);
    block_best<T, kHistThreads>(top, K, sc, best);
    if (threadIdx.x == 0) {
        Cand b[kMaxK];
#pragma unroll
        for (int i = 0; i < kMaxK; i++) b[i] = i < K ? best[i] : Cand{0, 0};
        // rows of the free slot's bit pattern: all ones in the type
        if (s_special) push<T>(b, K, Cand{s_special, (uint64_t)kFree});
        for (uint32_t r = 0; r < nan_n; r++)  // every NaN row is a bin of count 1
            push<T>(b, K, Cand{1ull, ubits(from_order_key<T>(nan_keys[r]))});
        HistResult* out = reinterpret_cast<HistResult*>(host.dst);
        out->ctl = HistCtl{s_distinct, s_special, s_nans, s_over ? kTooSmall : 0u, s_negzero};
#pragma unroll
        for (int i = 0; i < kMaxK; i++) out->top[i] = b[i];
    }
    host_out_done(host);
}

// The histogram's global table emptied (keys ~0, counts 0) and its control
// block cleared, in one launch.
__global__ __launch_bounds__(kBlock) void k_hist_init(GlobalTable table) {
    const size_t stride = (size_t)gridDim.x * kBlock;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i <= table.mask; i += stride) {
        table.keys[i] = kEmpty;
        table.counts[i] = 0;
    }
    if (blockIdx.x != 0) return;
    for (int i = threadIdx.x; i < kHllRegs; i += kBlock) table.hll[i] = 0;
    if (threadIdx.x == 0) *table.ctl = HistCtl{};
}

uint64_t pow2_at_least(uint64_t v) {
    uint64_t p = 1;
    while (p < v) p <<= 1;
    return p;
}

}  // namespace

void topk_most_frequent(Ctx* c, int dtype, const void* x, size_t n, int K, uint64_t* keys_bits_host,
                        int* n_distinct_host) {
    if (K < 1 || K > kMaxK) fail(DDJ_EINVAL, "top-K supports K in 1..4");
    if (n == 0) fail(DDJ_EINVAL, "top-K of an empty array");
    dispatch_native(dtype, [&](auto tag) {
        using T = decltype(tag);
        // fewer than K distinct values: the last real key repeats
        auto take = [&](const HistResult& f) {
            const int nd = (int)(f.ctl.distinct + (f.ctl.special ? 1 : 0) + f.ctl.nans);
            if (n_distinct_host) *n_distinct_host = nd;
            const int real = std::min(K, nd);
            for (int i = 0; i < K; i++) {
                uint64_t kb = f.top[i < real ? i : real - 1].key;
                if (std::is_floating_point<T>::value && kb == 0 && f.ctl.negzero)
                    kb = (sizeof(T) == 8) ? (1ull << 63) : (1ull << 31);
                keys_bits_host[i] = kb;
            }
        };
        HistResult found;
        if (n <= small_rows<T>()) {
            const HostOut ho = host_out(c);
            {
                KernelTimer kt_(c, "k_hist_small");
                hipLaunchKernelGGL(k_hist_small<T>, dim3(1), dim3(kHistThreads), 0, c->stream, static_cast<const T*>(x),
                                   (uint32_t)n, K, ho);
            }
            HIPC(hipGetLastError());
            memcpy(&found, wait_host_out(c, ho), sizeof found);
            if (!found.ctl.overflow) return take(found);
        }
        using Entry = HistEntry<HistKey<T>>;
        auto xs = static_cast<const T*>(x);
        // The keys that a full table (or k_hist_merge's) holds and has turned away.
        auto keys_seen = [&](const HistCtl& ctl, const DevBuf& hll) {
            uint32_t regs[kHllRegs];
            d2h(c, regs, hll.get(), sizeof regs);
            return ctl.distinct + (uint64_t)hll_estimate(regs);
        };
        uint64_t seen = 0;
        // One count in tiles of PER rows a thread by at most max_g workgroups, and
        // the merge: whether the tables held the keys.
        auto counted = [&](auto per, size_t max_g) {
            constexpr int PER = decltype(per)::value;
            const size_t rows = (size_t)PER * kHistThreads, g = std::min((n + rows - 1) / rows, max_g);
            // in four sizes, so that columns of every length share their blocks
            size_t room = 16;
            while (room < g) room *= 4;
            DevBuf info(c, sizeof(HistInfo) * g), off(c, 4 * (kHistParts + 1) * g), hll(c, 4 * kHllRegs),
                segs(c, sizeof(Entry) * seg_slots<T, PER>() * room);
            // up to 1M rows of 4 bytes the last workgroup merges (50 codes: one launch
            // of 22 us for two of 9 + 16); more workgroups have too many entries for
            // one (64M rows 70 us, two launches 53 + 17)
            HistTail tail;
            if (g <= (PER < 16 ? 128 : 64)) tail = HistTail{c->control->tickets, K, host_out(c)};
            {
                KernelTimer kt_(c, "k_hist_count");
                hipLaunchKernelGGL((k_hist_count<T, PER, false>), dim3((unsigned)g), dim3(kHistThreads), 0, c->stream, xs,
                                   n, GlobalTable{}, segs.get<Entry>(), off.get<uint32_t>(), info.get<HistInfo>(),
                                   hll.get<uint32_t>(), tail);
            }
            HIPC(hipGetLastError());
            if (tail.tickets) memcpy(&found, wait_host_out(c, tail.host), sizeof found);
            if (!tail.tickets || found.ctl.overflow == kNeedMerge) {
                DevBuf partials(c, sizeof(Cand) * K * kHistParts), part_ctl(c, 8 * kHistParts);
                const HostOut ho = host_out(c);
                {
                    KernelTimer kt_(c, "k_hist_merge");
                    hipLaunchKernelGGL(k_hist_merge<T>, dim3(kHistParts), dim3(kMergeThreads), 0, c->stream,
                                       segs.get<Entry>(), off.get<uint32_t>(), info.get<HistInfo>(), (uint32_t)g,
                                       (uint32_t)seg_slots<T, PER>(), K, partials.get<Cand>(), part_ctl.get<uint32_t>(),
                                       hll.get<uint32_t>(), c->control->tickets, ho);
                }
                HIPC(hipGetLastError());
                memcpy(&found, wait_host_out(c, ho), sizeof found);
            }
            if (found.ctl.overflow && found.ctl.distinct) seen = keys_seen(found.ctl, hll);  // the merge's tables filled
            return !found.ctl.overflow;
        };
        using Few = std::integral_constant<int, few_rows<T>()>;
        const size_t few = (size_t)Few::value * kHistThreads, cus = std::min<size_t>(c->cu_count, kMergeThreads);
        if (n <= few * cus) {
            if (counted(Few{}, cus)) return take(found);
        } else {
            if (counted(std::integral_constant<int, 16>{}, cus)) return take(found);
            // the merge takes the entries of up to kMergeThreads workgroups (4M int32
            // rows of 16,000 keys 244 us, 416 through the global table)
            if (Few::value < 16 && n <= few * kMergeThreads && counted(Few{}, kMergeThreads)) return take(found);
        }
        const size_t g = std::min((n + 16 * kHistThreads - 1) / (16 * kHistThreads), cus);
        DevBuf info(c, sizeof(HistInfo) * g);
        // more distinct keys than the LDS tables hold
        const uint64_t all_distinct = pow2_at_least(2 * (uint64_t)n + 2);
        uint64_t cap = std::min<uint64_t>(std::max<uint64_t>(1024, all_distinct),
                                          std::max<uint64_t>(1u << 16, pow2_at_least(2 * seen + 2)));
        for (int attempt = 0; attempt < 3; attempt++) {
            DevBuf keys(c, 8 * cap), counts(c, 8 * cap), ctl(c, sizeof(HistCtl)), hll(c, 4 * kHllRegs);
            const GlobalTable table{keys.get<unsigned long long>(), counts.get<unsigned long long>(), cap - 1,
                                    ctl.get<HistCtl>(), hll.get<uint32_t>()};
            kernel_bytes(c, "k_hist_init", 16.0 * (double)cap);
            const unsigned fg = (unsigned)std::min<uint64_t>((cap + kBlock - 1) / kBlock, (uint64_t)c->cu_count * 16);
            {
                KernelTimer kt_(c, "k_hist_init");
                hipLaunchKernelGGL(k_hist_init, dim3(fg), dim3(kBlock), 0, c->stream, table);
            }
            {
                KernelTimer kt_(c, "k_hist_count");
                hipLaunchKernelGGL((k_hist_count<T, 16, true>), dim3((unsigned)g), dim3(kHistThreads), 0, c->stream, xs, n,
                                   table, nullptr, nullptr, info.get<HistInfo>(), nullptr, HistTail{});
            }
            HIPC(hipGetLastError());
            // the top-K runs before the table's state is known, so that one
            // result brings both (it is dropped if the table filled)
            const unsigned tg = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((cap + kBlock - 1) / kBlock, 128));
            DevBuf partials(c, sizeof(Cand) * K * tg);
            const HostOut ho = host_out(c);
            {
                KernelTimer kt_(c, "k_hist_topk");
                hipLaunchKernelGGL(k_hist_topk<T>, dim3(tg), dim3(kBlock), 0, c->stream, table, K, partials.get<Cand>(),
                                   c->control->tickets, info.get<HistInfo>(), (uint32_t)g, ho);
            }
            HIPC(hipGetLastError());
            memcpy(&found, wait_host_out(c, ho), sizeof found);
            const HistCtl& h = found.ctl;
            if (h.overflow || h.distinct * 10 > cap * 7) {
                if (attempt == 2 || cap >= all_distinct) fail(DDJ_ENOMEM, "histogram table overflow");
                seen = h.overflow ? keys_seen(h, hll) : h.distinct;
                const uint64_t next = attempt == 0 ? std::min(all_distinct, pow2_at_least(2 * seen + 2)) : all_distinct;
                cap = std::max(next, std::min(all_distinct, 2 * cap));  // always grows
                continue;
            }
            return take(found);
        }
    });
}

}  // namespace ddj
