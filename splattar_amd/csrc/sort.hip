// Stable LSD radix sort of (key, u32 payload) pairs, 64- or 32-bit keys.
//
// Semantics of crates/gs-wgpu/src/sort.rs:17-327 (stable, element count read
// from a device buffer so it never round-trips to the host) but one 64-bit
// (tile || depth) key replaces the reference's two stable 32-bit sorts
// (binning.rs:5-8, 209-227). Each digit pass is reduce-then-scan over
// partitions of 1024 to 4096 keys, three kernels:
//   * upsweep: per-partition digit counts (per-wave LDS histograms), written
//     digit-major;
//   * scan: one block per digit turns its row of partition counts into
//     exclusive offsets and writes the digit's total;
//   * downsweep: ranks the partition's keys stably with wave64 ballots (8
//     ballots per key at 8-bit digits), permutes them through LDS into digit
//     order and writes each digit run at global start (exclusive scan of the
//     totals) + partition offset.
// Capacities up to 2^17 have at most 128 partitions: the downsweep sums the
// rows itself, without the scan. Up to 4096 pairs one workgroup does all
// passes. Latency bounds a pass up to about 1M keys (20k keys 16.8 -> 9.3 us,
// 250k 18.2 -> 14.3 against 4096 keys a partition and the scan always, three
// to four launches), HBM beyond (16M: 114 -> 109 us with one LDS buffer for
// keys and payloads in turn, 12 B a pair read, 8 written).
// No partition waits for another (a decoupled look-back walked ~6 rounds of
// 16 predecessor statuses per partition here and read ~1.8x the keys' bytes).
// Digit width is 4 or 8 bits (9 where the caller allows it); only the bit range
// [begin_bit, end_bit) is sorted, so a key whose high bits are known constant
// costs fewer passes. A count above the capacity sorts the first `capacity`
// pairs.
//
// Per pass HBM traffic: read (2 sizeof(K) + 4) B and write (sizeof(K) + 4) B
// per pair, plus 8 B per partition and digit of offsets.

#include "gs_internal.h"

namespace gs {

namespace {

constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / 64;
constexpr int kMaxItems = 8;                         // keys per thread at most
constexpr int kMaxPasses = 16;
constexpr uint32_t kFusedCap = 1u << 17;             // capacities whose downsweep sums the counts itself

// Keys per thread at n keys. A partition ranks its keys 64 a wave at a time,
// one round after another, so few keys are split over more workgroups; many
// keys take the longest partitions, whose digit runs are the longest. Measured
// with 2 / 4 / 8 (us a pass, 32-bit keys): 250k 15.1 / 16.8 / 17.7, 500k 17.9 /
// 18.0 / 19.0, 700k 19.6 / 18.2 / 19.6, 1M 22.5 / 19.7 / 20.2, 2M 36 / 26.5 /
// 25.5, 16M 212 / 141 / 109.
__host__ __device__ constexpr uint32_t sort_items(uint32_t n) {
    return n <= 1u << 19 ? 2u : n <= 1u << 20 ? 4u : 8u;
}
__host__ __device__ constexpr uint32_t sort_parts(uint32_t n) {
    const uint32_t part = kSortThreads * sort_items(n);
    return n / part + (n % part != 0u);
}
// The most partitions that any count up to the capacity has, a multiple of 4
// (rows of counts are read 16 B at a time).
uint32_t most_parts(uint32_t cap) {
    uint32_t m = sort_parts(cap);
    for (uint32_t c : {1u << 19, 1u << 20})
        if (c < cap) m = std::max(m, sort_parts(c));
    return (std::max(m, 1u) + 3u) & ~3u;
}

struct SortScratch {
    uint32_t hist[kMaxPasses * 256];  // per pass: digit totals
    // followed by uint32_t offsets[digits][parts] (digit-major partition counts,
    // then exclusive offsets)
};

__device__ __forceinline__ uint32_t* part_offsets(SortScratch* sc) {
    return reinterpret_cast<uint32_t*>(sc + 1);
}

// Wave-level match of the lanes whose digit d (RB bits) equals this lane's,
// among the lanes with ok set.
template <int RB>
__device__ __forceinline__ uint64_t digit_match(uint32_t d, bool ok) {
    uint64_t match = __ballot(ok);
#pragma unroll
    for (int b = 0; b < RB; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bal = __ballot(bit);
        match &= bit ? bal : ~bal;
    }
    return match;
}

// Exclusive scan over R <= 256 values held one per thread (threads >= R hold
// 0); every thread gets its own exclusive prefix.
template <uint32_t R>
__device__ __forceinline__ uint32_t block_exclusive_scan_digits(uint32_t v, uint32_t* s_tmp) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t incl = v;
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t t = __shfl_up(incl, o);
        if (lane >= o) incl += t;
    }
    if (lane == 63) s_tmp[wave] = incl;
    __syncthreads();
    uint32_t add = 0;
    for (int w = 0; w < wave; ++w) add += s_tmp[w];
    __syncthreads();
    return add + incl - v;
}

// Keys that the sort leaves out (with `drop`, in the first pass): items
// without entries, marked by the projection.
template <typename K>
__device__ __forceinline__ bool dropped(K key, bool drop) {
    return drop && key == (K)kDropKey;
}

template <typename K, int RB, int ITEMS>
__device__ __forceinline__ void upsweep_part(const K* __restrict__ kin, uint32_t n, uint32_t base, uint32_t shift,
                                             bool drop, uint32_t (&s_h)[kSortWaves][1 << RB]) {
    constexpr uint32_t R = 1u << RB;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    K key[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t idx = base + (uint32_t)r * kSortThreads + (uint32_t)tid;
        key[r] = idx < n ? kin[idx] : (K)0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t idx = base + (uint32_t)r * kSortThreads + (uint32_t)tid;
        const bool ok = idx < n && !dropped(key[r], drop);
        const uint32_t d = (uint32_t)(key[r] >> shift) & (R - 1u);
        const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
        const uint64_t live = __ballot(ok);
        if (__ballot(ok && d != d0) == 0ull) {
            if (lane == 0 && live != 0ull) atomicAdd(&s_h[wave][d0], (uint32_t)__popcll(live));
        } else if (ok) {
            atomicAdd(&s_h[wave][d], 1u);
        }
    }
}

// Partition `part`'s digit counts of the pass at `shift`: per-wave LDS
// histograms with plain atomics (a round whose live lanes share one digit
// adds its lane count once), summed per digit at the end.
template <typename K, int RB>
__global__ __launch_bounds__(kSortThreads) void upsweep_kernel(const K* __restrict__ kin,
                                                               const uint32_t* __restrict__ count,
                                                               uint32_t cap, uint32_t shift, uint32_t stride,
                                                               bool drop,
                                                               SortScratch* __restrict__ sc) {
    constexpr uint32_t R = 1u << RB;
    __shared__ uint32_t s_h[kSortWaves][R];
    const int tid = threadIdx.x;
    const uint32_t n = min(*count, cap);
    const uint32_t items = sort_items(n), parts = sort_parts(n);
    for (uint32_t part = blockIdx.x; part < parts; part += gridDim.x) {
        const uint32_t base = part * kSortThreads * items;
        for (uint32_t k = tid; k < kSortWaves * R; k += kSortThreads) (&s_h[0][0])[k] = 0u;
        if (items == 2) upsweep_part<K, RB, 2>(kin, n, base, shift, drop, s_h);
        else if (items == 4) upsweep_part<K, RB, 4>(kin, n, base, shift, drop, s_h);
        else upsweep_part<K, RB, 8>(kin, n, base, shift, drop, s_h);
        __syncthreads();
        uint32_t* off = part_offsets(sc);
        for (uint32_t k = tid; k < R; k += kSortThreads) {
            uint32_t c = 0;
#pragma unroll
            for (int w = 0; w < kSortWaves; ++w) c += s_h[w][k];
            off[(size_t)k * stride + part] = c;
        }
        __syncthreads();  // s_h is cleared for the next partition
    }
}

// One block per digit: row of partition counts -> exclusive offsets; the
// digit's total goes to hist[pass][digit].
constexpr int kScanPer = 8;
__global__ __launch_bounds__(256) void part_scan_kernel(const uint32_t* __restrict__ count, uint32_t cap,
                                                        uint32_t stride, uint32_t pass, uint32_t radix,
                                                        SortScratch* __restrict__ sc) {
    __shared__ uint32_t s_tmp[4];
    __shared__ uint32_t s_total;
    const uint32_t d = blockIdx.x;
    const int tid = threadIdx.x;
    const uint32_t nparts = sort_parts(min(*count, cap));
    uint32_t* row = part_offsets(sc) + (size_t)d * stride;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < nparts; base += 256 * kScanPer) {
        uint32_t v[kScanPer], sum = 0;
#pragma unroll
        for (int j = 0; j < kScanPer; ++j) {
            const uint32_t idx = base + (uint32_t)tid * kScanPer + j;
            v[j] = idx < nparts ? row[idx] : 0u;
            sum += v[j];
        }
        const uint32_t excl = block_exclusive_scan_digits<256>(sum, s_tmp);
        if (tid == 255) s_total = excl + sum;
        uint32_t run = carry + excl;
#pragma unroll
        for (int j = 0; j < kScanPer; ++j) {
            const uint32_t idx = base + (uint32_t)tid * kScanPer + j;
            if (idx < nparts) row[idx] = run;
            run += v[j];
        }
        __syncthreads();
        carry += s_total;
        __syncthreads();
    }
    if (tid == 0) sc->hist[pass * radix + d] = carry;
}

template <typename K, int RB>
struct DownsweepShared {
    uint32_t wave_hist[kSortWaves][1 << RB];   // running counts, then wave-exclusive
    uint32_t digit_start[1 << RB];             // block-local exclusive digit starts
    uint32_t out_base[1 << RB];                // global dest = out_base[d] + local pos
    uint32_t tmp[2][kSortWaves];
    uint32_t valid;                            // keys of the partition that are kept
    K buf[kSortThreads * kMaxItems];           // the keys in digit order, then the payloads
};

// part_off / hist_d: this partition's offset and the total of digit threadIdx.x.
template <typename K, int RB, int ITEMS>
__device__ __forceinline__ void downsweep_part(const K* __restrict__ kin, const uint32_t* __restrict__ vin,
                                               K* __restrict__ kout, uint32_t* __restrict__ vout, uint32_t n,
                                               uint32_t part, uint32_t shift, uint32_t part_off, uint32_t hist_d,
                                               uint32_t* __restrict__ kept, DownsweepShared<K, RB>& sm) {
    constexpr uint32_t R = 1u << RB;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool drop = kept != nullptr;
    // Load: wave w owns keys [base + 64 ITEMS w, base + 64 ITEMS (w+1)), ITEMS
    // rounds of 64 consecutive keys -> input order = (wave, round, lane).
    const uint32_t wbase = part * (kSortThreads * ITEMS) + (uint32_t)wave * (64u * ITEMS);
    K key[ITEMS];
    uint32_t rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t idx = wbase + (uint32_t)r * 64u + (uint32_t)lane;
        const bool ok = idx < n;
        key[r] = ok ? kin[idx] : (K)0;
    }
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    // Stable wave-level ranking with ballots.
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t idx = wbase + (uint32_t)r * 64u + (uint32_t)lane;
        const bool ok = idx < n && !dropped(key[r], drop);
        const uint32_t d = (uint32_t)(key[r] >> shift) & (R - 1u);
        const uint64_t match = digit_match<RB>(d, ok);
        const uint32_t before = (uint32_t)__popcll(match & lt_mask);
        const uint32_t total = (uint32_t)__popcll(match);
        uint32_t prev = 0;
        if (ok) prev = sm.wave_hist[wave][d];
        __builtin_amdgcn_wave_barrier();
        rank[r] = prev + before;
        if (ok && before == 0) sm.wave_hist[wave][d] = prev + total;
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // Per digit: wave-exclusive prefixes and the block count.
    uint32_t block_count = 0;
    if ((uint32_t)tid < R) {
        uint32_t run = 0;
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) {
            const uint32_t c = sm.wave_hist[w][tid];
            sm.wave_hist[w][tid] = run;
            run += c;
        }
        block_count = run;
    }
    // Exclusive scans of the block's counts and of the digit totals, together:
    // one barrier for both instead of four (1M pairs 79.0 -> 76.5 us for four
    // passes, 4M 146 -> 143, 64-bit 2M 214 -> 210 for eight).
    uint32_t digit_start = block_count, global_start = hist_d;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t a = __shfl_up(digit_start, o), b = __shfl_up(global_start, o);
        if (lane >= o) {
            digit_start += a;
            global_start += b;
        }
    }
    if (lane == 63) {
        sm.tmp[0][wave] = digit_start;
        sm.tmp[1][wave] = global_start;
    }
    __syncthreads();
    digit_start -= block_count;
    global_start -= hist_d;
    for (int w = 0; w < wave; ++w) {
        digit_start += sm.tmp[0][w];
        global_start += sm.tmp[1][w];
    }
    if ((uint32_t)tid < R) {
        sm.digit_start[tid] = digit_start;
        sm.out_base[tid] = global_start + part_off - digit_start;
    }
    if ((uint32_t)tid == R - 1u) {
        sm.valid = digit_start + block_count;
        if (drop && part == 0u) *kept = global_start + hist_d;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t idx = wbase + (uint32_t)r * 64u + (uint32_t)lane;
        if (idx < n && !dropped(key[r], drop)) {
            const uint32_t d = (uint32_t)(key[r] >> shift) & (R - 1u);
            rank[r] += sm.digit_start[d] + sm.wave_hist[wave][d];
            sm.buf[rank[r]] = key[r];
        } else {
            rank[r] = ~0u;
        }
    }
    __syncthreads();
    const uint32_t valid = sm.valid;
    uint32_t out[ITEMS], val[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t idx = wbase + (uint32_t)r * 64u + (uint32_t)lane;
        val[r] = idx < n ? vin[idx] : 0u;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = (uint32_t)(tid + r * kSortThreads);
        if (i < valid) {
            const K k = sm.buf[i];
            out[r] = sm.out_base[(uint32_t)(k >> shift) & (R - 1u)] + i;
            kout[out[r]] = k;
        }
    }
    __syncthreads();
    uint32_t* const vbuf = reinterpret_cast<uint32_t*>(sm.buf);
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
        if (rank[r] != ~0u) vbuf[rank[r]] = val[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const uint32_t i = (uint32_t)(tid + r * kSortThreads);
        if (i < valid) vout[out[r]] = vbuf[i];
    }
}

// FUSED: the counts are not scanned yet; thread d sums its digit's row (at
// most 128 counts, 16 B at a time) itself, which saves a launch: 20k keys 9.7
// us a pass against 13.1 with the scan, 120k 12.8 against 13.7; with 256
// counts a row (250k keys) the scan is faster, 15.1 against 15.7. `kept` (first pass
// of a sort that drops keys): receives the number of the others.
template <typename K, int RB, bool FUSED>
__global__ __launch_bounds__(kSortThreads) void downsweep_kernel(
    const K* __restrict__ kin, const uint32_t* __restrict__ vin, K* __restrict__ kout,
    uint32_t* __restrict__ vout, const uint32_t* __restrict__ count, uint32_t cap, uint32_t shift,
    uint32_t stride, uint32_t pass, const SortScratch* __restrict__ sc, uint32_t* __restrict__ kept) {
    constexpr uint32_t R = 1u << RB;
    __shared__ DownsweepShared<K, RB> sm;
    const int tid = threadIdx.x;
    const uint32_t n = min(*count, cap);
    const uint32_t part = blockIdx.x, items = sort_items(n), parts = sort_parts(n);
    if (part >= parts) {  // grid sized for the capacity
        if (kept != nullptr && part == 0u && tid == 0) *kept = 0u;
        return;
    }
    for (uint32_t k = tid; k < kSortWaves * R; k += kSortThreads) (&sm.wave_hist[0][0])[k] = 0u;
    // This partition's offset of every digit and the digit totals (read
    // early; used after the ranking).
    uint32_t part_off = 0u, hist_d = 0u;
    if ((uint32_t)tid < R) {
        const uint32_t* row = reinterpret_cast<const uint32_t*>(sc + 1) + (size_t)tid * stride;
        if constexpr (FUSED) {
#pragma unroll 4
            for (uint32_t j = 0; j < parts; j += 4) {
                const uint4 c = *reinterpret_cast<const uint4*>(row + j);  // stride is a multiple of 4
                const uint32_t v[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    hist_d += j + k < parts ? v[k] : 0u;
                    part_off += j + k < part ? v[k] : 0u;
                }
            }
        } else {
            part_off = row[part];
            hist_d = sc->hist[pass * R + tid];
        }
    }
    __syncthreads();
    if (items == 2) downsweep_part<K, RB, 2>(kin, vin, kout, vout, n, part, shift, part_off, hist_d, kept, sm);
    else if (items == 4) downsweep_part<K, RB, 4>(kin, vin, kout, vout, n, part, shift, part_off, hist_d, kept, sm);
    else downsweep_part<K, RB, 8>(kin, vin, kout, vout, n, part, shift, part_off, hist_d, kept, sm);
}

// A sort that one workgroup holds: 1024 threads, the pairs in registers, one
// LDS buffer through which first the keys and then the payloads take their
// new places.
constexpr int kSmallThreads = 1024, kSmallWaves = kSmallThreads / 64;
constexpr int kSmallItems = 4;
constexpr uint32_t kSmallCap = kSmallThreads * kSmallItems;

template <typename K, int RB>
struct SmallShared {
    K buf[kSmallCap];
    uint32_t wave_hist[kSmallWaves][1 << RB];
    uint32_t start[1 << RB];
    uint32_t tmp[kSmallWaves];
    uint32_t n;
};

// Rounds of 64 consecutive pairs that each wave holds: wave w's round r has
// pairs 64 (rounds w + r) .. + 63, so the waves share n pairs evenly.
__device__ __forceinline__ uint32_t small_rounds(uint32_t n) { return (n + kSmallThreads - 1) / kSmallThreads; }

// Sorts n <= kSmallCap pairs held in (wave, round, lane) order; the last pass
// writes them to kout (optional) and vout. Returns the number that is kept.
template <typename K, int RB>
__device__ __forceinline__ uint32_t small_sort(K (&key)[kSmallItems], uint32_t (&val)[kSmallItems], uint32_t n,
                                               uint32_t begin_bit, uint32_t passes, bool drop,
                                               K* kout, uint32_t* vout, SmallShared<K, RB>& sm) {
    constexpr uint32_t R = 1u << RB;
    constexpr int ITEMS = kSmallItems;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint32_t* const vbuf = reinterpret_cast<uint32_t*>(sm.buf);
    for (uint32_t p = 0; p < passes; ++p) {
        const uint32_t shift = begin_bit + p * RB, rounds = small_rounds(n);
        const uint32_t wbase = (uint32_t)wave * 64u * rounds + (uint32_t)lane;
        for (uint32_t k = tid; k < kSmallWaves * R; k += kSmallThreads) (&sm.wave_hist[0][0])[k] = 0u;
        __syncthreads();
        uint32_t pos[ITEMS];
        bool ok[ITEMS];
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            ok[r] = (uint32_t)r < rounds && wbase + 64u * (uint32_t)r < n && !dropped(key[r], drop && p == 0u);
            pos[r] = 0u;
            if ((uint32_t)r >= rounds) continue;
            const uint32_t d = (uint32_t)(key[r] >> shift) & (R - 1u);
            const uint64_t match = digit_match<RB>(d, ok[r]);
            const uint32_t before = (uint32_t)__popcll(match & lt_mask);
            uint32_t prev = 0;
            if (ok[r]) prev = sm.wave_hist[wave][d];
            __builtin_amdgcn_wave_barrier();
            pos[r] = prev + before;
            if (ok[r] && before == 0) sm.wave_hist[wave][d] = prev + (uint32_t)__popcll(match);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        uint32_t total = 0;
        if ((uint32_t)tid < R) {
#pragma unroll
            for (int w = 0; w < kSmallWaves; ++w) {
                const uint32_t c = sm.wave_hist[w][tid];
                sm.wave_hist[w][tid] = total;
                total += c;
            }
        }
        const uint32_t start = block_exclusive_scan_digits<R>(total, sm.tmp);
        if ((uint32_t)tid < R) sm.start[tid] = start;
        if ((uint32_t)tid == R - 1u) sm.n = start + total;
        __syncthreads();
        n = sm.n;
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            if (!ok[r]) continue;
            const uint32_t d = (uint32_t)(key[r] >> shift) & (R - 1u);
            pos[r] += sm.start[d] + sm.wave_hist[wave][d];
            sm.buf[pos[r]] = key[r];
        }
        __syncthreads();
        // The pairs' next places in (wave, round, lane) order, or the output.
        const bool final_pass = p + 1u == passes;
        const uint32_t next = (uint32_t)wave * 64u * small_rounds(n) + (uint32_t)lane;
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const uint32_t idx = final_pass ? (uint32_t)(tid + r * kSmallThreads) : next + 64u * (uint32_t)r;
            const bool in = idx < n && (final_pass || (uint32_t)r < small_rounds(n));
            key[r] = in ? sm.buf[idx] : (K)0;
            if (final_pass && in && kout != nullptr) kout[idx] = key[r];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r)
            if (ok[r]) vbuf[pos[r]] = val[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const uint32_t idx = final_pass ? (uint32_t)(tid + r * kSmallThreads) : next + 64u * (uint32_t)r;
            const bool in = idx < n && (final_pass || (uint32_t)r < small_rounds(n));
            val[r] = in ? vbuf[idx] : 0u;
            if (final_pass && in) vout[idx] = val[r];
        }
    }
    return n;
}

// After an even number of passes the output is the input's buffers: no
// __restrict__. Every pair is read before the first barrier.
template <typename K, int RB>
__global__ __launch_bounds__(kSmallThreads) void small_sort_kernel(const K* kin, const uint32_t* vin, K* kout,
                                                                   uint32_t* vout,
                                                                   const uint32_t* __restrict__ count, uint32_t cap,
                                                                   uint32_t begin_bit, uint32_t passes,
                                                                   uint32_t* __restrict__ kept) {
    __shared__ SmallShared<K, RB> sm;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t n = min(*count, cap), rounds = small_rounds(n);
    K key[kSmallItems];
    uint32_t val[kSmallItems];
#pragma unroll
    for (int r = 0; r < kSmallItems; ++r) {
        const uint32_t idx = (uint32_t)wave * 64u * rounds + 64u * (uint32_t)r + (uint32_t)lane;
        const bool in = (uint32_t)r < rounds && idx < n;
        key[r] = in ? kin[idx] : (K)0;
        val[r] = in ? vin[idx] : 0u;
    }
    const uint32_t m = small_sort<K, RB>(key, val, n, begin_bit, passes, kept != nullptr, kout, vout, sm);
    if (kept != nullptr && tid == 0) *kept = m;
}

// Longest-list-first order of up to kSmallCap tiles (as tile_order_keys_kernel
// and a 16-bit sort), and the cursors reset.
__global__ __launch_bounds__(kSmallThreads) void tile_order_kernel(const uint32_t* __restrict__ ranges,
                                                                   uint32_t tile_begin, uint32_t n_tiles,
                                                                   uint32_t* __restrict__ order,
                                                                   uint32_t* __restrict__ cursors) {
    __shared__ SmallShared<uint32_t, 8> sm;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t rounds = small_rounds(n_tiles);
    if (tid < 2 * (int)kTileQueues) cursors[(uint32_t)tid * kCursorStride] = 0u;
    uint32_t key[kSmallItems], val[kSmallItems];
#pragma unroll
    for (int r = 0; r < kSmallItems; ++r) {
        const uint32_t t = (uint32_t)wave * 64u * rounds + 64u * (uint32_t)r + (uint32_t)lane;
        const bool in = (uint32_t)r < rounds && t < n_tiles;
        const size_t g = (size_t)tile_begin + t;
        key[r] = in ? tile_order_key(ranges[2 * g + 1] - ranges[2 * g]) : 0u;
        val[r] = (uint32_t)g;
    }
    small_sort<uint32_t, 8>(key, val, n_tiles, 0, 2, false, nullptr, order, sm);
}

template <typename K>
__global__ __launch_bounds__(256) void copy_pairs_kernel(const K* __restrict__ sk,
                                                         const uint32_t* __restrict__ sv,
                                                         K* __restrict__ dk, uint32_t* __restrict__ dv,
                                                         const uint32_t* __restrict__ count, uint32_t cap) {
    const uint32_t n = min(*count, cap);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        dk[i] = sk[i];
        dv[i] = sv[i];
    }
}

template <typename K, int RB>
hipError_t run_passes(hipStream_t st, K* (&kb)[2], uint32_t* (&vb)[2], const uint32_t* count, uint32_t cap,
                             uint32_t begin_bit, uint32_t passes, SortScratch* sc, uint32_t* kept) {
    // One workgroup for all passes: 3000 keys 5.8 us a pass (64 bits: 5.2)
    // against 8.7 with two launches a pass and 15 with three; with twice the
    // pairs in it (8000) 10.7 against 9.4.
    if constexpr (RB <= 8) {
        if (cap <= kSmallCap) {
            const int dst = (int)(passes & 1u);
            hipLaunchKernelGGL((small_sort_kernel<K, RB>), dim3(1), dim3(kSmallThreads), 0, st, kb[0], vb[0], kb[dst],
                               vb[dst], count, cap, begin_bit, passes, kept);
            return hipGetLastError();
        }
    }
    const bool fused = cap <= kFusedCap;
    // A capacity far above the count launches workgroups that only leave (0.2
    // ns each): the upsweep takes partitions past 8192 workgroups in turn; in
    // the downsweep that loop costs 30 registers, and with them waves.
    const uint32_t grid = most_parts(cap), stride = grid;
    hipError_t e = hipSuccess;
    for (uint32_t p = 0; p < passes; ++p) {
        const uint32_t shift = begin_bit + p * RB;
        const int src = (int)(p & 1u), dst = 1 - src;
        const bool drop = kept != nullptr && p == 0;
        hipLaunchKernelGGL((upsweep_kernel<K, RB>), dim3(std::min(grid, 8192u)), dim3(kSortThreads), 0, st, kb[src],
                           count, cap, shift, stride, drop, sc);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (!fused) {
            hipLaunchKernelGGL(part_scan_kernel, dim3(1u << RB), dim3(256), 0, st, count, cap, stride, p, 1u << RB,
                               sc);
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
        auto* down = fused ? downsweep_kernel<K, RB, true> : downsweep_kernel<K, RB, false>;
        hipLaunchKernelGGL(down, dim3(grid), dim3(kSortThreads), 0, st, kb[src], vb[src], kb[dst], vb[dst], count,
                           cap, shift, stride, p, sc, drop ? kept : nullptr);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (drop) count = kept;
    }
    return hipSuccess;
}

// Digits of 9 bits where they save a pass and the caller's keys have no bits
// past end_bit (`exact`; other callers get whole 8-bit digits, as ever): 45 key
// bits in five passes instead of six (a binning of 1.1M 64-bit pairs 173 -> 164 us).
uint32_t digit_width(uint32_t cap, uint32_t bits, uint32_t digit_bits, bool exact) {
    const bool nine = exact && digit_bits == 8 && cap > kSmallCap && (bits + 8) / 9 < (bits + 7) / 8;
    return nine ? 9u : digit_bits;
}

template <typename K>
hipError_t radix_sort_impl(hipStream_t st, K* keys0, uint32_t* vals0, K* keys1, uint32_t* vals1,
                           const uint32_t* count, uint32_t capacity, uint32_t begin_bit,
                           uint32_t end_bit, uint32_t digit_bits, void* scratch,
                           int* result_in_alt, bool exact, uint32_t* kept) {
    SortScratch* sc = static_cast<SortScratch*>(scratch);
    if (digit_bits != 4 && digit_bits != 8) return hipErrorInvalidValue;
    if (end_bit <= begin_bit || end_bit > sizeof(K) * 8) return hipErrorInvalidValue;
    const uint32_t passes = radix_sort_passes(capacity, end_bit - begin_bit, digit_bits, exact);
    if (passes > (uint32_t)kMaxPasses) return hipErrorInvalidValue;
    *result_in_alt = (int)(passes & 1u);
    K* kb[2] = {keys0, keys1};
    uint32_t* vb[2] = {vals0, vals1};
    auto run = [&](auto fn) { return fn(st, kb, vb, count, capacity, begin_bit, passes, sc, kept); };
    const uint32_t width = digit_width(capacity, end_bit - begin_bit, digit_bits, exact);
    return width == 9 ? run(run_passes<K, 9>) : width == 8 ? run(run_passes<K, 8>) : run(run_passes<K, 4>);
}

}  // namespace

hipError_t launch_copy_pairs(hipStream_t st, const void* src_keys, const uint32_t* src_vals,
                             void* dst_keys, uint32_t* dst_vals, uint32_t key_bytes,
                             const uint32_t* count, uint32_t capacity) {
    uint32_t blocks = div_up(capacity ? capacity : 1, 256);
    if (blocks > 8192) blocks = 8192;
    if (key_bytes == 8)
        hipLaunchKernelGGL(copy_pairs_kernel<uint64_t>, dim3(blocks), dim3(256), 0, st,
                           static_cast<const uint64_t*>(src_keys), src_vals,
                           static_cast<uint64_t*>(dst_keys), dst_vals, count, capacity);
    else
        hipLaunchKernelGGL(copy_pairs_kernel<uint32_t>, dim3(blocks), dim3(256), 0, st,
                           static_cast<const uint32_t*>(src_keys), src_vals,
                           static_cast<uint32_t*>(dst_keys), dst_vals, count, capacity);
    return hipGetLastError();
}

uint32_t radix_sort_passes(uint32_t capacity, uint32_t bits, uint32_t digit_bits, bool exact) {
    const uint32_t width = digit_width(capacity, bits, digit_bits, exact);
    return (bits + width - 1) / width;
}

size_t sort_scratch_bytes(uint32_t capacity) {
    return sizeof(SortScratch) + (size_t)most_parts(capacity) * 512 * sizeof(uint32_t);  // 9-bit digits at most
}

hipError_t launch_radix_sort_u64(hipStream_t st, uint64_t* keys0, uint32_t* vals0, uint64_t* keys1,
                                 uint32_t* vals1, const uint32_t* count, uint32_t capacity,
                                 uint32_t begin_bit, uint32_t end_bit, uint32_t digit_bits,
                                 void* scratch, int* result_in_alt, bool exact) {
    return radix_sort_impl<uint64_t>(st, keys0, vals0, keys1, vals1, count, capacity, begin_bit,
                                     end_bit, digit_bits, scratch, result_in_alt, exact, nullptr);
}

hipError_t launch_radix_sort_u32(hipStream_t st, uint32_t* keys0, uint32_t* vals0, uint32_t* keys1,
                                 uint32_t* vals1, const uint32_t* count, uint32_t capacity,
                                 uint32_t begin_bit, uint32_t end_bit, uint32_t digit_bits,
                                 void* scratch, int* result_in_alt, bool exact, uint32_t* kept) {
    return radix_sort_impl<uint32_t>(st, keys0, vals0, keys1, vals1, count, capacity, begin_bit,
                                     end_bit, digit_bits, scratch, result_in_alt, exact, kept);
}

uint32_t tile_order_small_cap() { return kSmallCap; }

hipError_t launch_tile_order_small(hipStream_t st, const uint32_t* ranges, uint32_t tile_begin, uint32_t n_tiles,
                                   uint32_t* order, uint32_t* cursors) {
    if (n_tiles > kSmallCap) return hipErrorInvalidValue;
    hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(kSmallThreads), 0, st, ranges, tile_begin, n_tiles, order,
                       cursors);
    return hipGetLastError();
}

}  // namespace gs
