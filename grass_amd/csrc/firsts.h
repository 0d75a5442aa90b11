// First appearances: which positions of a sequence hold a (request, vertex) key for the first time, and
// how many such positions come before any other.
//
// Every position starts as a first (init: all ones) and is taken off the list at most once, while
// the positions are inserted into a table that keeps the smallest position of each key: by itself
// when its key already holds a smaller one, or by the position that displaces it.  Both only clear
// bits, so the order of the inserts does not matter, and no pass has to look every key up again
// once the table is complete.  64 positions share a word {bits, firsts before the word}: 16 bytes
// per 64 positions, so that the rank of any first is one load from memory that stays in the L2
// (2.9 MB for 11.5 M positions, where a prefix per position was 92 MB).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "devutil.h"
#include "scan.h"

namespace grass {

typedef ulonglong2 FirstWord;  // x: bit j = position 64 w + j is a first; y: firsts before the word

__device__ __forceinline__ void not_first(FirstWord* words, uint64_t p) {
    atomicAnd(&words[p >> 6].x, ~(1ull << (p & 63)));
}

// Firsts before position p.
__device__ __forceinline__ uint64_t first_rank(const FirstWord* __restrict__ words, uint64_t p) {
    const FirstWord w = words[p >> 6];
    return w.y + (uint64_t)__popcll(w.x & ((1ull << (p & 63)) - 1));
}

// Largest r in [lo, hi] with off[r] <= p (off ascending, off[lo] <= p).
__device__ __forceinline__ uint32_t segment_in(const uint64_t* __restrict__ off, uint32_t lo, uint32_t hi, uint64_t p) {
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo + 1) / 2;
        if (off[mid] <= p) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// The words a wave takes, one after the other: consecutive ones, so that the segment it is in (and the
// loads that find it, each waiting for the one before) serves many words.
struct WordChunk {
    uint64_t w, end;
};
template <int BLOCK>
__device__ __forceinline__ WordChunk wave_words(uint64_t n) {
    const uint64_t nwords = (n + kWave - 1) / kWave, waves = (uint64_t)gridDim.x * (BLOCK / kWave);
    const uint64_t wave = (uint64_t)blockIdx.x * (BLOCK / kWave) + threadIdx.x / kWave;
    const uint64_t per = (nwords + waves - 1) / waves, w = readfirstlane_u64(wave * per);
    return WordChunk{w, min(w + per, nwords)};
}

// The segment of each lane's position, for a wave that goes through consecutive words of 64 positions
// (n in all, R segments starting at off[]): the last segment found serves every word inside it.
struct SegmentCursor {
    uint32_t r = 0;
    uint64_t beg = 1, end = 0;  // positions of segment r
    __device__ __forceinline__ uint32_t of_lane(const uint64_t* __restrict__ off, uint32_t R, uint64_t w, uint64_t n) {
        const uint64_t p0 = w * kWave, last = min(p0 + kWave - 1, n - 1);
        if (p0 < beg || p0 >= end) {
            r = segment_in(off, 0, R - 1, p0);
            beg = off[r];
            end = r + 1 < R ? off[r + 1] : n;
        }
        if (last < end) return r;
        return segment_in(off, r, R - 1, min(p0 + (uint64_t)lane_id(), last));
    }
};

struct FirstsGen {
    const FirstWord* words;
    __device__ __forceinline__ uint64_t operator()(uint64_t w) const { return (uint64_t)__popcll(words[w].x); }
};

constexpr uint64_t kFirstsOneWg = 16384;  // words that one workgroup scans in a launch (1 M positions)

// firsts before off[r] for every r <= R (off[R] = n), and their total.
__device__ __forceinline__ void segment_firsts(const FirstWord* words, uint64_t n, uint64_t total,
                                               const uint64_t* __restrict__ off, uint32_t R, uint64_t* __restrict__ foff,
                                               uint64_t* count, uint32_t t, uint32_t threads) {
    for (uint32_t r = t; r <= R; r += threads) {
        const uint64_t p = off[r];
        foff[r] = p < n ? first_rank(words, p) : total;
    }
    if (t == 0 && count) *count = total;
}

// The counts of up to kFirstsOneWg words in one workgroup, and the segments' ranks.
static __global__ __launch_bounds__(1024) void firsts_scan_kernel(FirstWord* words, Count cnt,
                                                                  const uint64_t* __restrict__ off, uint32_t R,
                                                                  uint64_t* __restrict__ foff, uint64_t* count) {
    __shared__ uint32_t lds[1024 / kWave];
    constexpr uint32_t kPer = kFirstsOneWg / 1024;
    const uint64_t n = cnt.get();
    const uint32_t nw = (uint32_t)((n + kWave - 1) / kWave), per = (nw + 1023) / 1024;
    const uint32_t w0 = threadIdx.x * per;
    uint32_t c[kPer], s = 0;
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        c[i] = i < per && w0 + i < nw ? (uint32_t)__popcll(words[w0 + i].x) : 0u;
        s += c[i];
    }
    uint32_t total;
    uint32_t pre = block_exclusive_sum<uint32_t, 1024>(s, total, lds);
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        if (i < per && w0 + i < nw) words[w0 + i].y = pre;
        pre += c[i];
    }
    __syncthreads();  // the words' counts are read across the workgroup
    segment_firsts(words, n, total, off, R, foff, count, threadIdx.x, 1024);
}

// The same as marks of the scan (its items are the words).
struct SegmentMarks {
    const FirstWord* words;
    Count cnt;
    const uint64_t* off;
    uint64_t* foff;
    uint64_t* total;
    uint32_t count;  // R + 1
    __device__ __forceinline__ uint64_t at(uint32_t r) const {
        const uint64_t p = off[r];
        return p < cnt.get() ? p / kWave : ~0ull;
    }
    __device__ __forceinline__ void put(uint32_t r, uint64_t before) const {
        const uint64_t p = off[r];
        foff[r] = before + (p < cnt.get() ? (uint64_t)__popcll(words[p / kWave].x & ((1ull << (p & 63)) - 1)) : 0);
    }
    __device__ __forceinline__ void end(uint64_t t) const {
        if (total) *total = t;
    }
};

static __global__ __launch_bounds__(256) void firsts_segments_kernel(const FirstWord* words, Count cnt,
                                                                     const uint64_t* __restrict__ off, uint32_t R,
                                                                     uint64_t* __restrict__ foff, uint64_t* count) {
    const uint64_t n = cnt.get();
    const uint64_t total = words[(n + kWave - 1) / kWave].y;  // (the scan's total follows the last word)
    segment_firsts(words, n, total, off, R, foff, count, blockIdx.x * 256 + threadIdx.x, gridDim.x * 256);
}

// One workgroup's dedup of up to kOneWgEntries positions: table, firsts and ranks in LDS.  A slot is
// ((request << vb | vertex) << kOneWgPosBits) | position, all ones when empty (requests < 2^17, vertices <
// 2^31).  The table's memory is the caller's again once the ranks are made.
constexpr uint32_t kOneWgThreads = 1024;
constexpr uint32_t kOneWgPer = 8;  // positions of a thread: tid, tid + 1024, ...
constexpr uint32_t kOneWgEntries = kOneWgThreads * kOneWgPer;
constexpr uint32_t kOneWgPosBits = 13;
constexpr uint32_t kOneWgWords = kOneWgEntries / kWave;

// Slots for n entries (load <= 2/3), a power of two.
__host__ __device__ constexpr uint32_t one_wg_slots(uint32_t n) {
    uint32_t slots = 1024;
    while (slots < n + n / 2 + 2) slots <<= 1;
    return slots;
}

struct OneWgFirsts {
    unsigned long long* tab;            // one_wg_slots(n) slots
    unsigned long long bits[kOneWgWords];  // firsts of 64 positions each
    uint32_t pre[kOneWgWords];          // firsts before them
    uint32_t total;
    uint32_t mask, shift, vb;

    __device__ __forceinline__ uint32_t home(unsigned long long k) const {
        return (uint32_t)(((k + 1) * 0x9E3779B97F4A7C15ull) >> shift);
    }
    __device__ __forceinline__ uint32_t rank(uint32_t p) const {
        return pre[p / kWave] + (uint32_t)__popcll(bits[p / kWave] & ((1ull << (p & (kWave - 1))) - 1));
    }
    // Slot of (r, v), which position p enters.
    __device__ __forceinline__ uint32_t insert(uint32_t r, uint32_t v, uint32_t p) {
        const unsigned long long k = ((unsigned long long)r << vb) | v, w = (k << kOneWgPosBits) | p;
        uint32_t h = home(k);
        for (;;) {  // ends: more slots than entries
            const unsigned long long cur = atomicCAS(tab + h, ~0ull, w);
            if (cur == ~0ull) return h;
            if ((cur >> kOneWgPosBits) == k) {
                if (cur > w) atomicMin(tab + h, w);
                return h;
            }
            h = (h + 1) & mask;
        }
    }
    // First position of (r, v), or ~0 where it was never entered (after the inserts).
    __device__ __forceinline__ uint32_t first(uint32_t r, uint32_t v) const {
        const unsigned long long k = ((unsigned long long)r << vb) | v;
        uint32_t h = home(k);
        for (;;) {
            const unsigned long long cur = tab[h];
            if (cur == ~0ull) return ~0u;
            if ((cur >> kOneWgPosBits) == k) return (uint32_t)cur & (kOneWgEntries - 1);
            h = (h + 1) & mask;
        }
    }
};

// Empties the table for n positions.  Every function below is called by the whole workgroup.
__device__ __forceinline__ void one_wg_begin(OneWgFirsts& f, unsigned long long* tab, uint32_t n, uint32_t vb) {
    const uint32_t slots = one_wg_slots(n);
    for (uint32_t i = threadIdx.x; i < slots; i += kOneWgThreads) tab[i] = ~0ull;
    if (threadIdx.x == 0) {
        f.tab = tab;
        f.mask = slots - 1;
        f.shift = 64 - (31 - __clz(slots));
        f.vb = vb;
    }
    __syncthreads();
}

// After the inserts (slot[i] of position i * 1024 + tid, ~0 for none): which of the thread's positions are
// firsts (bit i), and the ranks of all.
__device__ __forceinline__ uint32_t one_wg_rank(OneWgFirsts& f, uint32_t n, const uint32_t* slot) {
    __syncthreads();
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t i = 0; i < kOneWgPer; ++i) {
        const uint32_t p = i * kOneWgThreads + threadIdx.x;
        const bool first = p < n && slot[i] != ~0u && ((uint32_t)f.tab[slot[i]] & (kOneWgEntries - 1)) == p;
        mine |= (first ? 1u : 0u) << i;
        const unsigned long long b = __ballot(first);
        if (lane_id() == 0) f.bits[p / kWave] = b;
    }
    __syncthreads();
    static_assert(kOneWgWords == 2 * kWave, "one wave scans two words a lane");
    if (threadIdx.x < kWave) {
        const uint32_t a = (uint32_t)__popcll(f.bits[2 * threadIdx.x]), b = (uint32_t)__popcll(f.bits[2 * threadIdx.x + 1]);
        const uint32_t inc = wave_inclusive_sum(a + b);
        f.pre[2 * threadIdx.x] = inc - a - b;
        f.pre[2 * threadIdx.x + 1] = inc - b;
        if (threadIdx.x == kWave - 1) f.total = inc;
    }
    __syncthreads();
    return mine;
}

// Words of a sequence of at most n_max positions, the entry after the last included.
inline uint64_t firsts_words(uint64_t n_max) { return (n_max + kWave - 1) / kWave + 1; }

// Fills the words' counts for n positions and the ranks of the R segments that start at off[] (off[R]
// = n; a scan of several workgroups takes fewer than kScanMarksMax of them along): foff[0..R], *count = all firsts.  Scratch: partials[scan_blocks(words)] and total[1].
inline hipError_t scan_firsts(FirstWord* words, Count n, uint64_t n_max, const uint64_t* off, uint32_t R,
                              uint64_t* foff, uint64_t* count, uint64_t* partials, uint64_t* total, hipStream_t s) {
    const uint64_t nw = firsts_words(n_max);
    if (nw <= kFirstsOneWg) {
        hipLaunchKernelGGL(firsts_scan_kernel, dim3(1), dim3(1024), 0, s, words, n, off, R, foff, count);
        return hipGetLastError();
    }
    Count in_words = n;
    in_words.shift = 6;
    if (R < kScanMarksMax)
        return exclusive_scan<2>(FirstsGen{words}, in_words, nw, (uint64_t*)words + 1, partials, total, s,
                                 SegmentMarks{words, n, off, foff, count, R + 1});
    hipError_t e = exclusive_scan<2>(FirstsGen{words}, in_words, nw, (uint64_t*)words + 1, partials, total, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(firsts_segments_kernel, dim3(std::min<uint32_t>(R / 256 + 1, 1024)), dim3(256), 0, s,
                       (const FirstWord*)words, n, off, R, foff, count);
    return hipGetLastError();
}

}  // namespace grass
