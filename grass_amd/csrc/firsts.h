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

// Segments of the 64 positions from 64 w (n in all, R segments): one search for the wave, and one
// per lane only where a segment ends inside the word.
__device__ __forceinline__ uint32_t segment_of_lane(const uint64_t* __restrict__ off, uint32_t R, uint64_t w, uint64_t n) {
    const uint64_t p0 = w * kWave;
    const uint32_t r0 = segment_in(off, 0, R - 1, p0);
    const uint64_t last = min(p0 + kWave - 1, n - 1);
    if (r0 + 1 == R || off[r0 + 1] > last) return r0;
    return segment_in(off, r0, R - 1, min(p0 + (uint64_t)lane_id(), last));
}

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

static __global__ __launch_bounds__(256) void firsts_segments_kernel(const FirstWord* words, Count cnt,
                                                                     const uint64_t* __restrict__ off, uint32_t R,
                                                                     uint64_t* __restrict__ foff, uint64_t* count) {
    const uint64_t n = cnt.get();
    const uint64_t total = words[(n + kWave - 1) / kWave].y;  // (the scan's total follows the last word)
    segment_firsts(words, n, total, off, R, foff, count, blockIdx.x * 256 + threadIdx.x, gridDim.x * 256);
}

// Words of a sequence of at most n_max positions, the entry after the last included.
inline uint64_t firsts_words(uint64_t n_max) { return (n_max + kWave - 1) / kWave + 1; }

// Fills the words' counts for n positions and the ranks of the R segments that start at off[] (off[R]
// = n): foff[0..R], *count = all firsts.  Scratch: partials[scan_blocks(words)] and total[1].
inline hipError_t scan_firsts(FirstWord* words, Count n, uint64_t n_max, const uint64_t* off, uint32_t R,
                              uint64_t* foff, uint64_t* count, uint64_t* partials, uint64_t* total, hipStream_t s) {
    const uint64_t nw = firsts_words(n_max);
    if (nw <= kFirstsOneWg) {
        hipLaunchKernelGGL(firsts_scan_kernel, dim3(1), dim3(1024), 0, s, words, n, off, R, foff, count);
        return hipGetLastError();
    }
    Count in_words = n;
    in_words.shift = 6;
    hipError_t e = exclusive_scan<2>(FirstsGen{words}, in_words, nw, (uint64_t*)words + 1, partials, total, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(firsts_segments_kernel, dim3(std::min<uint32_t>(R / 256 + 1, 1024)), dim3(256), 0, s,
                       (const FirstWord*)words, n, off, R, foff, count);
    return hipGetLastError();
}

}  // namespace grass
