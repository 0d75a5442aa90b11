// Reduce-then-scan exclusive prefix sum over a generated sequence of uint64 values.
//
// Launches with no inter-workgroup waiting: per-tile sums, then each tile re-generates its values
// and writes prefixes.  A sequence of at most kScanFoldMax tiles has each tile add up the tile sums
// before it itself (a few thousand cached values); a longer one scans the tile sums in one
// workgroup in between (a third launch).  Of at most kScanDirectMax tiles each generates the values
// before it itself and one launch does it all.  The length can be
// a host value or a device-resident count (so a sequence whose size a previous kernel
// produced needs no host round trip); the grid is sized for the host-side upper bound.
// Used for the record-length scan at load (replacing cub::DeviceScan::ExclusiveSum,
// LE/src/utils.hpp:337-342), CSR row pointers and sampler output offsets.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "devutil.h"

namespace grass {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;
constexpr uint64_t kScanTile = (uint64_t)kScanBlock * kScanItems;
constexpr uint64_t kScanFoldMax = 2048;  // tiles whose start each tile sums itself
// Tiles whose start each tile sums from the values (the generator must not read what is written): a
// launch saved against up to 48 more values per thread.  A full decode of R-MAT s14 (16 k rows, 148 k
// entries), whose calls the host's launches bound, went from 14.4 to 10.2 us with the one launch.
constexpr uint64_t kScanDirectMax = 4;
enum ScanMode { kScanDirect, kScanFold, kScanThree };

struct Count {
    uint64_t imm;
    const uint64_t* dev;  // when non-null the count is *dev
    uint32_t shift = 0;   // in units of 2^shift, rounded up
    __device__ __forceinline__ uint64_t get() const {
        return ((dev ? *dev : imm) + ((1ull << shift) - 1)) >> shift;
    }
};

template <class Gen>
__global__ __launch_bounds__(kScanBlock) void scan_reduce_kernel(Gen gen, Count cnt,
                                                                 uint64_t* partials) {
    __shared__ uint64_t lds[kScanBlock / kWave];
    const uint64_t n = cnt.get();
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
    uint64_t s = 0;
    if (base < n) {
#pragma unroll 4
        for (int j = 0; j < kScanItems; ++j) {
            uint64_t i = base + (uint64_t)j * kScanBlock + threadIdx.x;
            if (i < n) s += gen(i);
        }
    }
    s = block_sum<uint64_t, kScanBlock>(s, lds);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// One workgroup: partials[0..nb) -> exclusive prefixes in place; *total = sum.
// (A template so that every translation unit including this header may instantiate it.)
template <typename T>
__global__ __launch_bounds__(1024) void scan_partials_kernel(T* partials, uint64_t nb, T* total) {
    __shared__ T lds[1024 / kWave];
    const uint64_t per = (nb + 1023) / 1024;
    const uint64_t lo = threadIdx.x * per;
    T s = 0;
    for (uint64_t i = lo; i < lo + per && i < nb; ++i) s += partials[i];
    T tot;
    T pre = block_exclusive_sum<T, 1024>(s, tot, lds);
    for (uint64_t i = lo; i < lo + per && i < nb; ++i) {
        T t = partials[i];
        partials[i] = pre;
        pre += t;
    }
    if (threadIdx.x == 0 && total) *total = tot;
}

// 64-bit inclusive sum over the wave with DPP moves of the two halves (no LDS).
__device__ __forceinline__ uint64_t wave_inclusive_sum_u64(uint64_t x) {
#define GRASS_SCAN_STEP(CTRL, RM)                                                                  \
    x += ((uint64_t)dpp_move<CTRL, RM>((uint32_t)(x >> 32)) << 32) | dpp_move<CTRL, RM>((uint32_t)x)
    GRASS_SCAN_STEP(0x111, 0xf);
    GRASS_SCAN_STEP(0x112, 0xf);
    GRASS_SCAN_STEP(0x114, 0xf);
    GRASS_SCAN_STEP(0x118, 0xf);
    GRASS_SCAN_STEP(0x142, 0xa);
    GRASS_SCAN_STEP(0x143, 0xc);
#undef GRASS_SCAN_STEP
    return x;
}

// out[i] = sum of gen(0..i-1) for i < n, and out[n] = total.  Wave w of a tile takes
// kWave * kScanItems consecutive items in kScanItems rounds of kWave consecutive ones (coalesced
// loads and stores): its lanes' sums and one exchange of the wave sums give each wave its start,
// and each round is one DPP wave scan carried into the next (no workgroup scan per round).
// kScanFold: partials[] are the tile sums themselves (at most kScanFoldMax of them): each tile adds up
// those before it, and the tile holding item n - 1 also writes *total; kScanDirect: the same from the
// values themselves, partials[] unread; kScanThree: partials[] are
// the tiles' exclusive prefixes and *total was written with them.  Outputs lie STRIDE words apart.
//
// `marks` may name items whose prefixes are wanted by themselves (the ends of requests): once a tile's
// prefixes are written, its workgroup looks the marks that lie in it up, in place of a launch after
// the scan.  marks.at(r) is mark r's item, below n or (at the end) at least n; marks.put(r, prefix) takes
// it; marks.end(total) is called once, by a thread of the last tile.
struct NoMarks {
    static constexpr uint32_t count = 0;
    __device__ __forceinline__ uint64_t at(uint32_t) const { return 0; }
    __device__ __forceinline__ void put(uint32_t, uint64_t) const {}
    __device__ __forceinline__ void end(uint64_t) const {}
};
// Marks up to which the scan takes them: every tile reads all of them, so a thousand (four loads a thread,
// cached) cost less than a launch (4.7 us) and many thousands would not.  16 x 8192 seeds, two hops
// and blocks: 898 -> 887 us; 33 x 700 seeds, three hops: 975 -> 956.
constexpr uint32_t kScanMarksMax = 1024;

template <class Gen, ScanMode MODE, int STRIDE, class Marks>
__global__ __launch_bounds__(kScanBlock) void scan_write_kernel(Gen gen, Count cnt,
                                                                const uint64_t* partials,
                                                                uint64_t* total,
                                                                uint64_t* out, Marks marks) {
    constexpr bool FOLD = MODE != kScanThree;
    constexpr bool MARKS = !std::is_same<Marks, NoMarks>::value;
    __shared__ uint64_t wsum[kScanBlock / kWave];
    __shared__ uint64_t fold_lds[kScanBlock / kWave];
    const uint64_t n = cnt.get();
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
    if (base >= n) {
        if (base == 0 && threadIdx.x == 0) {  // empty sequence
            out[0] = 0;
            if (FOLD && total) *total = 0;
            if (MARKS) marks.end(0);
        }
        if (MARKS && base == 0)
            for (uint32_t r = threadIdx.x; r < marks.count; r += kScanBlock) marks.put(r, 0);
        return;
    }
    uint64_t mark = 0;  // of the first round, asked for early
    if (MARKS && threadIdx.x < marks.count) mark = marks.at(threadIdx.x);
    uint64_t start;
    if (FOLD) {
        uint64_t p = 0;
        if (MODE == kScanDirect) {
#pragma unroll 8
            for (uint64_t k = threadIdx.x; k < base; k += kScanBlock) p += gen(k);
        } else {
            for (uint64_t k = threadIdx.x; k < blockIdx.x; k += kScanBlock) p += partials[k];
        }
        start = block_sum<uint64_t, kScanBlock>(p, fold_lds);
    } else {
        start = partials[blockIdx.x];
    }
    const int lane = lane_id(), wid = threadIdx.x / kWave;
    const uint64_t wb = base + (uint64_t)wid * kWave * kScanItems + lane;
    uint64_t x[kScanItems];
    uint64_t s = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        const uint64_t i = wb + (uint64_t)j * kWave;
        x[j] = i < n ? gen(i) : 0;
        s += x[j];
    }
    const uint64_t st = wave_inclusive_sum_u64(s);
    if (lane == kWave - 1) wsum[wid] = st;
    __syncthreads();
    uint64_t carry = start;
    for (int w = 0; w < wid; ++w) carry += wsum[w];
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        const uint64_t i = wb + (uint64_t)j * kWave;
        const uint64_t inc = wave_inclusive_sum_u64(x[j]);
        if (i < n) out[i * STRIDE] = carry + inc - x[j];
        carry += readlane_u64(inc, kWave - 1);
    }
    if (threadIdx.x == 0 && base + kScanTile >= n) {
        if (FOLD) {
            uint64_t t = start;
            for (int w = 0; w < kScanBlock / kWave; ++w) t += wsum[w];
            out[n * STRIDE] = t;
            if (total) *total = t;
            if (MARKS) marks.end(t);
        } else {
            out[n * STRIDE] = *total;
            if (MARKS) marks.end(*total);
        }
    }
    if (MARKS) {
        __syncthreads();  // the prefixes are read across the workgroup
        const uint64_t next = base + kScanTile;
        for (uint32_t r = threadIdx.x; r < marks.count; r += kScanBlock) {
            if (r >= (uint32_t)kScanBlock) mark = marks.at(r);
            if (mark >= base && mark < next && mark < n) marks.put(r, out[mark * STRIDE]);
            else if (mark >= n && next >= n) marks.put(r, out[n * STRIDE]);
        }
    }
}

inline uint64_t scan_blocks(uint64_t n_max) { return n_max ? (n_max + kScanTile - 1) / kScanTile : 1; }

// Scratch: partials[scan_blocks(n_max)] and total[1].  DIRECT: the most tiles for one launch; 1 for a generator
// that gathers (13 k values by two dependent random loads each: 39 us in one launch, 20 in two).
template <int STRIDE = 1, uint64_t DIRECT = kScanDirectMax, class Gen, class Marks = NoMarks>
hipError_t exclusive_scan(Gen gen, Count cnt, uint64_t n_max, uint64_t* out, uint64_t* partials,
                          uint64_t* total, hipStream_t stream, Marks marks = Marks()) {
    const uint64_t nb = scan_blocks(n_max);
    if (nb <= DIRECT) {
        hipLaunchKernelGGL((scan_write_kernel<Gen, kScanDirect, STRIDE, Marks>), dim3((unsigned)nb), dim3(kScanBlock), 0, stream,
                           gen, cnt, (const uint64_t*)nullptr, total, out, marks);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(scan_reduce_kernel<Gen>, dim3((unsigned)nb), dim3(kScanBlock), 0, stream,
                       gen, cnt, partials);
    if (nb <= kScanFoldMax) {
        hipLaunchKernelGGL((scan_write_kernel<Gen, kScanFold, STRIDE, Marks>), dim3((unsigned)nb), dim3(kScanBlock), 0, stream,
                           gen, cnt, (const uint64_t*)partials, total, out, marks);
    } else {
        hipLaunchKernelGGL(scan_partials_kernel<uint64_t>, dim3(1), dim3(1024), 0, stream, partials, nb, total);
        hipLaunchKernelGGL((scan_write_kernel<Gen, kScanThree, STRIDE, Marks>), dim3((unsigned)nb), dim3(kScanBlock), 0, stream,
                           gen, cnt, (const uint64_t*)partials, total, out, marks);
    }
    return hipGetLastError();
}

// The two halves of a scan whose tiles' prefixes are kept: made once (prefixes[scan_blocks(n)], and the
// total after them), then any number of scans of the same values in one launch each.
template <class Gen>
hipError_t scan_prefixes(Gen gen, uint64_t n, uint64_t* prefixes, hipStream_t stream) {
    const uint64_t nb = scan_blocks(n);
    hipLaunchKernelGGL(scan_reduce_kernel<Gen>, dim3((unsigned)nb), dim3(kScanBlock), 0, stream, gen, Count{n, nullptr}, prefixes);
    hipLaunchKernelGGL(scan_partials_kernel<uint64_t>, dim3(1), dim3(1024), 0, stream, prefixes, nb, prefixes + nb);
    return hipGetLastError();
}
template <class Gen>
hipError_t scan_from_prefixes(Gen gen, uint64_t n, const uint64_t* prefixes, uint64_t* out, hipStream_t stream) {
    const uint64_t nb = scan_blocks(n);
    hipLaunchKernelGGL((scan_write_kernel<Gen, kScanThree, 1, NoMarks>), dim3((unsigned)nb), dim3(kScanBlock), 0, stream, gen,
                       Count{n, nullptr}, prefixes, const_cast<uint64_t*>(prefixes) + nb, out, NoMarks());
    return hipGetLastError();
}

}  // namespace grass
