// Device-side ingest: the R-MAT edge generator and graph_sort on the GPU, with the same results
// as grass_rmat_edges and grass_graph_sort on the host (graph_sort: LE/chunk_compress/
// graph_sort.cpp:22-82), so that R-MAT -> graph_sort -> grass_compress_device runs without the
// graph leaving HBM.
//
// graph_sort:
//   1. first[x] = the first stream position (2i for u, 2i + 1 for v of edge i; self loops skipped)
//      where id x appears -- an atomicMin that reads first, since most ids recur.
//   2. The ids that appear, sorted by first position (rocPRIM radix sort of (first, id) pairs),
//      get new ids 0, 1, ... in that order: the reference's numbering by first appearance.
//   3. Every edge becomes the key (a << nb | b) of its renumbered ends, nb bits each, undirected input
//      the smaller end first (a self loop: ~0, sorted to the end), and the keys are radix-sorted.
//   4. The distinct keys are counted per tile and written at their ranks; the row pointers follow from
//      where each first id's run starts.  Directed: these are the rows.
//   5. Undirected: a row is the ids below its vertex, then those above it.  The distinct keys are the
//      upper parts; sorted once more, by their larger end, they are the lower parts.
// R-MAT s22 (67 M edges): both directions' keys (a << 32 | b) took 1.04 ms to write, 5.5 to sort and 1.45
// to rank and place; half as many over fewer bits take 0.84, 2.4 and 0.53, the second sort 1.3 and
// the rows 0.43.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <rocprim/device/device_radix_sort.hpp>

#include "../../include/grass_ingest.h"
#include "blob.h"
#include "devutil.h"
#include "philox.h"
#include "runtime.h"
#include "scan.h"

namespace grass {
namespace {

constexpr int kIgBlock = 256;
constexpr unsigned kIgGrid = 8192;

// Edge i: level l picks quadrant (0,0)/(0,1)/(1,0)/(1,1) by word l % 4 of
// Philox(seed, {i_lo, i_hi, l / 4, 0x524D4154}) against the thresholds a, a + b, a + b + c (x 2^32).
__global__ __launch_bounds__(kIgBlock) void rmat_kernel(uint32_t scale, uint64_t m, uint64_t tA, uint64_t tAB,
                                                        uint64_t tABC, uint64_t seed, uint32_t* __restrict__ src,
                                                        uint32_t* __restrict__ dst) {
    for (uint64_t i = (uint64_t)blockIdx.x * kIgBlock + threadIdx.x; i < m; i += (uint64_t)gridDim.x * kIgBlock) {
        uint32_t u = 0, v = 0;
        U4 r{0, 0, 0, 0};
        for (uint32_t l = 0; l < scale; ++l) {
            if ((l & 3) == 0) r = philox4x32_10((uint32_t)i, (uint32_t)(i >> 32), l >> 2, 0x524D4154u, seed);
            const uint64_t x = (l & 3) == 0 ? r.x : (l & 3) == 1 ? r.y : (l & 3) == 2 ? r.z : r.w;
            u = (u << 1) | (uint32_t)(x >= tAB);
            v = (v << 1) | (uint32_t)((x >= tA && x < tAB) || x >= tABC);
        }
        src[i] = u;
        dst[i] = v;
    }
}

__global__ __launch_bounds__(kIgBlock) void max_id_kernel(const uint32_t* __restrict__ src,
                                                          const uint32_t* __restrict__ dst, uint64_t m,
                                                          unsigned int* __restrict__ out) {
    __shared__ uint32_t lds[kIgBlock / kWave];
    uint32_t mx = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * kIgBlock + threadIdx.x; i < m; i += (uint64_t)gridDim.x * kIgBlock)
        mx = max(mx, max(src[i], dst[i]));
    mx = block_max<uint32_t, kIgBlock>(mx, lds);
    if (threadIdx.x == 0) atomicMax(out, mx);
}

// Edges a thread takes at a time, kIgBlock apart: their loads are issued before any is used.
constexpr int kIgEdges = 4;
constexpr uint64_t kIgChunk = (uint64_t)kIgBlock * kIgEdges;
constexpr uint64_t kIgPart = 64ull << 10;  // edges of the first part; each part ends at four times the last one's end

// Edges c + e kIgBlock (e < kIgEdges) of a chunk; one past the end reads as a self loop of id 0.
struct EdgeBatch {
    uint32_t u[kIgEdges], v[kIgEdges];
    __device__ __forceinline__ EdgeBatch(const uint32_t* __restrict__ src, const uint32_t* __restrict__ dst, uint64_t c,
                                         uint64_t m) {
#pragma unroll
        for (int e = 0; e < kIgEdges; ++e) {
            const uint64_t i = c + (uint64_t)e * kIgBlock;
            u[e] = i < m ? src[i] : 0u;
            v[e] = i < m ? dst[i] : 0u;
        }
    }
};

// Bound by the lookups of two ids per edge, which for most of an edge list only find that the id has
// appeared before.  So the list goes in parts (kIgPart): after each, `seen` gets one bit per id that has
// appeared, half a megabyte where first[] has sixteen, and an id that a part finds there needs no
// more.  R-MAT s22, 67 M edges, 4.2 M ids: 1.15 ms with first[] looked up for every end, 0.83 with a first
// part of 2 M edges (300 us of it atomics to the same few ids), 0.62 with one of 64 k.
template <typename Pos>
__global__ __launch_bounds__(kIgBlock) void first_pos_kernel(const uint32_t* __restrict__ src,
                                                             const uint32_t* __restrict__ dst, uint64_t m0, uint64_t m,
                                                             const uint32_t* __restrict__ seen, Pos* first) {
    for (uint64_t c = m0 + (uint64_t)blockIdx.x * kIgChunk + threadIdx.x; c < m; c += (uint64_t)gridDim.x * kIgChunk) {
        const EdgeBatch b(src, dst, c, m);
        Pos fu[kIgEdges], fv[kIgEdges];
        uint32_t su[kIgEdges], sv[kIgEdges];
#pragma unroll
        for (int e = 0; e < kIgEdges; ++e) {
            su[e] = seen[b.u[e] >> 5] >> (b.u[e] & 31);
            sv[e] = seen[b.v[e] >> 5] >> (b.v[e] & 31);
        }
#pragma unroll
        for (int e = 0; e < kIgEdges; ++e) {
            fu[e] = su[e] & 1 ? (Pos)0 : __atomic_load_n(&first[b.u[e]], __ATOMIC_RELAXED);
            fv[e] = sv[e] & 1 ? (Pos)0 : __atomic_load_n(&first[b.v[e]], __ATOMIC_RELAXED);
        }
#pragma unroll
        for (int e = 0; e < kIgEdges; ++e) {
            const Pos pos = (Pos)(2 * (c + (uint64_t)e * kIgBlock));
            if (b.u[e] == b.v[e]) continue;
            if (fu[e] > pos) atomicMin(&first[b.u[e]], pos);
            if (fv[e] > pos + 1) atomicMin(&first[b.v[e]], (Pos)(pos + 1));
        }
    }
}

template <typename Pos>
__global__ __launch_bounds__(kIgBlock) void seen_bits_kernel(const Pos* __restrict__ first, uint64_t nid,
                                                             uint32_t* __restrict__ seen) {
    for (uint64_t x0 = (uint64_t)blockIdx.x * kIgBlock; x0 < nid; x0 += (uint64_t)gridDim.x * kIgBlock) {
        const uint64_t x = x0 + threadIdx.x;
        const unsigned long long bits = __ballot(x < nid && first[x] != (Pos)~0ull);
        if ((threadIdx.x & 31) == 0 && x < nid) seen[x >> 5] = (uint32_t)(bits >> (threadIdx.x & 32));
    }
}

template <typename Pos>
struct SeenGen {
    const Pos* first;
    __device__ __forceinline__ uint64_t operator()(uint64_t x) const { return first[x] != (Pos)~0ull; }
};

// The ids that appear, as (first position, id) pairs at their rank among the ids (any order).
template <typename Pos>
__global__ __launch_bounds__(kIgBlock) void seen_kernel(const Pos* __restrict__ first, uint64_t nid,
                                                        const uint64_t* __restrict__ rank, Pos* __restrict__ fkey,
                                                        uint32_t* __restrict__ fid) {
    for (uint64_t x = (uint64_t)blockIdx.x * kIgBlock + threadIdx.x; x < nid; x += (uint64_t)gridDim.x * kIgBlock) {
        const Pos f = first[x];
        if (f == (Pos)~0ull) continue;
        fkey[rank[x]] = f;
        fid[rank[x]] = (uint32_t)x;
    }
}

__global__ __launch_bounds__(kIgBlock) void newid_kernel(const uint32_t* __restrict__ fid, uint64_t n,
                                                         uint32_t* __restrict__ newid) {
    for (uint64_t k = (uint64_t)blockIdx.x * kIgBlock + threadIdx.x; k < n; k += (uint64_t)gridDim.x * kIgBlock)
        newid[fid[k]] = (uint32_t)k;
}

// Keys a << nb | b of the renumbered ends (undirected: the smaller end first), ~0 for a self loop.
__global__ __launch_bounds__(kIgBlock) void edge_keys_kernel(const uint32_t* __restrict__ src,
                                                             const uint32_t* __restrict__ dst, uint64_t m,
                                                             const uint32_t* __restrict__ newid, int directed,
                                                             uint32_t nb, unsigned long long* __restrict__ keys) {
    for (uint64_t c = (uint64_t)blockIdx.x * kIgChunk + threadIdx.x; c < m; c += (uint64_t)gridDim.x * kIgChunk) {
        const EdgeBatch e4(src, dst, c, m);
        uint32_t a[kIgEdges], b[kIgEdges];
#pragma unroll
        for (int e = 0; e < kIgEdges; ++e) {  // (the id of a self loop need not have a new one)
            a[e] = newid[e4.u[e]];
            b[e] = newid[e4.v[e]];
        }
#pragma unroll
        for (int e = 0; e < kIgEdges; ++e) {
            const uint64_t i = c + (uint64_t)e * kIgBlock;
            const bool swap = !directed && a[e] > b[e];
            const uint64_t hi = swap ? b[e] : a[e], lo = swap ? a[e] : b[e];
            if (i < m) keys[i] = e4.u[e] == e4.v[e] ? ~0ull : (hi << nb) | lo;
        }
    }
}

// Distinct keys of a sorted sequence, by waves of kUqWave consecutive ones.
constexpr int kUqRounds = 16, kUqBatch = 8, kUqBlock = 1024;
constexpr uint64_t kUqWave = (uint64_t)kUqRounds * kWave;
constexpr int kUqWaves = kUqBlock / kWave;
constexpr uint64_t kUqTile = kUqWave * kUqWaves;

struct KeyRounds {  // a wave's keys, a round of kWave at a time, kUqBatch rounds loaded together
    const unsigned long long* __restrict__ keys;
    uint64_t P, at;           // the lane's position in the next round to load
    uint64_t i;               // and in the current one
    unsigned long long prev;  // the key before the round's first
    unsigned long long k, kp;
    unsigned long long x[kUqBatch];
    __device__ __forceinline__ KeyRounds(const unsigned long long* p, uint64_t count, uint64_t base)
        : keys(p), P(count), at(base + lane_id()), i(0), k(0), kp(0) {
        prev = base ? keys[base - 1] : 0ull;
    }
    __device__ __forceinline__ void load() {
        i = at;
#pragma unroll
        for (int e = 0; e < kUqBatch; ++e, at += kWave) x[e] = at < P ? keys[at] : ~0ull;
    }
    // To round e of the batch: the key at i (~0 past the end), the one before it; whether it is the
    // first of its value.
    __device__ __forceinline__ bool next(int e) {
        if (e) i += kWave;
        k = x[e];
        kp = ((unsigned long long)dpp_move<0x138>((uint32_t)(k >> 32)) << 32) | dpp_move<0x138>((uint32_t)k);
        if (lane_id() == 0) kp = prev;
        prev = readlane_u64(k, kWave - 1);
        return k != ~0ull && (i == 0 || k != kp);
    }
};

__global__ __launch_bounds__(kUqBlock) void uniq_count_kernel(const unsigned long long* __restrict__ keys, uint64_t P,
                                                              uint32_t* __restrict__ wcount, uint64_t* __restrict__ tcount) {
    __shared__ uint64_t lds[kUqWaves];
    const uint64_t wave = (uint64_t)blockIdx.x * kUqWaves + threadIdx.x / kWave, base = wave * kUqWave;
    uint32_t count = 0;
    if (base < P) {
        KeyRounds r(keys, P, base);
        for (int t = 0; t < kUqRounds; t += kUqBatch) {
            r.load();
#pragma unroll
            for (int e = 0; e < kUqBatch; ++e) count += __popcll(__ballot(r.next(e)));
        }
    }
    if (lane_id() == 0) wcount[wave] = count;
    const uint64_t sum = block_sum<uint64_t, kUqBlock>(lane_id() == 0 ? count : 0u, lds);
    if (threadIdx.x == 0) tcount[blockIdx.x] = sum;
}

// rowptr[b .. a] = at for each lane with `on`: a lane's few by itself, long stretches (ids without
// entries) by the whole wave.
__device__ __forceinline__ void fill_rows(uint64_t* __restrict__ rowptr, bool on, uint32_t b, uint32_t a, uint64_t at) {
    const bool wide = on && a - b >= 16;
    for (unsigned long long w = __ballot(wide); w; w &= w - 1) {
        const int l = __ffsll(w) - 1;
        const uint32_t lo = lane_get(b, l), hi = lane_get(a, l);
        const uint64_t val = lane_get(at, l);
        for (uint32_t x = lo + lane_id(); x <= hi; x += kWave) rowptr[x] = val;
    }
    if (on && !wide)
        for (uint32_t x = b; x <= a; ++x) rowptr[x] = at;
}

// The distinct keys (or, `col`, their low ids) at their ranks, and the row pointers of their high ids: a
// position whose high id exceeds its predecessor's starts rows (predecessor's, its] at its rank.  The
// keys are sorted, so these runs cover the rows up to the last key's once; *tail is the row after it
// (undirected: most late ids have no larger neighbour; one lane filled their rows in 1.2 ms).
__global__ __launch_bounds__(kUqBlock) void uniq_write_kernel(const unsigned long long* __restrict__ keys, uint64_t P,
                                                              const uint32_t* __restrict__ wcount,
                                                              const uint64_t* __restrict__ tprefix, uint32_t nb,
                                                              uint64_t* __restrict__ rowptr,
                                                              uint64_t* __restrict__ tail,
                                                              unsigned long long* __restrict__ out,
                                                              uint32_t* __restrict__ col) {
    const uint32_t w = threadIdx.x / kWave;
    const uint64_t wave = (uint64_t)blockIdx.x * kUqWaves + w, base = wave * kUqWave;
    if (base > P) return;
    const uint32_t before = wave_inclusive_sum(lane_id() < (int)w ? wcount[wave - w + lane_id()] : 0u);
    uint64_t rank = tprefix[blockIdx.x] + lane_get(before, kWave - 1);
    KeyRounds r(keys, P, base);
    for (int t = 0; t < kUqRounds; t += kUqBatch) {
        r.load();
#pragma unroll
        for (int e = 0; e < kUqBatch; ++e) {
            const bool first = r.next(e);
            const unsigned long long lanes = __ballot(first);
            const uint64_t at = rank + lanes_below(lanes);
            rank += __popcll(lanes);
            if (first) {
                if (col) col[at] = (uint32_t)r.k & ((1u << nb) - 1);
                else out[at] = r.k;
            }
            const bool none = r.k == ~0ull, begins = r.i <= P && (r.i == 0 || (none ? r.kp != ~0ull : r.k >> nb != r.kp >> nb));
            const uint32_t b = r.i == 0 ? 0u : (uint32_t)(r.kp >> nb) + 1;
            fill_rows(rowptr, begins && !none, b, (uint32_t)(r.k >> nb), at);
            if (begins && none) *tail = b;
        }
    }
}

__global__ __launch_bounds__(kIgBlock) void rows_tail_kernel(const uint64_t* __restrict__ tail, uint64_t n, uint64_t M,
                                                             uint64_t* __restrict__ rowptr) {
    for (uint64_t x = *tail + (uint64_t)blockIdx.x * kIgBlock + threadIdx.x; x <= n; x += (uint64_t)gridDim.x * kIgBlock)
        rowptr[x] = M;
}

// Undirected: row v holds the ids below v, then those above it.  `up` are the distinct keys (a < b) by
// (a, b) with row starts upptr; `low` the same keys by (b, a).  The lower parts, and where they start:
__global__ __launch_bounds__(kIgBlock) void lower_kernel(const unsigned long long* __restrict__ low, uint64_t M, uint64_t n,
                                                         uint32_t nb, const uint64_t* __restrict__ upptr,
                                                         uint64_t* __restrict__ lowptr, uint32_t* __restrict__ col) {
    const uint32_t mask = (1u << nb) - 1;
    for (uint64_t j0 = (uint64_t)blockIdx.x * kIgBlock; j0 <= M; j0 += (uint64_t)gridDim.x * kIgBlock) {
        const uint64_t j = j0 + threadIdx.x;
        const unsigned long long k = j < M ? low[j] : 0ull;
        const uint32_t b = j < M ? (uint32_t)k & mask : (uint32_t)n;
        const uint32_t pb = j && j <= M ? ((uint32_t)low[j - 1] & mask) + 1 : 0u;
        if (j < M) col[j + upptr[b]] = (uint32_t)(k >> nb);
        fill_rows(lowptr, j <= M && pb <= b, pb, b, j);
    }
}

// and the upper parts; `rowptr` holds upptr and becomes the rows' starts.
__global__ __launch_bounds__(kIgBlock) void upper_kernel(const unsigned long long* __restrict__ up, uint64_t M, uint64_t n,
                                                         uint32_t nb, const uint64_t* __restrict__ lowptr,
                                                         uint64_t* __restrict__ rowptr, uint32_t* __restrict__ col) {
    const uint32_t mask = (1u << nb) - 1;
    const uint64_t t0 = (uint64_t)blockIdx.x * kIgBlock + threadIdx.x, threads = (uint64_t)gridDim.x * kIgBlock;
    for (uint64_t j = t0; j < M; j += threads) {
        const unsigned long long k = up[j];
        col[j + lowptr[(k >> nb) + 1]] = (uint32_t)k & mask;
    }
    for (uint64_t x = t0; x <= n; x += threads) rowptr[x] += lowptr[x];
}

int bits_for(uint64_t x) {  // bits needed to hold x
    int b = 0;
    while (b < 64 && (x >> b)) ++b;
    return b;
}

// 1-2: the new ids by first appearance (stream positions < 2m fit Pos, whose largest value is none).
template <typename Pos>
int number_ids(const uint32_t* src, const uint32_t* dst, uint64_t m, uint64_t nid, uint64_t rowptr_cap, hipStream_t s,
               uint64_t* d_tot, uint64_t* n_out, WorkMem& newid) {
    WorkMem d_first, d_seen, d_rank, d_fkey, d_fid, d_part;
    const uint64_t some = std::max<uint64_t>(nid, 1), words = (some + 31) / 32;
    if (d_first.alloc(some * sizeof(Pos), s) != hipSuccess || d_seen.alloc(words * 4, s) != hipSuccess || d_rank.alloc((nid + 1) * 8, s) != hipSuccess ||
        d_part.alloc((scan_blocks(some) + 2) * 8, s) != hipSuccess)
        return GRASS_ENOMEM;
    Pos* first = d_first.as<Pos>();
    uint64_t* rank = d_rank.as<uint64_t>();
    const unsigned gi = (unsigned)std::min<uint64_t>((nid + kIgBlock - 1) / kIgBlock + 1, kIgGrid);
    uint32_t* seen = d_seen.as<uint32_t>();
    hipLaunchKernelGGL(fill_kernel<Pos>, dim3(gi), dim3(kIgBlock), 0, s, first, nid, (Pos)~0ull);
    hipLaunchKernelGGL(fill_kernel<uint32_t>, dim3(std::min(gi, 1024u)), dim3(kIgBlock), 0, s, seen, words, 0u);
    for (uint64_t m0 = 0; m0 < m;) {
        const uint64_t m1 = std::min(m, std::max(kIgPart, 4 * m0));
        const unsigned gm = (unsigned)std::min<uint64_t>((m1 - m0 + kIgChunk - 1) / kIgChunk, kIgGrid);
        if (m0) hipLaunchKernelGGL(seen_bits_kernel<Pos>, dim3(gi), dim3(kIgBlock), 0, s, (const Pos*)first, nid, seen);
        hipLaunchKernelGGL(first_pos_kernel<Pos>, dim3(gm), dim3(kIgBlock), 0, s, src, dst, m0, m1, (const uint32_t*)seen,
                           first);
        m0 = m1;
    }
    hipError_t e = exclusive_scan(SeenGen<Pos>{first}, Count{nid, nullptr}, nid, rank, d_part.as<uint64_t>(), d_tot, s);
    uint64_t n = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&n, rank + nid, 8, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return status_of(e);
    *n_out = n;
    if (rowptr_cap < n + 1) return GRASS_ECAPACITY;
    if (d_fkey.alloc(std::max<uint64_t>(n, 1) * 2 * sizeof(Pos), s) != hipSuccess ||
        d_fid.alloc(std::max<uint64_t>(n, 1) * 8, s) != hipSuccess || newid.alloc(some * 4, s) != hipSuccess)
        return GRASS_ENOMEM;
    Pos* fk = d_fkey.as<Pos>();
    uint32_t* fid = d_fid.as<uint32_t>();
    hipLaunchKernelGGL(seen_kernel<Pos>, dim3(gi), dim3(kIgBlock), 0, s, (const Pos*)first, nid, (const uint64_t*)rank, fk,
                       fid);
    rocprim::double_buffer<Pos> kb(fk, fk + std::max<uint64_t>(n, 1));
    rocprim::double_buffer<uint32_t> vb(fid, fid + std::max<uint64_t>(n, 1));
    size_t tb = 0;
    const unsigned eb = (unsigned)std::max(1, bits_for(2 * m));
    e = rocprim::radix_sort_pairs(nullptr, tb, kb, vb, (size_t)n, 0u, eb, s);
    WorkMem tmp;
    if (e == hipSuccess && tmp.alloc(tb, s) != hipSuccess) return GRASS_ENOMEM;
    if (e == hipSuccess && n) e = rocprim::radix_sort_pairs(tmp.p, tb, kb, vb, (size_t)n, 0u, eb, s);
    if (e != hipSuccess) return status_of(e);
    const unsigned gn = (unsigned)std::min<uint64_t>((n + kIgBlock - 1) / kIgBlock + 1, kIgGrid);
    if (n)
        hipLaunchKernelGGL(newid_kernel, dim3(gn), dim3(kIgBlock), 0, s, (const uint32_t*)vb.current(), n, newid.as<uint32_t>());
    return status_of(hipGetLastError());
}

int graph_sort_device(const uint32_t* src, const uint32_t* dst, uint64_t m, int directed, hipStream_t s,
                      uint64_t* rowptr, uint64_t rowptr_cap, uint32_t* col, uint64_t col_cap, uint64_t* n_out,
                      uint64_t* m_out) {
    WorkMem small;
    if (small.alloc(64, s) != hipSuccess) return GRASS_ENOMEM;
    unsigned int* d_max = small.as<unsigned int>();
    uint64_t* d_tot = (uint64_t*)(small.as<char>() + 8);
    hipLaunchKernelGGL(fill_kernel<unsigned int>, dim3(1), dim3(64), 0, s, d_max, (uint64_t)1, 0u);
    const unsigned gm = (unsigned)std::min<uint64_t>((m + kIgBlock - 1) / kIgBlock + 1, kIgGrid);
    if (m) hipLaunchKernelGGL(max_id_kernel, dim3(gm), dim3(kIgBlock), 0, s, src, dst, m, d_max);
    unsigned int maxid = 0;
    hipError_t e = hipMemcpyAsync(&maxid, d_max, 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return status_of(e);
    if (maxid >= 0x80000000u) return GRASS_EINVAL;
    const uint64_t nid = m ? (uint64_t)maxid + 1 : 0;
    WorkMem d_newid;
    int rc = m < 0x7FFFFFFFull ? number_ids<unsigned int>(src, dst, m, nid, rowptr_cap, s, d_tot, n_out, d_newid)
                               : number_ids<unsigned long long>(src, dst, m, nid, rowptr_cap, s, d_tot, n_out, d_newid);
    if (rc) return rc;
    const uint64_t n = *n_out;

    // 3: one key per edge (undirected: of its ends in order) over the 2 nb bits it can set; ~0 still
    // sorts last, since the two ends differ
    const uint32_t nb = (uint32_t)std::max(1, bits_for(n ? n - 1 : 0));
    const uint64_t tiles = m / kUqTile + 1;  // of positions 0 .. m
    WorkMem d_keys, d_part;
    if (d_keys.alloc((m + 1) * 16, s) != hipSuccess || d_part.alloc(tiles * (8 + 4 * kUqWaves), s) != hipSuccess)
        return GRASS_ENOMEM;
    unsigned long long* keys = d_keys.as<unsigned long long>();
    uint64_t* tcount = d_part.as<uint64_t>();
    uint32_t* wcount = (uint32_t*)(tcount + tiles);
    if (m)
        hipLaunchKernelGGL(edge_keys_kernel, dim3((unsigned)std::min<uint64_t>((m + kIgChunk - 1) / kIgChunk, kIgGrid)),
                           dim3(kIgBlock), 0, s, src, dst, m, (const uint32_t*)d_newid.as<uint32_t>(), directed, nb, keys);
    rocprim::double_buffer<unsigned long long> kb(keys, keys + m + 1);
    size_t tb = 0;
    e = rocprim::radix_sort_keys(nullptr, tb, kb, (size_t)m, 0u, 2 * nb, s);
    {
        WorkMem tmp;
        if (e == hipSuccess && tmp.alloc(tb, s) != hipSuccess) return GRASS_ENOMEM;
        if (e == hipSuccess && m) e = rocprim::radix_sort_keys(tmp.p, tb, kb, (size_t)m, 0u, 2 * nb, s);
        if (e != hipSuccess) return status_of(e);
    }
    // 4: the distinct ones and their rows
    unsigned long long* sk = kb.current();
    unsigned long long* up = kb.alternate();
    hipLaunchKernelGGL(uniq_count_kernel, dim3((unsigned)tiles), dim3(kUqBlock), 0, s, (const unsigned long long*)sk, m,
                       wcount, tcount);
    hipLaunchKernelGGL(scan_partials_kernel<uint64_t>, dim3(1), dim3(1024), 0, s, tcount, tiles, d_tot);
    uint64_t M = 0;
    e = hipMemcpyAsync(&M, d_tot, 8, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return status_of(e);
    const uint64_t M_out = directed ? M : 2 * M;
    *m_out = M_out;
    if (col_cap < M_out || (M_out && !col)) return GRASS_ECAPACITY;
    hipLaunchKernelGGL(uniq_write_kernel, dim3((unsigned)tiles), dim3(kUqBlock), 0, s, (const unsigned long long*)sk, m,
                       (const uint32_t*)wcount, (const uint64_t*)tcount, nb, rowptr, d_tot + 1, up,
                       directed ? col : (uint32_t*)nullptr);
    hipLaunchKernelGGL(rows_tail_kernel, dim3((unsigned)std::min<uint64_t>(n / kIgBlock + 1, 1024)), dim3(kIgBlock), 0, s,
                       (const uint64_t*)(d_tot + 1), n, M, rowptr);
    if (!directed) {
        // 5: the same edges by their larger end (a stable sort over its bits)
        WorkMem d_low, tmp;
        if (d_low.alloc((n + 1) * 8, s) != hipSuccess) return GRASS_ENOMEM;
        e = rocprim::radix_sort_keys(nullptr, tb, (const unsigned long long*)up, sk, (size_t)M, 0u, nb, s);
        if (e == hipSuccess && tmp.alloc(tb, s) != hipSuccess) return GRASS_ENOMEM;
        if (e == hipSuccess && M)
            e = rocprim::radix_sort_keys(tmp.p, tb, (const unsigned long long*)up, sk, (size_t)M, 0u, nb, s);
        if (e != hipSuccess) return status_of(e);
        const unsigned gp = (unsigned)std::min<uint64_t>(std::max(M, n) / kIgBlock + 1, kIgGrid);
        hipLaunchKernelGGL(lower_kernel, dim3(gp), dim3(kIgBlock), 0, s, (const unsigned long long*)sk, M, n, nb,
                           (const uint64_t*)rowptr, d_low.as<uint64_t>(), col);
        hipLaunchKernelGGL(upper_kernel, dim3(gp), dim3(kIgBlock), 0, s, (const unsigned long long*)up, M, n, nb,
                           (const uint64_t*)d_low.as<uint64_t>(), rowptr, col);
        e = hipGetLastError();
        const hipError_t done = hipStreamSynchronize(s);
        return status_of(e == hipSuccess ? done : e);
    }
    e = hipGetLastError();
    const hipError_t done = hipStreamSynchronize(s);
    return status_of(e == hipSuccess ? done : e);
}

}  // namespace
}  // namespace grass

extern "C" {

int grass_rmat_edges_device(uint32_t scale, uint32_t edge_factor, double a, double b, double c, uint64_t seed,
                            int device, void* stream, uint32_t* src_dev, uint32_t* dst_dev) {
    if (scale == 0 || scale > 31 || edge_factor == 0 || !src_dev || !dst_dev) return GRASS_EINVAL;
    if (a < 0 || b < 0 || c < 0 || a + b + c > 1.0) return GRASS_EINVAL;
    const uint64_t m = (uint64_t)edge_factor << scale;
    const double two32 = 4294967296.0;
    const uint64_t tA = (uint64_t)(a * two32), tAB = (uint64_t)((a + b) * two32),
                   tABC = (uint64_t)((a + b + c) * two32);
    int prev = 0;
    (void)hipGetDevice(&prev);
    if (!grass::enter_device(device)) return GRASS_EDEVICE;
    const unsigned grid = (unsigned)std::min<uint64_t>((m + grass::kIgBlock - 1) / grass::kIgBlock, grass::kIgGrid);
    hipLaunchKernelGGL(grass::rmat_kernel, dim3(grid), dim3(grass::kIgBlock), 0, (hipStream_t)stream, scale, m, tA,
                       tAB, tABC, seed, src_dev, dst_dev);
    const int rc = grass::status_of(hipGetLastError());
    (void)hipSetDevice(prev);
    return rc;
}

int grass_graph_sort_device(const uint32_t* src_dev, const uint32_t* dst_dev, uint64_t m, int directed, int device,
                            void* stream, uint64_t* rowptr_dev, uint64_t rowptr_capacity, uint32_t* col_dev,
                            uint64_t col_capacity, uint64_t* n, uint64_t* m_out) {
    if (!n || !m_out || !rowptr_dev || (m && (!src_dev || !dst_dev)) || m >= (1ull << 34)) return GRASS_EINVAL;
    *n = *m_out = 0;
    int prev = 0;
    (void)hipGetDevice(&prev);
    if (!grass::enter_device(device)) return GRASS_EDEVICE;
    const int rc = grass::graph_sort_device(src_dev, dst_dev, m, directed, (hipStream_t)stream, rowptr_dev,
                                            rowptr_capacity, col_dev, col_capacity, n, m_out);
    (void)hipSetDevice(prev);
    return rc;
}

int grass_compress_on_device(const grass_csr* csr, int format, int device, grass_blob** graph, grass_blob** offset) {
    if (!csr || !graph || !offset || csr->n == 0) return GRASS_EINVAL;
    int prev = 0;
    (void)hipGetDevice(&prev);
    if (!grass::enter_device(device)) return GRASS_EDEVICE;
    int rc = GRASS_OK;
    {
        grass::WorkMem rp, cl;
        if (rp.alloc((csr->n + 1) * 8, nullptr) != hipSuccess || cl.alloc(std::max<uint64_t>(csr->m, 1) * 4, nullptr) != hipSuccess)
            rc = GRASS_ENOMEM;
        hipError_t e = hipSuccess;
        if (!rc) e = hipMemcpy(rp.p, csr->rowptr.data(), (csr->n + 1) * 8, hipMemcpyHostToDevice);
        if (!rc && e == hipSuccess && csr->m) e = hipMemcpy(cl.p, csr->col.data(), csr->m * 4, hipMemcpyHostToDevice);
        if (!rc && e != hipSuccess) rc = grass::status_of(e);
        if (!rc)
            rc = grass_compress_device(rp.as<uint64_t>(), cl.as<uint32_t>(), csr->n, format, device, nullptr, graph,
                                       offset);
    }
    (void)hipSetDevice(prev);
    return rc;
}

int grass_graph_sort_on_device(const uint32_t* src, const uint32_t* dst, uint64_t m, int directed, int device,
                               grass_csr** out) {
    if (!out || (m && (!src || !dst)) || m >= (1ull << 34)) return GRASS_EINVAL;
    *out = nullptr;
    uint32_t maxid = 0;
    for (uint64_t i = 0; i < m; ++i) maxid = std::max(maxid, std::max(src[i], dst[i]));
    if (maxid >= 0x80000000u) return GRASS_EINVAL;
    const uint64_t rcap = (uint64_t)maxid + 2, ccap = std::max<uint64_t>(directed ? m : 2 * m, 1);
    int prev = 0;
    (void)hipGetDevice(&prev);
    if (!grass::enter_device(device)) return GRASS_EDEVICE;
    int rc = GRASS_OK;
    grass_csr* csr = new (std::nothrow) grass_csr();
    if (!csr) rc = GRASS_ENOMEM;
    {
        grass::WorkMem ds, dd, rp, cl;
        if (!rc && (ds.alloc(std::max<uint64_t>(m, 1) * 4, nullptr) != hipSuccess ||
                    dd.alloc(std::max<uint64_t>(m, 1) * 4, nullptr) != hipSuccess || rp.alloc(rcap * 8, nullptr) != hipSuccess ||
                    cl.alloc(ccap * 4, nullptr) != hipSuccess))
            rc = GRASS_ENOMEM;
        hipError_t e = hipSuccess;
        if (!rc && m) e = hipMemcpy(ds.p, src, m * 4, hipMemcpyHostToDevice);
        if (!rc && m && e == hipSuccess) e = hipMemcpy(dd.p, dst, m * 4, hipMemcpyHostToDevice);
        if (!rc && e != hipSuccess) rc = grass::status_of(e);
        uint64_t n = 0, mo = 0;
        if (!rc)
            rc = grass_graph_sort_device(ds.as<uint32_t>(), dd.as<uint32_t>(), m, directed, device, nullptr,
                                         rp.as<uint64_t>(), rcap, cl.as<uint32_t>(), ccap, &n, &mo);
        if (!rc) {
            try {
                csr->n = n;
                csr->m = mo;
                csr->rowptr.resize(n + 1);
                csr->col.resize(mo);
            } catch (const std::bad_alloc&) {
                rc = GRASS_ENOMEM;
            }
        }
        if (!rc) e = hipMemcpy(csr->rowptr.data(), rp.p, (n + 1) * 8, hipMemcpyDeviceToHost);
        if (!rc && e == hipSuccess && mo) e = hipMemcpy(csr->col.data(), cl.p, mo * 4, hipMemcpyDeviceToHost);
        if (!rc && e != hipSuccess) rc = grass::status_of(e);
    }
    (void)hipSetDevice(prev);
    if (rc) {
        delete csr;
        return rc;
    }
    *out = csr;
    return GRASS_OK;
}

}  // extern "C"
