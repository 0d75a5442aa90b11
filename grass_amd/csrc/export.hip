// Sample export: k-hop mini-batch blocks (per-request local numbering), local ids of MDRW
// samples, and DLPack hand-over of MDRW results.
//
// k-hop blocks.  Request r's sequence is its seeds, then its hop-0 destinations, its hop-1
// destinations, ...; the sequences of all requests are laid end to end (request-major, starts
// Q[r]) so that one position space covers the batch.
//   1. rel_prepare_kernel (or, for very many requests, a few kernels and a scan): checks the batch's
//      offsets and fills Q, while other workgroups clear the table.
//   2. rel_insert_kernel: every position p inserts the key (r, vertex) into a hash table that keeps
//      the key's smallest position, and p stays on the list of first appearances (firsts.h) or takes
//      a larger one off it.  A scan of the list's words numbers the first appearances: the local id
//      of the vertex whose first position is f is rank(f) - rank(Q[r]).
//   3. rel_emit_kernel: writes each first appearance to nodes[rank(p)] and the local ids of every
//      batch edge (its destination is a position, its source a key looked up in the table).
// Every step is a data-parallel pass over the positions; the result does not depend on timing.
// A batch of few positions is one launch of one workgroup (rel_small_kernel).  A larger one is bound by
// the random atomics of the inserts, which the chip takes at 22 to 27 G/s whatever the table's size
// (a load of a slot and a CAS on it: 25.7 G/s), so a position touches the table once: 16 x 8192 seeds
// [25, 10] on R-MAT s24, 10.7 M positions, insert 435 us; a second pass that looked every key up again
// took 196 us more.  A large one therefore makes step 2 by partition (rel_part_*): 221 us with all its
// passes.  The emit, by lookups of the sources and loads a word ahead, is 150 us (229 without either).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <new>

#include "../../include/grass_export.h"
#include "devutil.h"
#include "firsts.h"
#include "runtime.h"
#include "scan.h"

namespace grass {
namespace {

constexpr int kExBlock = 256;
constexpr unsigned kExGrid = 4096;
constexpr uint32_t kNoId = 0xFFFFFFFFu;  // local id of a vertex that is not in the sample

struct RelReq {
    const uint32_t* seeds;
    uint64_t num;
    uint32_t hops;
};

// Open-addressing tables from (request r, vertex v) to the first position of v in r's sequence.
// Both have the same interface; the kernels below take either.  Linear probing from a
// multiplicative hash; a slot, once it holds a key, keeps it, and its position only decreases, so
// every slot ends at the minimum position whatever the order of the inserts.

// 16 bytes per slot: {key, first position}, key = ((r << 32) | v) + 1, key 0 = empty.  Takes any
// request count, vertex id and position; two atomics per new key (claim, then position).
struct RelTab16 {
    unsigned long long* slot;  // 2 * (mask + 1) words
    uint64_t mask;
    uint32_t shift;
    __device__ __forceinline__ static unsigned long long key(uint32_t r, uint32_t v) {
        return (((unsigned long long)r << 32) | v) + 1;
    }
    __device__ __forceinline__ unsigned long long* kp(uint64_t h) const { return slot + 2 * h; }
    __device__ __forceinline__ uint64_t home(unsigned long long k) const {
        return ((k * 0x9E3779B97F4A7C15ull) >> shift) & mask;
    }
    __device__ __forceinline__ void clear(uint64_t i) const {
        reinterpret_cast<ulonglong2*>(slot)[i] = make_ulonglong2(0ull, ~0ull);
    }
    // Whether p is its key's smallest position so far; the position it displaces is taken off `words`.
    __device__ __forceinline__ bool insert(uint32_t r, uint32_t v, uint64_t p, FirstWord* words, uint32_t* err) const {
        const unsigned long long k = key(r, v);
        uint64_t h = home(k);
        for (uint64_t probes = 0; probes <= mask; ++probes) {
            unsigned long long cur = __atomic_load_n(kp(h), __ATOMIC_RELAXED);
            if (cur == 0) {
                cur = atomicCAS(kp(h), 0ull, k);
                if (cur == 0) cur = k;
            }
            if (cur == k) {
                // read first: a repeat after the first occurrence needs no atomic
                if (__atomic_load_n(kp(h) + 1, __ATOMIC_RELAXED) < p) return false;
                const unsigned long long old = atomicMin(kp(h) + 1, (unsigned long long)p);
                if (old < p) return false;
                if (old != ~0ull) not_first(words, old);
                return true;
            }
            h = (h + 1) & mask;
        }
        atomicOr(err, 1u);  // cannot happen: slots > positions
        return false;
    }
    // First position of v in request r, where hint(p) was loaded for a position p that holds it.
    __device__ __forceinline__ uint32_t hint(uint64_t) const { return 0; }
    __device__ __forceinline__ uint64_t first_of(uint32_t, uint32_t r, uint32_t v) const { return first(r, v); }
    // First position of v in request r; ~0 when absent.
    __device__ __forceinline__ uint64_t first(uint32_t r, uint32_t v) const {
        const unsigned long long k = key(r, v);
        uint64_t h = home(k);
        for (uint64_t probes = 0; probes <= mask; ++probes) {
            const ulonglong2 kv = *(const ulonglong2*)kp(h);
            if (kv.x == k) return kv.y;
            if (kv.x == 0) break;
            h = (h + 1) & mask;
        }
        return ~0ull;
    }
};

// 8 bytes per slot when the request, the vertex and the position fit in one word:
// word = (((r << vb) | v) << pb) | position, all ones = empty (positions < 2^pb - 1 keep the low
// bits from being all ones).  A CAS claims an empty slot with the key and the position at once, and
// atomicMin on a word of the same key lowers only its position bits: one atomic per new key.
struct RelTab8 {
    unsigned long long* slot;  // mask + 1 words
    uint64_t mask;
    uint32_t shift, vb, pb;
    __device__ __forceinline__ uint64_t home(unsigned long long k) const {
        return (((k + 1) * 0x9E3779B97F4A7C15ull) >> shift) & mask;
    }
    __device__ __forceinline__ void clear(uint64_t i) const { slot[i] = ~0ull; }
    __device__ __forceinline__ bool insert(uint32_t r, uint32_t v, uint64_t p, FirstWord* words, uint32_t* err) const {
        if (vb < 32 && (v >> vb) != 0) {  // not a vertex of the graph
            atomicOr(err, 1u);
            return false;
        }
        const unsigned long long k = ((unsigned long long)r << vb) | v;
        const unsigned long long w = (k << pb) | p;
        uint64_t h = home(k);
        for (uint64_t probes = 0; probes <= mask; ++probes) {
            unsigned long long cur = __atomic_load_n(slot + h, __ATOMIC_RELAXED);
            if (cur == ~0ull) {
                cur = atomicCAS(slot + h, ~0ull, w);
                if (cur == ~0ull) return true;
            }
            if ((cur >> pb) == k) {
                if (cur < w) return false;
                const unsigned long long old = atomicMin(slot + h, w);
                if (old < w) return false;
                not_first(words, old & ((1ull << pb) - 1));
                return true;
            }
            h = (h + 1) & mask;
        }
        atomicOr(err, 1u);  // cannot happen: slots > positions
        return false;
    }
    __device__ __forceinline__ uint32_t hint(uint64_t) const { return 0; }
    __device__ __forceinline__ uint64_t first_of(uint32_t, uint32_t r, uint32_t v) const { return first(r, v); }
    __device__ __forceinline__ uint64_t first(uint32_t r, uint32_t v) const {
        if (vb < 32 && (v >> vb) != 0) return ~0ull;
        const unsigned long long k = ((unsigned long long)r << vb) | v;
        uint64_t h = home(k);
        for (uint64_t probes = 0; probes <= mask; ++probes) {
            const unsigned long long cur = slot[h];
            if (cur == ~0ull) break;
            if ((cur >> pb) == k) return cur & ((1ull << pb) - 1);
            h = (h + 1) & mask;
        }
        return ~0ull;
    }
};

// The batch as one position space.  Every offset row has been checked (rel_check_kernel) to be
// ascending and to end at or below the batch total before any pass reads through it, so every
// edge index e below is < total.
struct RelSeq {
    const RelReq* req;
    const uint64_t* off;  // batch offsets, hop-major [H][R + 1]
    const uint32_t* src;
    const uint32_t* dst;
    const uint64_t* Q;  // R + 1 request starts
    uint32_t R, H;
    uint32_t n;  // vertices of the graph: an id >= n is not a vertex
    // Vertex at position p of request r; e = its batch edge (~0 for a seed).
    __device__ __forceinline__ uint32_t at(uint64_t p, uint32_t r, uint64_t& e) const {
        uint64_t j = p - Q[r];
        const RelReq q = req[r];
        e = ~0ull;
        if (j < q.num) return q.seeds[j];
        j -= q.num;
        for (uint32_t h = 0; h < H; ++h) {
            const uint64_t e0 = off[(uint64_t)h * (R + 1) + r];
            const uint64_t c = off[(uint64_t)h * (R + 1) + r + 1] - e0;
            if (j < c) {
                e = e0 + j;
                return dst[e];
            }
            j -= c;
        }
        return n;  // past the request's edges (the checks reject such offsets first)
    }
};

// Checks the batch offsets against the requests before any pass reads through them: every row
// ascending and ending at or below `total`, no edges of request r at hops >= its hop count, and
// the sequence lengths summing to P.  Any failure sets *invalid, and the passes then touch
// nothing.
__device__ __forceinline__ bool rel_check(const uint64_t* __restrict__ off, const RelReq* __restrict__ req, uint32_t R,
                                          uint32_t H, uint64_t total, uint64_t t, uint64_t threads) {
    const uint64_t cells = (uint64_t)H * (R + 1);
    bool ok = true;
    for (uint64_t i = t; i < cells; i += threads) {
        const uint32_t h = (uint32_t)(i / (R + 1)), r = (uint32_t)(i % (R + 1));
        const uint64_t a = off[i];
        ok = ok && a <= total;
        if (r < R) {
            const uint64_t b = off[i + 1];
            ok = ok && a <= b && (h < req[r].hops || a == b);
        }
    }
    return ok;
}

// Length of request r's sequence: its seeds and its edges at every hop (only after the check).
__device__ __forceinline__ uint64_t rel_length(const RelReq* __restrict__ req, const uint64_t* __restrict__ off,
                                               uint32_t R, uint32_t H, uint32_t r) {
    uint64_t L = req[r].num;
    for (uint32_t h = 0; h < H; ++h) L += off[(uint64_t)h * (R + 1) + r + 1] - off[(uint64_t)h * (R + 1) + r];
    return L;
}

__global__ void rel_check_kernel(const uint64_t* __restrict__ off, const RelReq* __restrict__ req,
                                 uint32_t R, uint32_t H, uint64_t total, uint32_t* invalid) {
    if (!rel_check(off, req, R, H, total, (uint64_t)blockIdx.x * blockDim.x + threadIdx.x,
                   (uint64_t)gridDim.x * blockDim.x))
        atomicOr(invalid, 1u);
}

__global__ void rel_len_kernel(const RelReq* __restrict__ req, const uint64_t* __restrict__ off, uint32_t R,
                               uint32_t H, const uint32_t* __restrict__ invalid, uint64_t* __restrict__ len) {
    const uint32_t hops = *invalid ? 0 : H;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < R; r += gridDim.x * blockDim.x)
        len[r] = rel_length(req, off, R, hops, r);
}

// The sequence total must be the seeds plus the batch's edges: rows of different hops that
// overlap would make it larger.
__global__ void rel_total_kernel(const uint64_t* __restrict__ Q, uint32_t R, uint64_t P, uint32_t* invalid) {
    if (blockIdx.x == 0 && threadIdx.x == 0 && Q[R] != P) atomicOr(invalid, 1u);
}

struct LenGen {
    const uint64_t* len;
    __device__ __forceinline__ uint64_t operator()(uint64_t i) const { return len[i]; }
};

// The table's slots emptied and every position a first appearance.
template <class Tab>
__device__ __forceinline__ void rel_clear(const Tab& t, FirstWord* words, uint64_t nwords, uint64_t i0, uint64_t threads) {
    for (uint64_t i = i0; i < nwords; i += threads) words[i] = make_ulonglong2(~0ull, 0ull);
    for (uint64_t i = i0; i <= t.mask; i += threads) t.clear(i);
}

template <class Tab>
__global__ __launch_bounds__(1024) void rel_clear_kernel(Tab t, FirstWord* words, uint64_t nwords) {
    rel_clear(t, words, nwords, (uint64_t)blockIdx.x * 1024 + threadIdx.x, (uint64_t)gridDim.x * 1024);
}

constexpr uint32_t kPrepRequests = 8192;

// Partitions (rel_part_*): a request's sequence is cut into tiles of kPartTile positions, and its keys go
// by their hash into buckets of about kPartKeys, whose distinct ones fit a table of kPartSlots.
constexpr uint32_t kPartTile = 8192, kPartKeys = 2560, kPartSlots = 4096, kPartBuckets = 8192;
__host__ __device__ inline uint32_t part_buckets(uint64_t len) {
    const uint64_t b = (len + kPartKeys - 1) / kPartKeys;
    return (uint32_t)(b < kPartBuckets ? b : kPartBuckets);
}

// One workgroup of 1024: the offsets' check, the requests' starts Q, their total's check; tile0 and bkt0
// (or null): their first tiles and buckets.
__device__ __forceinline__ void rel_starts(const uint64_t* __restrict__ off, const RelReq* __restrict__ req, uint32_t R,
                                           uint32_t H, uint64_t total, uint64_t P, uint64_t* __restrict__ Q,
                                           uint32_t* __restrict__ tile0, uint32_t* __restrict__ bkt0, uint32_t* bad,
                                           uint32_t* invalid) {
    __shared__ uint64_t lds[1024 / kWave];
    const bool mine = H == 0 || rel_check(off, req, R, H, total, threadIdx.x, 1024);
    const bool ok = block_sum<uint64_t, 1024>(mine ? 0 : 1, lds) == 0;
    constexpr uint32_t kPer = kPrepRequests / 1024;
    const uint32_t per = (R + 1023) / 1024, r0 = threadIdx.x * per;
    uint64_t len[kPer], s = 0, parts = 0;  // parts: tiles << 32 | buckets
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        len[i] = i < per && r0 + i < R ? rel_length(req, off, R, ok ? H : 0, r0 + i) : 0;
        s += len[i];
        parts += ((len[i] + kPartTile - 1) / kPartTile << 32) | part_buckets(len[i]);
    }
    uint64_t sum, all = 0;
    uint64_t pre = block_exclusive_sum<uint64_t, 1024>(s, sum, lds);
    if (tile0) parts = block_exclusive_sum<uint64_t, 1024>(parts, all, lds);
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        if (i < per && r0 + i < R) {
            Q[r0 + i] = pre;
            if (tile0) {
                tile0[r0 + i] = (uint32_t)(parts >> 32);
                bkt0[r0 + i] = (uint32_t)parts;
            }
        }
        pre += len[i];
        parts += ((len[i] + kPartTile - 1) / kPartTile << 32) | part_buckets(len[i]);
    }
    if (threadIdx.x == 0) {
        Q[R] = sum;
        *bad = 0;
        const bool fits = ok && sum == P;
        *invalid = fits ? 0 : 1;
        if (tile0) {
            tile0[R] = fits ? (uint32_t)(all >> 32) : 0u;
            bkt0[R] = fits ? (uint32_t)all : 0u;
        }
    }
}

// Up to kPrepRequests requests: workgroup 0 checks the offsets, scans the lengths into Q and checks their
// total, while the others clear the table (with one workgroup, it does both): one launch where the
// steps by themselves are seven.
template <class Tab>
__global__ __launch_bounds__(1024) void rel_prepare_kernel(Tab t, FirstWord* words, uint64_t nwords,
                                                           const uint64_t* __restrict__ off,
                                                           const RelReq* __restrict__ req, uint32_t R, uint32_t H,
                                                           uint64_t total, uint64_t P, uint64_t* __restrict__ Q,
                                                           uint32_t* bad, uint32_t* invalid) {
    if (blockIdx.x || gridDim.x == 1)
        rel_clear(t, words, nwords, (uint64_t)(gridDim.x == 1 ? 0 : blockIdx.x - 1) * 1024 + threadIdx.x,
                  (uint64_t)(gridDim.x == 1 ? 1 : gridDim.x - 1) * 1024);
    if (blockIdx.x) return;
    rel_starts(off, req, R, H, total, P, Q, nullptr, nullptr, bad, invalid);
}

// Where a wave that goes through consecutive words is: the stretch of positions (a request's seeds,
// or its edges of one hop) it found last, whose vertices follow each other in one array.
struct RelCursor {
    uint64_t beg = 1, end = 0;  // positions of the stretch
    uint32_t r = 0;             // its request
    uint64_t e0 = 0;            // its first batch edge, ~0 for seeds
    const uint32_t* arr = nullptr;
    __device__ __forceinline__ void find(const RelSeq& q, uint64_t p) {
        r = segment_in(q.Q, 0, q.R - 1, p);
        const RelReq k = q.req[r];
        beg = q.Q[r];
        end = beg + k.num;
        arr = k.seeds;
        e0 = ~0ull;
        for (uint32_t h = 0; h < q.H && p >= end; ++h) {
            e0 = q.off[(uint64_t)h * (q.R + 1) + r];
            beg = end;
            end += q.off[(uint64_t)h * (q.R + 1) + r + 1] - e0;
            arr = q.dst + e0;
        }
    }
    // The vertex, request and batch edge (~0 for a seed) at the lane's position p <= last of word w.
    __device__ __forceinline__ uint32_t at(const RelSeq& q, uint64_t w, uint64_t p, uint64_t last, uint32_t& rr, uint64_t& e) {
        const uint64_t p0 = w * kWave;
        if (p0 < beg || p0 >= end) find(q, p0);
        if (last < end) {  // the whole word
            rr = r;
            e = e0 == ~0ull ? ~0ull : e0 + (p - beg);
            return arr[p - beg];
        }
        rr = segment_in(q.Q, r, q.R - 1, p);
        return q.at(p, rr, e);
    }
};

// One wave per 64 positions (a word of `words`).
template <class Tab>
__global__ __launch_bounds__(kExBlock) void rel_insert_kernel(RelSeq q, uint64_t P, Tab t, FirstWord* words,
                                                              const uint32_t* __restrict__ invalid, uint32_t* err) {
    if (*invalid) return;
    const WordChunk wc = wave_words<kExBlock>(P);
    RelCursor cur;
    for (uint64_t w = wc.w; w < wc.end; ++w) {
        const uint64_t p = w * kWave + lane_id(), last = min(w * kWave + kWave - 1, P - 1);
        uint32_t r;
        uint64_t e;
        const uint32_t v = cur.at(q, w, min(p, last), last, r, e);
        bool first = false;
        if (p < P) {
            if (v < q.n) first = t.insert(r, v, p, words, err);
            else atomicOr(err, 1u);  // a seed or destination that is not a vertex of the graph
        }
        const unsigned long long keep = __ballot(first);
        if (lane_id() == 0 && keep != ~0ull) atomicAnd(&words[w].x, keep);
    }
}

template <class Tab>
__global__ __launch_bounds__(kExBlock) void rel_emit_kernel(RelSeq q, uint64_t P, Tab t,
                                                            const FirstWord* __restrict__ words,
                                                            const uint64_t* __restrict__ node_off,
                                                            uint32_t* __restrict__ nodes, uint64_t cap,
                                                            uint32_t* __restrict__ lsrc, uint32_t* __restrict__ ldst,
                                                            const uint32_t* __restrict__ invalid, uint32_t* err) {
    if (*invalid) return;
    const WordChunk wc = wave_words<kExBlock>(P);
    RelCursor cur;
    // what a word's positions need that no lookup tells, loaded a word ahead
    struct Item {
        FirstWord fw;
        uint64_t e;  // ~0: a seed, or past the end
        uint32_t v, r, src, hint;
    };
    auto fetch = [&](uint64_t w) {
        Item it;
        it.fw = words[w];
        const uint64_t p = w * kWave + lane_id(), last = min(w * kWave + kWave - 1, P - 1);
        it.v = cur.at(q, w, min(p, last), last, it.r, it.e);
        if (p >= P) it.e = ~0ull;
        it.src = it.e != ~0ull ? q.src[it.e] : 0u;
        it.hint = t.hint(min(p, last));
        return it;
    };
    if (wc.w >= wc.end) return;
    Item next = fetch(wc.w);
    for (uint64_t w = wc.w; w < wc.end; ++w) {
        const Item it = next;
        if (w + 1 < wc.end) next = fetch(w + 1);
        const uint64_t p = w * kWave + lane_id();
        const bool first = (it.fw.x >> lane_id()) & 1;  // (not past the end)
        const uint64_t mine = it.fw.y + lanes_below(it.fw.x);
        if (first && mine < cap) nodes[mine] = it.v;
        if (it.e == ~0ull) continue;
        const uint64_t base = node_off[it.r];
        const uint64_t fd = first ? p : it.v < q.n ? t.first_of(it.hint, it.r, it.v) : ~0ull;
        const uint64_t fs = t.first(it.r, it.src);
        if (fd >= P || fs >= P) {  // a source that is neither a seed nor an earlier destination
            atomicOr(err, 1u);
            ldst[it.e] = lsrc[it.e] = kNoId;
            continue;
        }
        ldst[it.e] = (uint32_t)((first ? mine : first_rank(words, fd)) - base);
        lsrc[it.e] = (uint32_t)(first_rank(words, fs) - base);
    }
}

// The first appearances numbered, then the sampled vertices and the local ids of every edge.
template <class Tab>
hipError_t rel_number(const Tab& t, const RelSeq& q, uint64_t P, FirstWord* d_words, uint64_t* d_part, uint64_t* d_sc,
                      uint32_t* d_bad, grass_khop_blocks* out, hipStream_t s) {
    // node_off[r] = first appearances before request r; their total beside the other results
    hipError_t e = scan_firsts(d_words, Count{P, nullptr}, P, q.Q, q.R, out->node_off_dev, d_sc + 1, d_part, d_sc, s);
    if (e != hipSuccess || !P) return e;
    const unsigned gP = (unsigned)std::min<uint64_t>((P + kExBlock - 1) / kExBlock + 1, kExGrid);
    hipLaunchKernelGGL(rel_emit_kernel<Tab>, dim3(gP), dim3(kExBlock), 0, s, q, P, t, (const FirstWord*)d_words,
                       (const uint64_t*)out->node_off_dev, out->nodes_dev, out->node_capacity, out->lsrc_dev,
                       out->ldst_dev, (const uint32_t*)(d_bad + 1), d_bad);
    return hipGetLastError();
}

// Fills Q and clears the table, inserts every position, numbers the first appearances (scan) and
// writes the sampled vertices and the local ids of every edge.
template <class Tab>
hipError_t rel_build(const Tab& t, const RelSeq& q, uint64_t P, uint64_t* d_len, FirstWord* d_words, uint64_t* d_part,
                     uint64_t* d_sc, uint32_t* d_bad, const grass_khop_output* b, grass_khop_blocks* out,
                     hipStream_t s) {
    uint32_t* d_invalid = d_bad + 1;
    uint64_t* Q = const_cast<uint64_t*>(q.Q);
    const uint64_t nwords = firsts_words(P);
    const unsigned gC = 1 + (unsigned)std::min<uint64_t>((t.mask + 1) / 2048, 2048);
    if (q.R <= kPrepRequests) {
        hipLaunchKernelGGL(rel_prepare_kernel<Tab>, dim3(gC), dim3(1024), 0, s, t, d_words, nwords, q.off, q.req, q.R,
                           q.H, b->total, P, Q, d_bad, d_invalid);
    } else {
        hipLaunchKernelGGL(fill_kernel<uint32_t>, dim3(1), dim3(64), 0, s, d_bad, (uint64_t)2, 0u);
        const unsigned gR = (unsigned)std::min<uint64_t>((q.R + 255) / 256 + 1, 1024);
        if (q.H) hipLaunchKernelGGL(rel_check_kernel, dim3(1024), dim3(256), 0, s, q.off, q.req, q.R, q.H, b->total, d_invalid);
        hipLaunchKernelGGL(rel_len_kernel, dim3(gR), dim3(256), 0, s, q.req, q.off, q.R, q.H, (const uint32_t*)d_invalid,
                           d_len);
        hipError_t e = exclusive_scan(LenGen{d_len}, Count{q.R, nullptr}, q.R, Q, d_part, d_sc, s);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(rel_total_kernel, dim3(1), dim3(64), 0, s, q.Q, q.R, P, d_invalid);
        hipLaunchKernelGGL(rel_clear_kernel<Tab>, dim3(gC), dim3(1024), 0, s, t, d_words, nwords);
    }
    const unsigned gP = (unsigned)std::min<uint64_t>((P + kExBlock - 1) / kExBlock + 1, kExGrid);
    if (P)
        hipLaunchKernelGGL(rel_insert_kernel<Tab>, dim3(gP), dim3(kExBlock), 0, s, q, P, t, d_words,
                           (const uint32_t*)d_invalid, d_bad);
    return rel_number(t, q, P, d_words, d_part, d_sc, d_bad, out, s);
}

// ------------------------------------------------------------------ blocks by partition
// Random atomics on a table in memory bound the insert above, so where most keys are distinct and the
// table is far larger than the L2 the keys are first brought together: the positions of every bucket
// (a request's keys of one hash range) are written next to each other as {vertex, position}, and one
// workgroup deduplicates a bucket in LDS.  fpos[p] becomes the first position of p's key where that is
// not p; the bucket's table goes to memory for the lookups of the edges' sources.  10.7 M positions, R-MAT
// s24: prepare 13 us, count 30, scatter 68, dedup 90 (110 with its positions read and looked up twice), words 15.

struct RelParts {
    const uint32_t* tile0;  // R + 1: first tile, first bucket of each request
    const uint32_t* bkt0;
    uint32_t* bend;              // per bucket: count, then start, then (scattered) end of its positions
    unsigned long long* rec;     // (vertex << 32 | position), by bucket
    unsigned long long* tab;     // kPartSlots per bucket: such words, all ones = empty
    uint32_t* fpos;
    // Stands for the table in rel_emit_kernel.
    __device__ __forceinline__ uint32_t hint(uint64_t p) const { return fpos[p]; }
    __device__ __forceinline__ uint64_t first_of(uint32_t hint, uint32_t, uint32_t) const { return hint; }
    __device__ __forceinline__ uint64_t first(uint32_t r, uint32_t v) const;
};

__device__ __forceinline__ uint32_t part_hash(uint32_t v) {
    uint32_t h = v * 0x9E3779B1u;
    h ^= h >> 15;
    h *= 0x85EBCA77u;
    return h ^ (h >> 13);
}
// The bucket takes the hash's high bits, the first slot its low ones: one of every four, so that a
// lookup reads the four in one go (a wave waits for the longest of its lanes' probes).
__device__ __forceinline__ uint32_t part_slot(uint32_t h) { return h & (kPartSlots - 4); }
__device__ __forceinline__ uint32_t part_bucket(uint32_t h, uint32_t buckets) { return __umulhi(h, buckets); }

__device__ __forceinline__ uint64_t RelParts::first(uint32_t r, uint32_t v) const {
    const uint32_t b0 = bkt0[r], nb = bkt0[r + 1] - b0, h = part_hash(v);
    if (!nb || v == 0xFFFFFFFFu) return ~0ull;  // (no vertex; an empty slot's)
    const ulonglong2* t = (const ulonglong2*)(tab + (uint64_t)(b0 + part_bucket(h, nb)) * kPartSlots);
    for (uint32_t i = 0, s = part_slot(h); i < kPartSlots; i += 4, s = (s + 4) & (kPartSlots - 1)) {
        const ulonglong2 a = t[s / 2], b = t[s / 2 + 1];
        if ((uint32_t)(a.x >> 32) == v) return (uint32_t)a.x;
        if ((uint32_t)(a.y >> 32) == v) return (uint32_t)a.y;
        if ((uint32_t)(b.x >> 32) == v) return (uint32_t)b.x;
        if ((uint32_t)(b.y >> 32) == v) return (uint32_t)b.y;
        if (b.y == ~0ull) break;  // (a group fills in order)
    }
    return ~0ull;
}

__global__ __launch_bounds__(1024) void rel_part_prepare_kernel(RelParts t, uint32_t maxb, const uint64_t* __restrict__ off,
                                                                const RelReq* __restrict__ req, uint32_t R, uint32_t H,
                                                                uint64_t total, uint64_t P, uint64_t* __restrict__ Q,
                                                                uint32_t* bad, uint32_t* invalid) {
    if (blockIdx.x) {
        const uint64_t i0 = (uint64_t)(blockIdx.x - 1) * 1024 + threadIdx.x, threads = (uint64_t)(gridDim.x - 1) * 1024;
        for (uint64_t i = i0; i < P; i += threads) t.fpos[i] = ~0u;
        for (uint64_t i = i0; i < maxb; i += threads) t.bend[i] = 0;
        return;
    }
    rel_starts(off, req, R, H, total, P, Q, const_cast<uint32_t*>(t.tile0), const_cast<uint32_t*>(t.bkt0), bad, invalid);
}

// Batches that go by partition: kPartMin positions and a tile per request on average (GRASS_EXPORT_SLOT asks
// for a table in memory).  Whole mini-batch by table / by partition, us: R-MAT s24 [25, 10] one request
// of 365 k positions 158 / 187, of 677 k 204 / 223, four together 1.45 M 278 / 276, sixteen 1.6 M 314 / 288;
// s22 uniform 21 M 2088 / 1329; s16, most positions repeats, 3.7 M 540 / 451; 120 requests of 9.6 k 257 / 225.
constexpr uint64_t kPartMin = 1ull << 20;
constexpr int kPartBlock = 512;
constexpr int kPartPer = kPartTile / kPartBlock;
constexpr int kPartHeld = 8;  // a bucket's positions that a thread of its workgroup holds
constexpr uint32_t kPartHeldAll = kPartHeld * kPartBlock;
// The positions of a vertex that many repeat are one workgroup's work, 1.4 ns each past kPartHeldAll (2.4
// before they went by kPartHeld loads), where the table's inserts of a repeat are a read.  A bucket of more
// than kPartMost, unless others are as large, therefore sends the batch back to the table; the counts tell, and
// the batch has lost 0.1 ms.  A cycle of 2.4 M vertices, us by table / by partition without this / with it: one
// request of 12.3 M positions, one vertex 1 % of the seeds 661 / 853 / 767, 3 % 739 / 1326 / 870, 10 % 929 /
// 2910 / 1015, 50 % 2063 / 12180 / 2023; four requests of 0.7 M, 50 % each, 961 / 610 / 475.
constexpr uint32_t kPartMost = 1u << 17;
// Distinct vertices a request may have: the buckets' tables three quarters full.  By table / by partition,
// us, one request, seven eighths of its positions distinct: 23 M positions 1489 / 1150, 25 M 1613 / 1306, 28 M 1793 /
// 1604, 30 M 1909 / 2028; more than the tables hold, and most probes see every slot: 60 M 4255 / 157313.
constexpr uint64_t kPartDistinct = (uint64_t)kPartBuckets * (kPartSlots / 4 * 3);

// One workgroup per tile: counts its buckets' positions (SCATTER: takes room for them in each bucket,
// and writes them there).
template <bool SCATTER>
__global__ __launch_bounds__(kPartBlock) void rel_part_kernel(RelSeq q, RelParts t, uint32_t* err) {
    __shared__ uint32_t hist[kPartBuckets];
    __shared__ uint64_t beg[GRASS_KHOP_MAX_HOPS + 1];
    __shared__ const uint32_t* arr[GRASS_KHOP_MAX_HOPS + 1];
    if (blockIdx.x >= t.tile0[q.R]) return;
    uint32_t r = 0;
    for (uint32_t hi = q.R - 1; r < hi;) {  // the last request whose first tile is not after this one
        const uint32_t mid = r + (hi - r + 1) / 2;
        if (t.tile0[mid] <= blockIdx.x) r = mid;
        else hi = mid - 1;
    }
    const uint32_t b0 = t.bkt0[r], nb = t.bkt0[r + 1] - b0;
    const uint64_t p0 = q.Q[r] + (uint64_t)(blockIdx.x - t.tile0[r]) * kPartTile, p1 = min(p0 + kPartTile, q.Q[r + 1]);
    for (uint32_t i = threadIdx.x; i < nb; i += kPartBlock) hist[i] = 0;
    if (threadIdx.x == 0) {  // the stretches of the request's positions: its seeds, and its edges of each hop
        const RelReq k = q.req[r];
        beg[0] = q.Q[r];
        arr[0] = k.seeds;
        uint64_t at = q.Q[r] + k.num;
        for (uint32_t h = 0; h < q.H; ++h) {
            const uint64_t e0 = q.off[(uint64_t)h * (q.R + 1) + r];
            beg[h + 1] = at;
            arr[h + 1] = q.dst + e0;
            at += q.off[(uint64_t)h * (q.R + 1) + r + 1] - e0;
        }
    }
    __syncthreads();
    uint32_t v[kPartPer], at[kPartPer];
    bool bad = false;
#pragma unroll
    for (int i = 0; i < kPartPer; ++i) {
        const uint64_t p = p0 + (uint64_t)i * kPartBlock + threadIdx.x;
        v[i] = 0xFFFFFFFFu;
        if (p < p1) {
            uint32_t s = 0;
            for (uint32_t h = 1; h <= q.H; ++h) s = p >= beg[h] ? h : s;
            v[i] = arr[s][p - beg[s]];
            if (v[i] >= q.n) {  // a seed or destination that is not a vertex of the graph
                bad = true;
                v[i] = 0xFFFFFFFFu;
            }
        }
    }
    if (bad) atomicOr(err, 1u);
#pragma unroll
    for (int i = 0; i < kPartPer; ++i)
        if (v[i] != 0xFFFFFFFFu) at[i] = atomicAdd(&hist[part_bucket(part_hash(v[i]), nb)], 1u);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < nb; i += kPartBlock) {
        const uint32_t c = hist[i];
        if (c) {
            const uint32_t base = atomicAdd(&t.bend[b0 + i], c);
            if (SCATTER) hist[i] = base;
        }
    }
    if (!SCATTER) return;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPartPer; ++i) {
        const uint32_t p = (uint32_t)(p0 + (uint64_t)i * kPartBlock + threadIdx.x);
        if (v[i] != 0xFFFFFFFFu)
            t.rec[hist[part_bucket(part_hash(v[i]), nb)] + at[i]] = ((unsigned long long)v[i] << 32) | p;
    }
}

// Puts position w into the bucket's table: its slot, or kPartSlots when every slot holds another key.
__device__ __forceinline__ uint32_t part_insert(unsigned long long* tab, unsigned long long w) {
    uint32_t s = part_slot(part_hash((uint32_t)(w >> 32)));
    for (uint32_t probes = 0; probes < kPartSlots; ++probes, s = (s + 1) & (kPartSlots - 1)) {
        unsigned long long cur = *(volatile unsigned long long*)&tab[s];
        if (cur == ~0ull) cur = atomicCAS(&tab[s], ~0ull, w);
        if (cur == ~0ull) return s;
        if (((cur ^ w) >> 32) == 0) {
            if (cur > w) atomicMin(&tab[s], w);
            return s;
        }
    }
    return kPartSlots;
}

// The buckets' counts become their starts (one workgroup).  *invalid |= 2: few buckets hold so many
// positions that the workgroups of these would be the time (kPartMost); no tile and no bucket is left then.
__global__ __launch_bounds__(1024) void rel_part_starts_kernel(uint32_t* bend, uint32_t nb, uint32_t* tiles,
                                                               uint32_t* buckets, uint32_t* invalid) {
    constexpr uint32_t kWaves = 1024 / kWave;
    __shared__ uint32_t sums[kWaves], most[kWaves], past[kWaves];
    const uint32_t per = (nb + 1023) / 1024, lo = threadIdx.x * per, hi = min(lo + per, nb), wid = threadIdx.x / kWave;
    uint32_t sum = 0, m = 0, p = 0;  // the counts, the largest, and the positions that are not held
    for (uint32_t i = lo; i < hi; ++i) {
        const uint32_t c = bend[i];
        sum += c;
        m = max(m, c);
        p += c > kPartHeldAll ? c - kPartHeldAll : 0u;
    }
    const uint32_t inc = wave_inclusive_sum(sum);
    m = wave_max(m);
    p = wave_sum(p);
    if (lane_id() == kWave - 1) {
        sums[wid] = inc;
        most[wid] = m;
        past[wid] = p;
    }
    __syncthreads();
    uint32_t pre = inc - sum;
    for (uint32_t w = 0; w < wid; ++w) pre += sums[w];
    for (uint32_t i = lo; i < hi; ++i) {
        const uint32_t c = bend[i];
        bend[i] = pre;
        pre += c;
    }
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < kWaves; ++w) {
            m = max(m, most[w]);
            p += past[w];
        }
        if (m > kPartMost && 3ull * m > p) {
            *invalid |= 2u;
            *tiles = *buckets = 0;
        }
    }
}

// One workgroup per bucket, whose positions (but for those past kPartHeld per thread, mostly repeats) it
// holds in registers: loaded together, and not looked up again.  The others go through twice, kPartHeld
// loads at a time.  *invalid |= 2: more distinct keys than slots.
__global__ __launch_bounds__(kPartBlock) void rel_part_dedup_kernel(RelSeq q, RelParts t, uint32_t* invalid) {
    __shared__ unsigned long long tab[kPartSlots];
    const uint32_t k = blockIdx.x;
    if (k >= t.bkt0[q.R]) return;
    const uint32_t lo = (k ? t.bend[k - 1] : 0u) + threadIdx.x, hi = t.bend[k];
    unsigned long long w[kPartHeld];
    uint32_t s[kPartHeld];
    auto load = [&](uint32_t at) {
#pragma unroll
        for (int j = 0; j < kPartHeld; ++j) w[j] = at + j * kPartBlock < hi ? t.rec[at + j * kPartBlock] : ~0ull;
    };
    auto insert = [&]() {
        bool full = false;
#pragma unroll
        for (int j = 0; j < kPartHeld; ++j) {
            s[j] = w[j] != ~0ull ? part_insert(tab, w[j]) : 0u;
            full = full || s[j] == kPartSlots;
            s[j] &= kPartSlots - 1;
        }
        return full;
    };
    auto put = [&]() {
#pragma unroll
        for (int j = 0; j < kPartHeld; ++j) {
            if (w[j] == ~0ull) continue;
            const unsigned long long cur = tab[s[j]];
            if (cur < w[j]) t.fpos[(uint32_t)w[j]] = (uint32_t)cur;
        }
    };
    load(lo);
    for (uint32_t i = threadIdx.x; i < kPartSlots; i += kPartBlock) tab[i] = ~0ull;
    __syncthreads();
    bool full = false;
    if (lo + kPartHeldAll < hi) {
        for (uint32_t i = lo + kPartHeldAll; i < hi; i += kPartHeldAll) {
            load(i);
            full = insert() || full;
        }
        load(lo);
    }
    full = insert() || full;
    if (full) atomicOr(invalid, 2u);
    __syncthreads();
    put();
    for (uint32_t i = lo + kPartHeldAll; i < hi; i += kPartHeldAll) {
        load(i);
        insert();  // (already there)
        put();
    }
    unsigned long long* out = t.tab + (uint64_t)k * kPartSlots;
    for (uint32_t i = threadIdx.x; i < kPartSlots; i += kPartBlock) out[i] = tab[i];
}

__global__ __launch_bounds__(kExBlock) void rel_part_words_kernel(const uint32_t* __restrict__ fpos, uint64_t P,
                                                                  FirstWord* __restrict__ words) {
    const uint64_t nwords = (P + kWave - 1) / kWave, waves = (uint64_t)gridDim.x * (kExBlock / kWave);
    for (uint64_t w = ((uint64_t)blockIdx.x * kExBlock + threadIdx.x) / kWave; w < nwords; w += waves) {
        const uint64_t p = w * kWave + lane_id();
        const unsigned long long bits = __ballot(p < P && fpos[p] == ~0u);
        if (lane_id() == 0) words[w] = make_ulonglong2(bits, 0ull);
    }
}

hipError_t rel_build_parts(const RelParts& t, uint32_t maxb, const RelSeq& q, uint64_t P, FirstWord* d_words,
                           uint64_t* d_part, uint64_t* d_sc, uint32_t* d_bad, const grass_khop_output* b,
                           grass_khop_blocks* out, hipStream_t s) {
    const unsigned tiles = (unsigned)(P / kPartTile + q.R);
    uint32_t* d_invalid = d_bad + 1;
    hipLaunchKernelGGL(rel_part_prepare_kernel, dim3(1 + (unsigned)std::min<uint64_t>(P / 16384 + 1, 512)), dim3(1024), 0, s, t,
                       maxb, q.off, q.req, q.R, q.H, b->total, P, const_cast<uint64_t*>(q.Q), d_bad, d_invalid);
    hipLaunchKernelGGL(rel_part_kernel<false>, dim3(tiles), dim3(kPartBlock), 0, s, q, t, d_bad);
    hipLaunchKernelGGL(rel_part_starts_kernel, dim3(1), dim3(1024), 0, s, t.bend, maxb,
                       const_cast<uint32_t*>(t.tile0) + q.R, const_cast<uint32_t*>(t.bkt0) + q.R, d_invalid);
    hipLaunchKernelGGL(rel_part_kernel<true>, dim3(tiles), dim3(kPartBlock), 0, s, q, t, d_bad);
    hipLaunchKernelGGL(rel_part_dedup_kernel, dim3(maxb), dim3(kPartBlock), 0, s, q, t, d_invalid);
    const unsigned gP = (unsigned)std::min<uint64_t>((P + kExBlock - 1) / kExBlock + 1, kExGrid);
    hipLaunchKernelGGL(rel_part_words_kernel, dim3(gP), dim3(kExBlock), 0, s, (const uint32_t*)t.fpos, P, d_words);
    return rel_number(t, q, P, d_words, d_part, d_sc, d_bad, out, s);
}

// At most kOneWgEntries positions and 1024 requests: the whole build in one launch of one workgroup, the
// table in LDS.  reqs and result lie in host memory; result[0] = nodes, result[1] = 0 or 1 (the
// offsets are not the batch of these requests, an id is not a vertex, or a source is unknown).
__global__ __launch_bounds__(kOneWgThreads) void rel_small_kernel(RelSeq q, const RelReq* __restrict__ hreq,
                                                                  RelReq* dreq, uint64_t* Q, uint32_t P, uint64_t total,
                                                                  uint32_t vb, uint64_t* node_off,
                                                                  uint32_t* __restrict__ nodes, uint64_t cap,
                                                                  uint32_t* __restrict__ lsrc,
                                                                  uint32_t* __restrict__ ldst, uint64_t* result) {
    extern __shared__ unsigned long long rel_lds[];
    __shared__ OneWgFirsts f;
    __shared__ uint64_t lds[kOneWgThreads / kWave];
    const uint32_t t = threadIdx.x;
    if (t < q.R) dreq[t] = hreq[t];
    __syncthreads();
    const bool mine_ok = q.H == 0 || rel_check(q.off, q.req, q.R, q.H, total, t, kOneWgThreads);
    bool ok = block_sum<uint64_t, kOneWgThreads>(mine_ok ? 0 : 1, lds) == 0;
    uint64_t sum;
    const uint64_t len = t < q.R ? rel_length(q.req, q.off, q.R, ok ? q.H : 0, t) : 0;
    const uint64_t pre = block_exclusive_sum<uint64_t, kOneWgThreads>(len, sum, lds);
    ok = ok && sum == P;
    if (t < q.R) Q[t] = pre;
    if (t == 0) Q[q.R] = sum;
    if (!ok) {  // uniform: nothing below reads through the offsets
        if (t == 0) {
            result[0] = 0;
            result[1] = 1;
        }
        return;
    }
    one_wg_begin(f, rel_lds, P, vb);  // (its barrier also orders Q)
    uint32_t slot[kOneWgPer], rr[kOneWgPer], vv[kOneWgPer];
    uint64_t ee[kOneWgPer];
    bool bad = false;
#pragma unroll
    for (uint32_t i = 0; i < kOneWgPer; ++i) {
        const uint32_t p = i * kOneWgThreads + t;
        slot[i] = ~0u;
        if (p < P) {
            rr[i] = segment_in(q.Q, 0, q.R - 1, p);
            vv[i] = q.at(p, rr[i], ee[i]);
            if (vv[i] < q.n) slot[i] = f.insert(rr[i], vv[i], p);
            else bad = true;
        }
    }
    const uint32_t mine = one_wg_rank(f, P, slot);
#pragma unroll
    for (uint32_t i = 0; i < kOneWgPer; ++i) {
        const uint32_t p = i * kOneWgThreads + t;
        if (p >= P || slot[i] == ~0u) continue;
        const uint32_t first = (uint32_t)f.tab[slot[i]] & (kOneWgEntries - 1), id = f.rank(first);
        if (((mine >> i) & 1) && id < cap) nodes[id] = vv[i];
        if (ee[i] == ~0ull) continue;
        const uint32_t base = f.rank((uint32_t)q.Q[rr[i]]);
        const uint32_t src = q.src[ee[i]];
        const uint32_t fs = src < q.n ? f.first(rr[i], src) : ~0u;
        bad = bad || fs == ~0u;
        ldst[ee[i]] = id - base;
        lsrc[ee[i]] = fs == ~0u ? kNoId : f.rank(fs) - base;
    }
    for (uint32_t r = t; r <= q.R; r += kOneWgThreads) {
        const uint32_t p = (uint32_t)q.Q[r];
        node_off[r] = p < P ? f.rank(p) : f.total;
    }
    const uint64_t nbad = block_sum<uint64_t, kOneWgThreads>(bad ? 1 : 0, lds);
    if (t == 0) {
        result[0] = f.total;
        result[1] = nbad ? 1 : 0;
    }
}

// Whether a request may have more than kPartDistinct distinct vertices.
bool too_many_distinct(const grass_graph* g, const grass_khop_request* reqs, uint32_t R, uint64_t P) {
    if (std::min<uint64_t>(P, g->n) <= kPartDistinct) return false;
    for (uint32_t r = 0; r < R; ++r) {
        uint64_t front = std::min<uint64_t>(reqs[r].num_seeds, g->n), all = front;
        for (uint32_t h = 0; h < reqs[r].hops; ++h) {
            front = std::min<uint64_t>(front * std::min<uint64_t>(reqs[r].fanout[h], g->max_degree), g->n);
            all += front;
        }
        if (std::min<uint64_t>(all, P) > kPartDistinct) return true;
    }
    return false;
}

int khop_blocks(grass_graph* g, const grass_khop_request* reqs, uint32_t R, const grass_khop_output* b,
                grass_khop_blocks* out, hipStream_t s) {
    std::lock_guard<std::mutex> lock(g->mu);
    Workspace& ws = g->ws;
    out->nodes = 0;
    const uint32_t H = b->max_hops;
    if (H > GRASS_KHOP_MAX_HOPS || (H && !b->offsets_dev) || b->total > b->capacity || !out->node_off_dev)
        return GRASS_EINVAL;
    if (b->total && (!b->src_dev || !b->dst_dev || !out->lsrc_dev || !out->ldst_dev)) return GRASS_EINVAL;
    if (ws.reserve_stage(R * sizeof(RelReq) + 64) != hipSuccess) return GRASS_ENOMEM;
    RelReq* hreq = (RelReq*)ws.stage();
    uint64_t S = 0;
    for (uint32_t r = 0; r < R; ++r) {
        if (reqs[r].hops > H || (reqs[r].num_seeds && !reqs[r].seeds_dev)) return GRASS_EINVAL;
        hreq[r] = RelReq{reqs[r].seeds_dev, reqs[r].num_seeds, reqs[r].hops};
        S += reqs[r].num_seeds;
    }
    const uint64_t P = S + b->total;
    if (P && (!out->nodes_dev && out->node_capacity)) return GRASS_EINVAL;
    uint64_t slots = 1024;
    while (slots < P + P / 2 + 2) slots <<= 1;  // load <= 2/3: distinct keys <= positions
    const uint64_t nb = scan_blocks(std::max<uint64_t>(firsts_words(P), R));
    const size_t need = Carve::need(R * sizeof(RelReq)) + Carve::need(R * 8) + Carve::need((R + 1) * 8) +
                        Carve::need(firsts_words(P) * sizeof(FirstWord)) + Carve::need((nb + 2) * 8) +
                        Carve::need(64);
    // Packed 8-byte slots when the request, vertex and position bits fit one word; 16-byte slots
    // otherwise, or when GRASS_EXPORT_SLOT=16 asks for them.
    auto bits = [](uint64_t x) {
        uint32_t k = 0;
        while (k < 64 && (x >> k) != 0) ++k;
        return k;
    };
    const uint32_t rb = bits(R - 1), vb = std::max<uint32_t>(bits(g->n ? g->n - 1 : 0), 1u),
                   pb = std::max<uint32_t>(bits(P), 1u);  // positions < 2^pb - 1
    const char* force = getenv("GRASS_EXPORT_SLOT");
    const bool wide = rb + vb + pb > 64 || (force && strcmp(force, "16") == 0);
    if (ws.scratch.reserve(need) != hipSuccess) return GRASS_ENOMEM;
    const uint32_t maxb = (uint32_t)std::min<uint64_t>(P / kPartKeys + R, 0xFFFFFFFFull);
    auto carve_parts = [&](Carve& c, RelParts& t) {
        t.tile0 = c.take<uint32_t>(R + 1);
        t.bkt0 = c.take<uint32_t>(R + 1);
        t.bend = c.take<uint32_t>(maxb + 1);
        t.rec = c.take<unsigned long long>(P);
        t.tab = c.take<unsigned long long>((uint64_t)maxb * kPartSlots);
        t.fpos = c.take<uint32_t>(P);
    };
    // (a workgroup counts on in 32 bits past its bucket's last position)
    bool parts = P >= kPartMin && P + kPartHeldAll <= 0xFFFFFFFFull && R && R <= kPrepRequests && P / R >= kPartTile && !force &&
                 !too_many_distinct(g, reqs, R, P);
    if (parts) {
        Carve size(nullptr);
        RelParts t{};
        carve_parts(size, t);
        parts = ws.ht.reserve(size.off + 256) == hipSuccess;
    }
    if (!parts && ws.ht.reserve(slots * (wide ? 16 : 8)) != hipSuccess) return GRASS_ENOMEM;
    // this overwrites the k-hop dedup table's memory: the next k-hop batch clears it first
    ws.ht_gen = 0xFFFF;
    Carve cv(ws.scratch.ptr);
    RelReq* d_req = cv.take<RelReq>(R);
    uint64_t* d_len = cv.take<uint64_t>(R);
    uint64_t* d_Q = cv.take<uint64_t>(R + 1);
    FirstWord* d_words = cv.take<FirstWord>(firsts_words(P));
    uint64_t* d_part = cv.take<uint64_t>(nb + 2);
    uint64_t* d_sc = cv.take<uint64_t>(8);  // [0] scratch total, [1] node total, [2] error flags
    const uint32_t lg = (uint32_t)__builtin_ctzll(slots);

    hipError_t e = hipSuccess;
    uint64_t* hres = ws.result_slot();
    // (GRASS_EXPORT_SLOT asks for a table in memory)
    if (P && P <= kOneWgEntries && R && R <= kOneWgThreads && !force) {
        const size_t lds = (size_t)one_wg_slots((uint32_t)P) * 8;
        if (lds > 65536) {
            (void)hipFuncSetAttribute((const void*)rel_small_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            (void)hipGetLastError();
        }
        const RelSeq q{d_req, b->offsets_dev, b->src_dev, b->dst_dev, d_Q, R, H, (uint32_t)g->n};
        hipLaunchKernelGGL(rel_small_kernel, dim3(1), dim3(kOneWgThreads), lds, s, q, (const RelReq*)hreq, d_req, d_Q,
                           (uint32_t)P, b->total, vb, out->node_off_dev, out->nodes_dev, out->node_capacity, out->lsrc_dev,
                           out->ldst_dev, hres);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) return status_of(e);
        if (hres[1] != 0) return GRASS_EINVAL;
        out->nodes = hres[0];
        return out->nodes > out->node_capacity ? GRASS_ECAPACITY : GRASS_OK;
    }
    if (R) e = hipMemcpyAsync(d_req, hreq, R * sizeof(RelReq), hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return status_of(e);
    // the two halves of d_sc[2]: an id that is not a vertex, or an unknown source; and offsets that
    // do not fit the requests
    uint32_t* d_bad = (uint32_t*)(d_sc + 2);
    RelSeq q{d_req, b->offsets_dev, b->src_dev, b->dst_dev, d_Q, R, H, (uint32_t)g->n};
    if (parts) {
        Carve c(ws.ht.ptr);
        RelParts t{};
        carve_parts(c, t);
        e = rel_build_parts(t, maxb, q, P, d_words, d_part, d_sc, d_bad, b, out, s);
        if (e == hipSuccess) e = hipMemcpyAsync(hres, d_sc + 1, 16, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) return status_of(e);
        if (!(hres[1] >> 32 & 2)) {
            if (hres[1] != 0) return GRASS_EINVAL;
            out->nodes = hres[0];
            return out->nodes > out->node_capacity ? GRASS_ECAPACITY : GRASS_OK;
        }
        // a bucket's keys did not fit its table: the other way
        if (ws.ht.reserve(slots * (wide ? 16 : 8)) != hipSuccess) return GRASS_ENOMEM;
    }
    if (wide) {
        RelTab16 t{(unsigned long long*)ws.ht.ptr, slots - 1, 64 - lg};
        e = rel_build(t, q, P, d_len, d_words, d_part, d_sc, d_bad, b, out, s);
    } else {
        RelTab8 t{(unsigned long long*)ws.ht.ptr, slots - 1, 64 - lg, vb, pb};
        e = rel_build(t, q, P, d_len, d_words, d_part, d_sc, d_bad, b, out, s);
    }
    if (e != hipSuccess) return status_of(e);
    e = hipMemcpyAsync(hres, d_sc + 1, 16, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return status_of(e);
    // the offsets are not the batch of these requests (rows out of order or past the total, edges
    // at hops a request does not have, sizes that differ), an id is not a vertex, or an edge's
    // source is not among the request's earlier vertices
    if (hres[1] != 0) return GRASS_EINVAL;
    out->nodes = hres[0];
    return out->nodes > out->node_capacity ? GRASS_ECAPACITY : GRASS_OK;
}

// ------------------------------------------------------------------ MDRW local ids

// Rank of x in the ascending a[0, n); kNoId when absent.
__device__ __forceinline__ uint32_t rank_in(const uint32_t* __restrict__ a, uint64_t n, uint32_t x) {
    uint64_t lo = 0, hi = n;
    while (lo < hi) {
        const uint64_t mid = (lo + hi) / 2;
        if (a[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo < n && a[lo] == x ? (uint32_t)lo : kNoId;
}

__global__ __launch_bounds__(kExBlock) void mdrw_local_kernel(const uint64_t* __restrict__ eoff,
                                                              const uint32_t* __restrict__ esrc,
                                                              const uint32_t* __restrict__ edst, uint64_t E,
                                                              uint32_t I, const uint64_t* __restrict__ voff,
                                                              const uint32_t* __restrict__ verts,
                                                              uint32_t* __restrict__ lsrc,
                                                              uint32_t* __restrict__ ldst) {
    for (uint64_t e = (uint64_t)blockIdx.x * kExBlock + threadIdx.x; e < E; e += (uint64_t)gridDim.x * kExBlock) {
        const uint32_t i = segment_in(eoff, 0, I - 1, e);
        const uint32_t* V = verts + voff[i];
        const uint64_t nv = voff[i + 1] - voff[i];
        lsrc[e] = rank_in(V, nv, esrc[e]);
        ldst[e] = rank_in(V, nv, edst[e]);
    }
}

// ------------------------------------------------------------------ DLPack

struct DlHold {
    grass_dl_managed_tensor mt;
    int64_t shape[1];
    grass_mdrw_result* res;
};

void dl_release(grass_dl_managed_tensor* self) {
    if (!self) return;
    DlHold* h = (DlHold*)self->manager_ctx;
    grass_mdrw_result* res = h->res;
    delete h;
    res->release();
}

}  // namespace
}  // namespace grass

extern "C" {

int grass_khop_blocks_build(grass_graph* g, const grass_khop_request* reqs, uint32_t count,
                            const grass_khop_output* batch, grass_khop_blocks* out, void* stream) {
    if (!g || !batch || !out || (count && !reqs) || count > (1u << 17)) return GRASS_EINVAL;
    if (count == 0) {
        out->nodes = 0;
        return GRASS_OK;
    }
    int prev = 0;
    (void)hipGetDevice(&prev);
    if (!grass::enter_device(g->device)) return GRASS_EDEVICE;
    hipStream_t s = stream ? (hipStream_t)stream : g->stream;
    int rc = grass::khop_blocks(g, reqs, count, batch, out, s);
    (void)hipSetDevice(prev);
    return rc;
}

int grass_mdrw_local_edges(grass_graph* g, const grass_mdrw_result* res, int which, uint32_t* lsrc_dev,
                           uint32_t* ldst_dev, void* stream) {
    if (!g || !res || (which != GRASS_MDRW_EDGES_INDUCED && which != GRASS_MDRW_EDGES_STEPS)) return GRASS_EINVAL;
    const grass_mdrw_output& o = res->out;
    const bool ind = which == GRASS_MDRW_EDGES_INDUCED;
    const uint64_t E = ind ? o.induced : o.steps;
    if (E == 0 || o.count == 0) return GRASS_OK;
    if (!lsrc_dev || !ldst_dev) return GRASS_EINVAL;
    int prev = 0;
    (void)hipGetDevice(&prev);
    if (!grass::enter_device(g->device)) return GRASS_EDEVICE;
    hipStream_t s = stream ? (hipStream_t)stream : g->stream;
    const unsigned grid = (unsigned)std::min<uint64_t>((E + grass::kExBlock - 1) / grass::kExBlock, grass::kExGrid);
    hipLaunchKernelGGL(grass::mdrw_local_kernel, dim3(grid), dim3(grass::kExBlock), 0, s,
                       ind ? o.ind_off_dev : o.step_off_dev, ind ? o.ind_src_dev : o.step_src_dev,
                       ind ? o.ind_dst_dev : o.step_dst_dev, E, o.count, o.vert_off_dev, o.verts_dev, lsrc_dev,
                       ldst_dev);
    const int rc = grass::status_of(hipGetLastError());
    (void)hipSetDevice(prev);
    return rc;
}

int grass_mdrw_to_dlpack(grass_mdrw_result* res, int which, grass_dl_managed_tensor** out) {
    if (!res || !out || which < GRASS_MDRW_STEP_OFF || which > GRASS_MDRW_IND_DST) return GRASS_EINVAL;
    const grass_mdrw_output& o = res->out;
    const uint64_t no = (uint64_t)o.count + 1;
    const void* data[8] = {o.step_off_dev, o.step_src_dev, o.step_dst_dev, o.vert_off_dev,
                           o.verts_dev,    o.ind_off_dev,  o.ind_src_dev,  o.ind_dst_dev};
    const uint64_t len[8] = {no, o.steps, o.steps, no, o.verts, no, o.induced, o.induced};
    const bool offs = which == GRASS_MDRW_STEP_OFF || which == GRASS_MDRW_VERT_OFF || which == GRASS_MDRW_IND_OFF;
    grass::DlHold* h = new (std::nothrow) grass::DlHold();
    if (!h) return GRASS_ENOMEM;
    h->shape[0] = (int64_t)len[which];
    grass_dl_tensor& t = h->mt.dl_tensor;
    t.data = const_cast<void*>(data[which]);
    t.device = grass_dl_device{10, res->device};
    t.ndim = 1;
    t.dtype = grass_dl_dtype{0, (uint8_t)(offs ? 64 : 32), 1};
    t.shape = h->shape;
    t.strides = nullptr;
    t.byte_offset = 0;
    h->mt.manager_ctx = h;
    h->mt.deleter = grass::dl_release;
    res->refs.fetch_add(1, std::memory_order_relaxed);
    h->res = res;
    *out = &h->mt;
    return GRASS_OK;
}

}  // extern "C"
