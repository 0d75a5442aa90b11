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
// A batch of few positions is one launch of one workgroup (rel_small_kernel).  A large one is bound by
// the random atomics of the inserts, which the chip takes at 22 to 27 G/s whatever the table's size
// (a load of a slot and a CAS on it: 25.7 G/s), so a position touches the table once: 16 x 8192 seeds
// [25, 10] on R-MAT s24, 10.7 M positions, insert 435 us; a second pass that looked every key up again
// took 196 us more.  The emit is 223 us, most of it waiting on the source's lookup.
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

// Up to kPrepRequests requests: workgroup 0 checks the offsets, scans the lengths into Q and checks their
// total, while the others clear the table (with one workgroup, it does both): one launch where the
// steps by themselves are seven.
constexpr uint32_t kPrepRequests = 8192;
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
    __shared__ uint64_t lds[1024 / kWave];
    const bool mine = H == 0 || rel_check(off, req, R, H, total, threadIdx.x, 1024);
    const bool ok = block_sum<uint64_t, 1024>(mine ? 0 : 1, lds) == 0;
    constexpr uint32_t kPer = kPrepRequests / 1024;
    const uint32_t per = (R + 1023) / 1024, r0 = threadIdx.x * per;
    uint64_t len[kPer], s = 0;
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        len[i] = i < per && r0 + i < R ? rel_length(req, off, R, ok ? H : 0, r0 + i) : 0;
        s += len[i];
    }
    uint64_t sum;
    uint64_t pre = block_exclusive_sum<uint64_t, 1024>(s, sum, lds);
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        if (i < per && r0 + i < R) Q[r0 + i] = pre;
        pre += len[i];
    }
    if (threadIdx.x == 0) {
        Q[R] = sum;
        *bad = 0;
        *invalid = ok && sum == P ? 0 : 1;
    }
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
    for (uint64_t w = wc.w; w < wc.end; ++w) {
        const FirstWord fw = words[w];
        const uint64_t p = w * kWave + lane_id(), last = min(w * kWave + kWave - 1, P - 1);
        uint32_t r;
        uint64_t e;
        const uint32_t v = cur.at(q, w, min(p, last), last, r, e);
        if (p >= P) continue;
        const bool first = (fw.x >> lane_id()) & 1;
        const uint64_t mine = fw.y + lanes_below(fw.x);
        if (first && mine < cap) nodes[mine] = v;
        if (e == ~0ull) continue;
        const uint64_t base = node_off[r];
        const uint64_t fd = first ? p : v < q.n ? t.first(r, v) : ~0ull;
        const uint64_t fs = t.first(r, q.src[e]);
        if (fd >= P || fs >= P) {  // a source that is neither a seed nor an earlier destination
            atomicOr(err, 1u);
            ldst[e] = lsrc[e] = kNoId;
            continue;
        }
        ldst[e] = (uint32_t)((first ? mine : first_rank(words, fd)) - base);
        lsrc[e] = (uint32_t)(first_rank(words, fs) - base);
    }
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
    // node_off[r] = first appearances before request r; their total beside the other results
    hipError_t e = scan_firsts(d_words, Count{P, nullptr}, P, q.Q, q.R, out->node_off_dev, d_sc + 1, d_part, d_sc, s);
    if (e != hipSuccess || !P) return e;
    hipLaunchKernelGGL(rel_emit_kernel<Tab>, dim3(gP), dim3(kExBlock), 0, s, q, P, t, (const FirstWord*)d_words,
                       (const uint64_t*)out->node_off_dev, out->nodes_dev, out->node_capacity, out->lsrc_dev,
                       out->ldst_dev, (const uint32_t*)d_invalid, d_bad);
    return hipGetLastError();
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
    if (ws.scratch.reserve(need) != hipSuccess || ws.ht.reserve(slots * (wide ? 16 : 8)) != hipSuccess)
        return GRASS_ENOMEM;
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
