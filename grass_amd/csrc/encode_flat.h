// Encoding by slots.  Vertex v's record takes d + 1 consecutive slots, first slot rowptr[v] + v: one for
// its header, then one per field in stream order (LE: rocks, then seas; GT: list order).  A wave
// takes consecutive slots, 64 a pass, so lists of any length fill its lanes and the column ids are
// read in order.  Rows have to be strictly ascending with ids below 2^31 (the plan finds out), which
// keeps every value in 32 bits.  Bound by instruction issue (250 to 300 a pass).  Measured on R-MAT s22
// (2.4 M rows, 128 M entries, GT): a wave per vertex planned in 1.63 ms, wrote the image in 3.65 and made
// the resident stream of it in 3.2 more; by slots the plan takes 0.71 ms and the stream, straight from the
// rows, 0.81 (0.84 and 0.91 before passes inside one list kept its constants and skipped the placing).
#pragma once
#include <hip/hip_runtime.h>

#include "codec.h"
#include "devutil.h"

namespace grass {

// get_bit_num (compressor.hpp:16-22): bit length of |x|, 1 for 0.
__device__ __forceinline__ uint32_t bit_num(int64_t x) {
    if (x < 0) x = -x;
    return x == 0 ? 1u : 64u - (uint32_t)__clzll((unsigned long long)x);
}

// Length of the Elias-gamma code of x + 1 (compressor.hpp:411-417).
__device__ __forceinline__ uint32_t gamma_bits(uint64_t x) {
    return 2u * (63u - (uint32_t)__clzll((unsigned long long)(x + 1))) + 1u;
}

// Elias-gamma code of x + 1 (x + 1 < 2^32) at stream bit `at` of the pass buffer: L zero bits,
// then x + 1 in L + 1 bits.
__device__ __forceinline__ void put_gamma(uint32_t* B, uint64_t w0, uint64_t& at, uint32_t x) {
    const uint32_t y = x + 1;
    const uint32_t L = 31u - (uint32_t)__clz(y);
    put_field(B, w0, at + L, L + 1, y);
    at += 2 * L + 1;
}

constexpr int kFlatBlock = 256;
constexpr int kFlatWaves = kFlatBlock / kWave;
constexpr uint32_t kFlatPassMin = 4, kFlatPassMax = 32;  // passes per chunk
constexpr uint32_t kFlatLook = 32;                       // slots of a chunk's last pass past its own
// Words a pass of 64 slots touches: a field has at most 32 bits, a header at most 48 when the whole
// record is in the pass (d < 64; LE, d = 1: 66 and no field) and 114 otherwise, which at most two
// are; in the stream a payload's start skips at most 31 bits.  64 * 48 + 2 * 114 + 31 bits.
constexpr uint32_t kFlatWords = 112;

// Passes per chunk of consecutive slots: all waves get a few chunks of a large graph, and a chunk's
// look-ahead of half a pass is little of it.
__host__ __device__ __forceinline__ uint32_t flat_passes(uint64_t slots, uint64_t waves) {
    const uint64_t p = slots / (waves * kWave);
    return (uint32_t)(p < kFlatPassMin ? kFlatPassMin : p > kFlatPassMax ? kFlatPassMax : p);
}

// le_geometry and gt_geometry for d < 2^31 without a branch or a division (d >= 2, d >= 1): the root
// of a 31-bit number from a 1-ulp square root is off by at most one, and D / C is one of three values.
template <int FMT>
__device__ __forceinline__ void flat_geometry(uint32_t d, uint32_t& C, uint32_t& q, uint32_t& R) {
    const uint32_t D = FMT == kLE ? d - 1 : d;
    uint32_t s = (uint32_t)__builtin_amdgcn_sqrtf((float)D);
    int32_t r = (int32_t)(D - __umul24(s, s));
    if (r < 0) {
        r += 2 * (int32_t)s - 1;
        --s;
    } else if (r > 2 * (int32_t)s) {
        r -= 2 * (int32_t)s + 1;
        ++s;
    }
    // LE: C = s or s + 1 and q is C - 1 .. C + 1; GT: C = s (a square, q = s) or s + 1 and q = C - 2 .. C
    C = s + (FMT == kLE ? r > (int32_t)s : r > 0);
    const uint32_t lo = FMT == kLE ? C - 1 : C - 2;
    q = lo + (D >= __umul24(C, lo + 1)) + (D >= __umul24(C, lo + 2));
    R = D - __umul24(C, q);
}

// Position k -> chunk (block) c and index i in it (codec.h's split; LE: position d - 1 is rock C).
__device__ __forceinline__ void flat_pos(uint32_t k, uint32_t q, uint32_t R, uint32_t& c, uint32_t& i) {
    const uint32_t big = __umul24(R, q + 1);
    const bool lo = k < big;
    const uint32_t len = lo ? q + 1 : q, kk = lo ? k : k - big;
    const uint32_t b = udiv_chunk(kk, max(len, 1u));
    i = kk - __umul24(b, len);
    c = lo ? b : b + R;
}

// A list's constants, uniform over the wave: kept while whole passes lie in one list.
template <int FMT>
struct FlatList {
    uint32_t v = 0xFFFFFFFFu;  // whose they are
    uint32_t C, q, R;
    UDiv d1, d0;
    __device__ __forceinline__ void of(uint32_t vertex, uint32_t d) {
        if (vertex == v) return;
        v = vertex;
        flat_geometry<FMT>(d, C, q, R);
        C = (uint32_t)__builtin_amdgcn_readfirstlane((int)C);
        q = (uint32_t)__builtin_amdgcn_readfirstlane((int)q);
        R = (uint32_t)__builtin_amdgcn_readfirstlane((int)R);
        d1.init(q + 1);
        d0.init(q);
    }
    __device__ __forceinline__ void pos(uint32_t k, uint32_t& c, uint32_t& i) const {  // flat_pos
        const uint32_t big = R * (q + 1);
        const bool lo = k < big;
        UDiv u;
        u.d = lo ? q + 1 : q;
        u.m = lo ? d1.m : d0.m;
        const uint32_t kk = lo ? k : k - big, b = u.div(kk);
        i = kk - __umul24(b, u.d);
        c = lo ? b : b + R;
    }
};

// Residual of LE sea i of the chunk at list position s0 with L positions (le_residual for ascending rows).
__device__ __forceinline__ int32_t flat_residual(uint32_t x, uint32_t rl, uint32_t rr, uint32_t i, uint32_t L) {
    return (int32_t)(x - (rl + i * udiv_chunk(rr - rl, L)));
}

// A wave's place among the slots.
struct SlotWalk {
    const uint64_t* __restrict__ rowptr;
    uint64_t n;
    uint32_t cur;  // vertex of the pass's first slot
    uint64_t sc;   // its first slot
    uint64_t bj;   // one past the last slot of vertex cur + lane (~0 past the graph)

    __device__ __forceinline__ uint64_t first(uint64_t v) const { return rowptr[v] + v; }

    // To slot s: a search that probes 64 vertices a step.
    __device__ __forceinline__ void seek(uint64_t s) {
        const uint32_t lane = lane_id();
        uint64_t lo = 0, hi = n;  // first(lo) <= s < first(hi)
        while (hi - lo > 1) {
            const uint64_t step = (hi - lo + kWave - 1) / kWave, p = lo + (lane + 1) * step;
            const uint64_t below = __popcll(__ballot(p < hi && first(p) <= s));
            lo += below * step;
            hi = lo + step < hi ? lo + step : hi;
        }
        cur = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
        sc = readfirstlane_u64(first(cur));
        request();
    }
    __device__ __forceinline__ void request() {
        const uint64_t v = (uint64_t)cur + 1 + lane_id();
        bj = v <= n ? first(v) : ~0ull;
    }

    // The lanes' slots base + lane of lanes 0 .. last: j, their vertex's place among the 64 from `cur`
    // (each vertex writes its place to the lane of its first slot in the pass, and an inclusive
    // maximum gives every lane its vertex); k, the field's index in stream order, -1 at the header;
    // d; head, the first lane of its vertex in the pass.
    __device__ __forceinline__ void place(uint64_t base, uint32_t last, uint32_t* own, uint32_t& j, int32_t& k,
                                          uint32_t& d, uint32_t& head) const {
        const uint32_t lane = lane_id();
        const uint32_t rj = bj - sc > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)(bj - sc);
        const uint32_t pj = dpp_move<0x138>(rj);  // (lane 0: 0)
        const uint32_t e0 = (uint32_t)(base - sc);
        own[lane] = 0;
        wave_sync();
        if (rj > e0 && pj <= e0 + last) own[pj > e0 ? pj - e0 : 0u] = lane + 1;
        wave_sync();
        j = wave_inclusive_max(own[lane]) - 1;
        wave_sync();
        const uint32_t p = __shfl(pj, (int)j, kWave), e = __shfl(rj, (int)j, kWave);
        k = (int32_t)(e0 + lane - p) - 1;
        d = e - p - 1;
        head = p > e0 ? p - e0 : 0u;
    }
    // Whether slots base .. base + 63 are all fields of vertex cur.
    __device__ __forceinline__ bool in_list(uint64_t base) const {
        return base > sc && base + kWave <= readlane_u64(bj, 0);
    }
    // To the vertex of the slot after the last active lane's, which is at place jl: the next vertex when
    // that slot was its last (`end`), so that the 64 from `cur` always hold the next pass.
    __device__ __forceinline__ void advance(uint32_t jl, bool end) {
        jl += end;
        if (jl) {
            cur += jl;
            sc = readlane_u64(bj, (int)jl - 1);
        }
    }
};

// Inclusive OR (or sum) over the lanes head .. lane (a lane's head is its segment's first lane), the DPP
// tree of wave_inclusive_sum with the moves that would cross a segment's start left out.
struct SegmentScan {
    bool c1, c2, c4, c8, c16, c32;
    __device__ __forceinline__ explicit SegmentScan(uint32_t head) {
        const uint32_t lane = lane_id(), back = lane - head, row = lane & 15;
        c1 = back >= 1 && row >= 1;
        c2 = back >= 2 && row >= 2;
        c4 = back >= 4 && row >= 4;
        c8 = back >= 8 && row >= 8;
        c16 = (lane & 16) && head <= (lane & ~15u) - 1;
        c32 = lane >= 32 && head <= 31;
    }
    __device__ __forceinline__ uint32_t any(uint32_t x) const {
        uint32_t t = dpp_move<0x111>(x);
        x |= c1 ? t : 0u;
        t = dpp_move<0x112>(x);
        x |= c2 ? t : 0u;
        t = dpp_move<0x114>(x);
        x |= c4 ? t : 0u;
        t = dpp_move<0x118>(x);
        x |= c8 ? t : 0u;
        t = dpp_move<0x142, 0xa>(x);
        x |= c16 ? t : 0u;
        t = dpp_move<0x143, 0xc>(x);
        x |= c32 ? t : 0u;
        return x;
    }
    __device__ __forceinline__ uint32_t sum(uint32_t x) const {
        uint32_t t = dpp_move<0x111>(x);
        x += c1 ? t : 0u;
        t = dpp_move<0x112>(x);
        x += c2 ? t : 0u;
        t = dpp_move<0x114>(x);
        x += c4 ? t : 0u;
        t = dpp_move<0x118>(x);
        x += c8 ? t : 0u;
        t = dpp_move<0x142, 0xa>(x);
        x += c16 ? t : 0u;
        t = dpp_move<0x143, 0xc>(x);
        x += c32 ? t : 0u;
        return x;
    }
};

// The OR of all lanes, in lane 63 (the other lanes hold parts of it).
__device__ __forceinline__ uint32_t wave_or_last(uint32_t x) {
    x |= dpp_move<0x111>(x);
    x |= dpp_move<0x112>(x);
    x |= dpp_move<0x114>(x);
    x |= dpp_move<0x118>(x);
    x |= dpp_move<0x142, 0xa>(x);
    x |= dpp_move<0x143, 0xc>(x);
    return x;
}

// A plan's totals.
struct FlatStats {
    unsigned long long bits;     // of the .graph records
    unsigned long long longest;  // record, in bits
    unsigned long long flags;    // kFlatGeneral, kFlatImages
    unsigned long long max_degree;
    unsigned long long runs;   // decode runs (codec.h)
    unsigned long long words;  // of the GT stream
    unsigned long long m;
};
constexpr unsigned long long kFlatGeneral = 1;  // a row is not strictly ascending below 2^31
constexpr unsigned long long kFlatImages = 2;   // an id >= n, or a GT self loop at a block head (whose
                                                // .graph bytes hold another id)

// The fields' widths are the bit lengths of maxima, so of ORs: ors[v] (zero at first) becomes the OR of
// |rock - v| of the list's ends (LE) or |head - v| - 1 (GT) and of the residuals or gaps, and fps[v]
// first_pos, which the one entry that follows the last id below v tells.  A vertex inside a chunk is
// stored, one that chunks share ORed.
template <int FMT>
__global__ __launch_bounds__(kFlatBlock) void flat_plan_kernel(const uint64_t* __restrict__ rowptr,
                                                               const uint32_t* __restrict__ col, uint64_t n,
                                                               uint2* ors, uint32_t* __restrict__ fps,
                                                               FlatStats* stats) {
    __shared__ uint32_t own_lds[kFlatBlock];
    uint32_t* own = own_lds + (threadIdx.x & ~(kWave - 1));
    const uint32_t lane = lane_id();
    const uint64_t waves = (uint64_t)gridDim.x * kFlatWaves;
    const uint64_t wave = ((uint64_t)blockIdx.x * kFlatBlock + threadIdx.x) / kWave;
    const uint64_t slots = rowptr[n] + n;
    if (rowptr[0] != 0) {
        if (wave == 0 && lane == 0) atomicOr(&stats->flags, kFlatGeneral);
        return;
    }
    const uint64_t W = (uint64_t)flat_passes(slots, waves) * kWave;
    bool general = false, images = false;
    for (uint64_t s0 = wave * W; s0 < slots; s0 += waves * W) {
        const uint64_t s1 = s0 + W < slots ? s0 + W : slots;
        SlotWalk walk{rowptr, n};
        walk.seek(s0);
        const uint32_t before = walk.sc < s0 ? walk.cur : 0xFFFFFFFFu;  // a vertex begun by another chunk
        FlatList<FMT> list;
        uint32_t ca = 0, cb = 0;  // the ORs so far of the pass's first vertex
        uint32_t px = s0 - walk.sc >= 2 ? col[s0 - walk.cur - 2] : 0u;  // the id before the pass's first
        for (uint64_t base = s0; base < s1; base += kWave) {
            const uint32_t last = (uint32_t)(s1 - base < (uint64_t)kWave ? s1 - base - 1 : kWave - 1);
            uint32_t j, d, head, C, q, R, c, i;
            int32_t k;
            const bool whole = last == kWave - 1 && walk.in_list(base);  // the pass is in one list
            if (whole) {
                j = head = 0;
                k = (int32_t)(base - walk.sc) + (int32_t)lane - 1;
                d = (uint32_t)(readlane_u64(walk.bj, 0) - walk.sc) - 1;
                list.of(walk.cur, d);
                C = list.C;
                q = list.q;
                R = list.R;
                list.pos((uint32_t)k, c, i);
            } else {
                walk.place(base, last, own, j, k, d, head);
                flat_geometry<FMT>(d, C, q, R);
                flat_pos(k < 0 ? 0u : (uint32_t)k, q, R, c, i);
            }
            const bool end = k + 1 == (int32_t)d;
            const bool ended = __builtin_amdgcn_readlane((int)end, (int)last);
            const uint32_t v = walk.cur + j;
            if (!whole || ended) {
                walk.advance((uint32_t)__builtin_amdgcn_readlane((int)j, (int)last), ended);
                if (base + kWave < s1) walk.request();
            }
            const bool act = lane <= last, field = act && k >= 0;
            const uint64_t at = base + lane - v - 1;  // the entry (k >= 0)
            const uint32_t x = field ? col[at] : 0u;
            uint32_t prev = dpp_move<0x138>(x);
            if (lane == 0) prev = px;
            px = (uint32_t)__builtin_amdgcn_readlane((int)x, kWave - 1);
            uint32_t a = 0, b = 0;
            const uint32_t diff = x < v ? v - x : x - v;
            if (field) {
                general |= (x >> 31) || (k && x <= prev);
                images |= x >= n || (FMT == kGT && i == 0 && diff == 0);
                if (FMT == kGT) {
                    if (i == 0) a = diff ? diff - 1 : 1u;
                    else b = x - prev - 1;
                } else {
                    if (k == 0 || end) a = diff;
                    if (i) {
                        const uint32_t* r = col + (at - i);
                        const uint32_t L = c < R ? q + 1 : q;
                        const int32_t res = flat_residual(x, r[0], r[L], i, L);
                        b = (uint32_t)(res < 0 ? -res : res);
                    }
                }
                if (x < v ? end : !k || prev < v) fps[v] = x < v ? (FMT == kLE ? C + 1 : C) : c + (i != 0);
            }
            if (whole) {  // lane 63 alone can end the list
                a = wave_or_last(a) | ca;
                b = wave_or_last(b) | cb;
            } else {
                const SegmentScan seg(head);
                a = seg.any(a) | (j ? 0u : ca);
                b = seg.any(b) | (j ? 0u : cb);
            }
            if (act && end) {
                if (v == before) {
                    atomicOr(&ors[v].x, a);
                    atomicOr(&ors[v].y, b);
                } else {
                    ors[v] = make_uint2(a, b);
                }
            }
            ca = ended ? 0u : (uint32_t)__builtin_amdgcn_readlane((int)a, (int)last);
            cb = ended ? 0u : (uint32_t)__builtin_amdgcn_readlane((int)b, (int)last);
        }
        if (lane == 0 && (ca | cb)) {
            atomicOr(&ors[walk.cur].x, ca);
            atomicOr(&ors[walk.cur].y, cb);
        }
    }
    const unsigned long long f = (__ballot(general) ? kFlatGeneral : 0) | (__ballot(images) ? kFlatImages : 0);
    if (lane == 0 && f) atomicOr(&stats->flags, f);
}

// Widths, first_pos and lengths from the ORs: widths[v] = (f1 | f2 << 8 | header bits << 16, first_pos),
// len[v] = the record's bits, or the words of its payload in the GT stream.
template <int FMT, bool STREAM>
__global__ __launch_bounds__(kFlatBlock) void flat_vertex_kernel(const uint64_t* __restrict__ rowptr,
                                                                 const uint32_t* __restrict__ col, uint64_t n,
                                                                 const uint2* __restrict__ ors,
                                                                 const uint32_t* __restrict__ fps, uint32_t sh,
                                                                 uint64_t* __restrict__ len, uint2* __restrict__ widths,
                                                                 FlatStats* stats) {
    __shared__ unsigned long long lds[kFlatWaves];
    unsigned long long bits = 0, longest = 0, deg = 0, runs = 0, words = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * kFlatBlock + threadIdx.x; v < n; v += (uint64_t)gridDim.x * kFlatBlock) {
        const uint64_t base = rowptr[v];
        Hdr h;
        h.d = (uint32_t)(rowptr[v + 1] - base);
        h.f1 = h.f2 = h.fp = h.C = h.q = h.R = 0;
        h.pay = 0;
        uint32_t hb;
        uint64_t len_v;
        if (h.d >= (FMT == kLE ? 2u : 1u)) {
            flat_geometry<FMT>(h.d, h.C, h.q, h.R);
            const uint2 o = ors[v];
            h.fp = fps[v];
            h.f1 = bit_num(o.x);
            const uint32_t heads = FMT == kLE ? h.C + 1 : h.C;
            if (h.d > heads) h.f2 = bit_num(o.y);
            hb = gamma_bits(h.d) + gamma_bits(h.f1) + gamma_bits(h.f2) + gamma_bits(h.fp);
            len_v = hb + (uint64_t)heads * h.f1 + (uint64_t)(h.d - heads) * (FMT == kLE ? h.f2 + 1 : h.f2);
        } else {
            hb = FMT == kGT ? 4 * gamma_bits(0) : h.d ? gamma_bits(1) + gamma_bits(col[base]) : gamma_bits(0);
            len_v = hb;
        }
        widths[v] = make_uint2(h.f1 | (h.f2 << 8) | (hb << 16), h.fp);
        bits += len_v;
        longest = len_v > longest ? len_v : longest;
        deg = h.d > deg ? h.d : deg;
        runs += list_runs(FMT, h.d, h.C, h.q, run_shift(FMT, sh));
        if (STREAM) {
            len_v = (gtx_payload_bits(h, sh) + 31) >> 5;
            words += len_v;
        }
        len[v] = len_v;
    }
    bits = block_sum<unsigned long long, kFlatBlock>(bits, lds);
    runs = block_sum<unsigned long long, kFlatBlock>(runs, lds);
    if (STREAM) words = block_sum<unsigned long long, kFlatBlock>(words, lds);
    longest = block_max<unsigned long long, kFlatBlock>(longest, lds);
    deg = block_max<unsigned long long, kFlatBlock>(deg, lds);
    if (threadIdx.x == 0) {
        atomicAdd(&stats->bits, bits);
        atomicAdd(&stats->runs, runs);
        if (STREAM) atomicAdd(&stats->words, words);
        atomicMax(&stats->longest, longest);
        atomicMax(&stats->max_degree, deg);
        if (blockIdx.x == 0) stats->m = rowptr[n];
    }
}

// The header cache and the degrees of the resident graph (what the loader decodes from .graph).
template <int FMT>
__global__ __launch_bounds__(kFlatBlock) void flat_header_kernel(const uint64_t* __restrict__ rowptr,
                                                                 const uint32_t* __restrict__ col, uint64_t n,
                                                                 const uint64_t* __restrict__ start,
                                                                 const uint2* __restrict__ widths,
                                                                 uint4* __restrict__ hdr, uint32_t* __restrict__ deg) {
    for (uint64_t v = (uint64_t)blockIdx.x * kFlatBlock + threadIdx.x; v < n; v += (uint64_t)gridDim.x * kFlatBlock) {
        const uint64_t base = rowptr[v];
        const uint2 wd = widths[v];
        Hdr h;
        h.d = (uint32_t)(rowptr[v + 1] - base);
        h.f1 = wd.x & 0xFFu;
        h.f2 = (wd.x >> 8) & 0xFFu;
        h.fp = wd.y;
        h.C = h.q = h.R = 0;
        h.pay = FMT == kGT ? start[v] << 5 : start[v] + (wd.x >> 16);
        if (h.d >= (FMT == kLE ? 2u : 1u)) flat_geometry<FMT>(h.d, h.C, h.q, h.R);
        else if (FMT == kLE && h.d) h.f1 = col[base];
        hdr[v] = pack_hdr(h, FMT);
        deg[v] = h.d;
    }
}

// The words of a chunk's passes.  A chunk owns the words whose first bit its slots hold; its last pass
// reaches kFlatLook slots past them (a slot or the one after it has at least two bits, and the stream's
// padding ends a word) to complete the last of these: every word is stored once and nothing is ORed into
// memory.  A pass assembles its words in LDS; its partial last word is carried into the next.
template <bool SWAP>  // stored byte-swapped
struct FlatWindow {
    uint32_t* B;
    uint32_t* __restrict__ out;
    uint64_t from0, w0;  // bit of the chunk's first slot; word of the pass's first bit
    uint64_t pend_w;     // the carried word's index, ~0 when there is none
    uint32_t pend, nwords;

    __device__ __forceinline__ void store(uint64_t w, uint32_t x) const { out[w] = SWAP ? __builtin_bswap32(x) : x; }

    // Bits [from, to) are put next (put_field at B, w0).
    __device__ __forceinline__ void begin(bool first, uint64_t from, uint64_t to) {
        const uint32_t lane = lane_id();
        w0 = from >> 5;
        if (first) {
            from0 = from;
            pend_w = ~0ull;
        }
        if (pend_w != ~0ull && pend_w != w0) {  // completed by padding
            if (lane == 0 && pend_w << 5 >= from0) store(pend_w, pend);
            pend_w = ~0ull;
        }
        nwords = to > from ? (uint32_t)(((to - 1) >> 5) - w0 + 1) : pend_w == w0 ? 1u : 0u;
        for (uint32_t x = lane; x < nwords; x += kWave) B[x] = x == 0 && pend_w == w0 ? pend : 0u;
        wave_sync();
    }
    // The chunk's last pass stores the words that start before bit `end`.
    __device__ __forceinline__ void finish(bool last, uint64_t to, uint64_t end) {
        wave_sync();
        if (!last) end = to & ~31ull;
        for (uint32_t x = lane_id(); x < nwords; x += kWave) {
            const uint64_t bit = (w0 + x) << 5;
            if (bit >= from0 && bit < end) store(w0 + x, B[x]);
        }
        const bool part = !last && nwords && (to & 31);
        pend = part ? B[nwords - 1] : 0u;
        pend_w = part ? w0 + nwords - 1 : ~0ull;
        wave_sync();
    }
};

// GT stream: fields of a list's checkpoint positions before position i of block b (each takes 32 bits in
// place of f2).
__device__ __forceinline__ uint32_t flat_checkpoints(uint32_t b, uint32_t i, uint32_t q, uint32_t R, uint32_t sh) {
    const uint32_t lo = min(b, R);
    return __umul24(lo, q >> sh) + __umul24(b - lo, (q - 1) >> sh) + (i ? (i - 1) >> sh : 0u);
}

enum FlatOut { kFlatImage, kFlatResident };

// The words of the .graph image (kFlatImage: stored byte-swapped, as the file's bytes), or of the
// resident graph: LE the same words, GT the checkpointed payload stream (no headers; start[] in words).
template <int FMT, FlatOut OUT>
__global__ __launch_bounds__(kFlatBlock) void flat_write_kernel(const uint64_t* __restrict__ rowptr,
                                                                const uint32_t* __restrict__ col, uint64_t n,
                                                                const uint64_t* __restrict__ start,
                                                                const uint2* __restrict__ widths, uint32_t sh,
                                                                uint32_t* __restrict__ out) {
    constexpr bool STREAM = FMT == kGT && OUT == kFlatResident;
    __shared__ uint32_t own_lds[kFlatBlock];
    __shared__ uint32_t buf[kFlatWaves][kFlatWords + 1];
    uint32_t* own = own_lds + (threadIdx.x & ~(kWave - 1));
    FlatWindow<OUT == kFlatImage> win{buf[threadIdx.x / kWave], out};
    const uint32_t lane = lane_id();
    const uint64_t waves = (uint64_t)gridDim.x * kFlatWaves;
    const uint64_t slots = rowptr[n] + n;
    const uint32_t passes = flat_passes(slots, waves);
    const uint64_t W = (uint64_t)passes * kWave - kFlatLook;
    for (uint64_t s0 = ((uint64_t)blockIdx.x * kFlatBlock + threadIdx.x) / kWave * W; s0 < slots; s0 += waves * W) {
        SlotWalk walk{rowptr, n};
        walk.seek(s0);
        uint64_t st = 0;
        uint2 wd = make_uint2(0u, 0u);
        auto request = [&]() {
            if (walk.cur + (uint64_t)lane < n) {
                st = start[walk.cur + lane];
                wd = widths[walk.cur + lane];
            }
        };
        request();
        FlatList<FMT> list;
        uint32_t px = FMT == kGT && s0 - walk.sc >= 2 ? col[s0 - walk.cur - 2] : 0u;
        for (uint32_t t = 0; t < passes; ++t) {
            const uint64_t base = s0 + (uint64_t)t * kWave;
            if (base >= slots) break;
            const bool fin = t + 1 == passes || base + kWave >= slots;
            const uint32_t last = (uint32_t)(slots - base < (uint64_t)kWave ? slots - base - 1 : kWave - 1);
            uint32_t j, d, head, C, q, R, wx, fp = 0;
            int32_t k;
            uint64_t sv;
            const bool whole = last == kWave - 1 && walk.in_list(base);  // the pass is in one list
            if (whole) {
                j = 0;
                k = (int32_t)(base - walk.sc) + (int32_t)lane - 1;
                d = (uint32_t)(readlane_u64(walk.bj, 0) - walk.sc) - 1;
                list.of(walk.cur, d);
                C = list.C;
                q = list.q;
                R = list.R;
                wx = lane_get(wd.x, 0);
                sv = readlane_u64(st, 0);
            } else {
                walk.place(base, last, own, j, k, d, head);
                flat_geometry<FMT>(d, C, q, R);
                wx = __shfl(wd.x, (int)j, kWave);
                if (!STREAM) fp = __shfl(wd.y, (int)j, kWave);
                sv = ((uint64_t)__shfl((uint32_t)(st >> 32), (int)j, kWave) << 32) | __shfl((uint32_t)st, (int)j, kWave);
            }
            const uint32_t v = walk.cur + j;
            const bool ended = __builtin_amdgcn_readlane((int)(k + 1 == (int32_t)d), (int)last);
            if (!whole || ended) {
                walk.advance((uint32_t)__builtin_amdgcn_readlane((int)j, (int)last), ended);
                if (!fin) {
                    walk.request();
                    request();
                }
            }
            const bool act = lane <= last, field = act && k >= 0;
            const uint32_t f1 = wx & 0xFFu, f2 = (wx >> 8) & 0xFFu, hb = STREAM ? 0u : wx >> 16;
            const uint64_t pay = STREAM ? sv << 5 : sv + hb;
            const uint64_t row = base + lane - v - 1 - (int64_t)k;  // the list's first entry
            uint64_t at = pay;
            uint32_t wdt = 0, val = 0;
            if (FMT == kGT) {
                const uint32_t x = field ? col[row + k] : 0u;
                uint32_t prev = dpp_move<0x138>(x);
                if (lane == 0) prev = px;
                px = (uint32_t)__builtin_amdgcn_readlane((int)x, kWave - 1);
                uint32_t b, i;
                if (whole) list.pos((uint32_t)k, b, i);
                else flat_pos(k < 0 ? 0u : (uint32_t)k, q, R, b, i);
                const uint32_t diff = x < v ? v - x : x - v, heads = b + (i != 0);
                if (field) {
                    at = pay + __umul24(heads, f1) + (uint64_t)((uint32_t)k - heads) * f2;
                    val = i ? x - prev - 1 : diff ? diff - 1 : 1u;
                    wdt = i ? f2 : f1;
                    if (STREAM) {
                        at += (uint64_t)flat_checkpoints(b, i, q, R, sh) * (32 - f2);
                        if (i && !(i & ((1u << sh) - 1))) {
                            val = x;
                            wdt = 32;
                        }
                    }
                }
            } else if (field && d > 1) {
                const uint32_t* N = col + row;
                if ((uint32_t)k <= C) {
                    const uint32_t x = N[__umul24((uint32_t)k, q) + min((uint32_t)k, R)];
                    at = pay + __umul24((uint32_t)k, f1);
                    wdt = f1;
                    val = x < v ? v - x : x - v;
                } else {
                    // seas, chunk by chunk: R chunks of q of them, then chunks of q - 1
                    const uint32_t s = (uint32_t)k - C - 1, big = __umul24(R, q);
                    const bool lo = s < big;
                    const uint32_t len = lo ? q : q - 1, ss = lo ? s : s - big;
                    const uint32_t cc = udiv_chunk(ss, len), i = ss - __umul24(cc, len) + 1, c = lo ? cc : cc + R;
                    const uint32_t* r = N + (__umul24(c, q) + min(c, R));
                    const int32_t res = flat_residual(r[i], r[0], r[len + 1], i, len + 1);
                    at = pay + __umul24(C + 1, f1) + (uint64_t)s * (f2 + 1);
                    wdt = f2 + 1;
                    val = ((uint32_t)(res < 0 ? -res : res) << 1) | (res < 0 ? 1u : 0u);
                }
            }
            if (k < 0 && !STREAM) {
                at = sv;
                wdt = hb;
            }
            const uint64_t from = readlane_u64(at, 0), to = readlane_u64(at + wdt, (int)last);
            const uint64_t end = s0 + W < slots ? readlane_u64(at, kWave - kFlatLook) : ~0ull;  // (last pass)
            win.begin(t == 0, from, to);
            if (field) put_field(win.B, win.w0, at, wdt, wdt < 32 ? val & ((1u << wdt) - 1) : val);
            if (!STREAM && act && k < 0) {
                put_gamma(win.B, win.w0, at, d);
                if (FMT == kGT || d > 1) {
                    put_gamma(win.B, win.w0, at, f1);
                    put_gamma(win.B, win.w0, at, f2);
                    put_gamma(win.B, win.w0, at, fp);
                } else if (d) {
                    put_gamma(win.B, win.w0, at, col[row]);
                }
            }
            win.finish(fin, to, end);
        }
    }
}

}  // namespace grass
