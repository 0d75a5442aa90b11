// Full decode of the resident compressed graph to CSR (rowptr u64[n+1], col u32[m]).
//
// Run-parallel (LE, and GT with a checkpoint interval P <= 4): each wave64 owns a contiguous range
// of runs, a run being at most 4 consecutive positions that one lane decodes by itself -- LE: of one
// chunk, from the chunk's rock pair and one contiguous span of seas (LE/src/bcg.cuh:196-261 decodes
// a position at a time); GT: a block head or checkpoint and the gaps after it.  The outputs of a
// wave's 64 runs are consecutive, so they are staged in LDS and stored with coalesced writes.
//
// Slot-parallel (GT with P > 4): each wave owns a contiguous range of output slots (a tuning choice).
// When 64 consecutive slots lie in one list the wave reads that vertex's header once and divides
// through shared multiply-high reciprocals; otherwise each lane finds its vertex from the 64 row
// ends after the previous owner (one coalesced load and a register search).  Block heads and
// checkpoints are absolute and every other body is a gap, so the wave turns (absolute | gap+1)
// values into ids with a segmented prefix sum, carrying the running id from lane 63 into the next
// 64 slots (the cooperative decode of GT/src/bcg.cuh:171-345 and GT/src/grass.cu:525-553, without
// its per-warp cache limits).  A wave whose range starts between two absolute positions first backs
// up to the earlier one.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "devutil.h"
#include "runtime.h"
#include "scan.h"

namespace grass {

constexpr int kDecBlock = 256;

struct DegGen {
    const uint32_t* deg;
    __device__ __forceinline__ uint64_t operator()(uint64_t i) const { return deg[i]; }
};

// Largest v in [lo, hi] with rowptr[v] <= e.
__device__ __forceinline__ uint32_t owner_of(const uint64_t* __restrict__ rowptr, uint32_t lo,
                                             uint32_t hi, uint64_t e) {
    while (lo < hi) {
        uint32_t mid = lo + (hi - lo + 1) / 2;
        if (rowptr[mid] <= e) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// wstart[w] = the vertex that holds slot w * per_wave, the first slot of decode wave w: each
// vertex writes the waves that start inside its list.
__global__ __launch_bounds__(256) void wave_start_kernel(const uint64_t* __restrict__ rowptr, uint32_t n,
                                                         uint32_t per_wave, uint64_t waves,
                                                         uint32_t* __restrict__ wstart) {
    for (uint64_t v = (uint64_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (uint64_t)gridDim.x * 256) {
        const uint64_t b = rowptr[v], e = rowptr[v + 1];
        for (uint64_t w = (b + per_wave - 1) / per_wave; w < waves && w * per_wave < e; ++w)
            wstart[w] = (uint32_t)v;
    }
}

// A GT list in the device stream with its wave-uniform constants: block geometry, field
// widths, the bits of a (q + 1)- and of a q-position block, and shared divisors, so that an
// element costs two multiply-high divisions and one 32-bit window.
struct GtList {
    uint64_t pay;
    uint32_t v, f1, f2, fp, q, R, big, F1, F0, sh;
    UDiv d1, d0;
    __device__ __forceinline__ void init(const Hdr& h, uint32_t vv, uint32_t shift) {
        pay = h.pay;
        v = vv;
        f1 = h.f1;
        f2 = h.f2;
        fp = h.fp;
        q = h.q;
        R = h.R;
        sh = shift;
        big = (q + 1) * R;
        F1 = (uint32_t)gtx_field(h, q + 1, shift);
        F0 = (uint32_t)gtx_field(h, q, shift);
        d1.init(q + 1);
        d0.init(q);
    }
    // Element k: the absolute id at a block head or checkpoint (head = 1), else the gap + 1.  The
    // field's bit, width and kind are chosen first, so every lane issues the same one load.
    template <class Src>
    __device__ __forceinline__ uint32_t at(const Src& w, uint32_t k, int& head) const {
        uint32_t blk, i;
        uint64_t bo;
        if (k < big) {
            blk = d1.div(k);
            i = k - blk * (q + 1);
            bo = pay + (uint64_t)blk * F1;
        } else {
            const uint32_t kk = k - big, b2 = d0.div(kk);
            i = kk - b2 * q;
            blk = b2 + R;
            bo = pay + (uint64_t)R * F1 + (uint64_t)b2 * F0;
        }
        const uint32_t j = i - 1;
        const bool hd = i == 0, abs = !hd && (i & ((1u << sh) - 1)) == 0;
        const uint32_t off = hd ? 0u : f1 + j * f2 + (j >> sh) * (32 - f2);
        const uint32_t raw = w.read(bo + off, hd ? f1 : abs ? 32u : f2);
        head = hd || abs;
        return hd ? (blk >= fp ? v + raw + 1 : v - raw - 1) : abs ? raw : raw + 1;
    }
};

// Where the GT payload words come from: the stream in global memory, or a wave's LDS copy of the
// span of the stream its range of slots covers (L[0] is stream word W0).
struct GlobalWords {
    const uint32_t* __restrict__ w;
    __device__ __forceinline__ uint32_t read(uint64_t b, uint32_t nbits) const { return read_bits(w, b, nbits); }
};
struct LdsWords {
    const uint32_t* L;
    uint64_t W0;
    __device__ __forceinline__ uint32_t read(uint64_t b, uint32_t nbits) const {
        const uint32_t o = (uint32_t)((b >> 5) - W0);
        const uint64_t x = ((uint64_t)L[o] << 32) | L[o + 1];
        return (uint32_t)(x >> (32 - (uint32_t)(b & 31))) >> (32 - nbits);
    }
};

// gt_element (codec.h) on a word source.
template <class Src>
__device__ __forceinline__ uint32_t gt_element_src(const Src& w, const Hdr& h, uint32_t v, uint32_t blk, uint32_t i,
                                                   uint32_t sh, int& head) {
    const uint64_t bo = gtx_block_bit(h, blk, sh);
    const bool hd = i == 0, abs = !hd && (i & ((1u << sh) - 1)) == 0;
    const uint32_t raw = w.read(bo + gtx_field(h, i, sh), hd ? h.f1 : abs ? 32u : h.f2);
    head = hd || abs;
    return hd ? (blk >= h.fp ? v + raw + 1 : v - raw - 1) : abs ? raw : raw + 1;
}

// The slots [e0, e1) of one wave: vlo owns e0, vhi bounds the owner of e1 - 1, decoding starts
// at eb <= e0 (a run's absolute value); GT payload words come from `src`.
template <class Src>
__device__ __forceinline__ void decode_range(const DevGraph& g, const Src& src, const uint64_t* __restrict__ rowptr,
                                             uint32_t* __restrict__ col, uint64_t e0, uint64_t e1, uint64_t eb,
                                             uint32_t vlo, uint32_t vhi, uint32_t span) {
    const int lane = lane_id();
    uint32_t carry = 0;
    // owner of the iteration's first slot (a lower bound for every lane's) and its row bounds,
    // wave-uniform, reloaded only when it changes
    uint32_t cur = __builtin_amdgcn_readfirstlane(vlo);
    uint64_t rc = rowptr[cur], rn = rowptr[cur + 1];
    uint32_t hv = 0xFFFFFFFFu;  // vertex whose list constants are cached below
    Hdr uh;
    GtList gl;
    for (uint64_t base = eb; base < e1; base += kWave) {
        const uint64_t e = base + lane;
        const bool act = e < e1;
        const uint64_t ee = act ? e : e1 - 1;
        uint32_t x;
        int head = 1;
        if (base >= rc && base + (kWave - 1) < rn) {
            // the whole wave is inside one list: one header, shared constants, no owner search
            if (cur != hv) {
                hv = cur;
                load_hdr<kGT>(g, hv, uh);
                gl.init(uh, hv, g.cp_shift);
            }
            x = gl.at(src, (uint32_t)(ee - rc), head);
        } else {
            // Owner of slot ee: one coalesced load of the 64 row ends after `cur` (and, beside
            // it, of those 64 vertices' headers), then a 6-step search over them in registers;
            // slots more than 64 vertices past `cur` (only possible across vertices without
            // edges) fall back to a binary search of rowptr.  The owner's header then comes from
            // the lane that loaded it, and the next window's row bounds from the row ends.
            // (row ends as 32-bit offsets from the start of `cur`'s list, which is at or before
            // every slot of the iteration; one list is < 2^31 entries, larger offsets saturate)
            const uint64_t bj = (uint64_t)cur + 1 + lane <= g.n ? rowptr[cur + 1 + lane] : ~0ull;
            uint4 hj = make_uint4(0u, 0u, 0u, 0u);
            if (cur + (uint32_t)lane < g.n) hj = g.hdr[cur + lane];
            const uint32_t rj = bj - rc > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)(bj - rc);
            const uint32_t er = (uint32_t)(ee - rc);
            uint32_t pos = 0;
#pragma unroll
            for (uint32_t st = 32; st >= 1; st >>= 1) {
                const uint32_t t = __shfl(rj, (int)(pos + st - 1), kWave);
                if (t <= er) pos += st;
            }
            const uint32_t last = __shfl(rj, kWave - 1, kWave);
            if (pos == kWave - 1 && last <= er) pos = kWave;
            const uint32_t prev = __shfl(rj, (int)(pos > 0 ? pos - 1 : 0), kWave);
            const int src_lane = (int)(pos < (uint32_t)kWave ? pos : 0u);
            uint4 hv4 = make_uint4(__shfl(hj.x, src_lane, kWave), __shfl(hj.y, src_lane, kWave),
                                   __shfl(hj.z, src_lane, kWave), __shfl(hj.w, src_lane, kWave));
            uint32_t v;
            uint64_t vstart;
            if (pos < (uint32_t)kWave) {
                v = cur + pos;
                vstart = rc + (pos ? prev : 0u);
            } else {
                v = owner_of(rowptr, cur + kWave, vhi, ee);
                vstart = rowptr[v];
                hv4 = g.hdr[v];
            }
            const uint32_t p63 = (uint32_t)__builtin_amdgcn_readlane((int)pos, kWave - 1);
            if (p63 < (uint32_t)kWave) {
                if (p63) {
                    cur += p63;
                    rc = readlane_u64(bj, (int)p63 - 1);
                    rn = readlane_u64(bj, (int)p63);
                }
            } else {
                cur = __builtin_amdgcn_readlane((int)v, kWave - 1);
                rc = rowptr[cur];
                rn = rowptr[cur + 1];
            }
            const uint32_t k = (uint32_t)(ee - vstart);
            Hdr h;
            unpack_hdr<kGT>(hv4, h);
            uint32_t blk, i;
            gt_locate(h, k, blk, i);
            x = gt_element_src(src, h, v, blk, i, g.cp_shift, head);
        }
        if (lane == 0 && !head) {
            x += carry;
            head = 1;
        }
        x = short_segmented_sum(x, head, span);
        carry = (uint32_t)__builtin_amdgcn_readlane((int)x, kWave - 1);
        if (act && e >= e0) col[e] = x;
    }
}

// ---------------------------------------------------------------- runs (LE; GT with P <= 4)
// A run is at most 4 consecutive positions of a list that decode without any other run.
//   GT: a block head or a checkpoint and the gap fields after it up to the next one: the absolute
//       field and its gaps are one contiguous span of the stream.
//   LE: positions [4j, 4j + 4) of a chunk (the list's last position, rock C, is a chunk of one): the
//       chunk's rock pair, one division for its slope, and one contiguous span of at most 4 seas.
// The run kernel gives each lane one run: its slots and stream bits from the run's index in its list
// (no per-position division), its fields from one 16-byte load (a fifth word when they reach past
// it; LE: and one for the rock pair), its ids in registers (no cross-lane scan).  The 64 runs of a
// wave's pass fill consecutive output slots, which are staged in LDS and stored with coalesced
// writes.  Runs are numbered over the graph (roff = exclusive scan of runs per vertex) and every
// wave takes a fixed number of them, with its first vertex from a table like the slot-based one.
// Bound by instruction issue, then by the loads a pass waits for, so the geometry avoids branches
// and 32-bit multiplies, fields come off funnel shifts, a pass's output slots are a wave scan of its
// counts (no row pointers), and the next pass's run ends and headers are requested before the
// current pass decodes.  Measured on R-MAT, GT s24 (521 M entries) 1.05 -> 0.94 ms, 3.7 TB/s of the
// 3.5 GB it needs (a copy reaches 4.85); LE s22 (128 M) 0.62 ms with a lane per position, 0.38 by
// runs, 0.30 with the above.  Loading each lane's header by itself instead of 64 headers and a
// shuffle: GT 1.06 ms.

struct RunGen {  // runs of vertex i, from its header
    const uint4* hdr;
    int fmt;
    uint32_t sh;
    __device__ __forceinline__ uint64_t operator()(uint64_t i) const {
        const uint4 e = hdr[i];
        return list_runs(fmt, e.z, e.w & 0xFFFFu, e.y >> 16, sh);
    }
};

// One run's place: its positions [i0, i0 + cnt) of block (chunk) blk, which has len positions; GT:
// the stream bit of its absolute field.
struct RunAt {
    uint64_t bit;
    uint32_t cnt, blk, i0, len;
    uint32_t pos;  // position in the list of its first entry
};

// The list constants of run_at's division by the runs per block (nr1 for blocks of q + 1
// positions, nr0 for blocks of q): per lane with a float reciprocal, or shared by the wave.
struct RunDivLane {
    __device__ __forceinline__ uint32_t operator()(uint32_t n, uint32_t d, bool) const {
        return udiv_chunk(n, max(d, 1u));  // (LE, d = 1: no runs per chunk, the one run is run 0)
    }
};
struct RunDivShared {
    UDiv u1, u0;
    __device__ __forceinline__ uint32_t operator()(uint32_t n, uint32_t d, bool lo) const {
        UDiv u;
        u.d = d;
        u.m = lo ? u1.m : u0.m;
        return u.div(n);
    }
};

// Run rr (< the vertex's runs) of a vertex: R blocks of nr1 runs, then blocks of nr0 (LE: then the
// last rock, block C).  The block kind is chosen first, so lanes of both kinds share one division.
// C, q and a block's runs are below 2^16 and the field widths below 2^5, so all products but the
// bits of whole blocks are 24-bit multiplies (full rate, where 32-bit ones run at a quarter).
// P = 1 << sh positions per run; in a GT block, run j >= 1 starts f1 - 32 + j K bits after the head's
// field, K = 32 + (P - 1) f2 (the bits of a whole run), and a block of q positions has the bits of
// one of q + 1 less one field, which is a checkpoint when q is a multiple of P.
template <int FMT, class Div>
__device__ __forceinline__ RunAt run_at(const Hdr& h, uint32_t rr, uint32_t sh, const Div& div) {
    const uint32_t P1 = (1u << sh) - 1;
    const uint32_t nr1 = (h.q + 1 + P1) >> sh, nr0 = (h.q + P1) >> sh;
    const uint32_t bigr = __umul24(h.R, nr1);
    const bool lo = rr < bigr;
    const uint32_t t = lo ? rr : rr - bigr, nr = lo ? nr1 : nr0;
    const uint32_t b = div(t, nr, lo);
    const uint32_t j = t - __umul24(b, nr);
    RunAt a;
    a.blk = lo ? b : b + h.R;
    a.len = lo ? h.q + 1 : h.q;
    a.i0 = j << sh;
    a.pos = __umul24(b, a.len) + (lo ? 0u : __umul24(h.R, h.q + 1)) + a.i0;
    if (FMT == kLE && a.blk == h.C) a.len = 1;
    a.cnt = min(P1 + 1, a.len - a.i0);
    a.bit = 0;
    if (FMT == kGT) {
        const uint32_t K = 32 + __umul24(P1, h.f2);
        const uint32_t F1 = h.f1 + __umul24(h.q, h.f2) + __umul24(h.q >> sh, 32 - h.f2);
        const uint32_t F = lo ? F1 : F1 - ((h.q & P1) ? h.f2 : 32u);
        a.bit = h.pay + (uint64_t)b * F + (lo ? 0ull : (uint64_t)h.R * F1) + (j ? h.f1 - 32 + __umul24(j, K) : 0u);
    }
    return a;
}

// The ids of one GT run into out[0 .. cnt): the absolute field, then each gap + 1 added on.  One
// 16-byte load holds the field's offset in its word (< 32), a 32-bit field and three gaps of up to
// 21 bits; a fifth word is read when they need more.  (Ids past cnt are not meaningful.)
__device__ __forceinline__ void gt_run_ids(const uint32_t* __restrict__ w, const Hdr& h, uint32_t v, const RunAt& a,
                                           uint32_t out[kRunMax]) {
    const uint32_t* p = w + (a.bit >> 5);
    const Words4 q = *(const Words4*)p;
    const uint32_t s = (uint32_t)(a.bit & 31);
    const bool head = a.i0 == 0;
    const uint32_t aw = head ? h.f1 : 32u, f2 = h.f2;
    FieldReader f(q, s + aw + __umul24(a.cnt - 1, f2) > 128 ? p[4] : 0u, s);
    const uint32_t a0 = f.take(aw);  // f1 >= 1 for a vertex with entries
    const uint32_t x0 = head ? (a.blk >= h.fp ? v + a0 + 1 : v - a0 - 1) : a0;
    out[0] = x0;
    if (f2) {
        out[1] = x0 + f.take(f2) + 1;
        out[2] = out[1] + f.take(f2) + 1;
        out[3] = out[2] + f.take(f2) + 1;
    } else {  // (0-bit gap fields read as 0)
        out[1] = x0 + 1;
        out[2] = x0 + 2;
        out[3] = x0 + 3;
    }
}

// The ids of one LE run (le_get, codec.h, for each of its positions): rocks c and c + 1 in one
// window, the interpolation's slope once, and the run's seas, which follow each other.  Both loads
// are issued before either is used; the rock window of the last rock and the sea span of a run
// without seas lie at most four words past the record, inside the padded image.
__device__ __forceinline__ void le_run_ids(const uint32_t* __restrict__ w, const Hdr& h, uint32_t v, const RunAt& a,
                                           uint32_t out[kRunMax]) {
    if (h.d == 1) {
        out[0] = out[1] = out[2] = out[3] = h.f1;
        return;
    }
    const uint32_t c = a.blk, rb = h.f1, sw = h.f2 + 1;
    const uint32_t i1 = a.i0 ? a.i0 : 1u;  // first sea's position in the chunk
    const bool rock = a.i0 == 0;           // the run starts with the rock
    const uint32_t j = __umul24(h.q - 1, c) + min(c, h.R) + i1 - 1;
    const uint64_t rbit = h.pay + __umul24(c, rb);
    const uint64_t sbit = h.pay + __umul24(h.C + 1, rb) + (uint64_t)j * sw;
    const Words4 rq = *(const Words4*)(w + (rbit >> 5));
    const uint32_t* sp = w + (sbit >> 5);
    const Words4 sq = *(const Words4*)sp;
    const uint32_t ss = (uint32_t)(sbit & 31), rs = (uint32_t)(rbit & 31);
    const uint32_t w4 = ss + __umul24(a.cnt, sw) > 128 ? sp[4] : 0u;
    const uint32_t u0 = FieldReader::shl0(rq.x, rq.y, rs);
    const uint32_t u1 = FieldReader::shl0(rq.y, rq.z, rs);
    const uint32_t r1 = u0 >> (32 - rb), r2 = FieldReader::shl(u0, u1, rb) >> (32 - rb);
    const uint32_t A = c < h.fp ? v - r1 : v + r1;
    const uint32_t Z = c + 1 < h.fp ? v - r2 : v + r2;
    const uint32_t step = a.len > 1 ? udiv_chunk(Z - A, a.len) : 0u;
    FieldReader f(sq, w4, ss);
    uint32_t x = A + step * i1, e[kRunMax];
#pragma unroll
    for (uint32_t k = 0; k < kRunMax; ++k) {  // seas i1, i1 + 1, ...
        const uint32_t r = f.take(sw), mag = r >> 1;
        e[k] = x + ((r & 1) ? 0u - mag : mag);
        x += step;
    }
    out[0] = rock ? A : e[0];
    out[1] = rock ? e[0] : e[1];
    out[2] = rock ? e[1] : e[2];
    out[3] = rock ? e[2] : e[3];
}

// Wave w decodes runs [w * per_wave, ...) of the graph; rstart[w] is the vertex holding its first.
template <int FMT>
__global__ __launch_bounds__(kDecBlock) void decode_runs_kernel(DevGraph g, const uint64_t* __restrict__ rowptr,
                                                                const uint64_t* __restrict__ roff,
                                                                const uint32_t* __restrict__ rstart,
                                                                uint32_t* __restrict__ col, uint64_t nruns,
                                                                uint32_t per_wave, uint32_t sh) {
    __shared__ uint32_t stage_lds[(kDecBlock / kWave) * kWave * kRunMax];
    __shared__ uint32_t owner_lds[kDecBlock];
    uint32_t* L = stage_lds + (threadIdx.x / kWave) * (kWave * kRunMax);
    uint32_t* own = owner_lds + (threadIdx.x & ~(kWave - 1));
    const uint64_t wave = ((uint64_t)blockIdx.x * kDecBlock + threadIdx.x) / kWave;
    const int lane = lane_id();
    const uint64_t r0 = wave * per_wave;
    if (r0 >= nruns) return;  // uniform per wave
    const uint64_t r1 = r0 + per_wave < nruns ? r0 + per_wave : nruns;
    // the vertex of the pass's first run and its run bounds, wave-uniform
    uint32_t cur = __builtin_amdgcn_readfirstlane(rstart[wave]);
    uint64_t rc = roff[cur], rn = roff[cur + 1];
    uint32_t hv = 0xFFFFFFFFu;  // vertex whose list constants are cached below
    Hdr uh;
    RunDivShared ud;
    // the pass's first output slot: from the row pointer here, then carried from pass to pass
    uint64_t sb;
    {
        Hdr h;
        load_hdr<FMT>(g, cur, h);
        sb = rowptr[cur] + run_at<FMT>(h, (uint32_t)(r0 - rc), sh, RunDivLane{}).pos;
    }
    // run ends and headers of the 64 vertices from `cur`, requested a pass ahead
    uint64_t bj = 0;
    uint4 hj = make_uint4(0u, 0u, 0u, 0u);
    auto request = [&]() {
        bj = (uint64_t)cur + 1 + lane <= g.n ? roff[cur + 1 + lane] : ~0ull;
        if (cur + (uint32_t)lane < g.n) hj = g.hdr[cur + lane];
    };
    auto in_list = [&](uint64_t base) { return base >= rc && base + (kWave - 1) < rn; };
    if (!in_list(r0)) request();
    for (uint64_t base = r0; base < r1; base += kWave) {
        const uint64_t rho = base + lane;
        const bool act = rho < r1;
        const uint64_t rr = act ? rho : r1 - 1;
        RunAt a;
        Hdr h;
        uint32_t v;
        if (in_list(base)) {
            // the whole pass is in one list: one header, shared divisors
            if (cur != hv) {
                hv = cur;
                load_hdr<FMT>(g, hv, uh);
                const uint32_t P1 = (1u << sh) - 1;
                ud.u1.init((uh.q + 1 + P1) >> sh);
                ud.u0.init((uh.q + P1) >> sh);
            }
            h = uh;
            v = hv;
            a = run_at<FMT>(h, (uint32_t)(rr - rc), sh, ud);
        } else {
            // Vertex cur + j covers the pass's lanes from its first run on; each vertex that starts
            // a lane of the pass (or holds its first run) writes j + 1 into that lane's LDS slot,
            // and an inclusive max over the slots gives every lane its vertex (no search).  When
            // the 64 vertices end before the pass does (only across vertices without entries), each
            // lane searches the run offsets instead.
            const uint32_t rj = bj - rc > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)(bj - rc);
            const uint32_t pj = dpp_move<0x138>(rj);  // start of vertex cur + lane (lane 0: 0)
            const uint32_t e0 = (uint32_t)(base - rc);
            const uint32_t lastl = (uint32_t)(r1 - base < (uint64_t)kWave ? r1 - base - 1 : kWave - 1);
            const uint32_t elast = e0 + lastl;
            uint32_t ro;  // the lane's run in its vertex's list
            if ((uint32_t)__builtin_amdgcn_readlane((int)rj, kWave - 1) > elast) {
                const bool cand = rj > pj && rj > e0 && pj <= elast;
                own[lane] = 0;
                wave_sync();
                if (cand) own[pj > e0 ? pj - e0 : 0u] = lane + 1;
                wave_sync();
                int jo = (int)wave_inclusive_max(own[lane]) - 1;  // lane 0 always has a vertex
                wave_sync();
                const int jl = __builtin_amdgcn_readlane(jo, (int)lastl);
                jo = act ? jo : jl;
                v = cur + jo;
                ro = (uint32_t)(rr - rc) - __shfl(pj, jo, kWave);
                unpack_hdr<FMT>(make_uint4(__shfl(hj.x, jo, kWave), __shfl(hj.y, jo, kWave), __shfl(hj.z, jo, kWave),
                                           __shfl(hj.w, jo, kWave)), h);
                // the next pass starts at or after the last active lane's vertex
                if (jl) {
                    cur += jl;
                    rc = readlane_u64(bj, jl - 1);
                    rn = readlane_u64(bj, jl);
                }
            } else {
                v = owner_of(roff, cur, g.n - 1, rr);
                ro = (uint32_t)(rr - roff[v]);
                cur = (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lastl);
                rc = roff[cur];
                rn = roff[cur + 1];
                load_hdr<FMT>(g, v, h);
            }
            a = run_at<FMT>(h, ro, sh, RunDivLane{});
        }
        if (base + kWave < r1 && !in_list(base + kWave)) request();
        uint32_t ids[kRunMax];
        if (FMT == kLE) le_run_ids(g.w, h, v, a, ids);
        else gt_run_ids(g.w, h, v, a, ids);
        // the runs' slots follow each other: staged in LDS at the sum of the counts before, and
        // stored coalesced
        const uint32_t cnt = act ? a.cnt : 0u;
        const uint32_t inc = wave_inclusive_sum(cnt);
        const uint32_t o = inc - cnt, count = (uint32_t)__builtin_amdgcn_readlane((int)inc, kWave - 1);
#pragma unroll
        for (uint32_t k = 0; k < kRunMax; ++k)
            if (k < cnt) L[o + k] = ids[k];
        wave_sync();
        for (uint32_t k = lane; k < count; k += kWave) col[sb + k] = L[k];
        wave_sync();  // the stage is read before the next pass writes it
        sb += count;
    }
}

// LDS words a wave may copy its span into (the rest of a larger span is read from global memory).
constexpr uint32_t kDecStageMax = 2048;
__host__ __device__ constexpr uint32_t dec_stage_words(uint32_t per_wave) {
    return (per_wave < kDecStageMax ? per_wave : kDecStageMax) + 64;
}

// The slot-based kernel (GT, P > 4).  With stage != 0 the wave first copies the span of the payload stream its slots use (every
// field from its first run's absolute value to slot e1) into LDS with coalesced loads, all in
// flight together, when it fits `stage` words, and then decodes from LDS: no dependent global
// load per 64 slots.
__global__ __launch_bounds__(kDecBlock) void decode_csr_kernel(DevGraph g,
                                                               const uint64_t* __restrict__ rowptr,
                                                               const uint32_t* __restrict__ wstart,
                                                               uint32_t* __restrict__ col,
                                                               uint64_t m, uint32_t per_wave, uint32_t stage) {
    extern __shared__ uint32_t dec_lds[];
    const uint64_t wave = ((uint64_t)blockIdx.x * kDecBlock + threadIdx.x) / kWave;
    const int lane = lane_id();
    const uint64_t e0 = wave * per_wave;
    if (e0 >= m) return;  // uniform per wave
    const uint64_t e1 = e0 + per_wave < m ? e0 + per_wave : m;
    // owner of e0, and a bound on the owner of e1 - 1 (the next wave's first owner)
    const uint32_t vlo = wstart[wave];
    const uint32_t vhi = e1 < m ? wstart[wave + 1] : g.n - 1;
    // GT: an absolute value (block head or checkpoint) starts every run of at most P positions
    const uint32_t span = 1u << g.cp_shift;
    uint64_t eb = e0;
    const uint32_t sh = g.cp_shift;
    Hdr h;
    load_hdr<kGT>(g, vlo, h);
    uint32_t blk, i;
    gt_locate(h, (uint32_t)(e0 - rowptr[vlo]), blk, i);
    const uint32_t ib = i & ~(span - 1);
    eb = e0 - (i - ib);  // back to the block head or checkpoint
    if (stage) {
        // bits [B0, B1): from eb's field to slot e1's (the stream's end for the last wave);
        // a field read touches its word and the next, so words W0 ..= ((B1 - 1) >> 5) + 1
        const uint64_t B0 = gtx_block_bit(h, blk, sh) + gtx_field(h, ib, sh);
        Hdr hu;
        load_hdr<kGT>(g, vhi, hu);
        uint64_t B1;
        if (e1 < m) {
            uint32_t b1, i1;
            gt_locate(hu, (uint32_t)(e1 - rowptr[vhi]), b1, i1);
            B1 = gtx_block_bit(hu, b1, sh) + gtx_field(hu, i1, sh);
        } else {
            B1 = hu.pay + gtx_payload_bits(hu, sh);
        }
        const uint64_t W0 = B0 >> 5;
        const uint64_t NW = B1 > B0 ? ((B1 - 1) >> 5) + 2 - W0 : 0;
        if (NW && NW <= stage) {
            uint32_t* L = dec_lds + (threadIdx.x / kWave) * stage;
            const uint32_t nw = (uint32_t)NW;
            for (uint32_t c = 0; c < nw; c += 8 * kWave) {
                uint32_t t[8];
#pragma unroll
                for (uint32_t u = 0; u < 8; ++u) {
                    const uint32_t j = c + u * kWave + lane;
                    t[u] = j < nw ? g.w[W0 + j] : 0u;
                }
#pragma unroll
                for (uint32_t u = 0; u < 8; ++u) {
                    const uint32_t j = c + u * kWave + lane;
                    if (j < nw) L[j] = t[u];
                }
            }
            wave_sync();
            decode_range(g, LdsWords{L, W0}, rowptr, col, e0, e1, eb, vlo, vhi, span);
            return;
        }
    }
    decode_range(g, GlobalWords{g.w}, rowptr, col, e0, e1, eb, vlo, vhi, span);
}

int decode_csr(grass_graph* g, uint64_t* rowptr, uint32_t* col, hipStream_t s) {
    const uint64_t n = g->n, m = g->m;
    const uint64_t nb = scan_blocks(n);
    if (nb <= kScanDirectMax) {  // one launch, no partials
        const hipError_t e = exclusive_scan(DegGen{g->d_deg}, Count{n, nullptr}, n, rowptr, nullptr, nullptr, s);
        if (e != hipSuccess) return status_of(e);
    } else if (std::unique_lock<std::mutex> lock(g->mu); g->d_dpre) {  // one launch, the tiles' starts are there
        lock.unlock();
        const hipError_t e = scan_from_prefixes(DegGen{g->d_deg}, n, g->d_dpre, rowptr, s);
        if (e != hipSuccess) return status_of(e);
    } else {
        // The scan's partials have a buffer of their own, ordered between calls on the device:
        // each call's stream waits for the previous call's scan (on whatever stream) before its
        // own scan reuses the buffer, so no call waits on the host.
        if (!g->dec_ev && hipEventCreateWithFlags(&g->dec_ev, hipEventDisableTiming) != hipSuccess)
            return GRASS_ENOMEM;
        hipError_t e = hipStreamWaitEvent(s, g->dec_ev, 0);
        if (e != hipSuccess) return status_of(e);
        if (g->dec_part.reserve((nb + 4) * 8) != hipSuccess) return GRASS_ENOMEM;
        uint64_t* part = (uint64_t*)g->dec_part.ptr;
        e = exclusive_scan(DegGen{g->d_deg}, Count{n, nullptr}, n, rowptr, part, part + nb, s);
        if (e == hipSuccess) e = hipEventRecord(g->dec_ev, s);
        if (e != hipSuccess) return status_of(e);
    }
    if (m == 0 || !col) return GRASS_OK;
    const uint32_t per_wave = g->tune.decode_edges_per_wave.load(std::memory_order_relaxed);
    uint32_t slot = 0;
    while ((512u << slot) < per_wave && slot + 1 < kWaveStartSlots) ++slot;
    if ((512u << slot) != per_wave) return GRASS_EINVAL;
    // LE, and GT with P <= 4, decode by runs: about per_wave slots per wave, per_wave / P runs.  The
    // run offsets (a scan over the headers) are built once per graph; their total is known since load.
    // So are the starts of the row-pointer scan's tiles: R-MAT s16 (64 k rows, 1 M entries, bound by its
    // launches) 15.7 us a call with the tile sums, their scratch and its events in each, 10.4 without.
    const uint32_t sh = run_shift(g->fmt, g->cp_shift);
    const bool runs = (1u << sh) <= kRunMax;
    const uint32_t unit = runs ? per_wave >> sh : per_wave;
    const uint64_t units = runs ? g->dec_runs : m;
    const uint64_t waves = (units + unit - 1) / unit;
    const uint64_t blocks = (waves + kDecBlock / kWave - 1) / (kDecBlock / kWave);
    if (blocks > 0x7fffffffull) return GRASS_EINVAL;
    // The waves' first vertices depend only on the graph and per_wave: built once per per_wave
    // value from the row pointers (or the run offsets), complete before it is published, never
    // changed after.
    const uint64_t* uoff;
    const uint32_t* wstart;
    {
        std::lock_guard<std::mutex> lock(g->mu);
        uint64_t* r = g->d_roff;
        uint32_t* t = g->d_wstart[slot];
        uint64_t* d = g->d_dpre;
        const bool new_r = runs && !r, new_t = !t, new_d = !d && nb > kScanDirectMax;
        if (new_r || new_t || new_d) {
            WorkMem m_part;
            hipError_t e = hipSuccess;
            if (new_r) {
                if (m_part.alloc((nb + 4) * 8, s) != hipSuccess) return GRASS_ENOMEM;
                if (device_malloc((void**)&r, (n + 1) * 8) != hipSuccess) return GRASS_ENOMEM;
                uint64_t* part = m_part.as<uint64_t>();
                e = exclusive_scan(RunGen{g->d_hdr, g->fmt, sh}, Count{n, nullptr}, n, r, part, part + nb, s);
            }
            if (e == hipSuccess && new_t && device_malloc((void**)&t, (waves + 1) * 4) != hipSuccess) {
                t = nullptr;
                e = hipErrorOutOfMemory;
            }
            if (e == hipSuccess && new_t) {
                const unsigned grid = (unsigned)std::min<uint64_t>((n + 255) / 256, 16384);
                hipLaunchKernelGGL(wave_start_kernel, dim3(grid), dim3(256), 0, s, runs ? (const uint64_t*)r : (const uint64_t*)rowptr,
                                   (uint32_t)n, unit, waves, t);
                e = hipGetLastError();
            }
            if (e == hipSuccess && new_d && device_malloc((void**)&d, (nb + 1) * 8) != hipSuccess) {
                d = nullptr;
                e = hipErrorOutOfMemory;
            }
            if (e == hipSuccess && new_d) e = scan_prefixes(DegGen{g->d_deg}, n, d, s);
            const hipError_t done = hipStreamSynchronize(s);
            if (e == hipSuccess) e = done;
            if (e != hipSuccess) {
                if (new_d && d) (void)hipFree(d);
                if (new_r && r) (void)hipFree(r);
                if (new_t && t) (void)hipFree(t);
                return e == hipErrorOutOfMemory ? GRASS_ENOMEM : status_of(e);
            }
            g->d_roff = r;
            g->d_wstart[slot] = t;
            g->d_dpre = d;
        }
        uoff = runs ? (const uint64_t*)g->d_roff : (const uint64_t*)rowptr;
        wstart = g->d_wstart[slot];
    }
    if (runs && g->fmt == kLE) {
        hipLaunchKernelGGL(decode_runs_kernel<kLE>, dim3((unsigned)blocks), dim3(kDecBlock), 0, s, g->dev(),
                           (const uint64_t*)rowptr, uoff, wstart, col, units, unit, sh);
    } else if (runs) {
        hipLaunchKernelGGL(decode_runs_kernel<kGT>, dim3((unsigned)blocks), dim3(kDecBlock), 0, s, g->dev(),
                           (const uint64_t*)rowptr, uoff, wstart, col, units, unit, sh);
    } else {
        const uint32_t stage = dec_stage_words(per_wave);
        hipLaunchKernelGGL(decode_csr_kernel, dim3((unsigned)blocks), dim3(kDecBlock),
                           (size_t)stage * 4 * (kDecBlock / kWave), s, g->dev(), (const uint64_t*)rowptr, wstart,
                           col, m, per_wave, stage);
    }
    return status_of(hipGetLastError());
}

}  // namespace grass
