// Compressed-graph loader: files -> pinned host staging -> HBM, then on the device:
//   1. byte swap of the .graph and .offset images into big-endian word views,
//   2. record-length extraction from .offset fused into a reduce-then-scan (bit starts),
//   3. a validator that parses every record header, checks header + payload == record
//      length, and writes the degree array and the decoded-header cache,
//   4. GT: the checkpointed payload stream the samplers decode (flat_expand_kernel).
// Replaces loadGraph (LE/src/grass.cu:1015-1095), copyPartitionToGPU (LE/src/utils.hpp:328-353)
// with its decode_offset kernel (LE/src/bcg.cuh:284-329) and CUB scan.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <thread>
#include <vector>

#include "devutil.h"
#include "encode_flat.h"
#include "runtime.h"
#include "scan.h"

namespace grass {

__global__ void bswap_words_kernel(uint32_t* w, uint64_t nwords) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (; i < nwords; i += stride) w[i] = __builtin_bswap32(w[i]);
}

// Length field u of .offset: bits [8 + u*ubl, 8 + (u+1)*ubl) of the file, ubl in [1, 64]
// (LE/src/bcg.cuh:293-318 reads the same field across up to three words).
struct OffsetFieldGen {
    const uint32_t* ow;  // big-endian word view of the whole .offset file, padded
    uint32_t ubl;
    __device__ __forceinline__ uint64_t operator()(uint64_t u) const {
        uint64_t b = 8 + u * ubl;
        const uint32_t* p = ow + (b >> 5);
        uint32_t s = (uint32_t)(b & 31);
        uint64_t hi = ((uint64_t)p[0] << 32) | p[1];
        uint64_t win = s ? (hi << s) | (p[2] >> (32 - s)) : hi;
        return win >> (64 - ubl);
    }
};

constexpr int kValBlock = 256;

// stats: [0] sum of degrees, [1] max degree, [2] malformed records, [3] first malformed vertex,
// [4] decode runs of 1 << run_sh positions
template <int FMT>
__global__ __launch_bounds__(kValBlock) void validate_kernel(const uint32_t* __restrict__ w,
                                                             const uint64_t* __restrict__ start,
                                                             uint32_t n, uint64_t gbits,
                                                             uint32_t* __restrict__ deg,
                                                             uint4* __restrict__ hdr, uint32_t run_sh,
                                                             unsigned long long* stats) {
    __shared__ unsigned long long lds[kValBlock / kWave];
    unsigned long long sum = 0, mx = 0, bad = 0, runs = 0;
    for (uint32_t v = blockIdx.x * kValBlock + threadIdx.x; v < n; v += gridDim.x * kValBlock) {
        const uint64_t b0 = start[v], end = start[v + 1];
        uint64_t b = b0;
        // Every read below stays within [b0, end + 95] bits, inside the padded word view,
        // whatever the .offset held (a corrupt one may even wrap the 64-bit scan).
        bool ok = end > b0 && end <= gbits;
        Hdr h;
        h.d = h.f1 = h.f2 = h.fp = h.C = h.q = h.R = 0;
        ok = ok && gamma_checked(w, b, h.d) && b <= end;
        if (FMT == kLE) {
            if (ok && h.d >= 1) ok = gamma_checked(w, b, h.f1) && b <= end;
            if (ok && h.d == 1) ok = h.f1 < n;
            if (ok && h.d >= 2) {
                ok = gamma_checked(w, b, h.f2) && b <= end && gamma_checked(w, b, h.fp) && b <= end;
                if (ok) {
                    le_geometry(h.d, h.C, h.q, h.R);
                    ok = h.f1 >= 1 && h.f1 <= 31 && h.f2 <= 31 && h.fp <= h.C + 1;
                }
            }
        } else {
            ok = ok && gamma_checked(w, b, h.f1) && b <= end && gamma_checked(w, b, h.f2) &&
                 b <= end && gamma_checked(w, b, h.fp) && b <= end;
            if (ok && h.d) {
                gt_geometry(h.d, h.C, h.q, h.R);
                ok = h.f1 >= 1 && h.f1 <= 31 && h.f2 <= 31 && h.fp <= h.C &&
                     (h.f2 >= 1 || h.d == h.C);
            }
        }
        if (ok) {
            h.pay = b;
            ok = (b + payload_bits(FMT, h) == end) && h.d < 0x80000000u;
        }
        if (!ok) {
            ++bad;
            atomicMin(&stats[3], (unsigned long long)v);
            h.d = h.f1 = h.f2 = h.fp = h.C = 0;
            h.pay = b0;
        }
        deg[v] = h.d;
        hdr[v] = pack_hdr(h, FMT);
        sum += h.d;
        runs += list_runs(FMT, h.d, h.C, h.q, run_sh);
        mx = h.d > mx ? h.d : mx;
    }
    sum = block_sum<unsigned long long, kValBlock>(sum, lds);
    mx = block_max<unsigned long long, kValBlock>(mx, lds);
    bad = block_sum<unsigned long long, kValBlock>(bad, lds);
    runs = block_sum<unsigned long long, kValBlock>(runs, lds);
    if (threadIdx.x == 0) {
        atomicAdd(&stats[0], sum);
        atomicMax(&stats[1], mx);
        if (bad) atomicAdd(&stats[2], bad);
        atomicAdd(&stats[4], runs);
    }
}

// ------------------------------------------------------------------ GT payload stream

// Words of vertex v's payload in the device GT stream (P = 1 << shift).
struct GtxWordsGen {
    const uint4* hdr;
    uint32_t shift;
    __device__ __forceinline__ uint64_t operator()(uint64_t v) const {
        Hdr h;
        unpack_hdr<kGT>(hdr[v], h);
        return (gtx_payload_bits(h, shift) + 31) >> 5;
    }
};

// The GT payload stream from a .graph image: the same words as flat_write_kernel's from the rows.  `hdr`
// are the image's headers (payload bits in `w`), woff[] the payloads' first words in the stream,
// rowptr[] the degrees' prefix sums.  Heads and gaps are copied; a checkpoint's id is the sum over its
// block so far, a segmented sum over the lanes carried from pass to pass, which a chunk that starts
// inside a block begins with the fields before its own.  R-MAT s22 (128 M entries): 3.24 ms with a wave
// per vertex, 1.14 by slots.
__global__ __launch_bounds__(kFlatBlock) void flat_expand_kernel(const uint32_t* __restrict__ w,
                                                                 const uint64_t* __restrict__ rowptr,
                                                                 const uint4* __restrict__ hdr, uint64_t n,
                                                                 const uint64_t* __restrict__ woff, uint32_t sh,
                                                                 uint32_t* __restrict__ out) {
    __shared__ uint32_t own_lds[kFlatBlock];
    __shared__ uint32_t buf[kFlatWaves][kFlatWords + 1];
    uint32_t* own = own_lds + (threadIdx.x & ~(kWave - 1));
    FlatWindow<false> win{buf[threadIdx.x / kWave], out};
    const uint32_t lane = lane_id();
    const uint64_t waves = (uint64_t)gridDim.x * kFlatWaves;
    const uint64_t slots = rowptr[n] + n;
    const uint32_t passes = flat_passes(slots, waves);
    const uint64_t W = (uint64_t)passes * kWave - kFlatLook;
    for (uint64_t s0 = ((uint64_t)blockIdx.x * kFlatBlock + threadIdx.x) / kWave * W; s0 < slots; s0 += waves * W) {
        SlotWalk walk{rowptr, n};
        walk.seek(s0);
        uint64_t st = 0;
        uint4 hj = make_uint4(0u, 0u, 0u, 0u);
        auto request = [&]() {
            if (walk.cur + (uint64_t)lane < n) {
                st = woff[walk.cur + lane];
                hj = hdr[walk.cur + lane];
            }
        };
        request();
        uint32_t carry = 0;  // the id at the slot before the pass's first
        if (s0 - walk.sc >= 2) {
            Hdr h;
            unpack_hdr<kGT>(hdr[walk.cur], h);
            uint32_t b, i;
            flat_pos((uint32_t)(s0 - walk.sc) - 2, h.q, h.R, b, i);  // the field before the chunk's first
            const uint64_t bo = gt_file_block_bit(h, b);
            uint32_t sum = 0;
            for (uint32_t g = 1 + lane; g <= i; g += kWave) sum += read_bits0(w, bo + h.f1 + (uint64_t)(g - 1) * h.f2, h.f2) + 1;
            const uint32_t raw = read_bits(w, bo, h.f1);
            carry = wave_sum(sum) + (b >= h.fp ? walk.cur + raw + 1 : walk.cur - raw - 1);
        }
        for (uint32_t t = 0; t < passes; ++t) {
            const uint64_t base = s0 + (uint64_t)t * kWave;
            if (base >= slots) break;
            const bool fin = t + 1 == passes || base + kWave >= slots;
            const uint32_t last = (uint32_t)(slots - base < (uint64_t)kWave ? slots - base - 1 : kWave - 1);
            uint32_t j, d, head;
            int32_t k;
            walk.place(base, last, own, j, k, d, head);
            const uint32_t v = walk.cur + j;
            Hdr h;
            unpack_hdr<kGT>(make_uint4(__shfl(hj.x, (int)j, kWave), __shfl(hj.y, (int)j, kWave), d, __shfl(hj.w, (int)j, kWave)), h);
            const uint64_t sv = ((uint64_t)__shfl((uint32_t)(st >> 32), (int)j, kWave) << 32) | __shfl((uint32_t)st, (int)j, kWave);
            walk.advance((uint32_t)__builtin_amdgcn_readlane((int)j, (int)last),
                         __builtin_amdgcn_readlane((int)(k + 1 == (int32_t)d), (int)last));
            if (!fin) {
                walk.request();
                request();
            }
            const bool act = lane <= last, field = act && k >= 0;
            uint32_t b, i;
            flat_pos(k < 0 ? 0u : (uint32_t)k, h.q, h.R, b, i);
            const uint32_t heads = b + (i != 0), wf = i ? h.f2 : h.f1;
            const uint64_t off = __umul24(heads, h.f1) + (uint64_t)((uint32_t)k - heads) * h.f2;
            uint32_t raw = 0, x = 0;
            uint64_t at = sv << 5;
            uint32_t wdt = 0;
            if (field) {
                raw = read_bits(w, h.pay + off, wf);
                x = i ? raw + 1 : b >= h.fp ? v + raw + 1 : v - raw - 1;
                at += off + (uint64_t)flat_checkpoints(b, i, h.q, h.R, sh) * (32 - h.f2);
                wdt = wf;
            }
            // the ids: sums from the block's head, or from the carry where that lies in an earlier pass
            if (lane == 0 && field && i) x += carry;
            x = SegmentScan(!field ? lane : i <= lane ? lane - i : 0u).sum(x);
            carry = (uint32_t)__builtin_amdgcn_readlane((int)x, kWave - 1);
            if (i && !(i & ((1u << sh) - 1))) {
                raw = x;
                if (field) wdt = 32;
            }
            const uint64_t from = readlane_u64(at, 0), to = readlane_u64(at + wdt, (int)last);
            const uint64_t end = s0 + W < slots ? readlane_u64(at, kWave - kFlatLook) : ~0ull;  // (last pass)
            win.begin(t == 0, from, to);
            if (field) put_field(win.B, win.w0, at, wdt, raw);
            win.finish(fin, to, end);
        }
    }
}

struct DegreeGen {
    const uint32_t* deg;
    __device__ __forceinline__ uint64_t operator()(uint64_t v) const { return deg[v]; }
};

// The headers' payload bits moved from .graph to the stream.
__global__ __launch_bounds__(256) void gt_headers_kernel(const uint64_t* __restrict__ woff, uint64_t n,
                                                         uint4* __restrict__ hdr) {
    for (uint64_t v = (uint64_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (uint64_t)gridDim.x * 256) {
        uint4 e = hdr[v];
        const uint64_t pay = woff[v] << 5;
        e.x = (uint32_t)pay;
        e.y = (e.y & ~63u) | (uint32_t)(pay >> 32);
        hdr[v] = e;
    }
}

// Host threads that copy a chunk into pinned memory: GRASS_LOAD_THREADS in [1, 64], else up to 8.
unsigned load_threads() {
    if (const char* e = getenv("GRASS_LOAD_THREADS")) {
        const unsigned long t = strtoul(e, nullptr, 10);
        if (t >= 1 && t <= 64) return (unsigned)t;
    }
    return std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
}

// memcpy split over up to `threads` threads (slices of at least 4 MB); a thread that cannot be
// started leaves its slice to the calling thread.
void parallel_copy(void* dst, const uint8_t* src, uint64_t len, unsigned threads) {
    const uint64_t t = std::min<uint64_t>(threads, std::max<uint64_t>(1, len >> 22));
    if (t <= 1) {
        memcpy(dst, src, len);
        return;
    }
    const uint64_t step = ((len + t - 1) / t + 4095) & ~4095ull;
    std::vector<std::thread> pool;
    std::vector<uint64_t> mine = {0};
    for (uint64_t lo = step; lo < len; lo += step) {
        const uint64_t n = std::min(step, len - lo);
        try {
            pool.emplace_back([=] { memcpy((uint8_t*)dst + lo, src + lo, n); });
        } catch (...) {
            mine.push_back(lo);
        }
    }
    for (uint64_t lo : mine) memcpy((uint8_t*)dst + lo, src + lo, std::min(step, len - lo));
    for (std::thread& th : pool) th.join();
}

namespace {

constexpr uint64_t kChunk = 64ull << 20;  // pinned staging chunk

// Streams `src` into device memory through two pinned chunks so that the copy of chunk i+1
// overlaps the DMA of chunk i.  A source held in host memory is copied with several threads.
int stage_to_device(ByteSource& src, char* dst, hipStream_t stream, uint64_t* tail,
                    unsigned tail_len, uint8_t* tail_out) {
    const uint64_t total = src.size();
    if (total == 0) return GRASS_OK;
    if (const uint8_t* dev = src.device_data()) {  // already in device memory: one copy, no staging
        const uint64_t tl = std::min<uint64_t>(tail_len, total);
        hipError_t e = hipMemcpyAsync(dst, dev, total, hipMemcpyDeviceToDevice, stream);
        if (e == hipSuccess && tail_out && tl)
            e = hipMemcpyAsync(tail_out, dev + total - tl, tl, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (tail) *tail = tl;
        return e == hipSuccess ? GRASS_OK : GRASS_EDEVICE;
    }
    const uint64_t chunk = std::min<uint64_t>(kChunk, total);
    PinnedWork pinned[2];
    void* pin[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
    int rc = GRASS_OK;
    for (int i = 0; i < 2 && rc == GRASS_OK; ++i) {
        if (pinned[i].alloc(chunk) != hipSuccess) rc = GRASS_ENOMEM;
        else if (hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) != hipSuccess)
            rc = GRASS_EDEVICE;
        pin[i] = pinned[i].p;
    }
    uint64_t off = 0;
    int slot = 0;
    bool used[2] = {false, false};
    const uint8_t* mem = src.data();
    const unsigned threads = load_threads();
    while (rc == GRASS_OK && off < total) {
        uint64_t len = std::min(chunk, total - off);
        if (used[slot] && hipEventSynchronize(ev[slot]) != hipSuccess) { rc = GRASS_EDEVICE; break; }
        if (mem) parallel_copy(pin[slot], mem + off, len, threads);
        else if (!src.read(pin[slot], len)) { rc = GRASS_EIO; break; }
        // keep the last tail_len bytes of the stream on the host
        if (tail_out && off + len > total - std::min<uint64_t>(tail_len, total)) {
            uint64_t t0 = total - std::min<uint64_t>(tail_len, total);
            for (uint64_t i = std::max(off, t0); i < off + len; ++i)
                tail_out[i - t0] = ((uint8_t*)pin[slot])[i - off];
        }
        if (hipMemcpyAsync(dst + off, pin[slot], len, hipMemcpyHostToDevice, stream) != hipSuccess ||
            hipEventRecord(ev[slot], stream) != hipSuccess) {
            rc = GRASS_EDEVICE;
            break;
        }
        used[slot] = true;
        off += len;
        slot ^= 1;
    }
    if (tail) *tail = std::min<uint64_t>(tail_len, total);
    if (hipStreamSynchronize(stream) != hipSuccess && rc == GRASS_OK) rc = GRASS_EDEVICE;
    for (int i = 0; i < 2; ++i)
        if (ev[i]) (void)hipEventDestroy(ev[i]);
    return rc;
}

// Field u of .offset read on the host from the file's last `tlen` bytes.
uint64_t host_field(const uint8_t* tailb, uint64_t tlen, uint64_t file_bytes, uint64_t u,
                    uint32_t ubl) {
    uint64_t b = 8 + u * ubl;  // bit position in the file
    uint64_t first = file_bytes - tlen;
    uint64_t v = 0;
    for (uint32_t t = 0; t < ubl; ++t, ++b) {
        uint64_t byte = b >> 3;
        uint32_t bit = byte >= first && byte < file_bytes ? (tailb[byte - first] >> (7 - (b & 7))) & 1 : 0;
        v = (v << 1) | bit;
    }
    return v;
}

}  // namespace

int build_gt_stream(grass_graph* g, uint64_t* words);

int load_graph(grass_graph* g, ByteSource& gsrc, ByteSource& osrc) {
    const uint64_t gbytes = gsrc.size(), obytes = osrc.size();
    if (obytes < 2 || gbytes < 1) return GRASS_EFORMAT;
    if (8 * gbytes >= kMaxPayloadBits) return GRASS_EFORMAT;  // payload bits must fit the header cache
    hipStream_t s = g->stream;
    const uint64_t gwords = (gbytes + 3) / 4 + kPadWords;
    const uint64_t owords = (obytes + 3) / 4 + kPadWords;
    // The GT .graph words, the .offset words, the record starts and the scan's and the validator's
    // totals are used here only; the graph points at the first and third while it is being built.
    WorkMem m_words, m_off, m_start, m_tmp;
    struct Detach {
        grass_graph* g;
        ~Detach() {
            if (g->fmt == kGT) g->d_words = nullptr;
            g->d_start = nullptr;
        }
    } detach{g};
    if (g->fmt == kGT) {
        if (m_words.alloc(gwords * 4, s) != hipSuccess) return GRASS_ENOMEM;
        g->d_words = m_words.as<uint32_t>();
    } else if (device_malloc((void**)&g->d_words, gwords * 4) != hipSuccess) {
        return GRASS_ENOMEM;
    }
    if (m_off.alloc(owords * 4, s) != hipSuccess) return GRASS_ENOMEM;
    uint32_t* d_off = m_off.as<uint32_t>();
    int rc = GRASS_OK;
    // zero from the files' last partial words on (the images are copied over the start of them)
    if (hipMemsetAsync(g->d_words + gbytes / 4, 0, (gwords - gbytes / 4) * 4, s) != hipSuccess ||
        hipMemsetAsync(d_off + obytes / 4, 0, (owords - obytes / 4) * 4, s) != hipSuccess)
        return GRASS_EDEVICE;
    rc = stage_to_device(gsrc, (char*)g->d_words, s, nullptr, 0, nullptr);
    if (rc) return rc;
    uint8_t tailb[64];
    uint64_t tlen = 0;
    rc = stage_to_device(osrc, (char*)d_off, s, &tlen, sizeof(tailb), tailb);
    if (rc) return rc;

    // ubl = byte 0 of .offset; n = floor(8 (bytes - 1) / ubl) (LE/src/grass.cu:1071,1088),
    // minus trailing zero-length fields, which can only be padding (a record is >= 1 bit).
    uint8_t ubl = 0;
    if (hipMemcpy(&ubl, d_off, 1, hipMemcpyDeviceToHost) != hipSuccess) return GRASS_EDEVICE;
    if (ubl == 0 || ubl > 64) return GRASS_EFORMAT;
    uint64_t n = ((obytes - 1) * 8) / ubl;
    uint64_t tail_fields_max = std::min<uint64_t>(n, 7);
    for (uint64_t t = 0; t < tail_fields_max && n > 0; ++t) {
        if (8 + (n - 1) * (uint64_t)ubl < 8 * (obytes - tlen)) break;  // field not in the tail
        if (host_field(tailb, tlen, obytes, n - 1, ubl) != 0) break;
        --n;
    }
    if (n == 0 || n >= 0x80000000ull) return GRASS_EFORMAT;
    g->n = n;
    g->ubl = ubl;
    g->graph_bytes = gbytes;
    g->offset_bytes = obytes;

    const unsigned bsg = 2048;
    hipLaunchKernelGGL(bswap_words_kernel, dim3(bsg), dim3(256), 0, s, g->d_words, gwords);
    hipLaunchKernelGGL(bswap_words_kernel, dim3(bsg), dim3(256), 0, s, d_off, owords);

    if (m_start.alloc((n + 1) * 8, s) != hipSuccess) return GRASS_ENOMEM;
    g->d_start = m_start.as<uint64_t>();
    if (device_malloc((void**)&g->d_deg, n * 4) != hipSuccess) return GRASS_ENOMEM;
    const uint64_t hdr_bytes = n * 16;
    if (device_malloc((void**)&g->d_hdr, hdr_bytes) != hipSuccess) return GRASS_ENOMEM;
    const uint64_t nb = scan_blocks(n);
    if (m_tmp.alloc((nb + 8) * 8, s) != hipSuccess) return GRASS_ENOMEM;
    uint64_t* d_tmp = m_tmp.as<uint64_t>();  // partials[nb], total, stats[5]
    uint64_t* d_total = d_tmp + nb;
    unsigned long long* d_stats = (unsigned long long*)(d_tmp + nb + 2);
    unsigned long long init[5] = {0, 0, 0, ~0ull, 0};
    hipError_t e = hipMemcpyAsync(d_stats, init, sizeof(init), hipMemcpyHostToDevice, s);
    if (e == hipSuccess)
        e = exclusive_scan(OffsetFieldGen{d_off, ubl}, Count{n, nullptr}, n, g->d_start, d_tmp,
                           d_total, s);
    if (e == hipSuccess) {
        // (every workgroup adds to the same totals, one after another: 2.4 M vertices took 250 us with 9360
        // workgroups, 78 with 1024)
        unsigned grid = (unsigned)std::min<uint64_t>((n + kValBlock - 1) / kValBlock, 1024);
        if (g->fmt == kLE)
            hipLaunchKernelGGL(validate_kernel<kLE>, dim3(grid), dim3(kValBlock), 0, s, g->d_words,
                               g->d_start, (uint32_t)n, 8 * gbytes, g->d_deg, g->d_hdr,
                               run_shift(g->fmt, g->cp_shift), d_stats);
        else
            hipLaunchKernelGGL(validate_kernel<kGT>, dim3(grid), dim3(kValBlock), 0, s, g->d_words,
                               g->d_start, (uint32_t)n, 8 * gbytes, g->d_deg, g->d_hdr,
                               run_shift(g->fmt, g->cp_shift), d_stats);
        e = hipGetLastError();
    }
    uint64_t total = 0;
    unsigned long long stats[5] = {0, 0, 0, 0, 0};
    if (e == hipSuccess) e = hipMemcpyAsync(&total, d_total, 8, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(stats, d_stats, sizeof(stats), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return status_of(e);
    // records must cover the .graph bits up to < 8 bits of final padding
    if (total > 8 * gbytes || 8 * gbytes - total >= 8) return GRASS_EFORMAT;
    if (stats[2] != 0) return GRASS_EFORMAT;
    g->total_bits = total;
    g->m = stats[0];
    g->max_degree = stats[1];
    g->dec_runs = stats[4];
    uint64_t xwords = 0;
    if (g->fmt == kGT) {
        int rc2 = build_gt_stream(g, &xwords);
        if (rc2) return rc2;
    }
    // What stays resident is what the kernels read: the payload words (LE: the .graph image; GT:
    // the payload stream, which replaces the image), the header cache and the degrees.  The record
    // starts are folded into the header cache.
    g->device_bytes = (g->fmt == kGT ? xwords : gwords) * 4 + n * 4 + hdr_bytes;
    return GRASS_OK;
}

// Builds the device GT payload stream (g->d_gtx) from .graph and points the headers at it.
int build_gt_stream(grass_graph* g, uint64_t* words) {
    hipStream_t s = g->stream;
    const uint64_t n = g->n, nb = scan_blocks(n);
    WorkMem m_woff;  // n + 1 word offsets, n + 1 row starts, partials, total
    if (m_woff.alloc((2 * (n + 1) + nb + 2) * 8, s) != hipSuccess) return GRASS_ENOMEM;
    uint64_t* d_woff = m_woff.as<uint64_t>();
    uint64_t* d_row = d_woff + n + 1;
    uint64_t* d_part = d_row + n + 1;
    hipError_t e = exclusive_scan(GtxWordsGen{g->d_hdr, g->cp_shift}, Count{n, nullptr}, n, d_woff,
                                  d_part, d_part + nb, s);
    if (e == hipSuccess) e = exclusive_scan(DegreeGen{g->d_deg}, Count{n, nullptr}, n, d_row, d_part, d_part + nb, s);
    uint64_t total = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&total, d_woff + n, 8, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    uint32_t* out = nullptr;
    int rc = status_of(e);
    // payload bits must fit the header cache
    if (!rc && 32 * total >= kMaxPayloadBits) rc = GRASS_EFORMAT;
    if (!rc && device_malloc((void**)&out, (total + kPadWords) * 4) != hipSuccess) rc = GRASS_ENOMEM;
    if (!rc) {
        e = hipMemsetAsync(out + total, 0, kPadWords * 4, s);  // every word before is stored below
        if (e == hipSuccess) {
            int dev = 0, cus = 0;
            (void)hipGetDevice(&dev);
            (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
            hipLaunchKernelGGL(flat_expand_kernel, dim3((unsigned)std::max(cus, 1) * 8), dim3(kFlatBlock), 0, s,
                               (const uint32_t*)g->d_words, (const uint64_t*)d_row, (const uint4*)g->d_hdr, n,
                               (const uint64_t*)d_woff, g->cp_shift, out);
            hipLaunchKernelGGL(gt_headers_kernel, dim3((unsigned)std::min<uint64_t>((n + 255) / 256, 4096)), dim3(256), 0, s,
                               (const uint64_t*)d_woff, n, g->d_hdr);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        rc = status_of(e);
    }
    if (rc) {
        if (out) (void)hipFree(out);
        return rc;
    }
    g->d_gtx = out;
    *words = total + kPadWords;
    return GRASS_OK;
}

}  // namespace grass
