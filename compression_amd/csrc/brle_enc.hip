// Byte RLE encode for gfx950: one workgroup per chunk.
//
// Replaces brle::compress_gpu and its kernels (reference include/brle/
// brle.h:232-303: one thread runs the byte-at-a-time encoder of :129-230 per
// 256 KiB chunk, then a scan and a shift kernel pack the chunks).  The output
// is byte-identical to that encoder's.
//
// The encoder is a greedy state machine over the chunk's bytes: a pending
// group is empty, a literal group (up to 128 bytes; a third equal byte in a
// row ends it and starts a run) or a run (up to 130 equal bytes).  Cut the
// chunk into segments of equal bytes.  A segment always starts with n = 0..127
// pending literals (a run ends with its segment), and takes them to
//   * (n + L) mod 128 if its length L is 1 or 2;
//   * a value that depends on L alone if L >= 3 and n <= 125: its bytes are
//     runs of 130 and a rest, which is a run (3 or more) or literals;
//   * the same after 128 - n literals that fill the group, if n is 126 or 127.
// So any stretch of segments maps n to n' by {shift; the result for a shifted
// n below 126, for 126, for 127}, 29 bits, and such maps compose: the state
// machine is a prefix scan.  Per window of 32 KiB (32 bytes a thread):
//   1. each thread marks where segments start in its bytes, and a scan packs
//      those positions into a list: each ends the segment before it, so no
//      thread looks ahead.  The list's segments are dealt out evenly, the same
//      number to every thread, whatever bytes they cover;
//   2. each thread composes its segments' maps, and a scan gives the literals
//      pending before its first segment;
//   3. it counts the bytes its segments add, and a scan places them;
//   4. it writes them to the LDS copy of the output, which the workgroup
//      stores 16 bytes at a time.  A group's header byte is reserved with its
//      first literal and written by the segment that ends the group.
// Vector issue and the scans' latency bound it (four barriers a window), so a
// workgroup is as wide as the hardware allows; chunks of at most 2 or 8 KiB get
// one of 1 or 4 waves, with windows to match.  64 MiB of mean run length 12
// in 256 KiB chunks: 89 us for this kernel, 96 us a call (161 us for the kernel
// with each thread taking the segments that end in its own bytes, 22.0 ms with
// one lane walking a chunk).
// Groups go to a per-chunk slot of the work buffer; a scan kernel turns the
// chunk sizes into ptr[] and a shift kernel packs the slots into `data`.
#include "brle_load.h"
#include "mdz_device.h"
#include "mdz_internal.h"

namespace mdz {
namespace {

constexpr uint32_t kMinRun = 3, kMaxRun = 130, kMaxLit = 128;
constexpr uint32_t kPer = kBrlePer;             // bytes per thread and window

template <uint32_t kWaves>
struct EncLds {
    static constexpr uint32_t kThreads = kWaves * kWave;
    static constexpr uint32_t kWin = kThreads * kPer;
    static constexpr uint32_t kStage = kWin + kWin / 32 + 64;    // staged output bytes of a window
    alignas(16) uint32_t in[kWin / 4];
    alignas(16) uint32_t out[kStage / 4 + 8];
    uint16_t list[kWin];                        // window offsets where a segment ends
    uint32_t part[3][kWaves];
};

// Pending literals after a segment of L >= 3 bytes that starts as runs.
MDZ_DEV uint32_t rest_of(uint32_t L) {
    const uint32_t r = L % kMaxRun;
    return r < kMinRun ? r : 0;
}
// Output bytes of that segment: whole runs, then a run or a header and literals.
MDZ_DEV uint32_t run_bytes(uint32_t L) {
    const uint32_t r = L % kMaxRun;
    return 2 * (L / kMaxRun) + (r >= kMinRun ? 2 : r ? r + 1 : 0);
}

// A map of pending literals: bits 0..6 shift, then (bit 31 set) the results
// for a shifted count below 126, of 126 and of 127.
constexpr uint32_t kReset = 1u << 31;
MDZ_DEV uint32_t map_apply(uint32_t f, uint32_t n) {
    const uint32_t t = (n + f) & 127;
    const uint32_t r = f >> (t < 126 ? 7 : t == 126 ? 14 : 21);
    return f & kReset ? r & 127 : t;
}
MDZ_DEV uint32_t map_then(uint32_t f, uint32_t g) {      // f, then g
    const uint32_t shifted = (g & ~127u) | ((f + g) & 127);
    const uint32_t through = kReset | (f & 127) | map_apply(g, (f >> 7) & 127) << 7 |
                             map_apply(g, (f >> 14) & 127) << 14 | map_apply(g, (f >> 21) & 127) << 21;
    return f & kReset ? through : shifted;
}
MDZ_DEV uint32_t map_of(uint32_t L) {
    if (L < kMinRun) return L;
    const uint32_t b = L - 2 >= kMinRun ? rest_of(L - 2) : L - 2, c = L - 1 >= kMinRun ? rest_of(L - 1) : L - 1;
    return kReset | rest_of(L) << 7 | b << 14 | c << 21;
}
MDZ_DEV uint32_t wave_incl_maps(uint32_t v) {
    v = map_then(dpp_src<0x111, 0xf, 0u>(v), v);          // the identity is 0
    v = map_then(dpp_src<0x112, 0xf, 0u>(v), v);
    v = map_then(dpp_src<0x114, 0xf, 0u>(v), v);
    v = map_then(dpp_src<0x118, 0xf, 0u>(v), v);
    v = map_then(dpp_src<0x142, 0xa, 0u>(v), v);
    v = map_then(dpp_src<0x143, 0xc, 0u>(v), v);
    return v;
}
// The value of the lane below; `first` in lane 0.
MDZ_DEV uint32_t from_below(uint32_t v, uint32_t first) {
    const uint32_t r = (uint32_t)__shfl_up((int)v, 1, kWave);
    return lane_id() ? r : first;
}

// Output bytes of a segment of L bytes after n pending literals; n moves on.
MDZ_DEV uint32_t count_segment(uint32_t& n, uint32_t L) {
    uint32_t bytes = 0;
    if (L >= kMinRun && n >= 126) {             // the group fills up first
        bytes = kMaxLit - n;
        L -= bytes;
        n = 0;
    }
    if (L >= kMinRun) {
        bytes += run_bytes(L);
        n = rest_of(L);
    } else {
        bytes += L + (n == 0 && L ? 1u : 0u) + (n + L > kMaxLit ? 1u : 0u);
        n = (n + L) & (kMaxLit - 1);
    }
    return bytes;
}

// Writes that segment's bytes of value v at offset o (relative to the output
// so far) through put(offset, byte); returns the offset after them.
template <class Put>
MDZ_DEV int32_t write_segment(Put put, int32_t o, uint32_t& n, uint32_t L, uint32_t v) {
    auto literals = [&](uint32_t k) {
        for (; k; --k) {
            if (n == 0) ++o;                    // the header's place
            put(o++, v);
            if (++n == kMaxLit) {
                put(o - 1 - (int32_t)kMaxLit, kMaxLit + 127);
                n = 0;
            }
        }
    };
    if (L >= kMinRun && n >= 126) {
        const uint32_t fill = kMaxLit - n;
        literals(fill);
        L -= fill;
    }
    if (L < kMinRun) {
        literals(L);
        return o;
    }
    if (n) put(o - 1 - (int32_t)n, n + 127);
    n = 0;
    for (; L >= kMinRun; L -= min(L, kMaxRun)) {
        put(o, min(L, kMaxRun) - kMinRun);
        put(o + 1, v);
        o += 2;
    }
    literals(L);
    return o;
}

// Exclusive scan over the workgroup through part[kWaves]: `incl` is the wave's
// inclusive scan, `carry` comes before the workgroup's first thread and takes
// in its last.  One barrier; every row of 16 lanes then scans the parts.
template <uint32_t kWaves, class Then>
MDZ_DEV uint32_t block_scan(uint32_t* part, uint32_t incl, uint32_t& carry, Then then) {
    static_assert(kWaves <= 16, "the parts fit a row");
    const uint32_t wave = threadIdx.x / kWave;
    if (lane_id() == kWave - 1) part[wave] = incl;
    __syncthreads();
    const uint32_t w = lane_id() & 15;
    uint32_t v = w < kWaves ? part[min(w, kWaves - 1)] : 0u;
    v = then(dpp_src<0x111, 0xf, 0u>(v), v);              // 0 is every map's identity
    v = then(dpp_src<0x112, 0xf, 0u>(v), v);
    v = then(dpp_src<0x114, 0xf, 0u>(v), v);
    v = then(dpp_src<0x118, 0xf, 0u>(v), v);
    const uint32_t below = (uint32_t)__builtin_amdgcn_readlane((int)v, wave ? (int)wave - 1 : 0);
    const uint32_t before = wave ? then(carry, below) : carry;
    carry = then(carry, (uint32_t)__builtin_amdgcn_readlane((int)v, 15));
    return then(before, from_below(incl, 0));
}

// One chunk c, by the whole workgroup.
template <uint32_t kWaves>
MDZ_DEV void encode_chunk(EncLds<kWaves>& S, uint64_t c, const uint8_t* __restrict__ in, uint64_t in_bytes,
                          uint64_t chunk, uint64_t slot, uint8_t* __restrict__ work, uint64_t* __restrict__ sizes) {
    constexpr uint32_t kEncThreads = EncLds<kWaves>::kThreads, kWin = EncLds<kWaves>::kWin, kStage = EncLds<kWaves>::kStage;
    const uint32_t t = threadIdx.x;
    const uint64_t base = c * chunk;
    const uint32_t len = (uint32_t)min(chunk, in_bytes - base);
    const uint8_t* src = in + base;
    uint8_t* out = work + c * slot;
    const uint8_t* in8 = reinterpret_cast<const uint8_t*>(S.in);
    uint8_t* out8 = reinterpret_cast<uint8_t*>(S.out);
    const uint32_t skew = (uint32_t)((uintptr_t)src & 3);
    auto plus = [](uint32_t a, uint32_t b) { return a + b; };
    uint32_t open = 0;                          // start of the segment open before the window
    uint32_t state = 0;                         // map of the segments before the window: pending literals
    uint32_t last = 0x100;                      // the byte before the window
    uint64_t done = 0;                          // output bytes before the window
    uint64_t staged = 0;                        // the output from here on is in LDS, not yet in `out`
    for (uint32_t w0 = 0; w0 < len; w0 += min(kWin, len - w0)) {
        // 1. the thread's bytes: to LDS, and where they differ from the byte before
        const uint32_t wl = min(kWin, len - w0), at = kPer * t;
        uint32_t v[kPer / 4];
        if (at + kPer <= wl && ((uintptr_t)src & 15) == 0) {
            const uint4* p = reinterpret_cast<const uint4*>(src + w0 + at);
#pragma unroll
            for (uint32_t i = 0; i < kPer / 16; ++i) {
                const uint4 q = p[i];
                v[4 * i] = q.x, v[4 * i + 1] = q.y, v[4 * i + 2] = q.z, v[4 * i + 3] = q.w;
            }
        } else if (brle_whole_dwords(w0, at, len, skew)) {
            // whole dwords around the bytes, shifted together
            const uint32_t* p = reinterpret_cast<const uint32_t*>(src + w0 + at - skew);
            uint32_t lo = p[0];
#pragma unroll
            for (uint32_t i = 0; i < kPer / 4; ++i) {
                const uint32_t hi = p[i + 1];
                v[i] = alignbyte(hi, lo, skew);
                lo = hi;
            }
        } else {                                // the chunk's first or last bytes
#pragma unroll
            for (uint32_t i = 0; i < kPer; ++i) {
                const uint32_t b = at + i < wl ? src[w0 + at + i] : 0u;
                v[i / 4] = i & 3 ? v[i / 4] | b << (8 * (i & 3)) : b;
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < kPer / 4; ++i) S.in[at / 4 + i] = v[i];
        __syncthreads();
        uint32_t before = t ? in8[at - 1] : last, mask = 0;
#pragma unroll
        for (uint32_t i = 0; i < kPer / 4; ++i) {
            const uint32_t x = v[i] ^ (v[i] << 8 | (before & 0xFFu));
            const uint32_t nz = ((((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x) >> 7) & 0x01010101u;
            mask |= ((nz * 0x10204080u) >> 28) << (4 * i);
            before = v[i] >> 24;
        }
        if (w0 + t == 0) mask |= 1;             // the chunk's first byte opens a segment
        mask = at >= wl ? 0 : wl - at >= kPer ? mask : mask & ((1u << (wl - at)) - 1);
        // the segments that end in these bytes (position 0 ends none)
        const uint32_t ends = w0 + t == 0 ? mask & ~1u : mask;
        uint32_t count = 0;
        {
            const uint32_t mine = (uint32_t)__builtin_popcount(ends);
            uint32_t i = block_scan<kWaves>(S.part[0], wave_incl_scan_u32(mine), count, plus);
            for (uint32_t m = ends; m; m &= m - 1) S.list[i++] = (uint16_t)(at + (uint32_t)__builtin_ctz(m));
        }
        __syncthreads();
        const uint32_t share = (count + kEncThreads - 1) / kEncThreads, s0 = min(count, t * share), s1 = min(count, s0 + share);
        auto each = [&](auto fn) {
            uint32_t prev = s0 ? w0 + S.list[s0 - 1] : open;
            for (uint32_t i = s0; i < s1; ++i) {
                const uint32_t o = S.list[i], p = w0 + o;
                fn(p - prev, o);
                prev = p;
            }
        };
        // 2. literals pending before the thread's first segment
        uint32_t map = 0;
        each([&](uint32_t L, uint32_t) { map = map_then(map, map_of(L)); });
        uint32_t n = map_apply(block_scan<kWaves>(S.part[1], wave_incl_maps(map), state, map_then), 0);
        // 3. where its bytes go
        uint32_t bytes = 0, n3 = n;
        each([&](uint32_t L, uint32_t) { bytes += count_segment(n3, L); });
        uint32_t total = 0;
        const uint32_t off = block_scan<kWaves>(S.part[2], wave_incl_scan_u32(bytes), total, plus);
        // 4. write them.  LDS byte i holds output byte (staged & ~15) + i; what
        // does not fit there (long runs), and headers stored before, go straight out
        const uint64_t stage0 = staged & ~15ull;
        const bool fits = done + total - stage0 <= kStage;
        const int32_t held = (int32_t)(int64_t)(staged - done), shift = (int32_t)(int64_t)(done - stage0);
        if (!fits) {
            for (uint64_t i = staged + t; i < done; i += kEncThreads) out[i] = out8[i - stage0];
            __syncthreads();
        }
        auto put = [&](int32_t o, uint32_t b) {
            if (fits && o >= held) out8[o + shift] = (uint8_t)b;
            else out[(int64_t)done + o] = (uint8_t)b;
        };
        int32_t o = (int32_t)off;
        each([&](uint32_t L, uint32_t p) { o = write_segment(put, o, n, L, p ? in8[p - 1] : last); });
        last = in8[wl - 1];
        if (count) open = w0 + S.list[count - 1];
        __syncthreads();
        done += total;
        if (fits) {                             // store whole 16-byte units, keep the rest
            const uint64_t whole = w0 + wl == len ? done : max(done & ~15ull, staged);
            for (uint64_t u = stage0 + 16 * t; u < whole; u += 16 * kEncThreads) {
                const uint32_t i = (uint32_t)(u - stage0);
                if (u >= staged && u + 16 <= whole) {
                    *reinterpret_cast<uint4*>(out + u) = *reinterpret_cast<const uint4*>(out8 + i);
                } else {
                    for (uint32_t k = 0; k < 16; ++k)
                        if (u + k >= staged && u + k < whole) out[u + k] = out8[i + k];
                }
            }
            const uint32_t rest = (uint32_t)(done - whole);       // under 16 bytes
            const uint32_t keep = t < rest ? out8[(uint32_t)(whole - stage0) + t] : 0u;
            __syncthreads();
            if (t < rest) out8[(uint32_t)(whole & 15) + t] = (uint8_t)keep;
            staged = whole;
        } else {
            staged = done;
        }
    }
    // the last segment, and the literals still pending
    __syncthreads();
    uint32_t n = map_apply(state, 0);
    auto put = [&](int32_t o, uint32_t b) { out[(int64_t)done + o] = (uint8_t)b; };
    if (t == 0) {
        const int32_t o = write_segment(put, 0, n, len - open, last);
        if (n) put(o - 1 - (int32_t)n, n + 127);
        sizes[c] = done + (uint32_t)o;
    }
}

// Chunks beyond the grid's workgroups are taken in turn.
template <uint32_t kWaves>
__global__ __launch_bounds__(kWaves * kWave) void brle_encode_kernel(const uint8_t* __restrict__ in, uint64_t in_bytes,
                                                                     uint64_t n_chunks, uint64_t chunk, uint64_t slot,
                                                                     uint8_t* __restrict__ work,
                                                                     uint64_t* __restrict__ sizes) {
    __shared__ EncLds<kWaves> S;
    for (uint64_t c = blockIdx.x; c < n_chunks; c += gridDim.x) {
        encode_chunk<kWaves>(S, c, in, in_bytes, chunk, slot, work, sizes);
        __syncthreads();
    }
}

// ptr[0] = 0, ptr[c + 1] = ptr[c] + sizes[c]: one workgroup, each thread
// summing a contiguous run of chunks, then a scan of the thread sums.
constexpr uint32_t kScanThreads = 1024;

__global__ __launch_bounds__(kScanThreads) void brle_scan_kernel(const uint64_t* __restrict__ sizes, uint64_t n,
                                                                 uint64_t* __restrict__ ptr) {
    __shared__ uint64_t part[kScanThreads / kWave];
    const uint32_t t = threadIdx.x;
    const uint64_t per = (n + kScanThreads - 1) / kScanThreads;
    const uint64_t b = min(n, per * t), e = min(n, b + per);
    uint64_t s = 0;
    for (uint64_t i = b; i < e; ++i) s += sizes[i];
    const uint64_t incl = wave_incl_scan_u64(s);
    if (lane_id() == kWave - 1) part[t / kWave] = incl;
    __syncthreads();
    uint64_t before = 0;
    for (uint32_t w = 0; w < t / kWave; ++w) before += part[w];
    uint64_t run = before + incl - s;
    if (t == 0) ptr[0] = 0;
    for (uint64_t i = b; i < e; ++i) {
        run += sizes[i];
        ptr[i + 1] = run;
    }
}

// data[ptr[c], ptr[c + 1]) = work[c * slot, ...): dword stores at aligned
// destination addresses, each assembled from the two source dwords it spans.
// Few chunks are split over `gridDim.y` workgroups each, so that the chip is
// full (64 MiB in 256 chunks: 16 us with one workgroup per chunk).
constexpr uint32_t kShiftThreads = 256, kShiftGroups = 2048;

__global__ __launch_bounds__(kShiftThreads) void brle_shift_kernel(const uint8_t* __restrict__ work, uint64_t slot,
                                                                   const uint64_t* __restrict__ ptr,
                                                                   uint8_t* __restrict__ data) {
    const uint64_t c = blockIdx.x;
    const uint64_t d0 = ptr[c], n = ptr[c + 1] - d0;
    const uint8_t* s = work + c * slot;        // slot starts are 16-byte aligned
    uint8_t* d = data + d0;
    const uint32_t t = blockIdx.y * kShiftThreads + threadIdx.x, step = gridDim.y * kShiftThreads;
    const uint64_t head = min<uint64_t>((4 - ((uintptr_t)d & 3)) & 3, n);
    for (uint64_t i = t; i < head; i += step) d[i] = s[i];
    const uint64_t nw = (n - head) / 4;
    const uint32_t sk = (uint32_t)(head & 3);          // source skew of each destination dword
    const uint32_t* s4 = reinterpret_cast<const uint32_t*>(s + (head & ~3ull));
    uint32_t* d4 = reinterpret_cast<uint32_t*>(d + head);
    for (uint64_t i = t; i < nw; i += step) {
        // source bytes head + 4i .. + 3 lie in dwords i and i + 1 of s4 (the
        // slot is padded, so the second read stays inside it)
        d4[i] = sk ? alignbyte(s4[i + 1], s4[i], sk) : s4[i];
    }
    for (uint64_t i = head + 4 * nw + t; i < n; i += step) d[i] = s[i];
}

}  // namespace

int brle_compress_bound(uint64_t in_bytes, uint64_t chunk, uint64_t* n_chunks, uint64_t* work_bytes,
                        uint64_t* data_cap) {
    if (in_bytes == 0 || chunk == 0 || chunk > 0xFFFFFFF0ull) return MDZ_ERR_INVALID;
    const uint64_t n = (in_bytes - 1) / chunk + 1;
    const uint64_t worst = chunk + (chunk + kMaxLit - 1) / kMaxLit + 1;
    const uint64_t slot = (worst + 16 + 15) & ~15ull;
    if (n_chunks) *n_chunks = n;
    if (work_bytes) *work_bytes = n * slot + 8 * n;
    if (data_cap) *data_cap = in_bytes + n * ((chunk + kMaxLit - 1) / kMaxLit + 1);
    return MDZ_OK;
}

int brle_compress(const void* in, uint64_t in_bytes, uint64_t chunk, void* work, void* data, uint64_t* ptr,
                  hipStream_t s) {
    uint64_t n = 0, wb = 0;
    int rc = brle_compress_bound(in_bytes, chunk, &n, &wb, nullptr);
    if (rc) return rc;
    if (!in || !work || !data || !ptr || n > kMaxEncodeChunks) return MDZ_ERR_INVALID;
    const uint64_t slot = (wb - 8 * n) / n;
    uint64_t* sizes = reinterpret_cast<uint64_t*>(static_cast<uint8_t*>(work) + n * slot);
    // a workgroup no wider than its chunk's windows: 2, 8 or 32 KiB
    const uint32_t waves = chunk <= EncLds<1>::kWin ? 1 : chunk <= EncLds<4>::kWin ? 4 : 16;
    auto encode = waves == 1 ? brle_encode_kernel<1> : waves == 4 ? brle_encode_kernel<4> : brle_encode_kernel<16>;
    hipLaunchKernelGGL(encode, dim3((uint32_t)(n < (1u << 20) ? n : 1u << 20)), dim3(waves * kWave), 0, s,
                       static_cast<const uint8_t*>(in), in_bytes, n, chunk, slot, static_cast<uint8_t*>(work), sizes);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return record_hip(e, "brle_encode_kernel launch");
    hipLaunchKernelGGL(brle_scan_kernel, dim3(1), dim3(kScanThreads), 0, s, sizes, n, ptr);
    if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "brle_scan_kernel launch");
    const uint64_t most = (chunk + 4 * kShiftThreads - 1) / (4 * kShiftThreads), want = (kShiftGroups + n - 1) / n;
    hipLaunchKernelGGL(brle_shift_kernel, dim3((uint32_t)n, (uint32_t)(want < most ? want : most)), dim3(kShiftThreads), 0, s,
                       static_cast<const uint8_t*>(work), slot, ptr, static_cast<uint8_t*>(data));
    return record_hip(hipGetLastError(), "brle_shift_kernel launch");
}

}  // namespace mdz
