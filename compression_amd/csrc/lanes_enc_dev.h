// Scan and interleave kernels shared by the lane-transposed encoders (RLE v1,
// RLE v2, LZSS): chunk lengths -> offsets, and the 4-byte round-robin
// transpose of 32 lane streams (LZSS: in its sorted order) into a chunk (lane t's word r lands at word
// sum_t' min(words_t', r) + #{t' < t : words_t' > r}), tail zeroed to the
// chunk's 128-byte length.
#pragma once

#include "mdz_device.h"

namespace mdz {
namespace {

// A wave (one workgroup) per lane stream.  A chunk's 32 streams read the same
// input lines: units are numbered so that they run on one XCD (workgroups go
// to the XCDs in turn), whose L2 then reads each line once.
constexpr uint32_t kXcds = 8;

__host__ __device__ inline uint64_t lane_units(uint64_t n_chunks) {
    return (n_chunks + kXcds - 1) / kXcds * kXcds * 32;
}
MDZ_DEV bool lane_of_unit(uint64_t unit, uint64_t n_chunks, uint64_t& c, uint32_t& t) {
    t = (uint32_t)(unit / kXcds) % 32;
    c = unit / (kXcds * 32) * kXcds + unit % kXcds;
    return c < n_chunks;
}
inline dim3 lane_grid(uint64_t n_chunks) {       // the kernels stride over the units beyond it
    const uint64_t u = lane_units(n_chunks);
    return dim3((uint32_t)(u < (1u << 24) ? u : 1u << 24));
}

// Output of a lane stream that one thread encodes: stored by whole words, the
// last up to three bytes held back.  The stream's slot has room for the last
// word.
struct WordOut {
    uint8_t* out;
    uint32_t len = 0, held = 0;

    MDZ_DEV void put(uint32_t b) {               // b < 256
        held |= b << (8 * (len & 3));
        if ((++len & 3) == 0) {
            *reinterpret_cast<uint32_t*>(out + len - 4) = held;
            held = 0;
        }
    }
    MDZ_DEV void patch(uint32_t at, uint32_t b) {        // a byte put as 0
        if (at >= (len & ~3u)) held |= b << (8 * (at & 3));
        else out[at] = (uint8_t)b;
    }
    MDZ_DEV uint32_t finish() {                  // the stream's bytes
        if (len & 3) *reinterpret_cast<uint32_t*>(out + (len & ~3u)) = held;
        return len;
    }
};

// chunk_len[c]: the chunk's lanes rounded up to words, their sum to 128
// bytes.  Half a wave per chunk, a lane stream's words in each lane; all lanes
// of the wave take part, whether c < n or not.
MDZ_DEV void store_chunk_len(uint32_t words, uint64_t c, uint64_t n, uint64_t* __restrict__ chunk_len) {
    const uint32_t incl = wave_incl_scan_u32(words);
    const uint32_t low = (uint32_t)__builtin_amdgcn_readlane((int)incl, 31);
    if (c < n && threadIdx.x % 32 == 31) {
        const uint32_t total = lane_id() < 32 ? incl : incl - low;
        chunk_len[c] = ((uint64_t)total * 4 + 127) / 128 * 128;
    }
}

constexpr uint32_t kSizeThreads = 256, kSizeChunks = kSizeThreads / 32;

__global__ __launch_bounds__(kSizeThreads) void lanes_size_kernel(const uint64_t* __restrict__ col_len, uint64_t n,
                                                                  uint64_t* __restrict__ chunk_len) {
    const uint64_t c = (uint64_t)blockIdx.x * kSizeChunks + threadIdx.x / 32;
    store_chunk_len(c < n ? (uint32_t)((col_len[c * 32 + threadIdx.x % 32] + 3) / 4) : 0u, c, n, chunk_len);
}

constexpr uint32_t kScanThreads = 1024;

__global__ __launch_bounds__(kScanThreads) void lanes_scan_kernel(const uint64_t* __restrict__ sizes, uint64_t n,
                                                                  uint64_t* __restrict__ off, uint64_t* __restrict__ total,
                                                                  uint64_t last) {
    __shared__ uint64_t part[kScanThreads / kWave];
    const uint32_t t = threadIdx.x;
    const uint64_t per = (n + kScanThreads - 1) / kScanThreads;
    const uint64_t b = min(n, per * t), e = min(n, b + per);
    uint64_t s = 0;
    for (uint64_t i = b; i < e; ++i) s += sizes[i];
    const uint64_t incl = wave_incl_scan_u64(s);
    if (lane_id() == kWave - 1) part[t / kWave] = incl;
    __syncthreads();
    uint64_t run = 0;
    for (uint32_t w = 0; w < t / kWave; ++w) run += part[w];
    run += incl - s;
    if (t == 0) off[0] = 0;
    for (uint64_t i = b; i < e; ++i) {
        run += sizes[i];
        off[i + 1] = i + 1 == n && last != ~0ull ? last : run;
        if (i + 1 == n && total) *total = run;
    }
}

// Interleave.  Word r of slot t lands at base(r) + #{t' < t : words_t' > r},
// with base(r) = sum_t' min(words_t', r).  Per tile of 128 rounds base and the
// mask of slots still holding words are computed once per round, the slots'
// words are read along the streams (256 bytes a wave and load, 16 loads in
// flight), put in order in LDS (one word of padding per 32, or the 64 words of
// a load would share two banks) and stored along the chunk.  Few chunks are
// split over `parts` workgroups, tile by tile, so that the chip is full.
// 64 MiB of 4-byte RLE v1 values (512 chunks): 23 us, 113 us with one workgroup
// per chunk scattering words straight to memory.  Chunks of few rounds are
// stored straight from memory all the same, 32 words a half wave: a tile would
// be mostly empty (8192 chunks of 4 4-byte values a lane: 36 us with a tile,
// 15 us without; at 37 rounds both take 13 us for 2048 chunks).
constexpr uint32_t kIlvThreads = 256, kIlvWaves = kIlvThreads / kWave;
constexpr uint32_t kRoundTile = 2 * kWave;
constexpr uint32_t kDirectRounds = 32;           // rounds up to which no tile is made
constexpr uint32_t kIlvGroups = 2048;            // workgroups that fill the chip: 8 a CU

__global__ __launch_bounds__(kIlvThreads) void lanes_interleave_kernel(const uint8_t* __restrict__ work,
                                                                       uint64_t lane_slot,
                                                                       const uint64_t* __restrict__ col_len,
                                                                       const uint64_t* __restrict__ blk_off,
                                                                       const uint64_t* __restrict__ chunk_len,
                                                                       const uint8_t* __restrict__ lane_map,
                                                                       uint8_t* __restrict__ payload) {
    constexpr uint32_t kSlots = 32 / kIlvWaves;   // slots a wave reads
    __shared__ uint32_t words[32], bytes[32];
    __shared__ uint32_t rbase[kRoundTile + 1], rmask[kRoundTile];
    __shared__ uint32_t tile[kRoundTile * 33];
    const uint32_t tid = threadIdx.x, l = lane_id(), t0 = tid / kWave * kSlots;
    const uint64_t c = blockIdx.x;
    if (tid < 32) {
        bytes[tid] = (uint32_t)col_len[c * 32 + tid];
        words[tid] = (bytes[tid] + 3) / 4;
    }
    __syncthreads();
    uint32_t* dst = reinterpret_cast<uint32_t*>(payload + blk_off[c]);   // blk_off is a multiple of 128
    uint32_t total = 0, maxw = 0;
    for (uint32_t t = 0; t < 32; ++t) {
        total += words[t];
        maxw = max(maxw, words[t]);
    }
    // rbase[i] and rmask[i] of round r
    auto round = [&](uint32_t i, uint32_t r) {
        uint32_t base = 0, mask = 0;
        for (uint32_t u = 0; u < 32; ++u) {
            const uint32_t wu = words[u];
            base += wu < r ? wu : r;
            mask |= (wu > r ? 1u : 0u) << u;
        }
        rbase[i] = base;
        if (i < kRoundTile) rmask[i] = mask;
    };
    if (maxw <= kDirectRounds) {
        if (blockIdx.y) return;
        if (tid < maxw) round(tid, tid);
        __syncthreads();
        const uint32_t t = tid % 32;
        const uint32_t* src = reinterpret_cast<const uint32_t*>(
            work + (c * 32 + (lane_map ? lane_map[c * 32 + t] : t)) * lane_slot);
        for (uint32_t r = tid / 32; r < words[t]; r += kIlvThreads / 32) {
            const uint32_t have = bytes[t] - 4 * r, v = src[r];
            dst[rbase[r] + __builtin_popcount(rmask[r] & ((1u << t) - 1u))] =
                have < 4 ? v & ((1u << (8 * have)) - 1u) : v;
        }
        for (uint64_t q = total + tid; q < chunk_len[c] / 4; q += kIlvThreads) dst[q] = 0;
        return;
    }
    for (uint32_t r0 = blockIdx.y * kRoundTile; r0 < maxw; r0 += gridDim.y * kRoundTile) {
        uint32_t v[kSlots][2];
#pragma unroll
        for (uint32_t k = 0; k < kSlots; ++k) {
            const uint32_t t = t0 + k;
            // slot t holds lane_map[t]'s stream (identity without a map)
            const uint32_t* src = reinterpret_cast<const uint32_t*>(
                work + (c * 32 + (lane_map ? lane_map[c * 32 + t] : t)) * lane_slot);
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                const uint32_t r = r0 + kWave * h + l;
                v[k][h] = r < words[t] ? src[r] : 0u;
            }
        }
        if (tid <= kRoundTile) round(tid, r0 + tid);
        __syncthreads();
        const uint32_t first = rbase[0], count = rbase[kRoundTile] - first;
#pragma unroll
        for (uint32_t k = 0; k < kSlots; ++k) {
            const uint32_t t = t0 + k;
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                const uint32_t i = kWave * h + l, r = r0 + i;
                if (r < words[t]) {
                    const uint32_t have = bytes[t] - 4 * r;       // bytes of this word inside the stream
                    const uint32_t p = rbase[i] - first + __builtin_popcount(rmask[i] & ((1u << t) - 1u));
                    tile[p + p / 32] = have < 4 ? v[k][h] & ((1u << (8 * have)) - 1u) : v[k][h];
                }
            }
        }
        __syncthreads();
        for (uint32_t p = tid; p < count; p += kIlvThreads) dst[first + p] = tile[p + p / 32];
        __syncthreads();
    }
    if (blockIdx.y == 0) {
        const uint64_t clen = chunk_len[c];
        for (uint64_t q = total + tid; q < clen / 4; q += kIlvThreads) dst[q] = 0;
    }
}

inline dim3 interleave_grid(uint64_t n, uint64_t lane_slot) {
    const uint64_t tiles = (lane_slot / 4 + kRoundTile - 1) / kRoundTile, parts = (kIlvGroups + n - 1) / n;
    return dim3((uint32_t)n, (uint32_t)(parts < tiles ? parts : tiles));
}

}  // namespace
}  // namespace mdz
