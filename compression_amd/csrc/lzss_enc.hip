// LZSS encode for gfx950 (lane-transposed container).
//
// Replaces lzss::compress_gpu (reference include/lzss/lzss_gpu2.h:1952-2123:
// compress_init_func / compress_func_new per lane :332-494,511-707 with the
// window scan find_match :70-109, the lane sort :1063-1085 and the
// interleave :497-509).  Payload, col_len, col_map and blk_off equal that
// encoder's output byte for byte.
//
// Lane stream t of a chunk is chunk bytes 128 k + 4 t + j (j < 4).  It is
// encoded greedily: at each position the longest match of 3..34 bytes within
// the last 2047 bytes (never from position 0), ties to the oldest, else a
// literal; tokens in groups of 8 behind a flag byte.
//
// One wave encodes one lane stream.  The stream's bytes and an index of its
// positions live in LDS: `slot` lists the positions bucket by bucket (9 hash
// bits of 3 bytes), ascending inside a bucket.  A step searches two
// neighbouring positions, each half of the wave comparing 32 candidates of
// its position's bucket at once, oldest first; if the first becomes a literal
// the second's token follows in the same step, which about half of all tokens
// do.  A search ends when no younger candidate can be longer.  Only positions
// that the greedy parse reaches, and their successors, are searched, and what
// the whole wave shares (position, best matches, output offset) is scalar.
// What bounds it is instruction issue at the waves that LDS allows: 7.4 KiB
// per stream up to 2048 lane bytes (64 KiB chunks), 14 KiB beyond.  Lanes over
// 4096 bytes are indexed in windows of 4096 positions that advance by 2048.
// 64 MiB in 64 KiB chunks: 2.7 ms (3.4 ms with one position a step; 412 ms with
// one lane per stream and chains in global memory).  Streams of a few bytes are
// encoded by a thread each.
//
// A second kernel ranks a chunk's 32 lanes by length (descending, ties to
// the higher lane id) into col_map; the shared kernels scan the chunk
// lengths and interleave the sorted lanes.
#include "lanes_enc_dev.h"
#include "mdz_device.h"
#include "mdz_internal.h"

namespace mdz {
namespace {

constexpr uint32_t kHist = 2048, kMinLen = 3, kMaxLen = 34, kLenBits = 5;
constexpr uint32_t kHashBits = 9, kBuckets = 1u << kHashBits;

constexpr uint32_t kHalf = 32;                  // lanes that search one position

// One lane stream's window: kCap positions and the bytes a match at the last
// of them can reach.
template <uint32_t kCap>
struct LzStream {
    static constexpr bool kOld = kCap > kHist;  // candidates can be out of reach
    uint32_t data[(kCap + 64) / 4];
    uint16_t slot[kCap + kWave];                // positions by bucket, ascending; then kWave that are no candidates
    uint32_t bound[kBuckets / 2 + 1];           // u16: bucket h's slots are [bound[h], bound[h + 1])
    uint16_t first[kOld ? kBuckets : 2];        // first slot still within reach
};

// 4 and 8 bytes at byte p: whole dwords shifted together.  (A misaligned LDS
// read is one instruction too, but serialises the wave's lanes: with those the
// encoder spent 94 % of its time in LDS.)
MDZ_DEV uint32_t lds_u32(const uint32_t* w, uint32_t p) {
    const uint32_t k = p >> 2;
    return alignbyte(w[k + 1], w[k], p & 3);
}
MDZ_DEV uint64_t lds_u64(const uint32_t* w, uint32_t p) {
    const uint32_t k = p >> 2, w0 = w[k], w1 = w[k + 1], w2 = w[k + 2];
    return (uint64_t)alignbyte(w2, w1, p & 3) << 32 | alignbyte(w1, w0, p & 3);
}
// Of the low 3 bytes (a 24-bit multiply takes no others).
MDZ_DEV uint32_t lz_hash(uint32_t v) { return (uint32_t)__umul24(v, 0x9E3779u) >> (32 - kHashBits); }
// Zero bits below the lowest set one; all ones if there is none (v_ffbl_b32).
MDZ_DEV uint32_t ctz_or_max(uint32_t v) { return v ? (uint32_t)__builtin_ctz(v) : 0xFFFFFFFFu; }
MDZ_DEV uint32_t add_sat(uint32_t a, uint32_t b) { return __builtin_elementwise_add_sat(a, b); }
MDZ_DEV uint32_t lane_value_at(uint32_t v, uint32_t lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}

// Lists the window's positions [p0, p1) by bucket.
template <uint32_t kCap>
MDZ_DEV void lz_index(LzStream<kCap>& S, uint32_t p0, uint32_t p1, uint32_t l) {
    // While the slots are given out, the u16 at h + 1 counts bucket h.
    auto bump = [&](uint32_t h) {
        return (atomicAdd(&S.bound[(h + 1) >> 1], 1u << (16 * ((h + 1) & 1))) >> (16 * ((h + 1) & 1))) & 0xFFFFu;
    };
    for (uint32_t i = l; i <= kBuckets / 2; i += kWave) S.bound[i] = 0;
    wave_sync();
    for (uint32_t p = p0 + l; p < p1; p += kWave) bump(lz_hash(lds_u32(S.data, p)));
    wave_sync();
    {   // counts -> first slots: lane l holds the u16s [8 l, 8 l + 8); the last one is never read as a count
        constexpr uint32_t kPer = kBuckets / 2 / kWave;
        uint32_t c[kPer], sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < kPer; ++i) {
            c[i] = S.bound[l * kPer + i];
            sum += (c[i] & 0xFFFFu) + (c[i] >> 16);
        }
        // the u16 at h + 1 becomes bucket h's first slot: the counts before it
        uint32_t at = wave_incl_scan_u32(sum) - sum;
#pragma unroll
        for (uint32_t i = 0; i < kPer; ++i) {
            const uint32_t lo = at, hi = at + (c[i] & 0xFFFFu);
            at = hi + (c[i] >> 16);
            S.bound[l * kPer + i] = lo | hi << 16;
            if constexpr (LzStream<kCap>::kOld) {
                if (l || i) S.first[2 * (l * kPer + i) - 1] = (uint16_t)lo;
                S.first[2 * (l * kPer + i)] = (uint16_t)hi;
            }
        }
        if (l == kWave - 1) {
            S.bound[kBuckets / 2] = at;
            if constexpr (LzStream<kCap>::kOld) S.first[kBuckets - 1] = (uint16_t)at;
        }
    }
    wave_sync();
    // each slot given out moves its bucket's first slot: to the bucket's end
    for (uint32_t p = p0 + l; p < p1; p += kWave) S.slot[bump(lz_hash(lds_u32(S.data, p)))] = (uint16_t)p;
    wave_sync();
    // steps past the list's end read positions that are no candidates
    const uint32_t ns = p1 > p0 ? p1 - p0 : 0;
    S.slot[ns + l] = (uint16_t)(kCap - 1);
    // The 64 positions of one step may take their bucket's slots in any
    // order: put neighbours in order until none is out of it.
    for (;;) {
        bool moved = false;
#pragma unroll
        for (uint32_t odd = 0; odd < 2; ++odd) {
            for (uint32_t i = odd + 2 * l; i + 1 < ns; i += 2 * kWave) {
                const uint32_t a = S.slot[i], b = S.slot[i + 1];
                if (a > b && lz_hash(lds_u32(S.data, a)) == lz_hash(lds_u32(S.data, b))) {
                    S.slot[i] = (uint16_t)b;
                    S.slot[i + 1] = (uint16_t)a;
                    moved = true;
                }
            }
            wave_sync();
        }
        if (!__ballot(moved)) break;
    }
}

template <uint32_t kCap>
__global__ __launch_bounds__(kWave) void lzss_encode_kernel(const uint8_t* __restrict__ in, uint64_t n_chunks,
                                                            uint64_t chunk, uint64_t lane_slot,
                                                            uint8_t* __restrict__ work,
                                                            uint32_t* __restrict__ lane_len) {
    __shared__ LzStream<kCap> S;
    const uint32_t l = lane_id(), half = l / kHalf;
    const uint16_t* bounds = reinterpret_cast<const uint16_t*>(S.bound);
    const uint32_t n = (uint32_t)(chunk / 32);
    for (uint64_t unit = blockIdx.x; unit < lane_units(n_chunks); unit += gridDim.x) {
        uint64_t c;
        uint32_t t;
        if (!lane_of_unit(unit, n_chunks, c, t)) continue;
        const uint8_t* rows = in + c * chunk + 4 * t;
        uint8_t* out = work + (c * 32 + t) * lane_slot;
        uint32_t o = 1, flag_at = 0, ntok = 0, flags = 0;
        uint32_t cur = 0;                       // next position, counted from the window's start
        for (uint32_t w0 = 0;; w0 += kHist) {
            const uint32_t left = n - w0, stop = min(left, kCap);    // positions of the window
            wave_sync();
            for (uint32_t k = l; k < (kCap + 64) / 4; k += kWave)
                S.data[k] = w0 / 4 + k < n / 4 ? *reinterpret_cast<const uint32_t*>(rows + 128ull * (w0 / 4 + k)) : 0u;
            wave_sync();
            // position 0 is never a candidate, nor one with under 3 bytes left
            lz_index<kCap>(S, w0 ? 0u : 1u, min(stop, left >= kMinLen ? left - (kMinLen - 1) : 0u), l);
            while (cur < stop) {
                const uint32_t p = cur + half;
                const uint64_t here = lds_u64(S.data, p);
                const int32_t look = min((int32_t)(left - p), (int32_t)kMaxLen);  // longest match left
                const uint32_t h = lz_hash((uint32_t)here);
                uint32_t i = bounds[h];
                if constexpr (LzStream<kCap>::kOld) i = S.first[h];
                i += l % kHalf;
                const uint32_t e = bounds[h + 1];
                uint32_t len[2] = {0, 0}, from[2] = {0, 0};
                uint32_t least = kMinLen - 1;                // a match has to be longer
                for (;;) {
                    // Slots past the bucket's list hold positions of other 3 bytes,
                    // or none older than p: neither passes.
                    const uint32_t q = S.slot[i];
                    const int32_t cap = min((int32_t)(p - q), look);
                    const uint64_t x = lds_u64(S.data, q) ^ here;
                    // equal bytes, then at most cap; beyond 8 only if all 8 are equal
                    const uint32_t lo = ctz_or_max((uint32_t)x), hi = ctz_or_max((uint32_t)(x >> 32));
                    int32_t f = min((int32_t)(min(lo, add_sat(hi, 32u)) >> 3), cap);
                    if constexpr (LzStream<kCap>::kOld) f = p - q < kHist ? f : 0;
                    bool run = f > 8;
                    if (__ballot(run)) {
                        for (uint32_t j = 8; j < kMaxLen; j += 8) {
                            const uint64_t y = lds_u64(S.data, q + j) ^ lds_u64(S.data, p + j);
                            const int32_t g = (int32_t)(j + (y ? (uint32_t)__builtin_ctzll(y) >> 3 : 8u));
                            f = run ? min(g, cap) : f;
                            run = run && !y && cap > (int32_t)(j + 8);
                            if (!__ballot(run)) break;
                        }
                    }
                    // the oldest of the longest, in each half: each better one in turn
                    uint64_t m = __ballot(f > (int32_t)least);
#pragma unroll
                    for (uint32_t k = 0; k < 2; ++k) {
                        uint32_t mk = (uint32_t)(k ? m >> 32 : m);
                        while (mk) {
                            const uint32_t lane = kHalf * k + (uint32_t)__builtin_ctz(mk);
                            len[k] = lane_value_at((uint32_t)f, lane);
                            from[k] = lane_value_at(q, lane);
                            const uint64_t better = __ballot(f > (int32_t)len[k]);
                            mk = (uint32_t)(k ? better >> 32 : better);
                        }
                    }
                    // the next 32: if the last of these is in the list's middle and older
                    const uint64_t more = __ballot(i + 1 < e && q < p);
                    bool go0 = (more >> (kHalf - 1)) & 1, go1 = more >> (kWave - 1);
                    if constexpr (LzStream<kCap>::kOld) {
                        // a step wholly out of reach stays so for later positions
                        const uint64_t old = __ballot(q + kHist <= p);
                        if (go0 && (uint32_t)old == ~0u && l == kHalf - 1) S.first[h] = (uint16_t)(i + 1);
                        if (go1 && (uint32_t)(old >> 32) == ~0u && l == kWave - 1) S.first[h] = (uint16_t)(i + 1);
                    }
                    const uint32_t most = min(left - cur, kMaxLen);
                    go0 = go0 && len[0] < most;
                    go1 = go1 && len[1] < min(left - cur - 1, kMaxLen) && (go0 || !len[0]);
                    if (!go0 && !go1) break;
                    // a half that is done stays where it is and takes no more
                    const bool go = half ? go1 : go0;
                    least = go ? max(half ? len[1] : len[0], kMinLen - 1) : kWave;
                    i += go ? kHalf : 0;
                }
                // one token, and the successor's if it is a literal
#pragma unroll
                for (uint32_t k = 0; k < 2; ++k) {
                    if (len[k] == 0) {
                        if (l == kHalf * k) out[o] = (uint8_t)here;
                        flags |= 1u << ntok;
                        o += 1;
                        cur += 1;
                    } else {
                        const uint16_t v = (uint16_t)((cur - from[k]) << kLenBits | (len[k] - kMinLen));
                        if (l == 0) __builtin_memcpy(out + o, &v, 2);
                        o += 2;
                        cur += len[k];
                    }
                    if (++ntok == 8) {          // the next group's flag byte is reserved at once
                        if (l == 0) out[flag_at] = (uint8_t)flags;
                        flags = 0;
                        ntok = 0;
                        flag_at = o++;
                    }
                    if (k == 0 && (len[0] || cur >= stop)) break;
                }
                if constexpr (LzStream<kCap>::kOld) wave_sync();        // first[] before its next reader
            }
            if (stop == left) break;
            cur -= kHist;                       // the next window starts kHist positions on
        }
        if (l == 0) {
            out[flag_at] = (uint8_t)flags;
            lane_len[c * 32 + t] = o;
        }
    }
}

// Sorted slot of lane t: longer lanes first, equal lengths by higher lane id.
// Half a wave per chunk, `len` its lane lengths (the caller's own at len[t]).
MDZ_DEV void rank_lanes(const uint32_t* len, uint32_t t, uint64_t c, uint64_t n_chunks, uint64_t* __restrict__ col_len,
                        uint8_t* __restrict__ col_map, uint64_t* __restrict__ chunk_len) {
    const uint32_t mine = len[t];
    uint32_t rank = 0, words = 0;
    for (uint32_t u = 0; u < kHalf; ++u) {
        const uint32_t other = len[u];
        rank += (other > mine || (other == mine && u > t)) ? 1u : 0u;
        words += (other + 3) / 4;
    }
    if (c >= n_chunks) return;
    col_len[c * 32 + rank] = mine;
    col_map[c * 32 + rank] = (uint8_t)t;
    if (t == 0) chunk_len[c] = ((uint64_t)words * 4 + 127) / 128 * 128;
}

constexpr uint32_t kRankThreads = 256, kRankChunks = kRankThreads / kHalf;

__global__ __launch_bounds__(kRankThreads) void lzss_rank_kernel(const uint32_t* __restrict__ lane_len, uint64_t n_chunks,
                                                                 uint64_t* __restrict__ col_len,
                                                                 uint8_t* __restrict__ col_map,
                                                                 uint64_t* __restrict__ chunk_len) {
    __shared__ uint32_t len[kRankThreads];
    const uint32_t t = threadIdx.x % kHalf;
    const uint64_t c = (uint64_t)blockIdx.x * kRankChunks + threadIdx.x / kHalf;
    len[threadIdx.x] = c < n_chunks ? lane_len[c * 32 + t] : 0u;
    wave_sync();
    rank_lanes(len + (threadIdx.x - t), t, c, n_chunks, col_len, col_map, chunk_len);
}

// Short lane streams: a thread encodes one, its bytes in a column of LDS, half a
// wave per chunk; every earlier position is a candidate.  An index costs a wave
// the same however few positions it holds: 131072 chunks of 4 bytes a lane take
// 1810 us with a wave per stream and 56 us so, 16384 chunks of 32 bytes 950 and
// 130 us (Markov text).  A thread's time grows with the square of its bytes
// (129 us at 32) and few chunks do not fill the chip, so the more bytes the more
// chunks it takes: 1024 chunks of 32 bytes take 72 us a call with a wave per
// stream, 129 us so.  8 bytes take 12 us however few chunks there are, 14 us
// with a wave.
constexpr uint32_t kShortBytes = 8, kShortOfMany = 64, kShortChunks = kWave / kHalf;
inline bool short_lanes(uint32_t bytes, uint64_t n_chunks) {
    return bytes <= kShortBytes || (bytes <= kShortOfMany && n_chunks >= 2ull * bytes * bytes);
}

__global__ __launch_bounds__(kWave) void lzss_short_kernel(const uint8_t* __restrict__ in, uint64_t n_chunks,
                                                           uint64_t chunk, uint64_t lane_slot,
                                                           uint8_t* __restrict__ work, uint64_t* __restrict__ col_len,
                                                           uint8_t* __restrict__ col_map,
                                                           uint64_t* __restrict__ chunk_len) {
    __shared__ uint32_t data[kShortOfMany / 4 + 1][kWave];        // the last row is read, not used
    __shared__ uint32_t len[kWave];
    const uint32_t l = lane_id(), t = l % kHalf, n = (uint32_t)(chunk / 32);
    const uint64_t c = (uint64_t)blockIdx.x * kShortChunks + l / kHalf;
    uint32_t bytes = 0;
    if (c < n_chunks) {
        const uint8_t* rows = in + c * chunk + 4 * t;
        for (uint32_t k = 0; k < n / 4; ++k) data[k][l] = *reinterpret_cast<const uint32_t*>(rows + 128ull * k);
        auto at = [&](uint32_t p) { return alignbyte(data[p / 4 + 1][l], data[p / 4][l], p & 3); };   // 4 bytes
        WordOut o{work + (c * 32 + t) * lane_slot};
        o.put(0);
        uint32_t flag_at = 0, ntok = 0, flags = 0;
        for (uint32_t cur = 0; cur < n;) {
            const uint32_t here = at(cur);
            uint32_t best = kMinLen - 1, from = 0;
            // candidates four at a time, oldest first; position 0 is none, nor
            // one too near for a longer match
            const uint32_t most = min(n - cur, kMaxLen);
            uint32_t lo = data[0][l];
            for (uint32_t q4 = 0; q4 + best < cur && best < most; q4 += 4) {
                const uint32_t hi = data[q4 / 4 + 1][l];
                const uint32_t x0 = q4 ? (lo ^ here) << 8 : 1u, x1 = (alignbyte(hi, lo, 1) ^ here) << 8,
                               x2 = (alignbyte(hi, lo, 2) ^ here) << 8, x3 = (alignbyte(hi, lo, 3) ^ here) << 8;
                lo = hi;
                if (min(min(x0, x1), min(x2, x3))) continue;     // no 3 equal bytes
                for (uint32_t j = 0; j < 4; ++j) {
                    if (j == 0 ? x0 : j == 1 ? x1 : j == 2 ? x2 : x3) continue;
                    const uint32_t q = q4 + j, cap = q < cur ? min(cur - q, most) : 0u;
                    uint32_t f = 0;
                    while (f < cap) {
                        const uint32_t x = at(q + f) ^ at(cur + f);
                        f += x ? (uint32_t)__builtin_ctz(x) >> 3 : 4u;
                        if (x) break;
                    }
                    f = min(f, cap);
                    if (f > best) best = f, from = q;
                }
            }
            if (best < kMinLen) {
                flags |= 1u << ntok;
                o.put(here & 0xFFu);
                cur += 1;
            } else {
                const uint32_t v = (cur - from) << kLenBits | (best - kMinLen);
                o.put(v & 0xFFu);
                o.put(v >> 8);
                cur += best;
            }
            if (++ntok == 8) {                  // the next group's flag byte is reserved at once
                o.patch(flag_at, flags);
                flags = 0;
                ntok = 0;
                flag_at = o.len;
                o.put(0);
            }
        }
        o.patch(flag_at, flags);
        bytes = o.finish();
    }
    len[l] = bytes;
    wave_sync();
    rank_lanes(len + (l - t), t, c, n_chunks, col_len, col_map, chunk_len);
}

uint64_t lz_lane_slot(uint64_t chunk) {
    const uint64_t lb = chunk / 32;
    return (lb + lb / 8 + 16 + 15) & ~15ull;          // all literals: one flag byte per 8
}

}  // namespace

int lzss_compress_bound(uint64_t in_bytes, uint64_t chunk, uint64_t* n_chunks, uint64_t* work_bytes,
                        uint64_t* payload_cap) {
    // whole chunks only (a trailing partial chunk is dropped, as the reference
    // encoder drops it), at most 1 MiB.  Of the chunk * 2 bytes behind a chunk's
    // lane slots the encoder uses 128, the lane lengths; callers' buffers keep
    // their size.
    if (chunk == 0 || chunk % 128 || chunk > (1ull << 20) || in_bytes < chunk) return MDZ_ERR_INVALID;
    const uint64_t n = in_bytes / chunk;
    const uint64_t slot = lz_lane_slot(chunk);
    if (n_chunks) *n_chunks = n;
    if (work_bytes) *work_bytes = n * 32 * slot + n * chunk * 2 + 8 * n;
    if (payload_cap) *payload_cap = n * ((32 * slot + 127) / 128 * 128);
    return MDZ_OK;
}

int lzss_compress(const void* in, uint64_t in_bytes, uint64_t chunk, void* work, void* payload, uint64_t* col_len,
                  uint8_t* col_map, uint64_t* blk_off, hipStream_t s) {
    uint64_t n = 0;
    int rc = lzss_compress_bound(in_bytes, chunk, &n, nullptr, nullptr);
    if (rc) return rc;
    if (!in || !work || !payload || !col_len || !col_map || !blk_off || n > kMaxEncodeChunks) return MDZ_ERR_INVALID;
    if ((uintptr_t)in & 3) return MDZ_ERR_INVALID;   // lanes are read a dword at a time
    const uint64_t slot = lz_lane_slot(chunk);
    uint8_t* w = static_cast<uint8_t*>(work);
    uint32_t* lane_len = reinterpret_cast<uint32_t*>(w + n * 32 * slot);
    uint64_t* chunk_len = reinterpret_cast<uint64_t*>(w + n * 32 * slot + n * chunk * 2);
    const uint32_t lb = (uint32_t)(chunk / 32);
    hipError_t e;
    if (short_lanes(lb, n)) {
        hipLaunchKernelGGL(lzss_short_kernel, dim3((uint32_t)((n + kShortChunks - 1) / kShortChunks)), dim3(kWave), 0, s,
                           static_cast<const uint8_t*>(in), n, chunk, slot, w, col_len, col_map, chunk_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lzss_short_kernel launch");
    } else {
        auto encode = lb <= 1024 ? lzss_encode_kernel<1024> : lb <= 2048 ? lzss_encode_kernel<2048> : lzss_encode_kernel<4096>;
        hipLaunchKernelGGL(encode, lane_grid(n), dim3(kWave), 0, s, static_cast<const uint8_t*>(in), n, chunk, slot, w,
                           lane_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lzss_encode_kernel launch");
        hipLaunchKernelGGL(lzss_rank_kernel, dim3((uint32_t)((n + kRankChunks - 1) / kRankChunks)), dim3(kRankThreads), 0,
                           s, lane_len, n, col_len, col_map, chunk_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lzss_rank_kernel launch");
    }
    hipLaunchKernelGGL(lanes_scan_kernel, dim3(1), dim3(kScanThreads), 0, s, chunk_len, n, blk_off, nullptr, ~0ull);
    if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lanes_scan_kernel launch");
    hipLaunchKernelGGL(lanes_interleave_kernel, interleave_grid(n, slot), dim3(kIlvThreads), 0, s,
                       static_cast<const uint8_t*>(w), slot, col_len, blk_off, chunk_len, col_map,
                       static_cast<uint8_t*>(payload));
    return record_hip(hipGetLastError(), "lanes_interleave_kernel launch");
}

}  // namespace mdz
