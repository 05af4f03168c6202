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
// Half a wave encodes one lane stream, so a wave takes two neighbouring
// lanes and both share each instruction.  The stream's bytes and an index of
// its positions live in LDS: `slot` lists the positions bucket by bucket (9
// hash bits of 3 bytes), ascending inside a bucket.  At each token the 32
// lanes of the half compare 32 candidates of the token's bucket at once,
// oldest first, and a maximum over (length, age) picks the match; a search
// ends when no younger candidate can be longer.  Only the positions the
// greedy parse reaches are searched.  What bounds it is the dependent chain
// of LDS reads from one token to the next, so what counts is how many
// streams a CU holds: 7.2 KiB of LDS each up to 2048 lane bytes (64 KiB
// chunks), 13.4 KiB beyond.  Lanes over 4096 bytes are indexed in windows of
// 4096 positions that advance by 2048.
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
constexpr uint32_t kHalf = 32;                  // lanes that encode one stream
constexpr uint32_t kPairs = 16;                 // neighbouring lane pairs of a chunk
constexpr uint32_t kXcds = 8;

// One lane stream's window: kCap positions and the bytes a match at the last
// of them can reach.
template <uint32_t kCap>
struct LzStream {
    static constexpr bool kOld = kCap > kHist;  // candidates can be out of reach
    uint32_t data[(kCap + 64) / 4];
    uint16_t slot[kCap];                        // positions by bucket, ascending
    uint32_t end[kBuckets / 2];                 // u16 pairs: one past a bucket's last slot
    uint16_t first[kOld ? kBuckets : 2];        // first slot still within reach
};

MDZ_DEV uint32_t lds_u32(const uint8_t* p) {    // any alignment
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}
MDZ_DEV uint32_t lz_hash(uint32_t v) { return ((v & 0xFFFFFFu) * 2654435761u) >> (32 - kHashBits); }

// Maximum over each half of the wave, in every lane of the half.
MDZ_DEV uint32_t half_max_u32(uint32_t v) {
    v = max(v, dpp_src<0x128, 0xf, 0u>(v));     // row_ror 8, 4, 2, 1: each row of 16
    v = max(v, dpp_src<0x124, 0xf, 0u>(v));
    v = max(v, dpp_src<0x122, 0xf, 0u>(v));
    v = max(v, dpp_src<0x121, 0xf, 0u>(v));
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return max(r[0], r[1]);                     // rows 0 and 1, rows 2 and 3
}
MDZ_DEV uint32_t half_incl_scan_u32(uint32_t v) {
    v += dpp_src<0x111, 0xf, 0u>(v);
    v += dpp_src<0x112, 0xf, 0u>(v);
    v += dpp_src<0x114, 0xf, 0u>(v);
    v += dpp_src<0x118, 0xf, 0u>(v);
    v += dpp_src<0x142, 0xa, 0u>(v);            // row_bcast:15 into rows 1 and 3
    return v;
}
// The half's 32 bits of a ballot.
MDZ_DEV uint32_t half_ballot(bool b) {
    const uint64_t m = __ballot(b);
    return lane_id() < kHalf ? (uint32_t)m : (uint32_t)(m >> 32);
}

// Lists the window's positions [p0, p1) by bucket.  All 64 lanes; each half
// builds its own stream's index.
template <uint32_t kCap>
MDZ_DEV void lz_index(LzStream<kCap>& S, uint32_t p0, uint32_t p1, uint32_t sub) {
    const uint8_t* bytes = reinterpret_cast<const uint8_t*>(S.data);
    for (uint32_t i = sub; i < kBuckets / 2; i += kHalf) S.end[i] = 0;
    wave_sync();
    for (uint32_t p = p0 + sub; p < p1; p += kHalf) {
        const uint32_t h = lz_hash(lds_u32(bytes + p));
        atomicAdd(&S.end[h >> 1], 1u << (16 * (h & 1)));
    }
    wave_sync();
    {   // counts -> first slots, 16 buckets a lane
        constexpr uint32_t kPer = kBuckets / 2 / kHalf;
        uint32_t c[kPer], sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < kPer; ++i) {
            c[i] = S.end[sub * kPer + i];
            sum += (c[i] & 0xFFFFu) + (c[i] >> 16);
        }
        uint32_t at = half_incl_scan_u32(sum) - sum;
#pragma unroll
        for (uint32_t i = 0; i < kPer; ++i) {
            const uint32_t lo = at, hi = at + (c[i] & 0xFFFFu);
            at = hi + (c[i] >> 16);
            S.end[sub * kPer + i] = lo | hi << 16;
            if constexpr (LzStream<kCap>::kOld) {
                S.first[2 * (sub * kPer + i)] = (uint16_t)lo;
                S.first[2 * (sub * kPer + i) + 1] = (uint16_t)hi;
            }
        }
    }
    wave_sync();
    for (uint32_t p = p0 + sub; p < p1; p += kHalf) {   // each slot taken moves its bucket's end
        const uint32_t h = lz_hash(lds_u32(bytes + p));
        const uint32_t at = atomicAdd(&S.end[h >> 1], 1u << (16 * (h & 1)));
        S.slot[(at >> (16 * (h & 1))) & 0xFFFFu] = (uint16_t)p;
    }
    wave_sync();
    // The 32 positions of one step may take their bucket's slots in any
    // order: put neighbours in order until none is out of it.
    const uint32_t ns = p1 > p0 ? p1 - p0 : 0;
    for (;;) {
        bool moved = false;
#pragma unroll
        for (uint32_t odd = 0; odd < 2; ++odd) {
            for (uint32_t i = odd + 2 * sub; i + 1 < ns; i += 2 * kHalf) {
                const uint32_t a = S.slot[i], b = S.slot[i + 1];
                if (a > b && lz_hash(lds_u32(bytes + a)) == lz_hash(lds_u32(bytes + b))) {
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
    __shared__ LzStream<kCap> streams[2];
    const uint32_t l = lane_id(), sub = l & (kHalf - 1), half = l / kHalf;
    LzStream<kCap>& S = streams[half];
    const uint8_t* bytes = reinterpret_cast<const uint8_t*>(S.data);
    const uint16_t* ends = reinterpret_cast<const uint16_t*>(S.end);
    const uint32_t n = (uint32_t)(chunk / 32);
    // A chunk's 16 pairs read the same 128-byte rows: they run on one XCD
    // (workgroups go to the XCDs in turn), so its L2 reads each row once.
    const uint64_t units = (n_chunks + kXcds - 1) / kXcds * kXcds * kPairs;
    for (uint64_t unit = blockIdx.x; unit < units; unit += gridDim.x) {
        const uint32_t pair = (uint32_t)(unit / kXcds) % kPairs;
        const uint64_t c = unit / (kXcds * kPairs) * kXcds + unit % kXcds;
        if (c >= n_chunks) continue;
        const uint8_t* rows = in + c * chunk + 8 * pair;
        const uint64_t lane = c * 32 + 2 * pair + half;
        uint8_t* out = work + lane * lane_slot;
        uint32_t o = 1, flag_at = 0, ntok = 0, flags = 0;
        uint32_t cur = 0;                       // next position, counted from the window's start
        for (uint32_t w0 = 0;; w0 += kHist) {
            const uint32_t stop = min(n - w0, kCap);    // positions of the window
            wave_sync();
            for (uint32_t k = l; k < (kCap + 64) / 4; k += kWave) {
                uint32_t v[2] = {0, 0};
                if (w0 / 4 + k < n / 4) __builtin_memcpy(v, __builtin_assume_aligned(rows + 128ull * (w0 / 4 + k), 4), 8);
                streams[0].data[k] = v[0];
                streams[1].data[k] = v[1];
            }
            wave_sync();
            // position 0 is never a candidate, nor one with under 3 bytes left
            const uint32_t p0 = w0 ? 0u : 1u, left = n - w0;
            lz_index<kCap>(S, p0, min(stop, left >= kMinLen ? left - (kMinLen - 1) : 0u), sub);
            while (__ballot(cur < stop)) {
                const bool on = cur < stop;
                const uint32_t at = on ? cur : 0;
                const uint32_t word = lds_u32(bytes + at);
                const uint32_t h = lz_hash(word);
                const uint32_t look = on ? min(left - at, kMaxLen) : 0;    // longest match left
                const uint32_t lo = at >= kHist ? at - kHist + 1 : 0;
                uint32_t i, e = look >= kMinLen ? ends[h] : 0;
                if constexpr (LzStream<kCap>::kOld) i = S.first[h];
                else i = h ? ends[h - 1] : 0;
                uint32_t key = 0;               // length << 16 | 0xFFFF - position
                while (__ballot(i < e)) {
                    const uint32_t best = key >> 16;
                    const uint32_t q = i + sub < e ? S.slot[i + sub] : 0xFFFFu;
                    bool live = q < at && q >= lo;
                    const uint32_t cap = live ? min(at - q, look) : 0;
                    // a better match agrees on the byte after the best one's
                    // last, and on the two before it
                    const uint32_t probe = best >= kMinLen ? best - (kMinLen - 1) : 0;
                    live = live && cap > best;
                    const uint32_t qa = live ? q : 0;
                    const uint32_t x = lds_u32(bytes + qa + probe) ^ lds_u32(bytes + at + probe);
                    live = live && (x & 0xFFFFFFu) == 0;
                    uint32_t f = 0;
                    if (__ballot(live)) {
                        bool run = live;
                        while (__ballot(run)) {  // 8 bytes at a time
                            const uint32_t fa = run ? f : 0, qf = run ? q : 0;
                            uint64_t a, b;
                            __builtin_memcpy(&a, bytes + qf + fa, 8);
                            __builtin_memcpy(&b, bytes + at + fa, 8);
                            a ^= b;
                            f = !run ? f : a ? f + ((uint32_t)__builtin_ctzll(a) >> 3) : f + 8;
                            run = run && !a && f < cap;
                        }
                        f = min(f, cap);
                        const uint32_t mine = live && f > best && f >= kMinLen ? f << 16 | (0xFFFFu - q) : 0u;
                        key = max(key, half_max_u32(mine));
                    }
                    if constexpr (LzStream<kCap>::kOld) {
                        // a step wholly out of reach stays so for later positions
                        if (on && i + kHalf <= e && half_ballot(q < lo) == 0xFFFFFFFFu && sub == 0)
                            S.first[h] = (uint16_t)(i + kHalf);
                    }
                    i += kHalf;
                    // younger candidates: none, past the position, or too near to be longer
                    const uint32_t got = key >> 16;
                    const uint32_t reach = half_max_u32(q < at ? q : i - kHalf + sub < e ? 0xFFFFu : 0u);
                    if (got >= look || reach >= at || at - reach <= got) i = e;
                }
                if (on) {
                    const uint32_t len = key >> 16;
                    if (len == 0) {
                        if (sub == 0) out[o] = (uint8_t)word;
                        flags |= 1u << ntok;
                        o += 1;
                        cur += 1;
                    } else {
                        const uint32_t dist = at - (0xFFFFu - (key & 0xFFFFu));
                        const uint16_t v = (uint16_t)(dist << kLenBits | (len - kMinLen));
                        if (sub == 0) __builtin_memcpy(out + o, &v, 2);
                        o += 2;
                        cur += len;
                    }
                    if (++ntok == 8) {          // the next group's flag byte is reserved at once
                        if (sub == 0) out[flag_at] = (uint8_t)flags;
                        flags = 0;
                        ntok = 0;
                        flag_at = o++;
                    }
                }
                if constexpr (LzStream<kCap>::kOld) wave_sync();    // first[] before its next reader
            }
            if (stop == left) break;
            cur -= kHist;                       // the next window starts kHist positions on
        }
        if (sub == 0) {
            out[flag_at] = (uint8_t)flags;
            lane_len[lane] = o;
        }
    }
}

// Sorted slot of lane t: longer lanes first, equal lengths by higher lane id.
// Half a wave per chunk.
constexpr uint32_t kRankThreads = 256, kRankChunks = kRankThreads / kHalf;

__global__ __launch_bounds__(kRankThreads) void lzss_rank_kernel(const uint32_t* __restrict__ lane_len, uint64_t n_chunks,
                                                                 uint64_t* __restrict__ col_len,
                                                                 uint8_t* __restrict__ col_map,
                                                                 uint64_t* __restrict__ chunk_len) {
    __shared__ uint32_t len[kRankThreads];
    const uint32_t t = threadIdx.x % kHalf;
    const uint64_t c = (uint64_t)blockIdx.x * kRankChunks + threadIdx.x / kHalf;
    const uint32_t mine = c < n_chunks ? lane_len[c * 32 + t] : 0u;
    len[threadIdx.x] = mine;
    wave_sync();
    uint32_t rank = 0, words = 0;
    for (uint32_t u = 0; u < kHalf; ++u) {
        const uint32_t other = len[threadIdx.x - t + u];
        rank += (other > mine || (other == mine && u > t)) ? 1u : 0u;
        words += (other + 3) / 4;
    }
    if (c >= n_chunks) return;
    col_len[c * 32 + rank] = mine;
    col_map[c * 32 + rank] = (uint8_t)t;
    if (t == 0) chunk_len[c] = ((uint64_t)words * 4 + 127) / 128 * 128;
}

uint64_t lz_lane_slot(uint64_t chunk) {
    const uint64_t lb = chunk / 32;
    return (lb + lb / 8 + 16 + 15) & ~15ull;          // all literals: one flag byte per 8
}

}  // namespace

int lzss_compress_bound(uint64_t in_bytes, uint64_t chunk, uint64_t* n_chunks, uint64_t* work_bytes,
                        uint64_t* payload_cap) {
    // whole chunks only (a trailing partial chunk is dropped, as the reference
    // encoder drops it); lane positions fit the u16 chains
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
    if (!in || !work || !payload || !col_len || !col_map || !blk_off || n > (1ull << 24)) return MDZ_ERR_INVALID;
    if ((uintptr_t)in & 3) return MDZ_ERR_INVALID;   // lanes are read a dword at a time
    const uint64_t slot = lz_lane_slot(chunk);
    uint8_t* w = static_cast<uint8_t*>(work);
    uint32_t* lane_len = reinterpret_cast<uint32_t*>(w + n * 32 * slot);
    uint64_t* chunk_len = reinterpret_cast<uint64_t*>(w + n * 32 * slot + n * chunk * 2);
    const uint32_t lb = (uint32_t)(chunk / 32);
    const uint64_t units = (n + kXcds - 1) / kXcds * kXcds * kPairs;
    const dim3 grid((uint32_t)(units < (1u << 24) ? units : 1u << 24)), block(kWave);
    auto encode = lb <= 1024 ? lzss_encode_kernel<1024> : lb <= 2048 ? lzss_encode_kernel<2048> : lzss_encode_kernel<4096>;
    hipLaunchKernelGGL(encode, grid, block, 0, s, static_cast<const uint8_t*>(in), n, chunk, slot, w, lane_len);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return record_hip(e, "lzss_encode_kernel launch");
    hipLaunchKernelGGL(lzss_rank_kernel, dim3((uint32_t)((n + kRankChunks - 1) / kRankChunks)), dim3(kRankThreads), 0, s,
                       lane_len, n, col_len, col_map, chunk_len);
    if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lzss_rank_kernel launch");
    hipLaunchKernelGGL(lanes_scan_kernel, dim3(1), dim3(kScanThreads), 0, s, chunk_len, n, blk_off, nullptr, ~0ull);
    if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lanes_scan_kernel launch");
    hipLaunchKernelGGL(lanes_interleave_kernel, dim3((uint32_t)n), dim3(kIlvThreads), 0, s,
                       static_cast<const uint8_t*>(w), slot, col_len, blk_off, chunk_len, col_map,
                       static_cast<uint8_t*>(payload));
    return record_hip(hipGetLastError(), "lanes_interleave_kernel launch");
}

}  // namespace mdz
