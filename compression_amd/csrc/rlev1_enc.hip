// RLE v1 encode for gfx950 (lane-transposed container).
//
// Replaces rle_v1::compress_gpu and its kernels (reference include/rle_v1/
// rlev1.h:24-97: setup_deflate sizes every lane stream, reduction_scan runs
// one thread over the chunk sizes, deflate encodes again and interleaves).
// The payload, col_len and blk_off are byte-identical to that encoder's
// (compression_warp, include/rle_v1/encoder.h:607-1018).
//
// The encoder is greedy over a lane's values x: from the first value not yet
// written, p, a run starts if x[p], x[p+1], x[p+2] have one step in [-128,
// 127], and takes every value that continues it, at most 129; else x[p] is a
// literal, in groups of at most 127.  So the tokens follow from one bit per
// value, S[k]: x[k] continues the step of x[k-1] and x[k-2].
//   1. One wave per lane stream, 64 values at a time: the lanes compute S
//      (lane i the bit of value k = w + i) and decide value k - 2, whose run
//      or literal S[k] settles.  A scalar walk over the ballot of S, a few
//      steps per run, gives the run starts, the literals and the group
//      headers; a prefix sum over the lanes' byte counts places their bytes in
//      an LDS stage.  A header whose count is not known yet (a group or run
//      that goes on past the window) is written when it closes.  64 MiB of
//      4-byte values in 128 KiB chunks: 95 us, vector and scalar issue about
//      equal (1030 us with one lane encoding each stream).  Streams of a few
//      values are encoded by a thread each.
//   2. Small kernels sum the rounded lane lengths per chunk and scan them into
//      blk_off.
//   3. The lane streams are interleaved in the round-robin order of
//      encoder.h:564-588 (lanes_enc_dev.h).
#include <type_traits>

#include "lanes_enc_dev.h"
#include "mdz_device.h"
#include "mdz_internal.h"

namespace mdz {
namespace {

// eb little-endian bytes at `at` (bytes past the input read as 0): one load
// of the element's width when it is whole and aligned, else bytewise.
MDZ_DEV uint64_t load_elem(const uint8_t* in, uint64_t in_bytes, uint64_t at, uint32_t eb) {
    const uint8_t* p = in + at;
    if (at + eb <= in_bytes && ((uintptr_t)p & (eb - 1)) == 0) {
        if (eb == 8) return *reinterpret_cast<const uint64_t*>(p);
        if (eb == 4) return *reinterpret_cast<const uint32_t*>(p);
        if (eb == 2) return *reinterpret_cast<const uint16_t*>(p);
        return *p;
    }
    uint64_t v = 0;
    for (uint32_t b = 0; b < eb; ++b)
        if (at + b < in_bytes) v |= (uint64_t)in[at + b] << (8 * b);
    return v;
}

constexpr uint32_t kMinRunLen = 3, kMaxRunLen = 129, kMaxGroup = 127;
constexpr uint32_t kStageBytes = 4096;
constexpr uint32_t kWindowBytes = 64 * 11;      // most bytes a window adds

// The value of the lane below; `first` in lane 0.
MDZ_DEV uint32_t from_below(uint32_t v, uint32_t first) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)v, 0x138, 0xf, 0xf, false);   // wave_shr:1
}
MDZ_DEV uint64_t from_below(uint64_t v, uint64_t first) {
    return ((uint64_t)from_below((uint32_t)(v >> 32), (uint32_t)(first >> 32)) << 32) |
           from_below((uint32_t)v, (uint32_t)first);
}
MDZ_DEV uint32_t lane_at(uint32_t v, uint32_t lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane); }
MDZ_DEV uint64_t lane_at(uint64_t v, uint32_t lane) {
    return ((uint64_t)lane_at((uint32_t)(v >> 32), lane) << 32) | lane_at((uint32_t)v, lane);
}

template <int EB> struct Wide { typedef uint32_t T; };
template <> struct Wide<8> { typedef uint64_t T; };

// 0x100 | the step x - prev as a byte if it fits int8, else 0, in the element
// type's arithmetic as encoder.h evaluates it (u8/u16 promote to int; u32
// wraps to an unsigned difference, so only 0..127 fit; u64 wraps, signed).
template <int EB>
MDZ_DEV uint32_t step_code(typename Wide<EB>::T x, typename Wide<EB>::T prev) {
    const typename Wide<EB>::T d = x - prev;
    const bool fits = EB == 4 ? d < 128 : d + 128 < 256;
    return fits ? 0x100u | ((uint32_t)d & 0xFFu) : 0u;
}

// Values of lane t of chunk c: byte k*EB of the lane sits in line t + 32*(k*EB
// / line).  A chunk inside the input, aligned, with lines of a power of two:
// one load a value.
template <int EB>
struct LaneValues {
    typedef typename Wide<EB>::T T;
    typedef typename std::conditional<EB == 8, uint64_t, typename std::conditional<EB == 4, uint32_t,
            typename std::conditional<EB == 2, uint16_t, uint8_t>::type>::type>::type Elem;
    const uint8_t *in, *src;
    uint64_t in_bytes, base;
    uint32_t n, line, t, shift;
    bool plain;

    MDZ_DEV LaneValues(const uint8_t* in_, uint64_t in_bytes_, uint64_t c, uint64_t chunk, uint32_t line_, uint32_t t_)
        : in(in_), src(in_ + c * chunk), in_bytes(in_bytes_), base(c * chunk), n((uint32_t)(chunk / 32 / EB)),
          line(line_), t(t_), shift(31 - __builtin_clz(line_)),
          plain((line_ & (line_ - 1)) == 0 && (c + 1) * chunk <= in_bytes_ && ((uintptr_t)src & (EB - 1)) == 0) {}
    MDZ_DEV T operator()(uint32_t k) const {     // any value past the last
        if (plain) {
            const uint32_t o = min(k, n - 1) * EB;
            return *reinterpret_cast<const Elem*>(src + ((((uint64_t)(o >> shift) * 32 + t) << shift) | (o & (line - 1))));
        }
        if (k >= n) return 0;
        const uint32_t o = k * EB, r = o / line, j = o - r * line;
        return (T)load_elem(in, in_bytes, base + (t + 32ull * r) * line + j, EB);
    }
};

template <class T>
MDZ_DEV uint32_t leb_bytes(T v) {                // ceil(bits / 7), at least 1
    const uint32_t bits = sizeof(T) == 8 ? 64 - (uint32_t)__builtin_clzll((uint64_t)v | 1) : 32 - (uint32_t)__builtin_clz((uint32_t)v | 1);
    return ((bits + 6) * 37) >> 8;
}

// Output of a lane stream: bytes [base, at) are staged in LDS, those below are
// stored.  base is a multiple of 4.
struct LaneStage {
    uint8_t* stage;
    uint8_t* out;
    uint32_t base, at;

    MDZ_DEV void patch(uint32_t where, uint32_t b) {          // one byte, wave-uniform
        if (lane_id() == 0) {
            if (where >= base) stage[where - base] = (uint8_t)b;
            else out[where] = (uint8_t)b;
        }
    }
    MDZ_DEV void flush() {
        wave_sync();
        const uint32_t whole = (at - base) / 4, rest = (at - base) & 3;
        const uint32_t* s = reinterpret_cast<const uint32_t*>(stage);
        uint32_t* o = reinterpret_cast<uint32_t*>(out + base);
        for (uint32_t i = lane_id(); i < whole; i += kWave) o[i] = s[i];
        const uint32_t keep = s[whole];
        wave_sync();
        if (rest && lane_id() == 0) *reinterpret_cast<uint32_t*>(stage) = keep;
        wave_sync();
        base += 4 * whole;
    }
};

template <int EB>
__global__ __launch_bounds__(kWave) void rlev1_encode_kernel(const uint8_t* __restrict__ in, uint64_t in_bytes,
                                                             uint64_t n_chunks, uint64_t chunk, uint32_t line,
                                                             uint64_t lane_slot, uint8_t* __restrict__ work,
                                                             uint64_t* __restrict__ col_len) {
    typedef typename Wide<EB>::T T;
    __shared__ uint32_t stage[kStageBytes / 4 + 1];
    const uint32_t l = lane_id(), n = (uint32_t)(chunk / 32 / EB);
    for (uint64_t unit = blockIdx.x; unit < lane_units(n_chunks); unit += gridDim.x) {
        uint64_t c;
        uint32_t t;
        if (!lane_of_unit(unit, n_chunks, c, t)) continue;
        const LaneValues<EB> value(in, in_bytes, c, chunk, line, t);
        LaneStage w{reinterpret_cast<uint8_t*>(stage), work + (c * 32 + t) * lane_slot, 0, 0};
        uint32_t lit = 0, lit_at = 0;            // open literal group: values so far, header's offset
        uint32_t ones = 0, run_at = 0;           // open run: bits of S so far, count byte's offset
        uint32_t skip = 2;                       // lanes of the window before the first undecided value
        T x1 = 0, x2 = 0;                        // the two values before the window
        uint32_t s1 = 0;                         // step code of the last of them
        T next = value(l);
        for (uint32_t w0 = 0; w0 < n + 2; w0 += kWave) {
            const T x = next;
            next = value(w0 + kWave + l);
            const T p1 = from_below(x, x1), p2 = from_below(p1, x2);
            const uint32_t k = w0 + l, code = k && k < n ? step_code<EB>(x, p1) : 0u;
            const uint32_t below = from_below(code, s1);
            const uint64_t S = __ballot(code != 0 && code == below);
            x1 = lane_at(x, kWave - 1), x2 = lane_at(x, kWave - 2);
            s1 = lane_at(code, kWave - 1);
            const uint32_t end = min(n + 2 - w0, (uint32_t)kWave);     // lanes whose value k - 2 exists

            // the scalar walk: literals, run starts, headers, and the count
            // byte of each header that closes here
            uint64_t literals = 0, starts = 0, heads = 0;
            uint32_t head = 0;
            uint32_t group_lane = kWave, run_lane = kWave;             // openers in this window
            uint32_t j = skip;
            if (ones) {                          // a run goes on from the window before
                uint32_t more = ~S ? (uint32_t)__builtin_ctzll(~S) : kWave;
                more = min(more, kMaxRunLen - 2 - ones);
                ones += more;
                if (more == kWave) {
                    j = kWave;
                } else {
                    w.patch(run_at, ones + 2 - kMinRunLen);
                    j = more + 2;
                    ones = 0;
                }
            }
            while (j < end) {
                const uint64_t left = S >> j;
                const uint32_t s = left ? j + (uint32_t)__builtin_ctzll(left) : end, m = s - j;
                if (m) {
                    literals |= (m == 64 ? ~0ull : (1ull << m) - 1) << j;
                    uint32_t open = lit == 0 ? j : lit + m > kMaxGroup ? j + (kMaxGroup - lit) : kWave;
                    if (open < kWave) {          // a group opens at that lane; the one before is full
                        if (lit) {
                            if (group_lane < kWave) head = l == group_lane ? 256 - kMaxGroup : head;
                            else w.patch(lit_at, 256 - kMaxGroup);
                        }
                        heads |= 1ull << open;
                        group_lane = open;
                        lit = s - open;
                    } else {
                        lit += m;
                    }
                }
                j = s;
                if (s == end) break;
                if (lit) {                       // the run closes the group
                    if (group_lane < kWave) head = l == group_lane ? 256 - lit : head;
                    else w.patch(lit_at, 256 - lit);
                    lit = 0;
                    group_lane = kWave;
                }
                starts |= 1ull << s;
                const uint64_t rest = ~(S >> s);
                const uint32_t bits = rest ? (uint32_t)__builtin_ctzll(rest) : kWave;
                if (s + bits >= kWave) {         // may go on in the next window
                    ones = kWave - s;
                    run_lane = s;
                    j = kWave;
                } else {
                    head = l == s ? bits + 2 - kMinRunLen : head;
                    j = s + bits + 2;
                }
            }
            skip = j > kWave ? j - kWave : 0;

            // bytes: a literal's value, behind the group's header at its
            // first; a run's count, step and first value
            const bool is_lit = (literals >> l) & 1, is_run = (starts >> l) & 1, opens = (heads >> l) & 1;
            const uint32_t vb = leb_bytes(p2), pre = is_run ? 2 : opens ? 1 : 0;
            const uint32_t mine = is_lit || is_run ? pre + vb : 0;
            const uint32_t incl = wave_incl_scan_u32(mine);
            const uint32_t at = w.at + incl - mine;
            uint8_t* o = w.stage + (at - w.base);
            if (pre) o[0] = (uint8_t)head;
            if (is_run) o[1] = (uint8_t)code;
            T v = p2;
            for (uint32_t i = 0; __ballot(mine && i < vb); ++i) {
                if (mine && i < vb) o[pre + i] = (uint8_t)((uint32_t)v & 0x7Fu) | (i + 1 < vb ? 0x80u : 0u);
                v >>= 7;
            }
            if (group_lane < kWave) lit_at = lane_at(at, group_lane);
            if (run_lane < kWave) run_at = lane_at(at, run_lane);
            w.at += lane_at(incl, kWave - 1);
            if (w.at - w.base > kStageBytes - kWindowBytes) w.flush();
            wave_sync();
        }
        if (lit) w.patch(lit_at, 256 - lit);
        w.flush();
        if (l == 0) {
            if (w.at != w.base) *reinterpret_cast<uint32_t*>(w.out + w.base) = stage[0];
            col_len[c * 32 + t] = w.at;
        }
        wave_sync();
    }
}

// Short lane streams: a thread encodes one, value by value, half a wave per
// chunk.  No group or run of so few values is full.  A window of 64 values
// costs a wave the same whatever it holds: 65536 chunks of 2 4-byte values a
// lane take 811 us with a wave per stream and 34 us so, 3276 of 40 values 48 and
// 40 us.  One thread's values wait for each other, though: few chunks leave the
// chip empty either way, and there a wave is the faster from about 9 values a
// lane on (512 chunks of 16: 17 us a call against 19; 2048 chunks: 38 against 23).
// Bytes stay faster with a thread up to a whole window (4096 chunks of 64: 69 us
// against 98), wider values do not (2048 chunks of 64 8-byte values: 73 against 65).
constexpr uint32_t kShortThreads = 256, kShortChunks = kShortThreads / 32;
constexpr uint32_t kShortValues = 8, kShortOfMany = 40, kShortBytesOfMany = 64, kManyChunks = 2048;
static_assert(kShortBytesOfMany <= kMaxGroup && kShortBytesOfMany <= kMaxRunLen, "short streams fill no token");
inline bool short_lanes(uint64_t values, uint32_t eb, uint64_t n_chunks) {
    return values <= kShortValues ||
           (values <= (eb == 1 ? kShortBytesOfMany : kShortOfMany) && n_chunks >= kManyChunks);
}

template <int EB>
__global__ __launch_bounds__(kShortThreads) void rlev1_short_kernel(const uint8_t* __restrict__ in, uint64_t in_bytes,
                                                                    uint64_t n_chunks, uint64_t chunk, uint32_t line,
                                                                    uint64_t lane_slot, uint8_t* __restrict__ work,
                                                                    uint64_t* __restrict__ col_len,
                                                                    uint64_t* __restrict__ chunk_len) {
    typedef typename Wide<EB>::T T;
    const uint64_t c = (uint64_t)blockIdx.x * kShortChunks + threadIdx.x / 32;
    const uint32_t t = threadIdx.x % 32, n = (uint32_t)(chunk / 32 / EB);
    uint32_t len = 0;
    if (c < n_chunks) {
        const LaneValues<EB> value(in, in_bytes, c, chunk, line, t);
        WordOut o{work + (c * 32 + t) * lane_slot};
        uint32_t lit = 0, lit_at = 0;            // open literal group: values so far, header's offset
        auto varint = [&](T v) {
            for (; v > 0x7F; v >>= 7) o.put(((uint32_t)v & 0x7Fu) | 0x80u);
            o.put((uint32_t)v);
        };
        // x0, x1: the first value not yet written and its successor; s: x1's step code
        T x0 = value(0), x1 = value(1);
        uint32_t s = step_code<EB>(x1, x0), p = 0;
        while (p < n) {
            T x2 = value(p + 2);
            uint32_t s2 = p + 2 < n ? step_code<EB>(x2, x1) : 0;
            if (s && s2 == s) {
                if (lit) o.patch(lit_at, 256 - lit);
                lit = 0;
                uint32_t m = 2;
                do {                             // x2 is value p + m, in the run
                    ++m;
                    x1 = x2;
                    x2 = value(p + m);
                    s2 = p + m < n ? step_code<EB>(x2, x1) : 0;
                } while (s2 == s);
                o.put(m - kMinRunLen);
                o.put(s & 0xFFu);
                varint(x0);
                p += m;
                x0 = x2;
                x1 = value(p + 1);
                s = p + 1 < n ? step_code<EB>(x1, x0) : 0;
            } else {
                if (lit++ == 0) {
                    lit_at = o.len;
                    o.put(0);
                }
                varint(x0);
                ++p;
                x0 = x1;
                x1 = x2;
                s = s2;
            }
        }
        if (lit) o.patch(lit_at, 256 - lit);
        len = o.finish();
        col_len[c * 32 + t] = len;
    }
    store_chunk_len((len + 3) / 4, c, n_chunks, chunk_len);
}

uint64_t lane_slot_bytes(uint64_t chunk, uint32_t eb) {
    const uint64_t n = chunk / 32 / eb;
    return (n * 11 + 16 + 15) & ~15ull;          // LEB128 <= 10 bytes per value, plus headers
}

}  // namespace

int rlev1_compress_bound(uint64_t in_bytes, uint64_t chunk, uint32_t eb, uint32_t line, uint64_t* n_chunks,
                         uint64_t* work_bytes, uint64_t* payload_cap) {
    if (in_bytes == 0 || chunk % 32 || line == 0 || (chunk / 32) % line || line % eb ||
        (eb != 1 && eb != 2 && eb != 4 && eb != 8) || (chunk / 32) / eb < 2 || chunk > (1ull << 32))
        return MDZ_ERR_INVALID;
    const uint64_t n = (in_bytes + chunk - 1) / chunk;
    const uint64_t slot = lane_slot_bytes(chunk, eb);
    if (n_chunks) *n_chunks = n;
    if (work_bytes) *work_bytes = n * 32 * slot + 8 * n;
    if (payload_cap) *payload_cap = n * ((32 * slot + 127) / 128 * 128);
    return MDZ_OK;
}

int rlev1_compress(const void* in, uint64_t in_bytes, uint64_t chunk, uint32_t eb, uint32_t line, void* work,
                   void* payload, uint64_t* col_len, uint64_t* blk_off, hipStream_t s) {
    uint64_t n = 0;
    int rc = rlev1_compress_bound(in_bytes, chunk, eb, line, &n, nullptr, nullptr);
    if (rc) return rc;
    if (!in || !work || !payload || !col_len || !blk_off || n > kMaxEncodeChunks) return MDZ_ERR_INVALID;
    const uint64_t slot = lane_slot_bytes(chunk, eb);
    uint64_t* chunk_len = reinterpret_cast<uint64_t*>(static_cast<uint8_t*>(work) + n * 32 * slot);
    hipError_t e;
    if (short_lanes(chunk / 32 / eb, eb, n)) {
        auto encode = eb == 1 ? rlev1_short_kernel<1> : eb == 2 ? rlev1_short_kernel<2>
                    : eb == 4 ? rlev1_short_kernel<4> : rlev1_short_kernel<8>;
        hipLaunchKernelGGL(encode, dim3((uint32_t)((n + kShortChunks - 1) / kShortChunks)), dim3(kShortThreads), 0, s,
                           static_cast<const uint8_t*>(in), in_bytes, n, chunk, line, slot,
                           static_cast<uint8_t*>(work), col_len, chunk_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "rlev1_short_kernel launch");
    } else {
        auto encode = eb == 1 ? rlev1_encode_kernel<1> : eb == 2 ? rlev1_encode_kernel<2>
                    : eb == 4 ? rlev1_encode_kernel<4> : rlev1_encode_kernel<8>;
        hipLaunchKernelGGL(encode, lane_grid(n), dim3(kWave), 0, s, static_cast<const uint8_t*>(in), in_bytes, n,
                           chunk, line, slot, static_cast<uint8_t*>(work), col_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "rlev1_encode_kernel launch");
        hipLaunchKernelGGL(lanes_size_kernel, dim3((uint32_t)((n + kSizeChunks - 1) / kSizeChunks)), dim3(kSizeThreads),
                           0, s, col_len, n, chunk_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lanes_size_kernel launch");
    }
    hipLaunchKernelGGL(lanes_scan_kernel, dim3(1), dim3(kScanThreads), 0, s, chunk_len, n, blk_off, nullptr, ~0ull);
    if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lanes_scan_kernel launch");
    hipLaunchKernelGGL(lanes_interleave_kernel, interleave_grid(n, slot), dim3(kIlvThreads), 0, s,
                       static_cast<const uint8_t*>(work), slot, col_len, blk_off, chunk_len, nullptr,
                       static_cast<uint8_t*>(payload));
    return record_hip(hipGetLastError(), "lanes_interleave_kernel launch");
}

}  // namespace mdz
