// RLE v2 encode for gfx950 (lane-transposed container).
//
// Replaces rlev2::compress_gpu_transpose (reference include/rlev2/
// encoder_trans.h:428-537: block_encode :14-289 per lane, the transpose
// :291-349, the scans :466-492).  Payload, col_len and blk_off (blk_off[n]
// holding the uncompressed size, as the reference leaves it) equal that
// encoder's output byte for byte: run grouping of block_encode, the sub-mode
// choice of determineEncoding and the four writers (encoder.h:124-785).
//
// One wave per lane stream, whose q-th value is chunk element
// (q / RU) * 32 * RU + t * RU + q % RU.  A window of the stream's values sits
// in LDS.  block_encode's grouping depends on which neighbours are equal
// alone: a group that starts at s is
//   * a run if its first three values are equal: all values equal to them, at
//     most 128;
//   * else the literals up to the first three equal values in a row that lie
//     inside the group, at most 128.
// So per group the 64 lanes hold 128 values, two each, ballots of the equal
// neighbours give the group, and the sub-mode is chosen from ballots and
// counts: the 90th and 95th percentile tests take one count each, of the values
// that reach the next smaller width or the largest; only a patched group
// searches the width codes for its percentile, five counts.  Every writer packs
// most significant bit first, so all of them put fields at bit positions: the
// lanes or their fields into an LDS stage of big-endian words, which goes out
// in whole words.  A group costs about 300 instructions instead of its values'
// serial chain.  256 MiB of 8-byte values in 128 KiB chunks: 0.30 ms, bound by
// scalar and vector issue (1,900 and 1,060 instructions a stream) at 20 waves a
// CU (24.3 ms with one lane encoding each stream).  Streams of a few values are
// encoded by a thread each.  The scan and the interleave are the shared
// lane-encoder kernels (lanes_enc_dev.h).
#include <type_traits>

#include "lanes_enc_dev.h"
#include "mdz_device.h"
#include "mdz_internal.h"

namespace mdz {
namespace {

constexpr uint32_t kMinRepeat = 3, kMaxLit = 128, kMaxShortRepeat = 10;

constexpr uint32_t kStageWords = 640;            // output words staged per wave
constexpr uint32_t kGroupWords = 288;            // most words a group takes: 128 fields of 64 bits, headers, varints

// Values of the window: u32 storage when elements are 4 bytes or less,
// arithmetic always in 64 bits.
template <class LT>
struct V2EncLds {
    static constexpr uint32_t kVals = 4096 / sizeof(LT);
    LT val[kVals + kMaxLit];                     // the tail is read, not used
    uint32_t stage[kStageWords];
};

// The 5-bit width code of a bit width, and the widths each writer rounds to.
MDZ_DEV uint32_t width_code(uint32_t bits) {
    if (bits <= 1) return 0;
    if (bits <= 24) return bits - 1;
    if (bits <= 26) return 24;
    if (bits <= 28) return 25;
    if (bits <= 30) return 26;
    if (bits <= 32) return 27;
    if (bits <= 40) return 28;
    if (bits <= 48) return 29;
    if (bits <= 56) return 30;
    return 31;
}
MDZ_DEV uint32_t code_width(uint32_t code) {
    return code < 24 ? code + 1 : code < 28 ? 26 + 2 * (code - 24) : 40 + 8 * (code - 28);
}
MDZ_DEV uint32_t fixed_width(uint32_t bits) {            // nearest encodable width >= bits
    return code_width(width_code(bits));
}
MDZ_DEV uint32_t aligned_width(uint32_t bits) {          // 1, 2, 4, 8, 16, 24, 32, ... 64
    if (bits <= 1) return 1;
    if (bits <= 2) return 2;
    if (bits <= 4) return 4;
    if (bits <= 8) return 8;
    if (bits <= 16) return 16;
    if (bits <= 24) return 24;
    if (bits <= 32) return 32;
    return fixed_width(bits);                       // 40, 48, 56, 64
}
MDZ_DEV uint32_t value_width(uint64_t v) {               // fixed width of the bit length
    return fixed_width(v ? 64 - __builtin_clzll(v) : 0);
}

MDZ_DEV uint32_t bit_length(uint64_t v) { return v ? 64 - __builtin_clzll(v) : 0; }

MDZ_DEV uint32_t wave_max_u32(uint32_t v) {
    v = max(v, dpp_src<0x111, 0xf, 0u>(v));
    v = max(v, dpp_src<0x112, 0xf, 0u>(v));
    v = max(v, dpp_src<0x114, 0xf, 0u>(v));
    v = max(v, dpp_src<0x118, 0xf, 0u>(v));
    v = max(v, dpp_src<0x142, 0xa, 0u>(v));
    v = max(v, dpp_src<0x143, 0xc, 0u>(v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, kWave - 1);
}
template <int kCtrl, int kRowMask>
MDZ_DEV uint64_t dpp_min_u64(uint64_t v) {
    const uint64_t o = ((uint64_t)dpp_src<kCtrl, kRowMask, ~0u>((uint32_t)(v >> 32)) << 32) |
                       dpp_src<kCtrl, kRowMask, ~0u>((uint32_t)v);
    return min(v, o);
}
MDZ_DEV uint64_t wave_min_u64(uint64_t v) {
    v = dpp_min_u64<0x111, 0xf>(v);
    v = dpp_min_u64<0x112, 0xf>(v);
    v = dpp_min_u64<0x114, 0xf>(v);
    v = dpp_min_u64<0x118, 0xf>(v);
    v = dpp_min_u64<0x142, 0xa>(v);
    v = dpp_min_u64<0x143, 0xc>(v);
    return last_lane_u64(v);
}
MDZ_DEV uint64_t lane_u64(uint64_t v, int lane) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
}

// A group's values, lane l holding values l and 64 + l, and each one's
// predecessor; m0 and m1 are the lanes that hold one of its n values.
struct Group {
    uint64_t a0, a1, p0, p1;
    uint32_t n;
    uint64_t m0, m1;

    MDZ_DEV void take(uint32_t count) {
        n = count;
        m0 = n >= 64 ? ~0ull : (1ull << n) - 1;
        m1 = n >= 128 ? ~0ull : n > 64 ? (1ull << (n - 64)) - 1 : 0;
    }
    // Values for which the test holds; pairs: of value i - 1 and value i, i >= 1.
    template <class F> MDZ_DEV bool any(F f) const {
        return ((__ballot(f(a0)) & m0) | (__ballot(f(a1)) & m1)) != 0;
    }
    template <class F> MDZ_DEV bool any_pair(F f) const {
        return ((__ballot(f(p0, a0)) & m0 & ~1ull) | (__ballot(f(p1, a1)) & m1)) != 0;
    }
    // The largest width code that more than `below` of the n codes (c0, c1 per lane) reach.
    MDZ_DEV uint32_t code_at(uint32_t c0, uint32_t c1, uint32_t below) const {
        uint32_t c = 0;
#pragma unroll
        for (uint32_t bit = 16; bit; bit >>= 1) {
            const uint32_t k = (uint32_t)__popcll(__ballot(c0 >= (c | bit)) & m0) +
                               (uint32_t)__popcll(__ballot(c1 >= (c | bit)) & m1);
            if (k > below) c |= bit;
        }
        return c;
    }
    // How many of the codes are at least c.
    MDZ_DEV uint32_t at_least(uint32_t c0, uint32_t c1, uint32_t c) const {
        return (uint32_t)__popcll(__ballot(c0 >= c) & m0) + (uint32_t)__popcll(__ballot(c1 >= c) & m1);
    }
    MDZ_DEV uint32_t most(uint32_t c0, uint32_t c1) const {
        const uint32_t l = lane_id();
        return wave_max_u32(max(l < n ? c0 : 0u, 64 + l < n ? c1 : 0u));
    }
    // Values above the p-th percentile, as the reference counts them.
    MDZ_DEV uint32_t above(uint32_t p) const { return (n * (100 - p) - 1) / 100 + 1; }
};

// The lane stream's output: `bits` bits staged (big-endian words, zero past
// them), `words` words stored.
struct Sink {
    uint32_t* stage;
    uint8_t* out;
    uint64_t words = 0;
    uint32_t bits = 0;

    MDZ_DEV void start() {
        for (uint32_t i = lane_id(); i < kStageWords; i += kWave) stage[i] = 0;
        wave_sync();
    }
    // The low w bits (1..64) of v at bit `at` of the stage.
    MDZ_DEV void field(bool on, uint32_t at, uint64_t v, uint32_t w) {
        if (on) {
            const uint64_t top = v << (64 - w);
            const uint32_t sh = at & 31;
            const uint64_t hi = top >> sh;
            const uint32_t lo = sh ? (uint32_t)top << (32 - sh) : 0u;
            uint32_t* s = stage + (at >> 5);
            atomicOr(s, (uint32_t)(hi >> 32));
            if (w + sh > 32) {
                atomicOr(s + 1, (uint32_t)hi);
                if (w + sh > 64) atomicOr(s + 2, lo);
            }
        }
    }
    // A field of the whole wave's: v, bytes long.
    MDZ_DEV void bytes(uint64_t v, uint32_t count) {
        if (count) field(lane_id() == 0, bits, v, 8 * count);
        bits += 8 * count;
    }
    // LEB128, a lane per byte.
    MDZ_DEV void varint(uint64_t v) {
        const uint32_t len = max(1u, (bit_length(v) + 6) / 7), l = lane_id();
        const uint32_t b = (uint32_t)(v >> min(7 * l, 63u)) & 0x7Fu;
        field(l < len, bits + 8 * l, b | (l + 1 < len ? 0x80u : 0u), 8);
        bits += 8 * len;
    }
    MDZ_DEV void pad() { bits = (bits + 7) & ~7u; }
    // Stores the whole words and moves the rest to the stage's start.
    MDZ_DEV void flush() {
        wave_sync();
        const uint32_t full = bits >> 5, rest = stage[full];
        uint32_t* o = reinterpret_cast<uint32_t*>(out) + words;
        wave_sync();
        for (uint32_t i = lane_id(); i <= full; i += kWave) {
            if (i < full) o[i] = __builtin_bswap32(stage[i]);
            stage[i] = 0;
        }
        wave_sync();
        if (lane_id() == 0) stage[0] = rest;
        wave_sync();
        words += full;
        bits &= 31;
    }
    MDZ_DEV uint64_t finish() {                  // the stream's bytes
        flush();
        if (bits && lane_id() == 0) reinterpret_cast<uint32_t*>(out)[words] = __builtin_bswap32(stage[0]);
        return 4 * words + bits / 8;
    }
};

// The four writers (encoder.h:537-785); fields go out as the group's lanes hold them.
MDZ_DEV void short_repeat(Sink& o, uint64_t v, uint32_t n) {
    const uint32_t vbytes = (value_width(v) - 1) / 8 + 1;
    o.bytes(((vbytes - 1) << 3) | (n - kMinRepeat), 1);
    o.bytes(v, vbytes);
}
// f(i): value i of `count` values of w bits; lane l gives values l and 64 + l of them.
MDZ_DEV void fields(Sink& o, uint64_t v0, uint64_t v1, uint32_t count, uint32_t w) {
    const uint32_t l = lane_id();
    o.field(l < count, o.bits + l * w, v0, w);
    o.field(64 + l < count, o.bits + (64 + l) * w, v1, w);
    o.bits += count * w;
    o.pad();
}
MDZ_DEV uint32_t header(uint32_t mode, uint32_t code, uint32_t n) {
    return (mode | code << 1 | ((n - 1) & 0x100) >> 8) << 8 | ((n - 1) & 0xFF);
}
MDZ_DEV void direct(Sink& o, const Group& g, uint32_t code100) {
    const uint32_t w = aligned_width(code_width(code100));
    o.bytes(header(0x40, width_code(w), g.n), 2);
    fields(o, g.a0, g.a1, g.n, w);
}
MDZ_DEV void fixed_delta(Sink& o, uint64_t first, uint64_t step, uint32_t n) {
    o.bytes(header(0xC0, 0, n), 2);
    o.varint(first);
    o.varint((step << 1) ^ (uint64_t)((int64_t)step >> 63));         // zigzag
}
MDZ_DEV void delta(Sink& o, const Group& g, uint64_t first, uint64_t step, uint32_t delta_bits) {
    const uint32_t w = max(2u, aligned_width(delta_bits));
    o.bytes(header(0xC0, width_code(w), g.n), 2);
    o.varint(first);
    o.varint((step << 1) ^ (uint64_t)((int64_t)step >> 63));
    // the deltas from value 2 on: lane l holds those of values l and 64 + l
    const uint32_t l = lane_id();
    const uint64_t keep = ~0ull >> (64 - w);
    o.field(l >= 2 && l < g.n, o.bits + (l - 2) * w, (g.a0 - g.p0) & keep, w);
    o.field(64 + l < g.n, o.bits + (62 + l) * w, (g.a1 - g.p1) & keep, w);
    o.bits += (g.n - 2) * w;
    o.pad();
}
MDZ_DEV void patched(Sink& o, const Group& g, uint64_t base, uint32_t b95, uint32_t b100) {
    const uint64_t r0 = g.a0 - base, r1 = g.a1 - base;
    uint32_t pw = fixed_width(b100 - b95);
    if (pw == 64) {
        pw = 56;
        b95 = 8;
    }
    const uint64_t mask = (1ull << b95) - 1;
    const bool on0 = r0 > mask, on1 = r1 > mask;
    const uint64_t q0 = __ballot(on0) & g.m0, q1 = __ballot(on1) & g.m1;
    const uint32_t l = lane_id(), np = (uint32_t)__popcll(q0) + (uint32_t)__popcll(q1);
    // gaps from the patch before (the first one's from value 0)
    const uint64_t below = (1ull << l) - 1, u0 = q0 & below, u1 = q1 & below;
    const uint32_t gap0 = l - (u0 ? 63 - __builtin_clzll(u0) : 0);
    const uint32_t gap1 = 64 + l - (u1 ? 127 - __builtin_clzll(u1) : q0 ? 63 - __builtin_clzll(q0) : 0);
    const bool is0 = on0 && l < g.n, is1 = on1 && 64 + l < g.n;
    const uint32_t max_gap = wave_max_u32(max(is0 ? gap0 : 0u, is1 ? gap1 : 0u));
    const uint32_t pgw = value_width(max_gap);           // gaps stay below 128; no gap counts as 1 bit
    const uint32_t vbytes = value_width(base) / 8 + 1;
    o.bytes(header(0x80, width_code(b95), g.n), 2);
    o.bytes((((vbytes - 1) << 5) | width_code(pw)) << 8 | ((((pgw - 1) << 5) | np) & 0xFF), 2);
    if (vbytes > 8) o.bytes(0, 1);
    o.bytes(base, min(vbytes, 8u));
    fields(o, r0 & mask, r1 & mask, g.n, fixed_width(b95));
    const uint32_t w = fixed_width(pgw + pw);
    const uint32_t at0 = (uint32_t)__popcll(u0), at1 = (uint32_t)(__popcll(q0) + __popcll(u1));
    o.field(is0, o.bits + at0 * w, (uint64_t)gap0 << pw | r0 >> b95, w);
    o.field(is1, o.bits + at1 * w, (uint64_t)gap1 << pw | r1 >> b95, w);
    o.bits += np * w;
    o.pad();
}
// determineEncoding (encoder.h:366-535) of a literal group.
MDZ_DEV void literals(Sink& o, const Group& g) {
    const uint32_t c0 = width_code(bit_length(g.a0)), c1 = width_code(bit_length(g.a1));
    const uint64_t first = lane_u64(g.a0, 0);
    // the reference's signed-subtract safety test with INT8_MIN fails only
    // when min == 0 and max <= 128
    const bool narrow = g.n > kMinRepeat && g.any([](uint64_t v) { return v == 0; }) &&
                        !g.any([](uint64_t v) { return v > 128; });
    if (g.n > kMinRepeat && !narrow) {
        const uint64_t step = lane_u64(g.a0, 1) - first;
        if (!g.any_pair([&](uint64_t p, uint64_t v) { return v - p != step; })) {
            fixed_delta(o, first, step, g.n);
            return;
        }
        if (step && (!g.any_pair([](uint64_t p, uint64_t v) { return p > v; }) ||
                     !g.any_pair([](uint64_t p, uint64_t v) { return p < v; }))) {
            const uint32_t l = lane_id();
            const uint32_t most = wave_max_u32(max(l && l < g.n ? bit_length(g.a0 - g.p0) : 0u,
                                                   64 + l < g.n ? bit_length(g.a1 - g.p1) : 0u));
            delta(o, g, first, step, fixed_width(most));
            return;
        }
    }
    const uint32_t code100 = g.most(c0, c1);
    if (g.n > kMinRepeat && !narrow) {
        // the 90th percentile's width is over 1 below the largest: too few
        // values reach the widths that are not (widths step by 1 up to 24,
        // code 23, and by 2 or more beyond)
        const uint32_t near = code100 < 24 ? max(code100, 1u) - 1 : code100;
        if (g.at_least(c0, c1, near) <= g.above(90)) {
            const uint32_t l = lane_id();
            const uint64_t base = wave_min_u64(min(l < g.n ? g.a0 : ~0ull, 64 + l < g.n ? g.a1 : ~0ull));
            const uint32_t d0 = width_code(bit_length(g.a0 - base)), d1 = width_code(bit_length(g.a1 - base));
            const uint32_t r100 = g.most(d0, d1);
            if (g.at_least(d0, d1, r100) <= g.above(95)) {
                patched(o, g, base, code_width(g.code_at(d0, d1, g.above(95))), code_width(r100));
                return;
            }
        }
    }
    direct(o, g, code100);
}

// Element `el` of the chunk at byte `base`; a partial last value reads as 0.
MDZ_DEV uint64_t chunk_value(const uint8_t* in, uint64_t in_bytes, uint64_t base, uint64_t el, uint32_t eb) {
    const uint64_t off = base + el * eb;
    if (off + eb > in_bytes) return 0;
    const uint8_t* p = in + off;
    if (((uintptr_t)p & (eb - 1)) == 0) {                 // one load of the element's width
        if (eb == 8) return *reinterpret_cast<const uint64_t*>(p);
        if (eb == 4) return *reinterpret_cast<const uint32_t*>(p);
        if (eb == 2) return *reinterpret_cast<const uint16_t*>(p);
        return *p;
    }
    uint64_t v = 0;
    for (uint32_t b = 0; b < eb; ++b) v |= (uint64_t)p[b] << (8 * b);
    return v;
}

// Values [s, end) of lane t of the chunk at byte `base` to val[0, end - s).
// Where every value is whole, aligned and its line a power of two, eight loads
// a lane are in flight.
template <int EB, class LT>
MDZ_DEV void load_values(LT* val, const uint8_t* in, uint64_t in_bytes, uint64_t base, uint64_t chunk, uint32_t ru,
                         uint32_t t, uint32_t s, uint32_t end) {
    typedef typename std::conditional<EB == 8, uint64_t, typename std::conditional<EB == 4, uint32_t,
            typename std::conditional<EB == 2, uint16_t, uint8_t>::type>::type>::type E;
    const uint32_t l = lane_id();
    if (base + chunk <= in_bytes && ((uintptr_t)(in + base) & (EB - 1)) == 0 && (ru & (ru - 1)) == 0) {
        const E* v = reinterpret_cast<const E*>(in + base);
        const uint32_t sh = 31 - __builtin_clz(ru);
        for (uint32_t q0 = s; q0 < end; q0 += 8 * kWave) {
            E x[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) {
                const uint32_t q = min(q0 + i * kWave + l, end - 1);
                x[i] = v[((uint64_t)(q >> sh) * 32 + t) << sh | (q & (ru - 1))];
            }
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i)
                if (q0 + i * kWave + l < end) val[q0 + i * kWave + l - s] = (LT)x[i];
        }
        return;
    }
    for (uint32_t q = s + l; q < end; q += kWave) {
        const uint32_t line = q / ru;
        val[q - s] = (LT)chunk_value(in, in_bytes, base, ((uint64_t)line * 32 + t) * ru + (q - line * ru), EB);
    }
}

template <int EB>
__global__ __launch_bounds__(kWave) void rlev2_encode_kernel(const uint8_t* __restrict__ in, uint64_t in_bytes,
                                                             uint64_t n_chunks, uint64_t chunk, uint32_t ru,
                                                             uint64_t lane_slot, uint8_t* __restrict__ work,
                                                             uint64_t* __restrict__ col_len) {
    typedef typename std::conditional<EB == 8, uint64_t, uint32_t>::type LT;
    __shared__ V2EncLds<LT> S;
    constexpr uint32_t kVals = V2EncLds<LT>::kVals;
    const uint32_t l = lane_id(), nv = (uint32_t)(chunk / EB / 32);
    for (uint64_t unit = blockIdx.x; unit < lane_units(n_chunks); unit += gridDim.x) {
        uint64_t c;
        uint32_t t;
        if (!lane_of_unit(unit, n_chunks, c, t)) continue;
        Sink o{S.stage, work + (c * 32 + t) * lane_slot};
        o.start();
        uint32_t w0 = 0, end = 0;                // values [w0, end) are in LDS
        for (uint32_t s = 0; s < nv;) {
            if (end < nv && s + kMaxLit > end) {
                wave_sync();
                w0 = s;
                end = min(nv - s, kVals) + s;
                load_values<EB>(S.val, in, in_bytes, c * chunk, chunk, ru, t, s, end);
                wave_sync();
            }
            const uint32_t have = min(nv - s, kMaxLit), at = s - w0 + l;
            Group g;
            g.a0 = S.val[at], g.a1 = S.val[at + 64];
            g.p0 = S.val[at ? at - 1 : 0], g.p1 = S.val[at + 63];
            g.take(have);
            const uint64_t e0 = __ballot(g.a0 == g.p0) & g.m0 & ~1ull, e1 = __ballot(g.a1 == g.p1) & g.m1;
            // values that end three equal ones inside the group
            const uint64_t t0 = e0 & (e0 << 1), t1 = e1 & (e1 << 1 | e0 >> 63);
            if (o.bits > 32 * (kStageWords - kGroupWords)) o.flush();
            if (t0 & 4) {
                const uint64_t x0 = ~e0 & ~1ull, x1 = ~e1;
                const uint32_t n = x0 ? (uint32_t)__builtin_ctzll(x0) : x1 ? 64 + (uint32_t)__builtin_ctzll(x1) : 128;
                const uint64_t v = lane_u64(g.a0, 0);
                if (n <= kMaxShortRepeat) {
                    short_repeat(o, v, n);
                } else if (n == kMaxLit && v == 0) {     // a full run takes the literals' rules
                    g.take(n);
                    direct(o, g, 0);
                } else {
                    fixed_delta(o, v, 0, n);
                }
                s += n;
            } else {
                const uint32_t n = t0 ? (uint32_t)__builtin_ctzll(t0) - 2 : t1 ? 62 + (uint32_t)__builtin_ctzll(t1) : have;
                g.take(n);
                literals(o, g);
                s += n;
            }
        }
        const uint64_t len = o.finish();
        if (l == 0) col_len[c * 32 + t] = len;
        wave_sync();
    }
}

// Short lane streams: a thread encodes one, value by value, its values in a
// column of LDS, half a wave per chunk.  No group of so few values is full.  A
// group costs a wave the same however few values it holds: 131072 chunks of 1
// 8-byte value a lane take 2700 us with a wave per stream and 107 us so, 8192
// chunks of 16 values 231 and 165 us (the benchmark's column; constant values
// 143 and 13 us).  A thread's time grows with its values and few chunks do not
// fill the chip, so the more values the more chunks it takes: 256 chunks of 16
// 8-byte values take 22 us a call with a wave per stream and 127 us so.  Three
// values take 11 us however few chunks there are, 14 us with a wave.  Beyond 16
// values the benchmark's column is slower with a thread (24: 300 against 165
// us), bytes beyond 32 (48: 273 against 174 us).
constexpr uint32_t kShortValues = 3, kShortOfMany = 16, kShortBytesOfMany = 32, kShortChunks = kWave / 32;
static_assert(kShortBytesOfMany < kMaxLit, "short streams fill no group");
inline bool short_lanes(uint64_t values, uint32_t eb, uint64_t n_chunks) {
    return values <= kShortValues ||
           (values <= (eb == 1 ? kShortBytesOfMany : kShortOfMany) && n_chunks >= 192 * values);
}

// One thread's lane stream: values val[0..nv), strided by a wave, and output.
template <class LT>
struct ShortLane {
    const LT* val;
    WordOut o;
    uint32_t cur = 0, fill = 0;                  // bits of the byte being packed

    MDZ_DEV uint64_t at(uint32_t i) const { return val[i * kWave]; }
    MDZ_DEV void byte(uint64_t v) { o.put((uint32_t)v & 0xFFu); }
    // The low w bits of v, most significant first.
    MDZ_DEV void field(uint64_t v, uint32_t w) {
        while (w) {
            const uint32_t take = min(w, 8 - fill);
            w -= take;
            cur = cur << take | ((uint32_t)(v >> w) & ((1u << take) - 1u));
            if ((fill += take) == 8) pad();
        }
    }
    MDZ_DEV void pad() {
        if (fill) byte(cur << (8 - fill));
        cur = 0;
        fill = 0;
    }
    MDZ_DEV void bytes(uint64_t v, uint32_t count) {
        while (count) byte(v >> (8 * --count));
    }
    MDZ_DEV void varint(uint64_t v) {
        for (; v > 0x7F; v >>= 7) byte((v & 0x7F) | 0x80);
        byte(v);
    }
    // header, first value and zigzag step of a delta group
    MDZ_DEV void delta_head(uint32_t code, uint64_t first, uint64_t step, uint32_t n) {
        bytes(header(0xC0, code, n), 2);
        varint(first);
        varint((step << 1) ^ (uint64_t)((int64_t)step >> 63));
    }
    MDZ_DEV void run(uint64_t v, uint32_t n) {
        if (n > kMaxShortRepeat) return delta_head(0, v, 0, n);
        const uint32_t vbytes = (value_width(v) - 1) / 8 + 1;
        byte(((vbytes - 1) << 3) | (n - kMinRepeat));
        bytes(v, vbytes);
    }
    MDZ_DEV void direct(uint32_t s, uint32_t n, uint64_t all) {          // all: the values' bits
        const uint32_t w = aligned_width(value_width(all));
        bytes(header(0x40, width_code(w), n), 2);
        for (uint32_t i = 0; i < n; ++i) field(at(s + i), w);
        pad();
    }
    // How many of the offsets from base have a width code of at least c.
    MDZ_DEV uint32_t at_least(uint32_t s, uint32_t n, uint64_t base, uint32_t c) const {
        uint32_t k = 0;
        for (uint32_t i = 0; i < n; ++i) k += width_code(bit_length(at(s + i) - base)) >= c ? 1u : 0u;
        return k;
    }
    MDZ_DEV void patched(uint32_t s, uint32_t n, uint64_t base, uint32_t b95, uint32_t b100) {
        uint32_t pw = fixed_width(b100 - b95);
        if (pw == 64) {
            pw = 56;
            b95 = 8;
        }
        const uint64_t mask = (1ull << b95) - 1;
        uint32_t np = 0, prev = 0, max_gap = 0;
        for (uint32_t i = 0; i < n; ++i) {
            if (at(s + i) - base > mask) {
                max_gap = max(max_gap, i - prev);
                prev = i;
                ++np;
            }
        }
        const uint32_t pgw = value_width(max_gap), vbytes = value_width(base) / 8 + 1;
        bytes(header(0x80, width_code(b95), n), 2);
        bytes((((vbytes - 1) << 5) | width_code(pw)) << 8 | ((((pgw - 1) << 5) | np) & 0xFF), 2);
        if (vbytes > 8) byte(0);
        bytes(base, min(vbytes, 8u));
        for (uint32_t i = 0; i < n; ++i) field((at(s + i) - base) & mask, fixed_width(b95));
        pad();
        prev = 0;
        for (uint32_t i = 0; i < n; ++i) {
            const uint64_t r = at(s + i) - base;
            if (r > mask) {
                field((uint64_t)(i - prev) << pw | r >> b95, fixed_width(pgw + pw));
                prev = i;
            }
        }
        pad();
    }
    // The rules of literals() above for values [s, s + n).
    MDZ_DEV void literals(uint32_t s, uint32_t n) {
        const uint64_t first = at(s), step = n > 1 ? at(s + 1) - first : 0;
        uint64_t all = first, low = first, high = first, steps = 0, p = first;
        bool even = true, up = true, down = true;
        for (uint32_t i = 1; i < n; ++i) {
            const uint64_t v = at(s + i);
            all |= v;
            low = min(low, v);
            high = max(high, v);
            steps |= v - p;
            even = even && v - p == step;
            up = up && p <= v;
            down = down && p >= v;
            p = v;
        }
        if (n <= kMinRepeat || (low == 0 && high <= 128)) return direct(s, n, all);
        if (even) return delta_head(0, first, step, n);
        if (step && (up || down)) {
            const uint32_t w = max(2u, aligned_width(value_width(steps)));
            delta_head(width_code(w), first, step, n);
            for (uint32_t i = 2; i < n; ++i) field(at(s + i) - at(s + i - 1), w);
            return pad();
        }
        const uint32_t code = width_code(bit_length(all)), near = code < 24 ? max(code, 1u) - 1 : code;
        if (at_least(s, n, 0, near) <= (n * 10 - 1) / 100 + 1) {
            const uint32_t c100 = width_code(bit_length(high - low)), above = (n * 5 - 1) / 100 + 1;
            if (at_least(s, n, low, c100) <= above) {
                uint32_t c95 = 0;
                for (uint32_t bit = 16; bit; bit >>= 1)
                    if (at_least(s, n, low, c95 | bit) > above) c95 |= bit;
                return patched(s, n, low, code_width(c95), code_width(c100));
            }
        }
        direct(s, n, all);
    }
    MDZ_DEV uint32_t encode(uint32_t nv) {       // the stream's bytes
        for (uint32_t s = 0; s < nv;) {
            const uint64_t v = at(s);
            uint32_t n = 1;
            while (s + n < nv && at(s + n) == v) ++n;
            if (n >= kMinRepeat) {
                run(v, n);
            } else {                             // up to the first three equal values in a row
                uint32_t same = n;
                uint64_t p = v;
                for (; s + n < nv && same < kMinRepeat; ++n) {
                    const uint64_t x = at(s + n);
                    same = x == p ? same + 1 : 1;
                    p = x;
                }
                if (same == kMinRepeat) n -= kMinRepeat;
                literals(s, n);
            }
            s += n;
        }
        return o.finish();
    }
};

template <int EB>
__global__ __launch_bounds__(kWave) void rlev2_short_kernel(const uint8_t* __restrict__ in, uint64_t in_bytes,
                                                            uint64_t n_chunks, uint64_t chunk, uint32_t ru,
                                                            uint64_t lane_slot, uint8_t* __restrict__ work,
                                                            uint64_t* __restrict__ col_len,
                                                            uint64_t* __restrict__ chunk_len) {
    typedef typename std::conditional<EB == 8, uint64_t, uint32_t>::type LT;
    extern __shared__ __align__(8) uint8_t short_vals[];         // nv values per thread
    LT* val = reinterpret_cast<LT*>(short_vals);
    const uint32_t l = lane_id(), t = l % 32, nv = (uint32_t)(chunk / EB / 32);
    const uint64_t c = (uint64_t)blockIdx.x * kShortChunks + l / 32;
    uint32_t len = 0;
    if (c < n_chunks) {
        for (uint32_t q = 0, line = 0, at = 0; q < nv; ++q) {
            val[q * kWave + l] = (LT)chunk_value(in, in_bytes, c * chunk, ((uint64_t)line * 32 + t) * ru + at, EB);
            if (++at == ru) at = 0, ++line;
        }
        ShortLane<LT> e{val + l, WordOut{work + (c * 32 + t) * lane_slot}};
        len = e.encode(nv);
        col_len[c * 32 + t] = len;
    }
    store_chunk_len((len + 3) / 4, c, n_chunks, chunk_len);
}

uint64_t v2_lane_slot(uint64_t chunk, uint32_t eb) {
    return (chunk / eb / 32 * 10 + 64 + 15) & ~15ull;
}

}  // namespace

int rlev2_compress_bound(uint64_t in_bytes, uint64_t chunk, uint32_t eb, uint32_t ru, uint64_t* n_chunks,
                         uint64_t* work_bytes, uint64_t* payload_cap) {
    if (!(eb == 1 || eb == 2 || eb == 4 || eb == 8) || ru == 0 || chunk == 0 || chunk % (32ull * eb) ||
        (chunk / eb / 32) % ru || in_bytes == 0 || chunk > (1ull << 32))
        return MDZ_ERR_INVALID;
    const uint64_t n = (in_bytes + chunk - 1) / chunk;
    const uint64_t slot = v2_lane_slot(chunk, eb);
    if (n_chunks) *n_chunks = n;
    if (work_bytes) *work_bytes = n * 32 * slot + 8 * n;
    if (payload_cap) *payload_cap = n * ((32 * slot + 127) / 128 * 128);
    return MDZ_OK;
}

int rlev2_compress(const void* in, uint64_t in_bytes, uint64_t chunk, uint32_t eb, uint32_t ru, void* work,
                   void* payload, uint64_t* col_len, uint64_t* blk_off, uint64_t* payload_bytes, hipStream_t s) {
    uint64_t n = 0;
    int rc = rlev2_compress_bound(in_bytes, chunk, eb, ru, &n, nullptr, nullptr);
    if (rc) return rc;
    if (!in || !work || !payload || !col_len || !blk_off || n > kMaxEncodeChunks) return MDZ_ERR_INVALID;
    const uint64_t slot = v2_lane_slot(chunk, eb);
    uint64_t* chunk_len = reinterpret_cast<uint64_t*>(static_cast<uint8_t*>(work) + n * 32 * slot);
    hipError_t e;
    if (short_lanes(chunk / eb / 32, eb, n)) {
        auto encode = eb == 1 ? rlev2_short_kernel<1> : eb == 2 ? rlev2_short_kernel<2>
                    : eb == 4 ? rlev2_short_kernel<4> : rlev2_short_kernel<8>;
        hipLaunchKernelGGL(encode, dim3((uint32_t)((n + kShortChunks - 1) / kShortChunks)), dim3(kWave),
                           chunk / eb / 32 * kWave * (eb == 8 ? 8 : 4), s, static_cast<const uint8_t*>(in), in_bytes, n,
                           chunk, ru, slot, static_cast<uint8_t*>(work), col_len, chunk_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "rlev2_short_kernel launch");
    } else {
        auto encode = eb == 1 ? rlev2_encode_kernel<1> : eb == 2 ? rlev2_encode_kernel<2>
                    : eb == 4 ? rlev2_encode_kernel<4> : rlev2_encode_kernel<8>;
        hipLaunchKernelGGL(encode, lane_grid(n), dim3(kWave), 0, s, static_cast<const uint8_t*>(in), in_bytes, n, chunk,
                           ru, slot, static_cast<uint8_t*>(work), col_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "rlev2_encode_kernel launch");
        hipLaunchKernelGGL(lanes_size_kernel, dim3((uint32_t)((n + kSizeChunks - 1) / kSizeChunks)), dim3(kSizeThreads),
                           0, s, col_len, n, chunk_len);
        if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lanes_size_kernel launch");
    }
    // blk_off[n] holds the uncompressed size; the true payload end goes to *payload_bytes
    hipLaunchKernelGGL(lanes_scan_kernel, dim3(1), dim3(kScanThreads), 0, s, chunk_len, n, blk_off, payload_bytes,
                       in_bytes);
    if ((e = hipGetLastError()) != hipSuccess) return record_hip(e, "lanes_scan_kernel launch");
    hipLaunchKernelGGL(lanes_interleave_kernel, interleave_grid(n, slot), dim3(kIlvThreads), 0, s,
                       static_cast<const uint8_t*>(work), slot, col_len, blk_off, chunk_len, nullptr,
                       static_cast<uint8_t*>(payload));
    return record_hip(hipGetLastError(), "lanes_interleave_kernel launch");
}

}  // namespace mdz
