"""The work that users of the mdz library have it do, as timed cases.

A case is one call (or one launch) of a public entry point on inputs from the
library's own seeded generators: decode and encode of every codec, resident
in HBM and through the host entries, from one request of a few chunks to the
largest columns that the library's benchmark decodes.  All outputs are whole
bytes and integers, so every implementation has to give the same ones.

    listed()          the named cases
    draw(rng)         one more case of the same ranges
    prepare(case, s)  inputs and buffers of a case, on the GPU (seed s)
    run(state)        one pass; returns its outputs
    work(case)        bytes the pass cannot do without
    tolerance(case)   "exact" throughout
    exact(case, s)    None: no output is a rounded number
"""
from __future__ import annotations

import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from compression_amd import batch, brle, deflate, host, lzss, rle_v1, rlev2, sched
from compression_amd.lanes import DeviceLanes

KIB, MIB = 1 << 10, 1 << 20

# Per kind of call: smallest and largest raw size, and the share of the raw
# size that the generator's data encodes to (sizes the necessary traffic).
KINDS = {
    "rlev1_decode":      (16 * KIB, 64 * MIB, 0.53),
    "rlev1_host":        (16 * KIB, 16 * MIB, 0.53),
    "rlev1_encode":      (16 * KIB, 64 * MIB, 0.53),
    "rlev2_decode":      (16 * KIB, 256 * MIB, 0.32),
    "rlev2_encode":      (16 * KIB, 256 * MIB, 0.32),
    "rlev2_plain":       (16 * KIB, 256 * MIB, 0.31),
    "brle_decode":       (16 * KIB, 256 * MIB, 0.24),
    "brle_encode":       (16 * KIB, 64 * MIB, 0.24),
    "brle_trans_decode": (64 * KIB, 64 * MIB, 0.62),
    "batch_decode":      (1 * MIB, 1280 * MIB, 0.30),
    "lzss_decode":       (64 * KIB, 256 * MIB, 0.73),
    "lzss_plain":        (64 * KIB, 256 * MIB, 0.11),
    "lzss_encode":       (64 * KIB, 64 * MIB, 0.73),
    "inflate":           (16 * KIB, 1200 * MIB, 0.13),
}


def _case(kind, raw, chunk, elem=1, line=0, **more):
    """known: the caller passes the largest chunk's encoded size, as one that
    made the container itself can (RLE v1, RLE v2 and batched decode)."""
    return dict(kind=kind, bytes=raw, chunk=chunk, elem=elem, line=line, **more)


def listed():
    """Twelve cases; the sizes are the benchmark's own where it has the call."""
    named = {
        # a column of 32-bit keys, resident in HBM: the benchmark's 64 MiB RLE v1 decode
        "rlev1_decode_64MiB": _case("rlev1_decode", 64 * MIB, 128 * KIB, 4, 128, known=True),
        # the drop-in call of a program that holds a container file in host memory
        "rlev1_host_16MiB": _case("rlev1_host", 16 * MIB, 128 * KIB, 4, 32),
        # one request of three chunks, the last one cut short: latency
        "rlev2_decode_3_chunks": _case("rlev2_decode", 300_008, 128 * KIB, 8, 64, known=False),
        # two column types of a table in one persistent launch: the benchmark's
        # 1 GiB of 64-bit values (RLE v2) beside 256 MiB of bytes (byte RLE)
        "batch_decode_1280MiB": _case("batch_decode", 1280 * MIB, 128 * KIB, 8, 512, known=True),
        # ORC-like run streams, one per 32 KiB chunk
        "rlev2_plain_256MiB": _case("rlev2_plain", 256 * MIB, 32 * KIB, 8),
        # text with back-references, 64 KiB chunks, lane-transposed
        "lzss_decode_256MiB": _case("lzss_decode", 256 * MIB, 64 * KIB),
        # the same text, one stream per chunk
        "lzss_plain_256MiB": _case("lzss_plain", 256 * MIB, 64 * KIB),
        # zlib streams of 4 KiB to 4 MiB, 80 % dynamic, 10 % fixed, 10 % stored,
        # ordered by compressed size for the persistent launch
        "inflate_2048_streams": _case("inflate", 1200 * MIB, 4 * MIB, count=2048, sched=True, verify=False),
        # encode of each codec, resident in HBM: a table being written
        "rlev1_encode_64MiB": _case("rlev1_encode", 64 * MIB, 128 * KIB, 4, 128),
        "rlev2_encode_256MiB": _case("rlev2_encode", 256 * MIB, 128 * KIB, 8, 512),
        "brle_encode_64MiB": _case("brle_encode", 64 * MIB, 256 * KIB),
        "lzss_encode_64MiB": _case("lzss_encode", 64 * MIB, 64 * KIB),
    }
    return [dict(c, name=n) for n, c in named.items()]


def draw(rng):
    """A kind at random; sizes spread over the logarithm of its range, whole
    multiples of the element but seldom of the chunk."""
    kind = rng.choice(sorted(KINDS))
    lo, hi, _ = KINDS[kind]
    raw = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    if kind in ("rlev1_decode", "rlev1_host", "rlev1_encode"):
        elem = rng.choice((1, 2, 4, 8))
        line = rng.choice((32, 128, 512))
        chunk = rng.choice((16, 64, 128)) * KIB
        known = {"known": rng.random() < 0.5} if kind == "rlev1_decode" else {}
        return _case(kind, max(elem, raw // elem * elem), chunk, elem, line, **known)
    if kind in ("rlev2_decode", "rlev2_encode"):
        elem = rng.choice((1, 2, 4, 8))
        line = rng.choice((16, 64, 512))
        # whole READ_UNIT lines of 32 lanes
        chunk = max(32 * line * elem, rng.choice((32, 128)) * KIB)
        known = {"known": rng.random() < 0.5} if kind == "rlev2_decode" else {}
        return _case(kind, max(elem, raw // elem * elem), chunk, elem, line, **known)
    if kind == "rlev2_plain":
        return _case(kind, raw // 8 * 8, rng.choice((4, 8, 32, 128)) * KIB, 8)
    if kind in ("brle_decode", "brle_encode"):
        return _case(kind, raw, rng.choice((32, 128, 256) if kind == "brle_encode" else (32, 128)) * KIB)
    if kind == "batch_decode":
        return _case(kind, raw // 8 * 8, 128 * KIB, 8, rng.choice((64, 512)),
                     known=rng.random() < 0.5)
    if kind in ("lzss_decode", "lzss_encode", "brle_trans_decode"):
        # these formats hold whole chunks; an encoder's time grows with the chunk
        chunk = rng.choice((32, 64) if kind == "lzss_encode" else (32, 64, 128)) * KIB
        return _case(kind, max(1, raw // chunk) * chunk, chunk)
    if kind == "lzss_plain":
        return _case(kind, raw, rng.choice((32, 64, 128)) * KIB)
    top = rng.choice((64 * KIB, 512 * KIB, 4 * MIB))  # inflate
    count = int(math.exp(rng.uniform(0.0, math.log(2048))))
    mean = (top - 4 * KIB) / math.log(top / (4 * KIB))
    return _case(kind, int(count * mean), top, count=count, sched=rng.random() < 0.5, verify=rng.random() < 0.5)


# ----------------------------------------------------------------- inputs --

def _threads(fn, n, piece, dtype, seed):
    """n values of generator fn, made piece by piece (each piece has a seed of
    its own) on the host's cores."""
    out = np.empty(n, dtype)

    def fill(k):
        part = fn(min(piece, n - k * piece), seed * 1_000_003 + k)
        out[k * piece:k * piece + part.size] = part

    with ThreadPoolExecutor(host.default_threads()) as ex:
        list(ex.map(fill, range((n + piece - 1) // piece)))
    return out


def _ints_v1(raw, elem, seed):
    x = _threads(host.gen_rlev1_u32, raw // elem, 1 << 20, np.uint32, seed)
    return x if elem == 4 else x.astype({1: np.uint8, 2: np.uint16, 8: np.uint64}[elem])


def _ints_v2(raw, elem, seed):
    x = _threads(host.gen_rlev2_i64, raw // elem, 1 << 20, np.uint64, seed)
    return x if elem == 8 else x.astype({1: np.uint8, 2: np.uint16, 4: np.uint32}[elem])


def _runs(raw, seed):
    return _threads(host.gen_brle_u8, raw, 4 * MIB, np.uint8, seed)


def _text(raw, seed):
    return _threads(host.gen_lzss_markov, raw, 8 * MIB, np.uint8, seed)


def _dev(a, pad=0):
    t = torch.zeros(a.nbytes + pad, dtype=torch.uint8, device="cuda")
    t[:a.nbytes].copy_(torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)))
    return t


def _out(n):
    return torch.zeros(max(int(n), 1), dtype=torch.uint8, device="cuda")


def _words(n, dtype=torch.int64):
    return torch.zeros(max(int(n), 1), dtype=dtype, device="cuda")


class _Tensor:
    """A DeviceBuffer's memory for torch (kept alive by the tensor made from it)."""

    def __init__(self, buf, nbytes):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (int(nbytes),), "typestr": "|u1", "data": (buf.ptr, False),
                                         "version": 2}

    def tensor(self):
        return torch.as_tensor(self, device="cuda")


# ------------------------------------------------------------------ calls --

def _lanes(c, chunk, elem=1, line=4, col_map=None):
    return DeviceLanes(c.payload, c.blk_off, c.col_len, c.n_chunks, chunk, elem, line, col_map=col_map)


def _largest(case, blk_off, payload_bytes):
    """Largest chunk's encoded bytes, or 0 where the caller does not say."""
    off = np.append(blk_off[:-1], np.uint64(payload_bytes))
    return int(np.diff(off).max()) if case["known"] else 0


def _rlev1_decode(case, seed):
    c = host.rlev1_encode(_ints_v1(case["bytes"], case["elem"], seed), case["chunk"], case["line"])
    lanes = _lanes(c, case["chunk"], case["elem"], case["line"])
    dst, st = _out(c.raw_bytes), _words(c.n_chunks, torch.int32)

    most = _largest(case, c.blk_off, c.payload.size)

    def call():
        rle_v1.decompress(lanes, dst.data_ptr(), c.raw_bytes, st.data_ptr(), max_chunk_bytes=most)
        return dst, st
    return call


def _rlev1_host(case, seed):
    c = host.rlev1_encode(_ints_v1(case["bytes"], case["elem"], seed), case["chunk"], case["line"])
    blob = np.uint64(c.raw_bytes).tobytes() + c.payload.tobytes()

    def call():
        return np.frombuffer(rle_v1.decompress_gpu(blob, case["line"], case["chunk"], case["elem"], c.col_len,
                                                   c.blk_off), np.uint8)
    return call


def _rlev1_encode(case, seed):
    raw = case["bytes"]
    n, wb, cap = rle_v1.compress_bound(raw, case["chunk"], case["elem"], case["line"])
    src, work, pay = _dev(_ints_v1(raw, case["elem"], seed)), _out(wb), _out(cap)
    col, off = _words(32 * n), _words(n + 1)

    def call():
        rle_v1.compress(src.data_ptr(), raw, case["chunk"], case["elem"], case["line"], work.data_ptr(),
                        pay.data_ptr(), col.data_ptr(), off.data_ptr())
        return pay, col, off
    call.keep = work
    return call


def _rlev2_decode(case, seed):
    c = host.rlev2_encode(_ints_v2(case["bytes"], case["elem"], seed), case["chunk"], case["line"])
    lanes = _lanes(c, case["chunk"], case["elem"], case["line"])
    dst, st = _out(c.raw_bytes), _words(c.n_chunks, torch.int32)

    most = _largest(case, c.blk_off, c.payload_bytes)

    def call():
        rlev2.decompress(lanes, dst.data_ptr(), c.raw_bytes, st.data_ptr(), max_chunk_bytes=most)
        return dst, st
    return call


def _rlev2_encode(case, seed):
    raw = case["bytes"]
    n, wb, cap = rlev2.compress_bound(raw, case["chunk"], case["elem"], case["line"])
    src, work, pay = _dev(_ints_v2(raw, case["elem"], seed)), _out(wb), _out(cap)
    col, off, pb = _words(32 * n), _words(n + 1), _words(1)

    def call():
        rlev2.compress(src.data_ptr(), raw, case["chunk"], case["elem"], case["line"], work.data_ptr(),
                       pay.data_ptr(), col.data_ptr(), off.data_ptr(), pb.data_ptr())
        return pay, col, off, pb
    call.keep = work
    return call


def _rlev2_plain(case, seed):
    x = _ints_v2(case["bytes"], 8, seed) & np.uint64(0x7FFFFFFFFFFFFFFF)
    c = host.rlev2_plain_encode(x, case["chunk"])
    data, ptr = _dev(c.data, 16), _dev(c.ptr)
    dst, st = _out(c.raw_bytes), _words(c.n_chunks, torch.int32)

    def call():
        rlev2.decompress_plain(data.data_ptr(), c.data.size, ptr.data_ptr(), c.n_chunks, case["chunk"],
                               dst.data_ptr(), c.raw_bytes, st.data_ptr())
        return dst, st
    return call


def _brle_decode(case, seed):
    c = host.brle_encode(_runs(case["bytes"], seed), case["chunk"])
    b = brle.DeviceBrle(c.data, c.ptr, c.n_chunks, case["chunk"])
    dst, st = _out(c.raw_bytes), _words(c.n_chunks, torch.int32)

    def call():
        brle.decompress(b, dst.data_ptr(), c.raw_bytes, st.data_ptr())
        return dst, st
    return call


def _brle_encode(case, seed):
    raw = case["bytes"]
    n, wb, cap = brle.compress_bound(raw, case["chunk"])
    src, work, data, ptr = _dev(_runs(raw, seed)), _out(wb), _out(cap), _words(n + 1)

    def call():
        brle.compress(src.data_ptr(), raw, data.data_ptr(), ptr.data_ptr(), work.data_ptr(),
                      chunk_bytes=case["chunk"])
        return data, ptr
    call.keep = work
    return call


def _brle_trans_decode(case, seed):
    c = host.brle_trans_encode(_runs(case["bytes"], seed), case["chunk"])
    lanes = _lanes(c, case["chunk"], col_map=c.col_map)
    dst, st = _out(c.raw_bytes), _words(c.n_chunks, torch.int32)

    def call():
        brle.decompress_trans(lanes, dst.data_ptr(), c.raw_bytes, st.data_ptr())
        return dst, st
    return call


def _batch_decode(case, seed):
    ints = case["bytes"] // 5 * 4 // 8 * 8           # four fifths 64-bit values, one fifth bytes
    c2 = host.rlev2_encode(_ints_v2(ints, 8, seed), case["chunk"], case["line"])
    cb = host.brle_encode(_runs(case["bytes"] - ints, seed + 1), case["chunk"])
    lanes = _lanes(c2, case["chunk"], 8, case["line"])
    b = brle.DeviceBrle(cb.data, cb.ptr, cb.n_chunks, case["chunk"])
    d2, s2 = _out(c2.raw_bytes), _words(c2.n_chunks, torch.int32)
    d3, s3 = _out(cb.raw_bytes), _words(cb.n_chunks, torch.int32)
    job = batch.Batch(lanes, d2.data_ptr(), c2.raw_bytes, s2.data_ptr(), _largest(case, c2.blk_off, c2.payload_bytes), b, d3.data_ptr(), cb.raw_bytes,
                      s3.data_ptr())
    job.set_order(job.size_order())

    def call():
        job.submit()
        return d2, s2, d3, s3
    return call


def _lzss_decode(case, seed):
    c = host.lzss_encode(_text(case["bytes"], seed), case["chunk"])
    lanes = _lanes(c, case["chunk"], col_map=c.col_map)
    dst, st = _out(c.raw_bytes), _words(c.n_chunks, torch.int32)

    def call():
        lzss.decompress(lanes, dst.data_ptr(), c.raw_bytes, st.data_ptr())
        return dst, st
    return call


def _lzss_plain(case, seed):
    c = host.lzss_plain_encode(_text(case["bytes"], seed), case["chunk"])
    data, lens = _dev(c.data, 16), _dev(c.lens)
    dst, st = _out(c.raw_bytes), _words(c.n_chunks, torch.int32)

    def call():
        lzss.decompress_plain(data.data_ptr(), c.data.size, lens.data_ptr(), c.n_chunks, case["chunk"],
                              dst.data_ptr(), c.raw_bytes, st.data_ptr())
        return dst, st
    return call


def _lzss_encode(case, seed):
    raw = case["bytes"]
    n, wb, cap = lzss.compress_bound(raw, case["chunk"])
    src, work, pay = _dev(_text(raw, seed)), _out(wb), _out(cap)
    col, cmap, off = _words(32 * n), _out(32 * n), _words(n + 1)

    def call():
        lzss.compress(src.data_ptr(), raw, case["chunk"], work.data_ptr(), pay.data_ptr(), col.data_ptr(),
                      cmap.data_ptr(), off.data_ptr())
        return pay, col, cmap, off
    call.keep = work
    return call


def _inflate(case, seed):
    count, top = case["count"], case["chunk"]
    g = host.gen_deflate_batch(count, seed, 4 * KIB, top)
    # slots of each stream's size; the last one takes what is left of an
    # output whose size depends on the case alone
    caps = g.raw_len.copy()
    room = 16 * count + min(count * top, case["bytes"] + int(2 * top * math.sqrt(count)))
    caps[-1] = room - int(((caps[:-1] + np.uint64(15)) // np.uint64(16) * np.uint64(16)).sum())
    b = deflate.DeviceBatch(g.src, g.src_off, g.src_len, caps)
    b.dst.fill(0)                                     # the slots' alignment gaps are never written
    framing = deflate.HDR_ZLIB | (deflate.HDR_VERIFY if case["verify"] else 0)
    if case["sched"]:
        b.set_order(sched.lpt_order(g.src_len))
    dst = _Tensor(b.dst, b.dst.nbytes).tensor()
    st = _Tensor(b.status, b.count * deflate.STATUS.itemsize).tensor()

    def call():
        if case["sched"]:
            deflate.inflate_sched(b, framing)
        else:
            deflate.inflate(b, framing)
        return dst, st
    return call


_PREPARE = {
    "rlev1_decode": _rlev1_decode, "rlev1_host": _rlev1_host, "rlev1_encode": _rlev1_encode,
    "rlev2_decode": _rlev2_decode, "rlev2_encode": _rlev2_encode, "rlev2_plain": _rlev2_plain,
    "brle_decode": _brle_decode, "brle_encode": _brle_encode, "brle_trans_decode": _brle_trans_decode,
    "batch_decode": _batch_decode, "lzss_decode": _lzss_decode, "lzss_plain": _lzss_plain,
    "lzss_encode": _lzss_encode, "inflate": _inflate,
}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, int(seed))


def run(state):
    return state()


def work(case):
    """Compressed bytes once, raw bytes once, and the container's metadata."""
    raw = case["bytes"]
    meta = 48 * case["count"] if case["kind"] == "inflate" else 264 * max(1, raw // case["chunk"])
    return {"bytes": raw * (1.0 + KINDS[case["kind"]][2]) + meta, "flops": 0}


def tolerance(case):
    return "exact"


def exact(case, seed):
    return None
