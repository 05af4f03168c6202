"""GPU RLE v2 encoder (rlev2::compress_gpu_transpose, include/rlev2/
encoder_trans.h:428-537): payload, col_len and blk_off equal the host
restatement of the reference encoder byte for byte, and decode back."""
import numpy as np
import pytest

from compression_amd import host

pytestmark = pytest.mark.gpu


def _inputs():
    rng = np.random.default_rng(41)
    return {
        "generator_u64": host.gen_rlev2_i64(600_000, 42),
        "random_u32": rng.integers(0, 1 << 32, 300_000, dtype=np.uint64).astype(np.uint32),
        "repeats_u16": np.repeat(rng.integers(0, 60000, 30_000), rng.integers(1, 40, 30_000))[:400_000].astype(np.uint16),
        "ramp_u64": np.cumsum(rng.integers(-50, 51, 200_000)).astype(np.uint64),
        "zeros_u8": np.zeros(300_000, np.uint8),
        "outliers_u64": np.where(rng.random(250_000) < 0.05, rng.integers(0, 1 << 60, 250_000, dtype=np.uint64),
                                 rng.integers(0, 300, 250_000).astype(np.uint64)),
    }


@pytest.mark.parametrize("chunk,ru", [(131072, 512), (131072, 4), (65536, 1), (32768, 16)])
def test_matches_host_encoder(gpu, chunk, ru):
    from compression_amd import rlev2
    from compression_amd._lib import DeviceBuffer
    for name, data in _inputs().items():
        eb = data.dtype.itemsize
        if (chunk // eb // 32) % ru:
            continue
        raw = data.view(np.uint8)
        n, wb, cap = rlev2.compress_bound(raw.size, chunk, eb, ru)
        src = DeviceBuffer.from_array(raw)
        work, pay, pb = DeviceBuffer(wb), DeviceBuffer(cap), DeviceBuffer(8)
        col, off = DeviceBuffer(256 * n), DeviceBuffer(8 * (n + 1))
        print(f"rlev2 encode {name} chunk={chunk} ru={ru} n={n}", flush=True)
        rlev2.compress(src, raw.size, chunk, eb, ru, work, pay, col, off, pb)
        ref = host.rlev2_encode(data, chunk, ru)
        assert np.array_equal(off.download(8 * (n + 1)).view(np.uint64), ref.blk_off), name
        assert np.array_equal(col.download(256 * n).view(np.uint64), ref.col_len), name
        nbytes = int(pb.download(8).view(np.uint64)[0])
        assert nbytes == ref.payload_bytes, name
        assert pay.download(nbytes).tobytes() == ref.payload[:nbytes].tobytes(), name


def test_roundtrip_through_decoder(gpu):
    from compression_amd import rlev2
    from compression_amd._lib import DeviceBuffer
    from compression_amd.lanes import DeviceLanes
    data = host.gen_rlev2_i64(2_000_000, 43)
    raw = data.view(np.uint8)
    n, wb, cap = rlev2.compress_bound(raw.size, 131072, 8, 512)
    src = DeviceBuffer.from_array(raw)
    work, pay, pb = DeviceBuffer(wb), DeviceBuffer(cap), DeviceBuffer(8)
    col, off = DeviceBuffer(256 * n), DeviceBuffer(8 * (n + 1))
    rlev2.compress(src, raw.size, 131072, 8, 512, work, pay, col, off, pb)
    nbytes = int(pb.download(8).view(np.uint64)[0])
    lanes = DeviceLanes(pay.download(nbytes), off.download(8 * (n + 1)).view(np.uint64),
                        col.download(256 * n).view(np.uint64), n, 131072, 8, 512)
    dst, st = DeviceBuffer(raw.size), DeviceBuffer(4 * n)
    rlev2.decompress(lanes, dst, raw.size, st)
    assert (st.download(4 * n).view(np.int32) == 0).all()
    assert dst.download(raw.size).tobytes() == raw.tobytes()


def _shapes(n, seed):
    """Columns that meet every sub-mode at its limits: runs around 3, 10 and
    128 values, sorted and wrapping deltas, narrow values with zeros, patches."""
    rng = np.random.default_rng(seed)
    k = rng.choice([1, 2, 3, 4, 9, 10, 11, 12, 126, 127, 128, 129, 130, 131, 255, 256, 257, 300], n)
    v = rng.integers(0, 2**40, n).astype(np.uint64)
    v[::3] = 0
    steps = np.cumsum(rng.integers(0, 1000, n)).astype(np.uint64)
    seg, have = [], 0
    while have < n:
        m = int(rng.integers(1, 200))
        w = int(rng.integers(1, 63))
        s = rng.integers(0, 2**w, m)
        kind = rng.integers(0, 5)
        if kind == 0:
            s = s[0] // 2 + np.arange(m) * int(rng.integers(0, 100))
        elif kind == 1:
            s = np.where(rng.random(m) < 0.05, rng.integers(2**40, 2**62, m), s % 2**16)
        elif kind == 2:
            s = np.sort(s)[::int(rng.choice([1, -1]))]
        elif kind == 3:
            s = rng.integers(0, 2, m) * int(rng.integers(1, 300))
        seg.append(np.asarray(s, np.int64).view(np.uint64))
        have += m
    return {"runs": np.repeat(v, k)[:n], "up": steps, "down": np.uint64(1 << 62) - steps,
            "wrap": np.cumsum(rng.integers(0, 2**62, n).astype(np.uint64)), "zeros": np.zeros(n, np.uint64),
            "narrow": rng.integers(0, 130, n).astype(np.uint64), "mix": np.concatenate(seg)[:n]}


# lanes of 1 value to several LDS windows (512 values of 8 bytes, 1024 of less)
@pytest.mark.parametrize("dtype", [np.uint64, np.uint32, np.uint16, np.uint8])
@pytest.mark.parametrize("lane_values,ru", [(1, 1), (3, 3), (40, 4), (128, 16), (512, 512), (513, 27), (1300, 13),
                                            (4096, 64)])
def test_group_limits(gpu, dtype, lane_values, ru):
    from compression_amd import rlev2
    from compression_amd._lib import DeviceBuffer
    eb = np.dtype(dtype).itemsize
    chunk, nvals = 32 * lane_values * eb, min(32 * lane_values * 2 - 5, 200_000)
    for name, x in _shapes(max(nvals, 64), lane_values + eb).items():
        data = (x[:nvals] >> np.uint64(0 if eb == 8 else 5)).astype(dtype)
        raw = data.view(np.uint8)
        n, wb, cap = rlev2.compress_bound(raw.size, chunk, eb, ru)
        src, work, pay, pb = DeviceBuffer.from_array(raw), DeviceBuffer(wb), DeviceBuffer(cap), DeviceBuffer(8)
        col, off = DeviceBuffer(256 * n), DeviceBuffer(8 * (n + 1))
        print(f"rlev2 encode {name} {eb} bytes, {lane_values} lane values, ru={ru} n={n}", flush=True)
        rlev2.compress(src, raw.size, chunk, eb, ru, work, pay, col, off, pb)
        ref = host.rlev2_encode(data, chunk, ru)
        assert np.array_equal(off.download(8 * (n + 1)).view(np.uint64), ref.blk_off), name
        assert np.array_equal(col.download(256 * n).view(np.uint64), ref.col_len), name
        nbytes = int(pb.download(8).view(np.uint64)[0])
        assert nbytes == ref.payload_bytes, name
        assert pay.download(nbytes).tobytes() == ref.payload[:nbytes].tobytes(), name


# both forms of the encoder: a thread per lane stream up to 3 values, and up to
# 16 (bytes: 32) where there are 192 chunks or more per value; a wave beyond
@pytest.mark.parametrize("dtype", [np.uint64, np.uint32, np.uint16, np.uint8])
@pytest.mark.parametrize("lane_values,n_chunks", [(1, 5), (2, 5), (3, 5), (4, 767), (4, 769), (9, 1728), (16, 3071),
                                                  (16, 3073), (17, 3265), (32, 6145), (33, 6336)])
def test_short_lanes(gpu, dtype, lane_values, n_chunks):
    from compression_amd import rlev2
    from compression_amd._lib import DeviceBuffer
    eb = np.dtype(dtype).itemsize
    chunk, nvals = 32 * lane_values * eb, 32 * lane_values * n_chunks - 5
    rng = np.random.default_rng(lane_values + n_chunks + eb)
    m = nvals + 5
    kinds = dict(_shapes(m, lane_values + eb))
    kinds["outliers"] = np.where(rng.random(m) < 0.08, rng.integers(2**30, 2**64, m, dtype=np.uint64),
                                 rng.integers(1, 2**int(rng.integers(1, 20)), m).astype(np.uint64))
    kinds["repeats"] = np.repeat(rng.integers(0, 2**50, m), rng.integers(1, 14, m))[:m].astype(np.uint64)
    for name, x in kinds.items():
        # lane t's values are t, t + 32, ...: make neighbours of x one lane's
        x = x.reshape(n_chunks, 32, lane_values).swapaxes(1, 2).reshape(-1)[:nvals]
        data = (x >> np.uint64(0 if eb == 8 else 5)).astype(dtype)
        raw = data.view(np.uint8)
        n, wb, cap = rlev2.compress_bound(raw.size, chunk, eb, 1)
        src, work, pay, pb = DeviceBuffer.from_array(raw), DeviceBuffer(wb), DeviceBuffer(cap), DeviceBuffer(8)
        col, off = DeviceBuffer(256 * n), DeviceBuffer(8 * (n + 1))
        print(f"rlev2 encode {name} {eb} bytes, {lane_values} lane values n={n}", flush=True)
        rlev2.compress(src, raw.size, chunk, eb, 1, work, pay, col, off, pb)
        ref = host.rlev2_encode(data, chunk, 1)
        assert n == n_chunks and np.array_equal(off.download(8 * (n + 1)).view(np.uint64), ref.blk_off), name
        assert np.array_equal(col.download(256 * n).view(np.uint64), ref.col_len), name
        nbytes = int(pb.download(8).view(np.uint64)[0])
        assert nbytes == ref.payload_bytes, name
        assert pay.download(nbytes).tobytes() == ref.payload[:nbytes].tobytes(), name


def test_more_streams_than_workgroups(gpu):
    """The wave form strides over its lane streams beyond 2^24 workgroups
    (524,288 chunks): a period of 7 chunks, repeated, against the period's own
    encoding."""
    from compression_amd import rlev2
    from compression_amd._lib import DeviceBuffer
    lane_values, periods = 33, 524_288 // 7 + 2
    chunk = 32 * lane_values
    one = _shapes(7 * chunk, 19)["mix"].astype(np.uint8)
    data = np.tile(one, periods)
    n, wb, cap = rlev2.compress_bound(data.size, chunk, 1, 1)
    src, work, pay, pb = DeviceBuffer.from_array(data), DeviceBuffer(wb), DeviceBuffer(cap), DeviceBuffer(8)
    col, off = DeviceBuffer(256 * n), DeviceBuffer(8 * (n + 1))
    print(f"rlev2 encode {n} chunks", flush=True)
    rlev2.compress(src, data.size, chunk, 1, 1, work, pay, col, off, pb)
    ref = host.rlev2_encode(one, chunk, 1)
    got, size = off.download(8 * (n + 1)).view(np.uint64), int(ref.payload_bytes)
    assert n == 7 * periods > 524_288 and got[-1] == data.size
    assert int(pb.download(8).view(np.uint64)[0]) == size * periods
    assert np.array_equal(got[:-1].reshape(periods, 7),
                          ref.blk_off[:7] + np.uint64(size) * np.arange(periods, dtype=np.uint64)[:, None])
    assert (col.download(256 * n).view(np.uint64).reshape(periods, -1) == ref.col_len).all()
    assert (pay.download(size * periods).reshape(periods, -1) == ref.payload[:size]).all()


# inputs that start between elements, in both forms (3 and 130 lane values)
@pytest.mark.parametrize("dtype,skip", [(np.uint16, 1), (np.uint32, 1), (np.uint32, 2), (np.uint64, 3), (np.uint64, 4)])
@pytest.mark.parametrize("lane_values", [3, 130])
def test_unaligned_input(gpu, dtype, skip, lane_values):
    from compression_amd import rlev2
    from compression_amd._lib import DeviceBuffer
    eb = np.dtype(dtype).itemsize
    chunk = 32 * lane_values * eb
    raw = _shapes(32 * lane_values * 7, lane_values)["mix"].astype(dtype).view(np.uint8)
    data = np.frombuffer(raw[skip:skip + (raw.size - skip) // eb * eb].tobytes(), dtype)
    n, wb, cap = rlev2.compress_bound(data.nbytes, chunk, eb, 1)
    src, work, pay, pb = DeviceBuffer.from_array(raw), DeviceBuffer(wb), DeviceBuffer(cap), DeviceBuffer(8)
    col, off = DeviceBuffer(256 * n), DeviceBuffer(8 * (n + 1))
    print(f"rlev2 encode unaligned {eb} bytes skip {skip}", flush=True)
    rlev2.compress(src.ptr + skip, data.nbytes, chunk, eb, 1, work, pay, col, off, pb)
    ref = host.rlev2_encode(data, chunk, 1)
    assert np.array_equal(off.download(8 * (n + 1)).view(np.uint64), ref.blk_off)
    assert np.array_equal(col.download(256 * n).view(np.uint64), ref.col_len)
    nbytes = int(pb.download(8).view(np.uint64)[0])
    assert nbytes == ref.payload_bytes and pay.download(nbytes).tobytes() == ref.payload[:nbytes].tobytes()
