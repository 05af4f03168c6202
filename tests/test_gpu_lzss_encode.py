"""GPU LZSS encoder (lzss::compress_gpu, include/lzss/lzss_gpu2.h:1952-2123):
payload, sorted col_len, col_map and blk_off equal the host restatement of
the reference encoder byte for byte, and decode back."""
import numpy as np
import pytest

from compression_amd import host

pytestmark = pytest.mark.gpu


def _inputs():
    rng = np.random.default_rng(51)
    return {
        "markov": host.gen_lzss_markov(3_000_000, 52),
        "random": rng.integers(0, 256, 1_000_000).astype(np.uint8),
        "low_alphabet": rng.integers(0, 3, 1_000_000).astype(np.uint8),
        "periodic": (np.arange(1_500_000) // 7 % 256).astype(np.uint8),
        "zeros": np.zeros(700_000, np.uint8),
    }


@pytest.mark.parametrize("chunk", [131072, 65536, 4096])
def test_matches_host_encoder(gpu, chunk):
    from compression_amd import lzss
    from compression_amd._lib import DeviceBuffer
    for name, data in _inputs().items():
        n, wb, cap = lzss.compress_bound(data.size, chunk)
        src = DeviceBuffer.from_array(data)
        work, pay = DeviceBuffer(wb), DeviceBuffer(cap)
        col, cmap, off = DeviceBuffer(256 * n), DeviceBuffer(32 * n), DeviceBuffer(8 * (n + 1))
        print(f"lzss encode {name} chunk={chunk} n={n}", flush=True)
        lzss.compress(src, data.size, chunk, work, pay, col, cmap, off)
        ref = host.lzss_encode(data, chunk)
        got_off = off.download(8 * (n + 1)).view(np.uint64)
        assert np.array_equal(got_off, ref.blk_off), name
        assert np.array_equal(col.download(256 * n).view(np.uint64), ref.col_len), name
        assert np.array_equal(cmap.download(32 * n), ref.col_map), name
        assert pay.download(int(got_off[-1])).tobytes() == ref.payload[:int(got_off[-1])].tobytes(), name


def test_host_form_roundtrip(gpu):
    from compression_amd import lzss
    data = host.gen_lzss_markov(5 * 131072 + 1000, 53)
    payload, blobs = lzss.compress_gpu(data.tobytes())
    ref = host.lzss_encode(data, 131072)
    assert payload == ref.payload[:int(ref.blk_off[-1])].tobytes()
    assert blobs[0] == np.uint64(131072).tobytes() and blobs[1] == ref.blk_off.tobytes()
    assert blobs[2] == ref.col_len.tobytes() and blobs[3] == ref.col_map.tobytes()
    assert lzss.decompress_gpu(payload, blobs) == data[:5 * 131072].tobytes()


# lane bytes at the edges of the encoder's LDS windows (1024, 2048, 4096
# positions), the windows that advance by 2048 above, and the smallest lanes
@pytest.mark.parametrize("lane_bytes", [4, 8, 40, 1024, 1028, 2044, 2048, 2052, 4096, 4100, 6144, 10240, 32768])
def test_window_edges(gpu, lane_bytes):
    from compression_amd import lzss
    from compression_amd._lib import DeviceBuffer
    chunk = 32 * lane_bytes
    size = max(3 * chunk, min(20 * chunk, 400_000))
    rng = np.random.default_rng(lane_bytes)
    far = np.zeros(size, np.uint8)                 # matches at the far end of the history
    far[:] = np.tile(rng.integers(0, 256, 2045 * 32), -(-size // (2045 * 32)))[:size]
    for name, data in {"markov": host.gen_lzss_markov(size, lane_bytes), "far": far,
                       "pairs": rng.integers(0, 2, size).astype(np.uint8),
                       "zeros": np.zeros(size, np.uint8)}.items():
        n, wb, cap = lzss.compress_bound(size, chunk)
        src, work, pay = DeviceBuffer.from_array(data), DeviceBuffer(wb), DeviceBuffer(cap)
        col, cmap, off = DeviceBuffer(256 * n), DeviceBuffer(32 * n), DeviceBuffer(8 * (n + 1))
        print(f"lzss encode {name} lane_bytes={lane_bytes} n={n}", flush=True)
        lzss.compress(src, size, chunk, work, pay, col, cmap, off)
        ref = host.lzss_encode(data, chunk)
        assert np.array_equal(off.download(8 * (n + 1)).view(np.uint64), ref.blk_off), name
        assert np.array_equal(col.download(256 * n).view(np.uint64), ref.col_len), name
        assert np.array_equal(cmap.download(32 * n), ref.col_map), name
        assert pay.download(int(ref.blk_off[-1])).tobytes() == ref.payload[:int(ref.blk_off[-1])].tobytes(), name


# both forms of the encoder: a thread per lane stream up to 8 bytes, and up to
# 64 where there are at least 2 * bytes * bytes chunks; a wave per stream beyond
@pytest.mark.parametrize("lane_bytes,n_chunks", [(4, 3), (8, 7), (12, 7), (12, 287), (12, 288), (32, 2047), (32, 2049),
                                                 (64, 8191), (64, 8193), (68, 9248)])
def test_short_lanes(gpu, lane_bytes, n_chunks):
    from compression_amd import lzss
    from compression_amd._lib import DeviceBuffer
    chunk = 32 * lane_bytes
    size = n_chunks * chunk
    rng = np.random.default_rng(lane_bytes + n_chunks)
    kinds = {"markov": host.gen_lzss_markov(size, lane_bytes), "pairs": rng.integers(0, 2, size).astype(np.uint8),
             "mixed": np.where(rng.random(size) < 0.1, rng.integers(0, 256, size), 7).astype(np.uint8),
             "random": rng.integers(0, 256, size).astype(np.uint8), "zeros": np.zeros(size, np.uint8)}
    for name, data in kinds.items():
        n, wb, cap = lzss.compress_bound(size, chunk)
        src, work, pay = DeviceBuffer.from_array(data), DeviceBuffer(wb), DeviceBuffer(cap)
        col, cmap, off = DeviceBuffer(256 * n), DeviceBuffer(32 * n), DeviceBuffer(8 * (n + 1))
        print(f"lzss encode {name} lane_bytes={lane_bytes} n={n}", flush=True)
        lzss.compress(src, size, chunk, work, pay, col, cmap, off)
        ref = host.lzss_encode(data, chunk)
        assert np.array_equal(off.download(8 * (n + 1)).view(np.uint64), ref.blk_off), name
        assert np.array_equal(col.download(256 * n).view(np.uint64), ref.col_len), name
        assert np.array_equal(cmap.download(32 * n), ref.col_map), name
        assert pay.download(int(ref.blk_off[-1])).tobytes() == ref.payload[:int(ref.blk_off[-1])].tobytes(), name


def test_more_streams_than_workgroups(gpu):
    """The wave form strides over its lane streams beyond 2^24 workgroups
    (524,288 chunks): a period of 7 chunks, repeated, against the period's own
    encoding."""
    from compression_amd import lzss
    from compression_amd._lib import DeviceBuffer
    chunk, periods = 32 * 68, 524_288 // 7 + 2
    one = host.gen_lzss_markov(7 * chunk, 23)
    data = np.tile(one, periods)
    n, wb, cap = lzss.compress_bound(data.size, chunk)
    src, work, pay = DeviceBuffer.from_array(data), DeviceBuffer(wb), DeviceBuffer(cap)
    col, cmap, off = DeviceBuffer(256 * n), DeviceBuffer(32 * n), DeviceBuffer(8 * (n + 1))
    print(f"lzss encode {n} chunks", flush=True)
    lzss.compress(src, data.size, chunk, work, pay, col, cmap, off)
    ref = host.lzss_encode(one, chunk)
    got, size = off.download(8 * (n + 1)).view(np.uint64), int(ref.blk_off[7])
    assert n == 7 * periods > 524_288
    assert np.array_equal(got[:-1].reshape(periods, 7),
                          ref.blk_off[:7] + np.uint64(size) * np.arange(periods, dtype=np.uint64)[:, None])
    assert (col.download(256 * n).view(np.uint64).reshape(periods, -1) == ref.col_len).all()
    assert (cmap.download(32 * n).reshape(periods, -1) == ref.col_map).all()
    assert (pay.download(size * periods).reshape(periods, -1) == ref.payload[:size]).all()
