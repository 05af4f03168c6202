"""The byte RLE encoder's choice of dword loads (compression_amd/csrc/
brle_load.h), compiled for the host: at every thread of a chunk's first and
last windows the loads that the rule allows stay inside the chunk, and where
they do it allows them.  Chunks may be up to 0xFFFFFFF0 bytes long."""
import ctypes
import subprocess

import pytest

from compression_amd import build

PER = 32
SOURCE = r"""
#include "brle_load.h"
// Loads outside the chunk that the rule allows, plus refused ones a dword or more inside it.
extern "C" uint64_t wrong(uint32_t win, uint32_t len, uint32_t skew) {
    const uint32_t last = (len - 1) / win * win, starts[3] = {0, last >= win ? last - win : 0, last};
    uint64_t bad = 0;
    for (uint32_t w0 : starts)
        for (uint32_t at = 0; at < win; at += mdz::kBrlePer) {
            const int64_t first = (int64_t)w0 + at - skew, end = first + mdz::kBrlePer + 4;
            const bool allowed = mdz::brle_whole_dwords(w0, at, len, skew);
            bad += allowed ? first < 0 || end > (int64_t)len : first >= 0 && end + 4 <= (int64_t)len;
        }
    return bad;
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("brle_load")
    (d / "rule.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{build.CSRC}", "-o", str(d / "rule.so"),
                    str(d / "rule.cpp")], check=True)
    fn = ctypes.CDLL(str(d / "rule.so")).wrong
    fn.argtypes, fn.restype = [ctypes.c_uint32] * 3, ctypes.c_uint64
    return fn


# windows of 1, 4 and 16 waves; chunks of more than 8 KiB take the widest alone
@pytest.mark.parametrize("win,lens", [
    (64 * PER, (1, 31, 35, 36, 37, 2047, 2048)),
    (256 * PER, (2049, 4095, 8191, 8192)),
    (1024 * PER, (8193, 32767, 32768, 32769, 65541, 262144, 1 << 31, 0xFFFF0001, 0xFFFF7FFF, 0xFFFF8000, 0xFFFF8001,
                  0xFFFF8024, 0xFFFFF000, 0xFFFFF001, 0xFFFFFFDB, 0xFFFFFFE0, 0xFFFFFFE4, 0xFFFFFFEF, 0xFFFFFFF0))])
@pytest.mark.parametrize("skew", [0, 1, 2, 3])
def test_dword_loads_stay_inside(rule, win, lens, skew):
    assert [n for n in lens if rule(win, n, skew)] == []
