"""`ojk_spread` (which tile a workgroup of the copied f16 tile takes), compiled for the host."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

KERNELS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ojas-engine_amd", "csrc", "kernels")
SOURCE = """#include "ojk_spread.h"
extern "C" void spread(unsigned gx, unsigned gy, unsigned rows, unsigned tokens, int *out) {
    for (unsigned y = 0; y < gy; y++)
        for (unsigned x = 0; x < gx; x++, out += 3) {
            unsigned r, t, s;
            if (ojk_spread(x & 7, y * (gx >> 3) + (x >> 3), rows, tokens, gy, r, t, s)) out[0] = (int)r, out[1] = (int)t, out[2] = (int)s;
            else out[0] = out[1] = out[2] = -1;
        }
}
"""


@pytest.fixture(scope="module")
def spread(tmp_path_factory):
    d = tmp_path_factory.mktemp("spread")
    (d / "s.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-shared", "-fPIC", "-O1", "-I", KERNELS, "-o", str(d / "s.so"), str(d / "s.cpp")])
    fn = ctypes.CDLL(str(d / "s.so")).spread

    def run(gx, gy, rows, tokens):
        out = np.empty((gy * gx, 3), np.int32)
        fn(gx, gy, rows, tokens, out.ctypes.data_as(ctypes.c_void_p))
        return out
    return run


@pytest.mark.parametrize("rows", [1, 2, 4, 7, 8, 9, 17, 32, 55, 112, 250])
@pytest.mark.parametrize("tokens", [1, 2, 3, 5, 16])
@pytest.mark.parametrize("slices", [1, 3, 16, 20])
def test_every_tile_once_and_no_xcd_more_than_its_share(spread, rows, tokens, slices):
    """Each tile of the grid's 8 ceil(row tiles / 8) x token tiles x slices is taken by one workgroup, the eight XCDs' counts
    (linear workgroup number modulo 8) differ by one at most, workgroups without one come last, and where there are whole groups of eight row tiles the
    token tiles of one are on one XCD."""
    gx = -(-rows // 8) * 8 * tokens
    got = spread(gx, slices, rows, tokens)
    taken = got[:, 0] >= 0
    r, t, s = got[taken].T
    key = (r * tokens + t) * slices + s
    assert np.array_equal(np.sort(key), np.arange(rows * tokens * slices))
    shares = np.array([np.count_nonzero(taken[x::8]) for x in range(8)])
    assert shares.max() - shares.min() <= 1, shares
    for x in range(8):                                      # workgroups without a tile come last on their XCD
        assert np.all(taken[x::8][:shares[x]])
    xcd = np.nonzero(taken)[0] % 8
    in_group = r < rows // 8 * 8
    assert np.array_equal(xcd[in_group], r[in_group] % 8)
