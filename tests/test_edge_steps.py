"""Steps through the last edge positions that a graph may have (2^32 - 3): the
header the kernels use, compiled for the host."""
import ctypes
import os
import subprocess

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wedge_amd", "csrc")

# the loop of a wavefront over a tile, writing every position its lanes take;
# stops after max positions
DRIVER = r"""
#include "wg_span.h"
uint32_t steps(uint32_t b, uint32_t e, uint32_t width, uint32_t* out, uint32_t max)
{
    uint32_t n = 0;
    for (uint32_t p = b, len; (len = wg_step(p, e, width)) != 0u; p += len)
        for (uint32_t lane = 0; lane < width; ++lane)
            if (lane < len) {
                if (n == max)
                    return n + 1;
                out[n++] = p + lane;
            }
    return n;
}
"""


def test_steps_end_where_positions_wrap(tmp_path):
    src, lib = tmp_path / "steps.c", tmp_path / "steps.so"
    src.write_text(DRIVER)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-I", CSRC, "-o", str(lib), str(src)], check=True)
    f = ctypes.CDLL(str(lib)).steps
    f.restype = ctypes.c_uint32
    f.argtypes = [ctypes.c_uint32] * 3 + [ctypes.c_void_p, ctypes.c_uint32]
    for top in (2**32 - 2, 2**32 - 3, 2**32 - 64, 2**32 - 65, 1000):
        for count in (0, 1, 2, 63, 64, 65, 127, 128, 129, 512):
            for width in (64, 1024):
                out = np.zeros(600, np.uint32)
                n = f(top - count, top, width, out.ctypes.data, out.size)
                assert n == count, (top, count, width)
                assert np.array_equal(out[:n].astype(np.uint64), np.arange(top - count, top, dtype=np.uint64))
