"""The cut kernels' truth-table placement, four bits per lane (tt_nibble), against
the one in a piece (tt_place_stretch, which is checked against the oracle), both
of culs_amd/csrc/tt_place.h compiled for the host: all 16 phases, every table
over the phase's variables, all four lanes."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "culs_amd", "csrc", "tt_place.h")
HELPER = r"""
#define __host__
#define __device__
#define __forceinline__ inline
#include "%s"
extern "C" int differ(int n, const uint32_t *t, int phase) {
    int bad = 0;
    for (int i = 0; i < n; i++) {
        uint32_t x = 0;
        for (uint32_t k = 0; k < 4; k++) x |= tt_nibble(t[i], phase, k << 6 | (k >> 1) << 4 | (k & 1u) << 2) << 4 * k;
        bad += x != (tt_place_stretch(t[i], tt_place_entry(phase)) & 0xFFFFu);
    }
    return bad;
}
"""


@pytest.fixture(scope="module")
def differ(tmp_path_factory):
    d = tmp_path_factory.mktemp("nibble")
    (d / "n.cpp").write_text(HELPER % HEADER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", str(d / "libn.so"), str(d / "n.cpp")], check=True)
    return ctypes.CDLL(str(d / "libn.so")).differ


@pytest.mark.parametrize("phase", range(16))
def test_nibbles(differ, phase):
    k = bin(phase).count("1")
    t = np.arange(1 << (1 << k), dtype=np.uint32)
    for j in range(k, 4):           # the table does not depend on the other variables
        t |= t << np.uint32(1 << j)
    assert differ(len(t), ctypes.c_void_p(t.ctypes.data), phase) == 0
