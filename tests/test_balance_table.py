"""Room of the balance's node table (balance_table_slots, culs_amd/csrc/
gls_internal.h), compiled for the host: a power of two, at most a quarter full
where that is small, and never more than twice what half full takes, nor 2^32
slots (whose last index means none) where 2^31 are half full."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def slots(tmp_path_factory):
    d = tmp_path_factory.mktemp("slots")
    (d / "s.cpp").write_text('#include "gls_internal.h"\n'
                             'extern "C" uint64_t slots(uint64_t n) { return balance_table_slots(n); }\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "culs_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                    "-o", str(d / "libs.so"), str(d / "s.cpp")], check=True)
    f = ctypes.CDLL(str(d / "libs.so")).slots
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_uint64]
    return f


@pytest.mark.parametrize("bits", range(0, 32))
def test_slots(slots, bits):
    for n in (1 << bits, (1 << bits) + 1, (3 << bits) // 2, (2 << bits) - 17):
        s = slots(n)
        assert s & (s - 1) == 0 and s >= 2 * n
        if n <= (1 << 29) - 16:
            assert s >= 4 * n and s <= max(1024, 8 * (n + 16))
        elif n <= (1 << 30) - 16:
            assert s == 1 << 31
        elif n <= (1 << 31) - 16:
            assert s == 1 << 32
