"""The host side of the array fetch (culs_amd/csrc/transfer.hip), compiled for
the host and linked with a stand-in for the HIP runtime whose device memory is
the host's: what the fetch does where pinned memory cannot be had, and on which
device it and the copy of a graph run.  Sizes on both sides of the staging (2 MiB
in all) and of its pieces (4 MiB of an array), both literal conventions, arrays
left out."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "culs_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

RUNTIME = r"""
#include "gls_internal.h"
#include <atomic>
#include <cstdlib>
#include <cstring>

static bool g_pinned;
static thread_local int t_device;          // the thread's current device
static std::atomic<int> g_elsewhere;       // allocations, launches and events on another one than the context's
constexpr int DEVICE = 3;
static void here() { if (t_device != DEVICE) g_elsewhere++; }

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    here();
    *p = g_pinned ? malloc(n) : nullptr;
    return g_pinned ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipGetDevice(int *d) { *d = t_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { here(); *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { here(); return hipErrorUnknown; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipUnregisterFatBinary(void **) {}

int run_fetch(int pinned, int32_t nPIs, int32_t n, int32_t nPOs, uint32_t *g0, uint32_t *g1, uint32_t *gp, uint32_t *f0,
              uint32_t *f1, uint32_t *pos, int32_t conv) {
    g_pinned = pinned != 0;
    gls_ctx ctx;
    ctx.device = DEVICE;
    DevGraph g;
    g.nObjs = n;
    g.nPIs = nPIs;
    g.nPOs = nPOs;
    g.f0 = g0;
    g.f1 = g1;
    g.pos = gp;
    const int rc = dev_graph_fetch(&ctx, g, f0, f1, pos, conv);
    transfer_free(&ctx);
    return rc;
}

// a copy and fetches of all sizes by a thread on `device`; returns the device that
// it is left on, or -1 if something ran elsewhere
int run_on(int device, int32_t n, uint32_t *words, uint32_t *out) {
    g_elsewhere = 0;
    t_device = device;
    gls_ctx ctx;
    ctx.device = DEVICE;
    DevGraph g;
    g.nObjs = n;
    g.nPIs = 1;
    g.nPOs = 0;
    g.f0 = g.f1 = g.level = g.pos = words;
    for (int pinned = 0; pinned < 2; pinned++) {
        g_pinned = pinned != 0;
        (void)dev_graph_copy(&ctx, g, g);
        (void)dev_graph_fetch(&ctx, g, out, nullptr, nullptr, 0);
    }
    const int left = t_device;
    t_device = DEVICE;
    transfer_free(&ctx);
    return g_elsewhere ? -1 : left;
}
}
int gls_fail(gls_ctx *, int code, const char *, ...) { return code; }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("transfer")
    (d / "runtime.cpp").write_text(RUNTIME)
    flags = [HIPCC, "-O1", "-std=c++17", "-fPIC", "-x", "hip", "--offload-host-only", "-Wno-everything", "-I" + SRC,
             "-I" + os.path.join(ROOT, "include")]
    objs = []
    for src in (os.path.join(SRC, "transfer.hip"), d / "runtime.cpp"):
        objs.append(str(d / (os.path.basename(src) + ".o")))
        subprocess.run(flags + ["-c", str(src), "-o", objs[-1]], check=True)
    # the device code of the kernels, which nothing here launches
    name = next(x.split()[-1] for x in subprocess.run(["nm", objs[0]], stdout=subprocess.PIPE, text=True, check=True)
                .stdout.splitlines() if "__hip_fatbin_" in x and " U " in x)
    so = str(d / "libtransfer.so")
    subprocess.run(["g++", "-shared", "-o", so] + objs + ["-Wl,--defsym=%s=0" % name, "-Wl,-Bsymbolic", "-pthread"], check=True)
    return ctypes.CDLL(so)


def ptr(a):
    return ctypes.c_void_p(a.ctypes.data if a is not None else None)


SIZES = [(100, 7), (180_000, 524288 - 360000), (1_048_576, 20), (1_048_577, 20), (5_000_001, 1_200_000)]


@pytest.mark.parametrize("pinned", [False, True], ids=["without", "pinned"])
@pytest.mark.parametrize("n,nPOs", SIZES)
@pytest.mark.parametrize("conv", [0, 1])
def test_fetch(host, pinned, n, nPOs, conv):
    if pinned and 4 * (2 * n + nPOs) <= 2 << 20:
        pytest.skip("goes by kernels, which the stand-in does not run")
    rng = np.random.default_rng(n)
    graph = [rng.integers(0, 50, k, dtype=np.uint32) for k in (n, n, nPOs)]
    want = [np.where(x < 2, 1 - x.astype(np.int64), x).astype(np.uint32) if conv else x for x in graph]
    for left_out in (None, 0, 1, 2):
        out = [None if i == left_out else np.full(len(x), 77, np.uint32) for i, x in enumerate(graph)]
        rc = host.run_fetch(int(pinned), 3, n, nPOs, *map(ptr, graph), *map(ptr, out), conv)
        assert rc == 0
        assert all(o is None or np.array_equal(o, w) for o, w in zip(out, want))


@pytest.mark.parametrize("n", [100, 3_000_000])
@pytest.mark.parametrize("device", [0, 3, 5])
def test_thread_on_another_device(host, n, device):
    words, out = np.zeros(n, np.uint32), np.zeros(n, np.uint32)
    assert host.run_on(device, n, ptr(words), ptr(out)) == device
