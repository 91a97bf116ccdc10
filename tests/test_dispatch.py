"""Which kernels a call launches, on the CPU: the library is loaded over a few
HIP entry points of its own (stream capture, memory and kernel launch) that
record launches instead of making them and can run out of memory. The operands
are addresses that nothing reads."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

FAKE = r"""
#include <dlfcn.h>
#include <cstddef>
#include <cstring>
struct dim3 { unsigned x, y, z; };
typedef void* st;
static dim3 g, b; static size_t sh; static st s;
static char log_[1 << 16];
static int no_memory;
static size_t next = 1u << 28;
extern "C" {
st capturing = (st)0x1000;
void fake_no_memory(int v) { no_memory = v; }
const char* fake_log() { return log_; }
void fake_clear() { log_[0] = 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int) { return 0; }
int hipGetLastError() { return 0; }
int hipPeekAtLastError() { return 0; }
int hipStreamIsCapturing(st x, int* c) { *c = x == capturing; return 0; }
int hipThreadExchangeStreamCaptureMode(int* m) { *m = 0; return 0; }
int hipMalloc(void** p, size_t n) {
    if (no_memory) return 2;
    *p = (void*)next;
    next += (n + 255) / 256 * 256;
    return 0;
}
int __hipPushCallConfiguration(dim3 a, dim3 c, size_t m, st x) { g = a; b = c; sh = m; s = x; return 0; }
int __hipPopCallConfiguration(dim3* a, dim3* c, size_t* m, st* x) { *a = g; *c = b; *m = sh; *x = s; return 0; }
int hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, st) {
    Dl_info i;
    std::strcat(log_, dladdr(f, &i) && i.dli_sname ? i.dli_sname : "?");
    std::strcat(log_, "\n");
    return 0;
}
}
"""

# Names of a call's kernels, or the code of its error.
CHILD = r"""
import ctypes as C, json, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
from brain_amd import load
lib = load()
fake.fake_log.restype = C.c_char_p
A, CAP = 1 << 20, 0x1000
kernels = ("pad_rows", "expand_q4", "gemm_i8_dma", "gemm_i8_kernel", "splitk_reduce")
def run(stream, m, k, n, q4=False, mem=True, off=0):
    fake.fake_no_memory(0 if mem else 1)
    fake.fake_clear()
    fn = lib.bh_matmul_q4_dyn if q4 else lib.bh_matmul_i8_dyn
    rc = fn(stream, A + off, 2 * A, A, A, None, A, 0, m, k if q4 else k // 4, n)
    names = fake.fake_log().decode().split()
    return [next(x for x in kernels if x in n) for n in names] if rc == 0 else rc
out = []
for c in json.loads(sys.stdin.read()):
    if c[0] == "reserve":
        fake.fake_no_memory(0)
        out.append(lib.bh_reserve_workspace(*c[1:]))
    else:
        out.append(run(*c[1:2], *c[2:5], **c[5]))
print(json.dumps(out))
"""

CAP = 0x1000
PER_THREAD = 2
PADDED = ["pad_rows", "gemm_i8_dma"]
STAGED = ["gemm_i8_kernel"]
SPLIT = ["gemm_i8_dma", "splitk_reduce"]
RAGGED, LONG = (65, 1000, 257), (128, 3072, 1024)  # unsplit; split over K


@pytest.fixture(scope="module")
def dispatch(tmp_path_factory):
    d = tmp_path_factory.mktemp("fakehip")
    src, so = d / "fake.cpp", d / "libfakehip.so"
    src.write_text(FAKE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", str(src), "-o", str(so), "-ldl"], check=True)

    def run(calls):
        """calls: ("run", stream, m, k, n, options) or ("reserve", stream, m, kg, n), in one process."""
        p = subprocess.run([sys.executable, "-c", CHILD, str(so)], input=json.dumps(calls), capture_output=True,
                           text=True, cwd=ROOT)
        assert p.returncode == 0, p.stderr
        return json.loads(p.stdout.splitlines()[-1])

    return run


@pytest.mark.parametrize("q4", [False, True])
def test_without_memory_the_kernels_that_need_none(dispatch, q4):
    o = dict(q4=q4)
    got = dispatch([("run", 0, *RAGGED, dict(o, mem=False)), ("run", 0, *LONG, dict(o, mem=False)),
                    ("run", 0, *LONG, dict(o, mem=False, off=4)), ("run", 0, 40, 6152, 64, dict(o, mem=False)),
                    ("run", 0, *RAGGED, o), ("run", 0, *LONG, o), ("run", 0, *LONG, dict(o, mem=False))])
    assert got == [STAGED, ["gemm_i8_dma"], STAGED, STAGED, PADDED, SPLIT, SPLIT]


def test_captured_and_per_thread_calls_share_no_padded_copies(dispatch):
    big = ("run", CAP + 0x1000, 4096, 1000, 4096, {})
    got = dispatch([big, ("run", CAP, *RAGGED, {}), ("run", CAP, *RAGGED, dict(q4=True)),
                    ("run", CAP, *LONG, dict(off=4, q4=True)), ("run", PER_THREAD, *RAGGED, {}),
                    ("run", CAP, 200, 8192, 1024, dict(q4=True))])
    assert got == [PADDED, STAGED, STAGED, STAGED, STAGED, ["gemm_i8_dma"]]


def test_int4_splits(dispatch):
    """Weights expanded to int8 from 6144 rows where there is a workspace; column ranges where 256x256 tiles would leave most of a round empty;
    K split where 16 q would not fit one i32 sum (unless there are no slabs for
    it); padded copies in column ranges from the size their bound allows."""
    q4 = dict(q4=True)
    dma = ["gemm_i8_dma"]
    calls = [
        (("run", 0, 4096, 4096, 22016, q4), dma * 2), (("run", 0, 4096, 4096, 22016, {}), dma * 2),
        (("run", 0, 300, 131200, 64, q4), SPLIT), (("run", 0x3000, 300, 131200, 64, dict(q4, mem=False)), STAGED),
        (("run", CAP, 200, 131200, 64, q4), STAGED), (("run", 0, 4096, 131200, 4096, q4), STAGED),
        (("run", 0, 300, 9952, 151936, q4), PADDED * 2), (("run", 0, 200, 9960, 151936, q4), STAGED),
        (("run", 0x3000, 8192, 4096, 11008, dict(q4, mem=False)), dma * 2),
        (("run", CAP, 8192, 4096, 11008, q4), dma * 2),
        (("run", 0, 8192, 4096, 11008, q4), ["expand_q4"] + dma * 2),
        (("reserve", CAP + 0x1000, 8192, 1024, 11008), 0),
    ]
    assert dispatch([c for c, _ in calls]) == [want for _, want in calls]
