"""The staged state transfers (csrc/cles_stage.cpp) against a HIP stub on the
CPU: every row arrives, the padding is left alone, and the calling thread's
current device is the one it had, also after a failed copy and where neither
pinned memory nor every thread's buffer is to be had (no GPU is touched)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "cles_internal.h"

static thread_local int current = 0;
static std::atomic<bool> pinned{true}, broken{false};
static std::atomic<int> wrong_device{0};

extern "C" {
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)8; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (!pinned) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (current != 1) wrong_device++;
    if (broken) return hipErrorUnknown;
    std::memcpy(d, s, n);
    return hipSuccess;
}
}

static int check(int64_t n0, int64_t n1, int64_t n2, int64_t C)
{
    const int64_t h = 2, p0 = n0 + 2 * h, p1 = n1 + 2 * h, p2 = n2 + 2 * h, NP = p0 * p1 * p2;
    std::vector<double> host(NP * C), back(NP * C, 7.0), dev(n0 * n1 * n2 * C);
    for (size_t i = 0; i < host.size(); i++) host[i] = (double)i;
    cles::View3 v;
    v.n[0] = n0; v.n[1] = n1; v.n[2] = n2;
    v.s[0] = 1; v.s[1] = p0; v.s[2] = p0 * p1;
    const int64_t org = h + p0 * (h + p1 * h);
    cles::HostStage stage;
    stage.transfer(false, 1, nullptr, dev.data(), v, C, NP, host.data() + org);
    stage.transfer(true, 1, nullptr, dev.data(), v, C, NP, back.data() + org);
    int bad = 0;
    for (int64_t c = 0; c < C; c++)
        for (int64_t k = 0; k < p2; k++)
            for (int64_t j = 0; j < p1; j++)
                for (int64_t i = 0; i < p0; i++) {
                    const bool in = i >= h && i < h + n0 && j >= h && j < h + n1 && k >= h && k < h + n2;
                    const int64_t o = i + p0 * (j + p1 * (k + p2 * c));
                    bad += back[o] != (in ? host[o] : 7.0);
                }
    return bad;
}

int main()
{
    int bad = 0, threw = 0;
    hipSetDevice(3);
    bad += check(9, 1, 1, 5) + check(33, 29, 31, 5) + check(129, 130, 65, 6);
    std::printf("device %d\n", current);
    pinned = false;
    bad += check(129, 130, 65, 6);
    std::printf("device %d\n", current);
    broken = true;
    try {
        bad += check(129, 130, 65, 6);
    } catch (const cles::Error &e) {
        threw = e.code;
    }
    std::printf("device %d\n", current);
    std::printf("bad %d wrong %d threw %d\n", bad, wrong_device.load(), threw == CLES_ERR_HIP);
}
"""


def test_transfers_leave_the_current_device(tmp_path):
    src = tmp_path / "stage.cpp"
    src.write_text(PROGRAM)
    pkg = os.path.join(ROOT, "compactles.jl_amd")
    exe = tmp_path / "stage"
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(pkg, "csrc"), str(src),
                    os.path.join(pkg, "csrc", "cles_stage.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.split("\n")
    assert out[:4] == ["device 3"] * 3 + ["bad 0 wrong 0 threw 1"]
