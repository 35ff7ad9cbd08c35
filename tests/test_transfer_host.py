"""The host side of long transfers (csrc/eup_transfer.h) with the runtime calls and kernels replaced by
host code: every byte arrives at its place for sizes around the pieces, both ways, also where helper
threads cannot be had (CPU)."""
import os
import subprocess

import pytest

from euplectella_hpc_amd import build

HARNESS = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>
#include "eup_transfer.h"

// the allocations of the main thread that fail: from the countdown's end on, `failures` of them
static thread_local int countdown = -1, failures = 0;
void *operator new(std::size_t n)
{
    if (countdown > 0) --countdown;
    else if (countdown == 0 && failures > 0) { --failures; throw std::bad_alloc(); }
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
}
namespace eup {
int hip_check(Handle *, hipError_t e, const char *) { return e == hipSuccess ? 0 : EUP_EHIP; }
int transfer_ready(Handle *h, int64_t bytes)
{
    std::free(h->pinned);
    h->pinned = static_cast<char *>(std::calloc(1, (size_t)bytes)); // exactly what was asked for
    h->pinned_len = bytes;
    return 0;
}
}

int main()
{
    using namespace eup;
    int bad = 0, runs = 0;
    const int64_t units[] = {8, 4, 12 * 256};
    for (int fail = 0; fail < 8; ++fail) // 0: none; else helper 1, 2 or 3 and none or all after it, the fourth
        for (int64_t unit : units)
            for (int64_t pieces = 0; pieces < 11; ++pieces)
                for (int64_t extra : {int64_t(1), int64_t(4), unit - 4, int64_t(500000)}) {
                    const int64_t most = kMovePiece / unit * unit, bytes = pieces * most + extra;
                    if (bytes == 0) continue; // no caller moves nothing
                    std::vector<char> device((size_t)bytes), host((size_t)bytes);
                    for (int in = 0; in < 2; ++in) {
                        for (int64_t b = 0; b < bytes; ++b) {
                            (in ? host : device)[(size_t)b] = (char)(b * 2654435761u >> 13);
                            (in ? device : host)[(size_t)b] = 0;
                        }
                        Handle h;
                        char *dev = device.data();
                        countdown = fail ? (fail - 1) / 2 : -1;
                        failures = fail ? (fail % 2 ? 1 : 100) : 0;
                        int rc;
                        if (in)
                            rc = transfer<true>(&h, host.data(), bytes, unit, [=](int64_t at, int64_t len, char *p) { std::memcpy(dev + at, p, (size_t)len); });
                        else
                            rc = transfer<false>(&h, host.data(), bytes, unit, [=](int64_t at, int64_t len, char *p) { std::memcpy(p, dev + at, (size_t)len); });
                        countdown = -1;
                        ++runs;
                        if (rc || device != host) ++bad;
                        std::free(h.pinned);
                    }
                }
    std::printf("%d transfers, %d wrong\n", runs, bad);
    return bad != 0;
}
"""


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    if not os.path.exists(build.hipcc()):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("transfer")
    src, exe = d / "transfer_check.hip", d / "transfer_check"
    src.write_text(HARNESS)
    subprocess.run([build.hipcc(), "--offload-arch=gfx950", "--offload-host-only", "-O2", "-std=c++17", "-w",
                    "-I", os.path.join(build.HERE, "csrc"), str(src), "-lpthread", "-o", str(exe)], check=True)
    return str(exe)


def test_every_byte_arrives_with_and_without_helpers(harness):
    res = subprocess.run([harness], capture_output=True, text=True, timeout=240)
    assert res.returncode == 0, res.stdout + res.stderr
    assert " 0 wrong" in res.stdout
