"""The pinned staging copies (CPU only): psim_stage.hip compiled for the host
against a stream that runs what is enqueued only when it is waited for, so that a
half of the buffer reused too early, or read too early, shows.  Arrays around
the sizes of the buffer (8 MiB), with as much pinned memory as asked for, with
too little to grow, and with none."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "proteinsim2015_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <vector>
#include "psim_stage.hip"

// ---- a runtime whose stream runs when it is waited for
static std::vector<std::function<void()>> queue;
static size_t ran = 0, limit = 0, pinned = 0;
static std::map<void *, size_t> blocks, marks;
static void run(size_t to) { while (ran < to) queue[ran++](); }
extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (pinned + n > limit) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    std::memset(*p, 0xee, n);
    blocks[*p] = n;
    pinned += n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    if (ran != queue.size() || !blocks.count(p)) std::abort();   // still in use, or not ours
    pinned -= blocks[p];
    blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    queue.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { run(queue.size()); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void *)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { marks[(void *)e] = queue.size(); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { run(marks[(void *)e]); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
}
namespace psim {
void host_copy(void *d, const void *s, size_t n) { std::memcpy(d, s, n); }
}

int main(int argc, char **argv)
{
    limit = std::strtoull(argv[1], nullptr, 10);
    const size_t first = std::strtoull(argv[2], nullptr, 10);
    psim::HostStage h;
    (void)psim::stage_reserve(h, first);
    const size_t held = h.cap;
    std::vector<std::vector<unsigned char>> host, dev;
    std::vector<psim::Xfer> x;
    for (int k = 3; k < argc; ++k) {
        const size_t n = std::strtoull(argv[k], nullptr, 10);
        host.emplace_back(n);
        dev.emplace_back(n);
        for (size_t i = 0; i < n; ++i) dev.back()[i] = (unsigned char)(i * 131 + k + (i >> 13));
    }
    for (size_t k = 0; k < host.size(); ++k)
        x.push_back({host[k].data(), dev[k].data(), dev[k].size()});
    for (int pass = 0; pass < 2; ++pass) {   // the buffer as the pass before left it
        for (auto &v : host) std::memset(v.data(), 0, v.size());
        if (psim::stage_read(h, nullptr, x.data(), (int)x.size())) return 1;
        if (host != dev) return 2;
        for (auto &v : host)
            for (auto &c : v) c ^= 0x5a;
        for (auto &v : dev) std::memset(v.data(), 0, v.size());
        if (psim::stage_write(h, nullptr, x.data(), (int)x.size())) return 3;
        run(queue.size());
        if (host != dev) return 4;
    }
    std::printf("%zu %zu\n", held, h.cap);
    psim::stage_free(h);
    return pinned ? 5 : 0;
}
"""

MIB = 1 << 20
ARRAYS = [
    [1], [4096], [24, 24 * 170], [8 * MIB], [8 * MIB - 64, 64], [8 * MIB - 63, 64],
    [8 * 3 * 69904] * 5, [8 * 3 * 69905] * 5, [8 * 3 * 69906] * 5,
    [4 * MIB, 4 * MIB + 1], [20 * MIB + 12345, 7, 3 * MIB], [1, 9 * MIB, 1],
]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("stage")
    src, exe = d / "stage.cpp", d / "stage"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I",
                           "/opt/rocm/include", "-I", CSRC, str(src), "-o", str(exe)])
    return str(exe)


def copy(program, limit, first, arrays):
    r = subprocess.run([program, str(limit), str(first), *map(str, arrays)],
                       capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
    return tuple(map(int, r.stdout.split()))


@pytest.mark.parametrize("arrays", ARRAYS)
def test_pinned(program, arrays):
    held, cap = copy(program, 1 << 40, 1, arrays)
    assert held == 4096 and 4096 <= cap <= 8 * MIB


@pytest.mark.parametrize("arrays", ARRAYS)
def test_no_more_pinned_memory(program, arrays):
    """64 KiB made with the context, nothing beyond: more rounds through it."""
    held, cap = copy(program, 65536 + 4096, 65536, arrays)
    assert held == cap == 65536


@pytest.mark.parametrize("arrays", ARRAYS)
def test_no_pinned_memory(program, arrays):
    assert copy(program, 0, 8 * MIB, arrays) == (0, 0)
