"""Device memory that contexts and batches keep between calls is given back when another
allocation needs it, and only what no run uses: the library's allocator on the host, over
stand-ins for the HIP calls that count the bytes of a small device."""
import os
import subprocess
import tempfile

import sandengine_amd as S

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = r"""
#include "CSRC/se_internal.hpp"
#include <cstdio>
#include <cstdlib>
#include <map>
static std::map<void*, size_t> g_live;
static size_t g_free = 100;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (n > g_free) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = std::malloc(1);
    g_live[*p] = n;
    g_free -= n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    if (!g_live.count(p)) { printf("free of an unknown address\n"); exit(1); }
    g_free += g_live[p];
    g_live.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
}
#define CHECK(c) if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; }
using namespace se_rt;
static void hold(Pool::Block& b, size_t n) { if (hipMalloc(&b.mem, n) == hipSuccess) b.bytes = n; }
int main() {
    void *p = nullptr, *q = nullptr;
    auto a = make_pool(0), b = make_pool(0), other = make_pool(1);
    Pool::Block idle, busy;
    a->arenas.push_back(&idle);
    b->arenas.push_back(&busy);
    hold(a->scratch, 30);
    hold(idle, 20);
    hold(busy, 10);
    hold(other->scratch, 10);
    busy.busy = true;
    CHECK(device_alloc(0, &p, 30) == hipSuccess && a->scratch.mem && idle.mem);  // fits beside them
    CHECK(device_alloc(0, &q, 50) == hipSuccess);                                // in their place
    CHECK(!a->scratch.mem && !a->scratch.bytes && !idle.mem && busy.mem && other->scratch.mem && g_free == 0);
    CHECK(hipFree(q) == hipSuccess && device_alloc(0, &q, 51) != hipSuccess && !q);  // a run's and another device's stay
    CHECK(busy.mem && other->scratch.mem);
    busy.busy = false;
    CHECK(device_alloc(0, &q, 60) == hipSuccess && !busy.mem);
    CHECK(hipFree(q) == hipSuccess && hipFree(p) == hipSuccess);
    hold(b->scratch, 40);
    b->arenas.clear();
    b.reset();  // the last owner frees what is left
    CHECK(g_free == 90);
    CHECK(device_alloc(0, &q, 95) != hipSuccess && device_alloc(0, &q, 90) == hipSuccess);
    CHECK(hipFree(q) == hipSuccess);
    printf("ok\n");
    return 0;
}
"""


def test_kept_memory_is_given_back():
    csrc, pkg = os.path.join(ROOT, "sandengine_amd", "csrc"), os.path.dirname(S.__file__)
    with tempfile.TemporaryDirectory() as d:
        cpp, exe = os.path.join(d, "kept.cpp"), os.path.join(d, "kept")
        with open(cpp, "w") as f:
            f.write(MAIN.replace("CSRC", csrc))
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-w", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                               "-o", exe, cpp, "-L" + pkg, "-l:libsandengine_hip.so", "-Wl,-rpath," + pkg,
                               "-Wl,--allow-shlib-undefined"])
        p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout + p.stderr
