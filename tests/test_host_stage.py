"""The crossing of large host arrays through pinned buffers (csrc/host_stage.hpp), compiled against
a stand-in of the runtime with two devices in host memory (CPU test): contents, the caller's
current device, failing copies and buffers taken by another context."""
import os
import subprocess

from conftest import PKG

RUNTIME = r"""
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
enum hipError_t { hipSuccess, hipErrorInvalidHandle, hipErrorUnknown };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum { hipEventDisableTiming, hipHostMallocPortable };
struct Owned { int device; };
typedef Owned *hipStream_t, *hipEvent_t;
inline thread_local int current = 0;        // per thread, device 0 in a new one
inline std::atomic<int> copies{0}, fail_at{-1};
inline hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { *p = malloc(n); return hipSuccess; }
inline hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = new Owned{current}; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    return e->device == s->device ? hipSuccess : hipErrorInvalidHandle;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (copies++ == fail_at) return hipErrorUnknown;
    memcpy(d, s, n);
    return hipSuccess;
}
"""

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "host_stage.hpp"
using namespace rpcf_host;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
static unsigned char at(size_t i, int salt) { return (unsigned char)(i * 2654435761u >> 11) + salt; }

// out and back in through padded host rows; false: contents or the padding changed
static bool round_trip(int device, size_t rows, size_t row, size_t pitch, int salt, bool* staged) {
    Owned stream{device};
    std::vector<char> dev(rows * row), host(rows * pitch, 77), back(rows * row, 0);
    for (size_t i = 0; i < dev.size(); i++) dev[i] = at(i, salt);
    for (int out = 1; out >= 0; out--) {
        char* d = out ? dev.data() : back.data();
        if (staged_copy(device, &stream, d, host.data(), rows, row, pitch, out, staged) != hipSuccess) return false;
        if (*staged) continue;
        if (out) copy_rows(host.data(), pitch, d, row, rows, row);
        else copy_rows(d, row, host.data(), pitch, rows, row);
    }
    if (back != dev) return false;
    for (size_t r = 0; r < rows; r++)
        for (size_t k = row; k < pitch; k++)
            if (host[r * pitch + k] != 77) return false;
    return true;
}

int main() {
    bool staged;
    stage_ref(1);
    // whole and partial pieces, rows that do not divide a piece, one row a piece
    const size_t sizes[][3] = {{8 << 10, 1 << 10, 1 << 10}, {8192, 1040, 1088}, {9001, 2064, 2064}, {5, 2 << 20, 2 << 20}};
    for (auto& s : sizes)
        for (int own : {0, 1})
            for (int context : {0, 1}) {
                current = own;
                CHECK(round_trip(context, s[0], s[1], s[2], own, &staged) && staged);
                CHECK(current == own);
            }
    // a copy that fails on any thread
    for (int n = 0; n < 8; n++) {
        current = 1, copies = 0, fail_at = n;
        Owned stream{0};
        std::vector<char> dev(16 << 20), host(16 << 20);
        for (bool out : {false, true}) {
            copies = 0;
            CHECK(staged_copy(0, &stream, dev.data(), host.data(), 16 << 10, 1 << 10, 1 << 10, out, &staged) != hipSuccess);
            CHECK(staged && current == 1);
        }
    }
    fail_at = -1;
    // below the least size, and with the buffers taken: left to the caller
    CHECK(round_trip(0, 100, 1 << 10, 1 << 10, 3, &staged) && !staged);
    {
        std::lock_guard<std::mutex> taken(g_stage_mu);
        CHECK(round_trip(0, 8 << 10, 1 << 10, 1 << 10, 4, &staged) && !staged);
    }
    // contexts of two devices that cross at once
    bool ok[4] = {};
    std::vector<std::thread> th;
    for (int t = 0; t < 4; t++)
        th.emplace_back([&ok, t] {
            ok[t] = true;
            for (int i = 0; i < 6; i++) {
                bool way;
                ok[t] = ok[t] && round_trip(t & 1, 8200, 1040, 1040 + 16 * t, t + i, &way);
            }
        });
    for (auto& t : th) t.join();
    CHECK(ok[0] && ok[1] && ok[2] && ok[3]);
    stage_ref(-1);
    CHECK(g_stage == nullptr);
    printf("ok\n");
}
"""


def test_staged_copies(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "stage.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "stage")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-class-memaccess", "-pthread", "-I", str(tmp_path), "-I",
                    os.path.join(PKG, "csrc"), "-o", exe, str(tmp_path / "stage.cpp")], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout + out.stderr
