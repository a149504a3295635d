"""The transfer of states (gpu-vah_amd/csrc/vah_transfer.h) on the CPU, against a stand-in
for the runtime whose asynchronous copies happen as late as they may: when their stream
is waited for.  A slot read before its copy or refilled before it, a chunk left out, a
row or a gap misplaced and a write past a buffer all show; built with the address and
undefined-behaviour checks, and with the thread checks for the shares that several
threads take."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "gpu-vah_amd", "csrc", "vah_transfer.h")

RUNTIME = r'''
#pragma once
#include <stdlib.h>
#include <string.h>
#include <deque>
#include <mutex>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
struct Pending { void *dst; const void *src; size_t n; };
struct FakeStream { std::mutex m; std::deque<Pending> q; };
typedef FakeStream *hipStream_t;
inline bool g_refuse_pinned = false;
inline hipError_t hipHostMalloc(void **p, size_t n) { *p = g_refuse_pinned ? nullptr : malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
inline hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    std::lock_guard<std::mutex> l(st->m);
    st->q.push_back({d, s, n});
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t st) {
    std::lock_guard<std::mutex> l(st->m);
    for (const Pending &p : st->q) memcpy(p.dst, p.src, p.n);
    st->q.clear();
    return hipSuccess;
}
'''

# the layout of vah_host_common.h
COMMON = r'''
#pragma once
namespace vah_host {
struct Layout {
    int nx, ny, nz, ncx, ncy, ncz;
    long ncell, fs;
    Layout(int nx_, int ny_, int nz_)
        : nx(nx_), ny(ny_), nz(nz_), ncx(nx_ + 4), ncy(ny_ + 4), ncz(nz_ > 1 ? nz_ + 4 : 1) {
        ncell = (long)ncx * ncy * ncz;
        fs = (ncell + 63) / 64 * 64;
    }
};
}
'''

MAIN = r'''
#include "vah_transfer.h"
#include <stdio.h>
using namespace vah_host;
static double value(long k) { return 1.0 + 1e-3 * (double)k; }
static int round_trip(Transfer &T, int nx, int ny, int nz, bool ghosts) {
    const Layout L(nx, ny, nz);
    const Rows R = ghosts ? Rows(L) : Rows(nx, ny, nz);
    const long n = (long)nx * ny * nz, fs = ghosts ? L.fs : n;
    const int nf[3] = {15, 1, 4};
    FakeStream st;
    std::vector<std::vector<double>> dev, src, dst;
    std::vector<Segment> up, down;
    for (int s = 0; s < 3; ++s) {
        dev.emplace_back(nf[s] * fs, -7.0);
        src.emplace_back(nf[s] * n);
        dst.emplace_back(nf[s] * n, -1.0);
        for (long k = 0; k < (long)src[s].size(); ++k) src[s][k] = value(k + s);
        up.push_back({dev[s].data(), nf[s], nullptr, src[s].data()});
        down.push_back({dev[s].data(), nf[s], dst[s].data(), nullptr});
    }
    if (T.upload(0, &st, R, up) != hipSuccess) return 1;
    const long g = ghosts ? 2 : 0, gz = ghosts && nz > 1 ? 2 : 0;
    for (int s = 0; s < 3; ++s)
        for (int f = 0; f < nf[s]; ++f)
            for (long c = 0; c < fs; ++c) {
                const long i = c % (nx + 2 * g) - g, r = c / (nx + 2 * g), j = r % (ny + 2 * g) - g, k = r / (ny + 2 * g) - gz;
                const bool in = i >= 0 && i < nx && j >= 0 && j < ny && k >= 0 && k < nz;
                const double want = in ? src[s][((f * (long)nz + k) * ny + j) * nx + i] : 0.0;
                if (dev[s][f * fs + c] != want) return 2;
            }
    if (T.download(0, &st, R, down) != hipSuccess) return 3;
    if (!st.q.empty()) return 4;
    return src == dst ? 0 : 5;
}
int main() {
    const int shapes[][3] = {{1, 1, 1}, {1, 9, 1}, {33, 1, 1}, {7, 5, 2}, {41, 37, 1}, {161, 165, 1}, {140001, 1, 1},
                             {45, 50, 60}};
    for (int refuse = 0; refuse < 2; ++refuse) {
        g_refuse_pinned = refuse;
        Transfer shared;  // one object through all sizes, and one of its own for each
        for (auto &s : shapes)
            for (int ghosts = 0; ghosts < 2; ++ghosts) {
                Transfer own;
                const int a = round_trip(shared, s[0], s[1], s[2], ghosts), b = round_trip(own, s[0], s[1], s[2], ghosts);
                if (a || b) {
                    printf("%d x %d x %d ghosts %d refused %d: %d %d\n", s[0], s[1], s[2], ghosts, refuse, a, b);
                    return 1;
                }
            }
    }
    return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("checks", [("-fsanitize=address,undefined", "-fno-sanitize-recover=undefined"),
                                    ("-fsanitize=thread",)], ids=["address", "thread"])
def test_round_trips_with_late_copies(tmp_path, checks):
    d = tmp_path
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "vah_host_common.h").write_text(COMMON)
    shutil.copy(HEADER, d)
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", *checks, "-I", str(d), "-o", str(d / "t"),
                    str(d / "main.cpp")], check=True, capture_output=True, text=True)
    r = subprocess.run([str(d / "t")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout + r.stderr)[-3000:]
