"""The C++ launchers' workspace under stream capture (kf/flash_attn.hpp), on
the host: the header is compiled against a stand-in HIP runtime and C ABI.

Allocating during a capture is an error, so a call that runs without a
workspace, if slower, has to be captured without one when its stream has none
yet; one that cannot do without still asks for it.
"""
import os
import shutil
import subprocess

import pytest

INCLUDE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include")

HIP = r"""
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstdlib>
typedef struct S* hipStream_t;
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorStreamCaptureUnsupported = 900 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone, hipStreamCaptureStatusActive };
inline bool g_capturing = false;
inline int g_mallocs = 0;
inline size_t g_memory = SIZE_MAX;   // the largest allocation that succeeds
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t busy() { return g_capturing ? hipErrorStreamCaptureUnsupported : hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return busy(); }
inline hipError_t hipStreamSynchronize(hipStream_t) { return busy(); }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline int g_frees = 0;
inline void* g_freed[1000];
// (Kept, so that no later buffer has a freed one's address.)
inline hipError_t hipFree(void* p) { g_freed[g_frees++] = p; return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t n) {
    if (g_capturing) return hipErrorStreamCaptureUnsupported;
    if (n > g_memory) return hipErrorOutOfMemory;
    ++g_mallocs;
    *p = malloc(n);
    return hipSuccess;
}
inline hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
"""

MAIN = r"""
#include "kf/flash_attn.hpp"
#include <cstdio>
// The call needs `least` bytes and runs best with `best`.
static size_t least, best, got;
static void* got_ws;
extern "C" {
int kf_last_hip_error(void) { return 0; }
int kf_launch_flash_attn(const uint16_t*, const uint16_t*, const uint16_t*, float*, int, int, int, int, int,
                         void*) { return 0; }
int kf_attn_plan(int, int, int, int, int, int, kf_attn_plan_t* p) {
    p->workspace_bytes = best;
    p->path = least ? KF_PATH_DECODE_SPLIT : KF_PATH_DECODE;
    p->num_splits = 4;
    return KF_OK;
}
size_t kf_attn_workspace_bytes_lens(int, int, int, int, int, int) { return best; }
size_t kf_attn_decode_paged_workspace_bytes(int, int, int, int, int, int, int) { return best; }
static int take(void* ws, size_t n) {
    if (least && (!ws || n < least)) return KF_ERR_WORKSPACE;
    got = ws ? n : 0;
    got_ws = ws;
    return KF_OK;
}
int kf_attn_fwd(const void*, const void*, const void*, float*, float*, float*, int, int, int, int, int, int,
                void* ws, size_t n, void*) { return take(ws, n); }
int kf_attn_fwd_ex(const void*, const void*, const void*, void*, float*, float*, int, int, int, int, int, int,
                   const int*, int, void* ws, size_t n, void*) { return take(ws, n); }
int kf_attn_decode_paged(const void*, const void*, const void*, const int*, const int*, void*, float*, float*,
                         int, int, int, int, int, int, int, int, int, void* ws, size_t n, void*) {
    return take(ws, n);
}
}
static hipError_t call(int i, long stream, size_t need, size_t want) {
    least = need; best = want; got = 99999;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    int lens = 1;
    if (i == 0) return launch_flash_attn(nullptr, nullptr, nullptr, nullptr, 1, 1, 1, 1, 1, 16, s);
    if (i == 1) return kf::attn_fwd_ex(nullptr, nullptr, nullptr, nullptr, 1, 1, 1, 1, 1, 16, &lens, 0, s);
    return kf::attn_decode_paged(nullptr, nullptr, nullptr, nullptr, &lens, nullptr, 1, 1, 1, 1, 16, 16, 1, 1, 0, s);
}
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
"""

UNDER_CAPTURE = r"""
int main() {
    for (int i = 0; i < 3; ++i) {
        const long s = 8 * i;
        g_capturing = true;                                    // no buffer yet
        CHECK(call(i, s + 1, 0, 512) == hipSuccess && got == 0);
        CHECK(call(i, s + 1, 256, 512) == hipErrorStreamCaptureUnsupported);
        g_capturing = false;
        CHECK(call(i, s + 2, 256, 256) == hipSuccess && got == 256);
        g_capturing = true;                                    // a smaller one
        CHECK(call(i, s + 2, 256, 512) == hipSuccess && got == 256);
        CHECK(call(i, s + 2, 0, 512) == hipSuccess && got == 256);
        g_capturing = false;                                   // it grows again
        CHECK(call(i, s + 2, 256, 512) == hipSuccess && got == 512);
        const int n = g_mallocs;
        CHECK(call(i, s + 2, 256, 512) == hipSuccess && g_mallocs == n);
    }
    // Every entry of the cache taken: none is released under capture.
    for (long s = 100; s < 140; ++s) CHECK(call(1, s, 16, 16) == hipSuccess);
    g_capturing = true;
    CHECK(call(1, 200, 0, 512) == hipSuccess && got == 0);
    g_capturing = false;
    std::printf("ok\n");
    return 0;
}
"""


# A buffer handed out under capture belongs to the graph: what later calls free
# (on growth, on release of the entry) never includes it.
CAPTURED_BUFFERS = r"""
static bool freed(void* p) {
    for (int i = 0; i < g_frees; ++i)
        if (g_freed[i] == p) return true;
    return false;
}
int main() {
    for (int i = 0; i < 3; ++i) {
        const long s = 8 * i;
        // Captured with less than its best, then an eager call of the same shape.
        CHECK(call(i, s + 1, 256, 256) == hipSuccess);
        void* const small = got_ws;
        g_capturing = true;
        CHECK(call(i, s + 1, 256, 512) == hipSuccess && got_ws == small);
        g_capturing = false;
        CHECK(call(i, s + 1, 256, 512) == hipSuccess && got == 512 && got_ws != small && !freed(small));
        // Captured at its best, then a larger call.
        void* const best_ws = got_ws;
        g_capturing = true;
        CHECK(call(i, s + 1, 256, 512) == hipSuccess && got_ws == best_ws);
        g_capturing = false;
        CHECK(call(i, s + 1, 1024, 1024) == hipSuccess && got == 1024 && !freed(best_ws));
        // The buffer that followed was not captured: it goes as it grows.
        void* const eager = got_ws;
        CHECK(call(i, s + 1, 2048, 2048) == hipSuccess && freed(eager));
    }
    // Every entry released: the captured buffer stays, the others go.
    CHECK(call(1, 99, 16, 16) == hipSuccess);
    void* const kept = got_ws;
    g_capturing = true;
    CHECK(call(1, 99, 16, 16) == hipSuccess && got_ws == kept);
    g_capturing = false;
    CHECK(call(1, 100, 16, 16) == hipSuccess);
    void* const gone = got_ws;
    for (long s = 101; s < 140; ++s) CHECK(call(1, s, 16, 16) == hipSuccess);
    CHECK(!freed(kept) && freed(gone));
    std::printf("ok\n");
    return 0;
}
"""

# No memory for a call's best: it runs without a workspace, or with the partials
# of its plan (4 splits of one row at D = 16: 256 bytes, and 256 for each of the
# two statistics).
OUT_OF_MEMORY = r"""
int main() {
    for (int i = 0; i < 3; ++i) {
        const long s = 8 * i;
        g_memory = 1000;
        CHECK(call(i, s + 1, 0, 4096) == hipSuccess && got == 0);
        CHECK(call(i, s + 1, 768, 4096) == hipSuccess && got == 768);
        CHECK(call(i, s + 1, 768, 4096) == hipSuccess && got == 768);
        CHECK(call(i, s + 1, 768, 768) == hipSuccess && got == 768);
        g_memory = 700;
        CHECK(call(i, s + 2, 768, 4096) == hipErrorOutOfMemory);
        CHECK(call(i, s + 2, 768, 768) == hipErrorOutOfMemory);
        g_memory = SIZE_MAX;
        CHECK(call(i, s + 2, 768, 4096) == hipSuccess && got == 4096);
    }
    std::printf("ok\n");
    return 0;
}
"""
BODIES = {"under_capture": UNDER_CAPTURE, "captured_buffers": CAPTURED_BUFFERS, "out_of_memory": OUT_OF_MEMORY}


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
@pytest.mark.parametrize("body", list(BODIES))
def test_launchers_under_capture(tmp_path, body):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN + BODIES[body])
    exe = tmp_path / "main"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{tmp_path}", f"-I{INCLUDE}", str(tmp_path / "main.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
