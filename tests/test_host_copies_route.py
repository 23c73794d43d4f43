"""The routes of hip_h2d, hip_d2h and hip_d2h_rows (hip_backend.c) without a
GPU: the file is compiled against a stand-in of the HIP runtime whose device
memory is host memory and which writes down every transfer's host address.

Pageable memory goes through the context's pinned staging at small sizes, and
downloads from 2 MiB on; memory that the runtime knows (pinned or managed, as
hipPointerGetAttributes says) is what the transfer itself reads or writes, at
every size.  Bytes arrive whole either way."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM_INC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")
pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(ROCM_INC, "hip", "hip_runtime_api.h")),
                                reason="HIP headers not present")

HARNESS = r"""
#include "hip_backend.c"
static char *known, *known_end;          /* the range the runtime knows */
static const char *user, *user_end;      /* the caller's memory */
static int direct, other;                /* transfers to or from the caller's memory, and the rest */
static void* seen(const void* p) { if ((char*)p >= user && (char*)p < user_end) direct++; else other++; return (void*)p; }
hipError_t hipMemcpyHtoDAsync(hipDeviceptr_t d, const void* s, size_t n, hipStream_t st) { (void)st; memcpy(d, seen(s), n); return hipSuccess; }
hipError_t hipMemcpyDtoHAsync(void* d, hipDeviceptr_t s, size_t n, hipStream_t st) { (void)st; memcpy(seen(d), s, n); return hipSuccess; }
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind k, hipStream_t st) {
    (void)k; (void)st;
    seen(d);
    for (size_t r = 0; r < h; r++) memcpy((char*)d + r * dp, (const char*)s + r * sp, w);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    memset(a, 0, sizeof(*a));
    a->type = (char*)p >= known && (char*)p < known_end ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
#define OK(name, args) hipError_t name args { return hipSuccess; }
#pragma GCC diagnostic ignored "-Wunused-parameter"
OK(hipSetDevice, (int d)) OK(hipStreamSynchronize, (hipStream_t s)) OK(hipStreamDestroy, (hipStream_t s))
OK(hipStreamCreateWithFlags, (hipStream_t* s, unsigned f)) OK(hipStreamWaitEvent, (hipStream_t s, hipEvent_t e, unsigned f))
OK(hipEventCreateWithFlags, (hipEvent_t* e, unsigned f)) OK(hipEventDestroy, (hipEvent_t e))
OK(hipEventRecord, (hipEvent_t e, hipStream_t s)) OK(hipMemsetD8Async, (hipDeviceptr_t p, unsigned char v, size_t n, hipStream_t s))
OK(hipModuleLoadData, (hipModule_t* m, const void* p)) OK(hipModuleUnload, (hipModule_t m))
OK(hipModuleGetFunction, (hipFunction_t* f, hipModule_t m, const char* n))
OK(hipModuleLaunchKernel, (hipFunction_t f, unsigned a, unsigned b, unsigned c, unsigned d, unsigned e, unsigned g, unsigned s,
                           hipStream_t st, void** p, void** x))
OK(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor, (int* n, hipFunction_t f, int b, size_t s))
OK(hipDeviceGetAttribute, (int* v, hipDeviceAttribute_t a, int d))
const char* hipGetErrorName(hipError_t e) { return ""; }
const char* hipGetErrorString(hipError_t e) { return ""; }

/* argv: image, then what (up, down, rows), known (0/1), bytes or rows, row bytes, pitch */
int main(int argc, char** argv) {
    HipCtx c = hip_init(NULL, argv[1]);
    hip_set_current(&c);
    for (int i = 2; i + 4 < argc; i += 5) {
        const int rows = argv[i][0] == 'r', up = argv[i][0] == 'u';
        const u64 n = strtoull(argv[i + 2], NULL, 10), rb = strtoull(argv[i + 3], NULL, 10),
                  pitch = strtoull(argv[i + 4], NULL, 10);
        const u64 host = rows ? n * rb : n, dev = rows ? n * pitch : n;
        unsigned char *h = malloc(host + 1), *d = malloc(dev + 1);
        for (u64 b = 0; b < dev; b++) d[b] = (unsigned char)(b * 7 + b / 251);
        for (u64 b = 0; b < host; b++) h[b] = (unsigned char)(b * 5 + b / 253);
        known = known_end = NULL;
        user = (char*)h; user_end = (char*)h + host;
        if (argv[i + 1][0] == '1') { known = (char*)h; known_end = (char*)h + host; }
        direct = other = 0;
        int ok = 1;
        if (up) {
            hip_h2d(d, h, n);
            ok = memcmp(h, d, n) == 0;
        } else if (!rows) {
            hip_d2h(h, d, n);
            ok = memcmp(h, d, n) == 0;
        } else {
            hip_d2h_rows(h, d, pitch, rb, n);
            for (u64 r = 0; r < n; r++) ok = ok && memcmp(h + r * rb, d + r * pitch, rb) == 0;
        }
        printf("%d %d %d\n", ok, direct, other);
        free(h);
        free(d);
    }
    hip_shutdown(&c);
    return 0;
}
"""
KB, MB = 1 << 10, 1 << 20


@pytest.fixture(scope="module")
def copies(tmp_path_factory):
    d = tmp_path_factory.mktemp("copies")
    (d / "h.c").write_text(HARNESS)
    (d / "image").write_bytes(b"x")
    subprocess.run(["gcc", "-std=c11", "-O1", "-D__HIP_PLATFORM_AMD__", "-D_DEFAULT_SOURCE",
                    "-I" + os.path.join(ROOT, "turkce-llm_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                    "-I" + ROCM_INC, str(d / "h.c"), "-o", str(d / "h"), "-pthread"], check=True)

    def run(calls):
        out = subprocess.run([str(d / "h"), str(d / "image")] + [str(v) for c in calls for v in c], check=True,
                             capture_output=True, text=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]

    return run


SIZES = [1, 4 * KB, 128 * KB, 128 * KB + 1, MB, 2 * MB - 1, 2 * MB, 4 * MB + 5, 9 * MB]
ROWS = [(3, 10, 16), (64, 31769 * 4, 31772 * 4), (33, 100, 100), (5, 4 * MB + 4, 4 * MB + 16)]


def test_memory_the_runtime_knows_goes_direct(copies):
    calls = [(what, 1, n, 0, 0) for what in ("up", "down") for n in SIZES] + [("rows", 1, *r) for r in ROWS]
    for call, (ok, direct, other) in zip(calls, copies(calls)):
        assert ok and direct >= 1 and other == 0, (call, direct, other)


def test_pageable_memory_is_staged(copies):
    calls = [(what, 0, n, 0, 0) for what in ("up", "down") for n in SIZES] + [("rows", 0, *r) for r in ROWS]
    for call, (ok, direct, other) in zip(calls, copies(calls)):
        what, _, n = call[:3]
        staged = what == "rows" or n <= 128 * KB or (what == "down" and n >= 2 * MB)
        assert ok and (direct, other > 0) == ((0, True) if staged else (1, False)), (call, direct, other)
