/* hip_backend.c -- HIP module-API backend (see include/hip_backend.h).
 *
 * Role of cuda/cuda_backend.c (cuda_backend.c:15-161): fatal error check,
 * kernel image load, allocation, synchronous copies and launch helpers.
 */
#include "hip_backend.h"

#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#define STAGE_BLOCK (4ull << 20)   /* bytes of each of a context's two staging buffers */

struct HipAllocList {
    pthread_mutex_t lock;
    void** ptrs;
    u64 count;
    u64 cap;
    void* image;   /* the loaded code object's bytes, owned until hip_shutdown */
    pthread_mutex_t stage_lock;   /* held by a copy from its first use of stage to its last */
    u8* stage[2];  /* pinned, STAGE_BLOCK bytes each, freed by hip_shutdown */
};

struct HipSide {
    hipStream_t stream;
    hipEvent_t fork, join;
    hipEvent_t mark[HIP_SIDE_MARKS];
    i32 active;
};

static _Thread_local HipCtx* tls_ctx = NULL;

static void fatal_exit(void) {
    fflush(stdout);
    fflush(stderr);
    _exit(1);
}

/* Same convention as the reference (cuda_backend.c:23-34): name what failed,
 * the error's name and description, and end the process. */
static void check(hipError_t r, const char* what) {
    if (r != hipSuccess) {
        fprintf(stderr, "[HIP ERROR] %s -> %s: %s\n", what, hipGetErrorName(r), hipGetErrorString(r));
        fatal_exit();
    }
}

/* The code object is read into memory the context owns and keeps until
 * hip_shutdown has unloaded the module: the HSA loader may keep referring to
 * the bytes a code object was loaded from (a reader created from memory
 * must outlive the loaded object), so they must not live in an arena the
 * caller may reset or free while the module is loaded. */
static void* read_image(const char* path, u64* out_size) {
    FILE* f = fopen(path, "rb");
    if (!f) {
        fprintf(stderr, "[HIP ERROR] cannot open kernel image: %s\n", path);
        fatal_exit();
    }
    fseek(f, 0, SEEK_END);
    long size = ftell(f);
    fseek(f, 0, SEEK_SET);
    u8* buf = (u8*)malloc((size_t)size + 1);
    if (!buf) {
        fprintf(stderr, "[HIP ERROR] out of host memory for kernel image: %s\n", path);
        fatal_exit();
    }
    size_t got = fread(buf, 1, (size_t)size, f);
    fclose(f);
    if (got != (size_t)size) {
        fprintf(stderr, "[HIP ERROR] short read of kernel image: %s\n", path);
        fatal_exit();
    }
    buf[size] = 0;
    *out_size = (u64)size;
    return buf;
}

HipCtx hip_init_on_device(Allocator* scratch, const char* image_path, i32 device_index) {
    HipCtx c;
    memset(&c, 0, sizeof(c));
    i32 count = 0;
    check(hipGetDeviceCount(&count), "hipGetDeviceCount");
    if (count < 1) {
        fprintf(stderr, "[HIP ERROR] no HIP device found\n");
        fatal_exit();
    }
    if (device_index < 0 || device_index >= count) {
        fprintf(stderr, "[HIP ERROR] device index %d exceeds the %d visible devices\n", device_index, count);
        fatal_exit();
    }
    c.device = device_index;
    check(hipSetDevice(device_index), "hipSetDevice");
    (void)scratch;   /* the reference reads the image into it; here the context owns the bytes */
    u64 size;
    void* image = read_image(image_path, &size);
    check(hipModuleLoadData(&c.module, image), "hipModuleLoadData");
    check(hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking), "hipStreamCreateWithFlags");
    c.allocs = (HipAllocList*)calloc(1, sizeof(HipAllocList));
    pthread_mutex_init(&c.allocs->lock, NULL);
    pthread_mutex_init(&c.allocs->stage_lock, NULL);
    c.allocs->image = image;
    for (int i = 0; i < 2; i++)
        check(hipHostMalloc((void**)&c.allocs->stage[i], STAGE_BLOCK, hipHostMallocDefault), "hipHostMalloc");
    return c;
}

HipCtx hip_init(Allocator* scratch, const char* image_path) {
    return hip_init_on_device(scratch, image_path, 0);
}

i32 hip_device_count(void) {
    i32 count = 0;
    check(hipGetDeviceCount(&count), "hipGetDeviceCount");
    return count;
}

void hip_shutdown(HipCtx* c) {
    if (!c->allocs) return;
    check(hipSetDevice(c->device), "hipSetDevice");
    check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
    if (c->side) check(hipStreamSynchronize(c->side->stream), "hipStreamSynchronize");
    for (u64 i = 0; i < c->allocs->count; i++)
        if (c->allocs->ptrs[i]) check(hipFree(c->allocs->ptrs[i]), "hipFree");
    void* image = c->allocs->image;
    free(c->allocs->ptrs);
    for (int i = 0; i < 2; i++)
        check(hipHostFree(c->allocs->stage[i]), "hipHostFree");
    pthread_mutex_destroy(&c->allocs->lock);
    pthread_mutex_destroy(&c->allocs->stage_lock);
    free(c->allocs);
    c->allocs = NULL;
    if (c->side) {
        check(hipStreamSynchronize(c->side->stream), "hipStreamSynchronize");
        for (i32 i = 0; i < HIP_SIDE_MARKS; i++) check(hipEventDestroy(c->side->mark[i]), "hipEventDestroy");
        check(hipEventDestroy(c->side->fork), "hipEventDestroy");
        check(hipEventDestroy(c->side->join), "hipEventDestroy");
        check(hipStreamDestroy(c->side->stream), "hipStreamDestroy");
        free(c->side);
        c->side = NULL;
    }
    check(hipStreamDestroy(c->stream), "hipStreamDestroy");
    check(hipModuleUnload(c->module), "hipModuleUnload");
    free(image);
    if (tls_ctx == c) tls_ctx = NULL;
}

void hip_set_current(HipCtx* c) {
    check(hipSetDevice(c->device), "hipSetDevice");
    tls_ctx = c;
}

static HipCtx* current(const char* what) {
    if (!tls_ctx) {
        fprintf(stderr, "[HIP ERROR] %s: no context is current on this thread\n", what);
        fatal_exit();
    }
    return tls_ctx;
}

hipStream_t hip_current_stream(void) { return current("hip_current_stream")->stream; }

u32 hip_cu_count(void) {
    int n = 0;
    check(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, current("hip_cu_count")->device),
          "hipDeviceGetAttribute(multiprocessor count)");
    return (u32)n;
}

u32 hip_blocks_per_cu(hipFunction_t f, u32 block_threads) {
    int n = 0;
    check(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, (int)block_threads, 0),
          "hipModuleOccupancyMaxActiveBlocksPerMultiprocessor");
    return (u32)n;
}

hipFunction_t hip_get_kernel(HipCtx* c, const char* name) {
    hipFunction_t f;
    hipError_t r = hipModuleGetFunction(&f, c->module, name);
    if (r != hipSuccess) {
        fprintf(stderr, "[HIP ERROR] hipModuleGetFunction(%s) -> %s: %s\n", name, hipGetErrorName(r),
                hipGetErrorString(r));
        fatal_exit();
    }
    return f;
}

hipDeviceptr_t hip_alloc(u64 bytes) {
    HipCtx* c = current("hip_alloc");
    void* p = NULL;
    check(hipMalloc(&p, bytes ? bytes : 4), "hipMalloc");
    HipAllocList* l = c->allocs;
    pthread_mutex_lock(&l->lock);
    if (l->count == l->cap) {
        l->cap = l->cap ? l->cap * 2 : 256;
        l->ptrs = (void**)realloc(l->ptrs, l->cap * sizeof(void*));
    }
    l->ptrs[l->count++] = p;
    pthread_mutex_unlock(&l->lock);
    return p;
}

void hip_free(hipDeviceptr_t p) {
    HipCtx* c = current("hip_free");
    HipAllocList* l = c->allocs;
    pthread_mutex_lock(&l->lock);
    for (u64 i = l->count; i-- > 0;) {
        if (l->ptrs[i] == p) { l->ptrs[i] = l->ptrs[--l->count]; break; }
    }
    pthread_mutex_unlock(&l->lock);
    check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
    if (c->side) check(hipStreamSynchronize(c->side->stream), "hipStreamSynchronize");
    check(hipFree(p), "hipFree");
}

/* Small and large host copies of pageable memory go through pinned staging of
 * the context's own: one to or from pageable memory costs the runtime far more than its bytes.
 * Measured on MI355X, direct -> staged: upload of 4 KB 14 -> 13 us, 64 KB 33
 * -> 10; download of 4 KB 22 -> 11, 64 KB 37 -> 11, 16 MB of padded rows 1600
 * -> 302 and the copy out of the staging, which host threads share (fresh
 * pages fault at 0.8 us each, in parallel).  A 128-token prompt's 16 MB of
 * logits 2.55 -> 1.6 ms in all, 64 rows of a decoder's logits (one copy, where
 * each row was one) 1.2 ms less.  Between STAGED_SMALL and COPY_THREADED a
 * loop over one buffer is faster staged too (192 KB: upload 84 -> 16 us), but
 * the matmul node with its operands and results in a fresh arena is slower
 * (128x384x1024: 730 us of copies and products direct, 855 staged), and large
 * uploads cost as much either way (16 MB 598 / 721 us): those go direct. */
#define STAGED_SMALL (128ull << 10)
#define COPY_THREADED (2ull << 20)     /* below it one host thread copies out */
#define COPY_MIN_PART (512ull << 10)   /* a host thread's share at least */
#define COPY_THREADS 8

static u8** stage_acquire(HipCtx* c) {
    pthread_mutex_lock(&c->allocs->stage_lock);
    return c->allocs->stage;
}

static void stage_release(HipCtx* c) { pthread_mutex_unlock(&c->allocs->stage_lock); }

/* Memory that the runtime does not know.  What it knows (pinned, managed or
 * device memory) a transfer reaches by itself: pinned downloads of 2 MB 87 ->
 * 45 us, 16 MB 518 -> 303, 16 MB of padded rows 513 -> 293 against staging
 * them too.  And the host must not touch device memory.  The question costs
 * 0.1 us. */
static int pageable(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();   /* no error of the caller's */
    return 1;
}

/* Bytes [from, to) of packed rows of row_bytes, from staged rows `pitch` apart. */
typedef struct CopyPart { u8* dst; const u8* src; u64 from, to, row_bytes, pitch; } CopyPart;

static void* copy_part(void* arg) {
    const CopyPart* c = (const CopyPart*)arg;
    for (u64 o = c->from; o < c->to;) {
        const u64 r = o / c->row_bytes, at = o % c->row_bytes;
        u64 n = c->row_bytes - at;
        if (n > c->to - o) n = c->to - o;
        memcpy(c->dst + o, c->src + r * c->pitch + at, n);
        o += n;
    }
    return NULL;
}

static void copy_rows(u8* dst, const u8* src, u64 pitch, u64 row_bytes, u64 rows) {
    const u64 bytes = rows * row_bytes;
    u64 nt = bytes < COPY_THREADED ? 1 : bytes / COPY_MIN_PART;
    if (nt > COPY_THREADS) nt = COPY_THREADS;
    const u64 per = ((bytes + nt - 1) / nt + 63) & ~63ull;
    CopyPart part[COPY_THREADS];
    pthread_t th[COPY_THREADS];
    int started[COPY_THREADS];
    for (u64 i = 0; i < nt; i++) {
        const u64 from = i * per < bytes ? i * per : bytes;
        part[i] = (CopyPart){ dst, src, from, from + per < bytes ? from + per : bytes, row_bytes, pitch };
        started[i] = i > 0 && pthread_create(&th[i], NULL, copy_part, &part[i]) == 0;
    }
    copy_part(&part[0]);
    for (u64 i = 1; i < nt; i++) {
        if (started[i]) pthread_join(th[i], NULL);
        else copy_part(&part[i]);
    }
}

void hip_h2d(hipDeviceptr_t dst, const void* src, u64 bytes) {
    HipCtx* c = current("hip_h2d");
    /* no host address: the runtime's error */
    const int staged = src && bytes > 0 && bytes <= STAGED_SMALL && pageable(src);
    if (staged) {
        u8* stage = stage_acquire(c)[0];
        memcpy(stage, src, bytes);
        src = stage;
    }
    check(hipMemcpyHtoDAsync(dst, (void*)src, bytes, c->stream), "hipMemcpyHtoDAsync");
    check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
    if (staged) stage_release(c);
}

/* `rows` rows of at most STAGE_BLOCK bytes, `block` rows to a staging block:
 * one block's transfer runs while the one before it is copied out. */
static void d2h_blocks(HipCtx* c, u8* dst, const u8* src, u64 pitch, u64 row_bytes, u64 rows, u64 block) {
    u8** stage = stage_acquire(c);
    u64 n = 0, done = 0;   /* rows of the block in flight; rows before it */
    for (u64 i = 0;; i++) {
        const u64 at = done + n, next = rows - at < block ? rows - at : block;
        if (n || !next) check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
        if (next)
            check(hipMemcpyDtoHAsync(stage[i & 1], (hipDeviceptr_t)(src + at * pitch),
                                     (next - 1) * pitch + row_bytes, c->stream), "hipMemcpyDtoHAsync");
        if (n) copy_rows(dst + done * row_bytes, stage[(i & 1) ^ 1], pitch, row_bytes, n);
        if (!next) break;
        done = at;
        n = next;
    }
    stage_release(c);
}

void hip_d2h(void* dst, hipDeviceptr_t src, u64 bytes) {
    HipCtx* c = current("hip_d2h");
    if (!dst || (bytes > STAGED_SMALL && bytes < COPY_THREADED) || !pageable(dst)) {
        check(hipMemcpyDtoHAsync(dst, src, bytes, c->stream), "hipMemcpyDtoHAsync");
        check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
        return;
    }
    const u64 whole = bytes / STAGE_BLOCK, rest = bytes % STAGE_BLOCK;
    if (whole || !rest) d2h_blocks(c, (u8*)dst, (const u8*)src, STAGE_BLOCK, STAGE_BLOCK, whole, 1);
    if (rest) d2h_blocks(c, (u8*)dst + (bytes - rest), (const u8*)src + (bytes - rest), rest, rest, 1, 1);
}

void hip_d2h_rows(void* dst, hipDeviceptr_t src, u64 pitch, u64 row_bytes, u64 rows) {
    HipCtx* c = current("hip_d2h_rows");
    if (dst && pitch > row_bytes && row_bytes > 0 && rows > 0 && !pageable(dst)) {
        check(hipMemcpy2DAsync(dst, row_bytes, src, pitch, row_bytes, rows, hipMemcpyDeviceToHost, c->stream),
              "hipMemcpy2DAsync");
        check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
    } else if (dst && pitch <= STAGE_BLOCK && pitch > row_bytes && row_bytes > 0) {
        d2h_blocks(c, (u8*)dst, (const u8*)src, pitch, row_bytes, rows, STAGE_BLOCK / pitch);
    } else if (pitch == row_bytes) {
        hip_d2h(dst, src, rows * row_bytes);
    } else {
        for (u64 r = 0; r < rows; r++)
            hip_d2h(dst ? (u8*)dst + r * row_bytes : NULL, (hipDeviceptr_t)((u8*)src + r * pitch), row_bytes);
    }
}

void hip_launch(hipFunction_t f, u32 gx, u32 gy, u32 gz, u32 bx, u32 by, u32 bz, u32 shared_bytes,
                void** params) {
    HipCtx* c = current("hip_launch");
    if (gx == 0 || gy == 0 || gz == 0) return;
    hipStream_t st = (c->side && c->side->active) ? c->side->stream : c->stream;
    check(hipModuleLaunchKernel(f, gx, gy, gz, bx, by, bz, shared_bytes, st, params, NULL),
          "hipModuleLaunchKernel");
}

static int side_serial;

void hip_side_serial(i32 on) { side_serial = on != 0; }

void hip_side_begin(void) {
    HipCtx* c = current("hip_side_begin");
    if (side_serial) return;
    if (!c->side) {
        HipSide* s = (HipSide*)calloc(1, sizeof(HipSide));
        check(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking), "hipStreamCreateWithFlags");
        check(hipEventCreateWithFlags(&s->fork, hipEventDisableTiming), "hipEventCreateWithFlags");
        check(hipEventCreateWithFlags(&s->join, hipEventDisableTiming), "hipEventCreateWithFlags");
        for (i32 i = 0; i < HIP_SIDE_MARKS; i++)
            check(hipEventCreateWithFlags(&s->mark[i], hipEventDisableTiming), "hipEventCreateWithFlags");
        c->side = s;
    }
    check(hipEventRecord(c->side->fork, c->stream), "hipEventRecord");
    check(hipStreamWaitEvent(c->side->stream, c->side->fork, 0), "hipStreamWaitEvent");
    c->side->active = 1;
}

static void check_mark(i32 mark, const char* what) {
    if (mark < 0 || mark >= HIP_SIDE_MARKS) {
        fprintf(stderr, "[HIP ERROR] %s: side mark %d out of range\n", what, mark);
        fatal_exit();
    }
}

void hip_side_end(i32 mark) {
    HipCtx* c = current("hip_side_end");
    check_mark(mark, "hip_side_end");
    if (side_serial) return;
    if (!c->side || !c->side->active) {
        fprintf(stderr, "[HIP ERROR] hip_side_end without hip_side_begin\n");
        fatal_exit();
    }
    check(hipEventRecord(c->side->mark[mark], c->side->stream), "hipEventRecord");
    c->side->active = 0;
}

void hip_main_wait(i32 mark) {
    HipCtx* c = current("hip_main_wait");
    check_mark(mark, "hip_main_wait");
    if (side_serial || !c->side) return;   /* no side stream, or nothing queued on it */
    check(hipStreamWaitEvent(c->stream, c->side->mark[mark], 0), "hipStreamWaitEvent");
}

void hip_side_join(void) {
    HipCtx* c = current("hip_side_join");
    if (!c->side) return;
    check(hipEventRecord(c->side->join, c->side->stream), "hipEventRecord");
    check(hipStreamWaitEvent(c->stream, c->side->join, 0), "hipStreamWaitEvent");
}

#define BLOCK_1D 256u

void hip_launch_1d(hipFunction_t f, u32 n, void** params) {
    hip_launch(f, (n + BLOCK_1D - 1) / BLOCK_1D, 1, 1, BLOCK_1D, 1, 1, 0, params);
}

void hip_launch_1d_shared(hipFunction_t f, u32 n, u32 block_size, u32 shared_bytes, void** params) {
    hip_launch(f, (n + block_size - 1) / block_size, 1, 1, block_size, 1, 1, shared_bytes, params);
}

#define BLOCK_2D 16u

void hip_launch_2d(hipFunction_t f, u32 rows, u32 cols, void** params) {
    hip_launch(f, (cols + BLOCK_2D - 1) / BLOCK_2D, (rows + BLOCK_2D - 1) / BLOCK_2D, 1, BLOCK_2D, BLOCK_2D, 1,
               0, params);
}

void hip_memset_zero(hipDeviceptr_t p, u64 bytes) {
    HipCtx* c = current("hip_memset_zero");
    check(hipMemsetD8Async(p, 0, bytes, c->stream), "hipMemsetD8Async");
}

void hip_sync(void) {
    HipCtx* c = current("hip_sync");
    check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
    if (c->side) check(hipStreamSynchronize(c->side->stream), "hipStreamSynchronize");
}
