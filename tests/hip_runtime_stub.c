/* A stand-in for the HIP runtime, for tests of libaxhip.so's host side without a GPU: loaded with RTLD_GLOBAL before the library, whose runtime calls
 * then come here.  It reports one gfx950 device of 256 CUs with `stub_free` bytes free, hands out addresses that nothing may touch, runs no kernel, notes
 * every launch, and refuses what the runtime refuses: allocations beyond what is free, and grids of 2^32 threads and more.  An error stays until
 * hipGetLastError is called, as ROCm 7 keeps it. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#define MOST 4096
typedef struct {
    char kernel[256];
    uint32_t grid[3], block[3];
    uint64_t shared, args[7];      /* of attention: Q, K, V, O, L, heads, sequence */
    int32_t order;                 /* and in which its tiles go out */
} Launch;
static Launch launches[MOST];
static int count;
static hipError_t sticky = hipSuccess;
static size_t left = (size_t)1 << 50;
static uintptr_t next_address = (uintptr_t)1 << 44;
static struct { uintptr_t at; size_t bytes; } held[MOST];
static struct { const void *host; char name[256]; } functions[MOST];
static int functions_n;
static struct { dim3 grid, block; size_t shared; hipStream_t stream; } pending;

static hipError_t note(hipError_t e) {
    if (e != hipSuccess) sticky = e;
    return e;
}

/* ---- for the test ---- */
void stub_set_free(size_t bytes) { left = bytes; }
int stub_launches(void) { return count; }
void stub_forget_launches(void) { count = 0; }
const Launch *stub_launch(int i) { return i >= 0 && i < count && i < MOST ? &launches[i] : NULL; }

/* ---- the runtime ---- */
void **__hipRegisterFatBinary(const void *data) {
    static void *handle;
    (void)data;
    return &handle;
}
void __hipUnregisterFatBinary(void **modules) { (void)modules; }
void __hipRegisterFunction(void **modules, const void *host, char *device, const char *name, unsigned limit, void *tid, void *bid, dim3 *block, dim3 *grid, int *size) {
    (void)modules, (void)device, (void)limit, (void)tid, (void)bid, (void)block, (void)grid, (void)size;
    if (functions_n == MOST) abort();
    functions[functions_n].host = host;
    strncpy(functions[functions_n++].name, name, 255);
}
void __hipRegisterVar(void **modules, void *var, char *host, char *device, int ext, size_t size, int constant, int global) {
    (void)modules, (void)var, (void)host, (void)device, (void)ext, (void)size, (void)constant, (void)global;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    pending.grid = grid, pending.block = block, pending.shared = shared, pending.stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
    *grid = pending.grid, *block = pending.block, *shared = pending.shared, *stream = pending.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *function, dim3 grid, dim3 block, void **args, size_t shared, hipStream_t stream) {
    (void)stream;
    const uint64_t most = (uint64_t)1 << 32;
    if (!grid.x || !grid.y || !grid.z || (uint64_t)block.x * block.y * block.z > 1024 || shared > 160 * 1024) return note(hipErrorInvalidConfiguration);
    if ((uint64_t)grid.x * block.x >= most || (uint64_t)grid.y * block.y >= most || (uint64_t)grid.z * block.z >= most) return note(hipErrorInvalidConfiguration);
    if (count < MOST) {
        Launch *l = &launches[count];
        memset(l, 0, sizeof *l);
        for (int i = 0; i < functions_n; i++)
            if (functions[i].host == function) memcpy(l->kernel, functions[i].name, sizeof l->kernel);
        l->grid[0] = grid.x, l->grid[1] = grid.y, l->grid[2] = grid.z;
        l->block[0] = block.x, l->block[1] = block.y, l->block[2] = block.z;
        l->shared = shared;
        for (int i = 0; i < 7 && strstr(l->kernel, "k_sdpa"); i++) memcpy(&l->args[i], args[i], 8);
        if (strstr(l->kernel, "k_sdpaI")) memcpy(&l->order, args[12], 4);
    }
    count++;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = sticky;
    sticky = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : e == hipErrorOutOfMemory ? "out of memory" : e == hipErrorInvalidConfiguration ? "invalid configuration" : "an error"; }
hipError_t hipMalloc(void **ptr, size_t bytes) {
    int i = 0;
    while (i < MOST && held[i].at) i++;
    if (bytes > left || i == MOST) return note(hipErrorOutOfMemory);
    left -= bytes;
    held[i].at = next_address, held[i].bytes = bytes;
    *ptr = (void *)next_address;
    next_address += (bytes + 4095) / 4096 * 4096;
    return hipSuccess;
}
hipError_t hipFree(void *ptr) {
    if (!ptr) return hipSuccess;
    for (int i = 0; i < MOST; i++)
        if (held[i].at == (uintptr_t)ptr) {
            left += held[i].bytes;
            held[i].at = 0;
            return hipSuccess;
        }
    return note(hipErrorInvalidValue);
}
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total) {
    *free_bytes = left, *total = (size_t)288 << 30;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) { return d == 0 ? hipSuccess : note(hipErrorInvalidDevice); }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *prop, int d) {
    (void)d;
    memset(prop, 0, sizeof *prop);
    strcpy(prop->gcnArchName, "gfx950:sramecc+:xnack-");
    prop->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **ptr, const void *symbol) {
    (void)symbol;
    *ptr = (void *)((uintptr_t)1 << 43);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *function, hipFuncAttribute attribute, int value) {
    (void)function, (void)attribute, (void)value;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) {
    (void)p, (void)v, (void)n;
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s) {
    (void)s;
    return hipMemset(p, v, n);
}
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind kind) {
    (void)to, (void)from, (void)n, (void)kind;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind kind, hipStream_t s) {
    (void)s;
    return hipMemcpy(to, from, n, kind);
}
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t)(uintptr_t)64;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    (void)e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    (void)e, (void)s;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    (void)e;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
    (void)a, (void)b;
    *ms = 0.0f;
    return hipSuccess;
}
