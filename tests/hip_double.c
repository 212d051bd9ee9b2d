/* A double of the HIP runtime for tests of the library's host code without a
 * device: memory is the host's, copies are memcpy, launches do nothing.
 * hip_double_fail(name, after, code): the call of `name` after the next `after`
 * ones returns `code`. */
#include <stdlib.h>
#include <string.h>

static char fail_name[64];
static int fail_after = -1, fail_code;

void hip_double_fail(const char* name, int after, int code) {
    strncpy(fail_name, name, sizeof(fail_name) - 1);
    fail_after = after;
    fail_code = code;
}

/* How many calls the failure is still away (-1: it has been). */
int hip_double_left(void) { return fail_after; }

static int status(const char* name) {
    return fail_after >= 0 && strcmp(name, fail_name) == 0 && fail_after-- == 0 ? fail_code : 0;
}

static int handle(const char* name, void** p) {
    *p = (void*)name;
    return status(name);
}

static int allocate(const char* name, void** p, size_t bytes) {
    const int s = status(name);
    *p = s == 0 ? calloc(1, bytes) : NULL;
    return s;
}

static int release(void* p) {
    free(p);
    return 0;
}

static int copy(const char* name, void* d, const void* s, size_t bytes) {
    memcpy(d, s, bytes);
    return status(name);
}

static int set(int* v, int to) {
    *v = to;
    return 0;
}

#define HANDLE(name, ...) int name(void** p, ##__VA_ARGS__) { return handle(#name, p); }
#define PLAIN(name, ...) int name(__VA_ARGS__) { return status(#name); }

HANDLE(hipEventCreate)
HANDLE(hipEventCreateWithFlags, unsigned f)
HANDLE(hipStreamCreateWithFlags, unsigned f)
PLAIN(hipEventDestroy, void* e)
PLAIN(hipEventRecord, void* e, void* s)
PLAIN(hipEventSynchronize, void* e)
PLAIN(hipStreamDestroy, void* s)
PLAIN(hipStreamQuery, void* s)
PLAIN(hipStreamSynchronize, void* s)
PLAIN(hipGetLastError, void)
PLAIN(hipSetDevice, int d)
int hipMalloc(void** p, size_t n) { return allocate("hipMalloc", p, n); }
int hipHostMalloc(void** p, size_t n, unsigned f) { return allocate("hipHostMalloc", p, n); }
int hipFree(void* p) { return release(p); }
int hipHostFree(void* p) { return release(p); }
int hipMemcpy(void* d, const void* s, size_t n, int k) { return copy("hipMemcpy", d, s, n); }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* t) {
    return copy("hipMemcpyAsync", d, s, n);
}
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return status("hipMemset"); }
int hipMemsetAsync(void* d, int v, size_t n, void* t) {
    memset(d, v, n);
    return status("hipMemsetAsync");
}
int hipGetDevice(int* d) { return set(d, 0); }
int hipGetDeviceCount(int* n) { return set(n, 1); }
int hipDeviceGetAttribute(int* v, int a, int d) { return set(v, 256); }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int b, size_t l) {
    return set(n, 1);
}
int hipGetDevicePropertiesR0600(void* p, int d) {
    memset(p, 0, 1472);   /* sizeof(hipDeviceProp_t) */
    return 0;
}
int hipEventElapsedTime(float* ms, void* a, void* b) {
    *ms = 1.0f;
    return status("hipEventElapsedTime");
}
const char* hipGetErrorString(int e) { return e == 0 ? "no error" : "an error"; }
/* not offered: pointer attributes, symbols, graphs */
#define ABSENT(name) int name(void) { return 1; }
ABSENT(hipPointerGetAttributes)
ABSENT(hipMemGetAddressRange)
ABSENT(hipGetSymbolAddress)
ABSENT(hipStreamBeginCapture)
ABSENT(hipStreamEndCapture)
ABSENT(hipGraphDestroy)
ABSENT(hipGraphExecDestroy)
ABSENT(hipGraphInstantiate)
ABSENT(hipGraphLaunch)
/* launches */
struct dims { unsigned x, y, z; };
int __hipPushCallConfiguration(struct dims g, struct dims b, size_t l, void* s) { return 0; }
int __hipPopCallConfiguration(struct dims* g, struct dims* b, size_t* l, void** s) {
    memset(g, 0, sizeof(*g));
    memset(b, 0, sizeof(*b));
    *l = 0;
    *s = NULL;
    return 0;
}
int hipLaunchKernel(const void* f, struct dims g, struct dims b, void** a, size_t l, void* s) {
    return status("hipLaunchKernel");
}
void** __hipRegisterFatBinary(const void* data) {
    static void* module;
    return &module;
}
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}
void __hipUnregisterFatBinary(void** m) {}
