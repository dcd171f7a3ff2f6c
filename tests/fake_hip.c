/* A HIP runtime without a GPU, for tests of the host code in libvpbs: device memory is host memory (zeroed),
 * kernels are counted and not run, and allocations can be made to fail. Loaded with RTLD_GLOBAL before
 * libvpbs, whose calls then come here. One thread at a time. */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { SUCCESS = 0, INVALID_VALUE = 1, OUT_OF_MEMORY = 2, MAX_BLOCKS = 4096, MAX_KERNELS = 8192 };

static struct {
    void *p;
    size_t bytes;
} blocks[MAX_BLOCKS];
static int nblocks;
static long mallocs;            /* hipMalloc calls */
static long fail_at = -1;       /* the call that fails, counted from 1 */
static const char *fail_call;   /* or any call of this name */
static int last_error;

static struct {
    const void *host;
    char *name;
    long launches;
} kernels[MAX_KERNELS];
static int nkernels;

/* Control, called by the tests. */
long fake_mallocs(void) { return mallocs; }
void fake_fail_malloc(long n) { fail_at = n > 0 ? mallocs + n : -1; }
void fake_fail_call(const char *name) {
    free((void *)fail_call);
    fail_call = name ? strdup(name) : NULL;
}
int fake_blocks(size_t *bytes, int max) {
    for (int i = 0; i < nblocks && i < max; i++) bytes[i] = blocks[i].bytes;
    return nblocks;
}
long fake_launches(const char *part) { /* of kernels with this in their (mangled) name */
    long n = 0;
    for (int i = 0; i < nkernels; i++)
        if (strstr(kernels[i].name, part)) n += kernels[i].launches;
    return n;
}

static int result(const char *name) {
    if (fail_call && !strcmp(fail_call, name)) return last_error = INVALID_VALUE;
    return SUCCESS;
}

int hipMalloc(void **p, size_t n) {
    mallocs++;
    if (mallocs == fail_at || nblocks == MAX_BLOCKS || !(*p = calloc(1, n ? n : 1))) return last_error = OUT_OF_MEMORY;
    blocks[nblocks].p = *p;
    blocks[nblocks++].bytes = n;
    return SUCCESS;
}
int hipFree(void *p) {
    if (!p) return SUCCESS;
    for (int i = 0; i < nblocks; i++)
        if (blocks[i].p == p) {
            blocks[i] = blocks[--nblocks];
            free(p);
            return SUCCESS;
        }
    return last_error = INVALID_VALUE; /* not allocated, or freed before */
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    (void)flags;
    return (*p = calloc(1, n)) ? SUCCESS : OUT_OF_MEMORY;
}
int hipHostFree(void *p) {
    free(p);
    return SUCCESS;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned flags) {
    (void)flags;
    *d = h;
    return result("hipHostGetDevicePointer");
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
    (void)kind;
    if (n && (!d || !s)) return last_error = INVALID_VALUE;
    memmove(d, s, n);
    return SUCCESS;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) {
    (void)stream;
    return hipMemcpy(d, s, n, kind);
}
int hipMemset(void *d, int v, size_t n) {
    if (n && !d) return last_error = INVALID_VALUE;
    memset(d, v, n);
    return SUCCESS;
}
int hipMemsetAsync(void *d, int v, size_t n, void *stream) {
    (void)stream;
    return hipMemset(d, v, n);
}
int hipGetSymbolAddress(void **p, const void *symbol) {
    static char memory[(size_t)64 << 20];
    (void)symbol;
    *p = memory;
    return SUCCESS;
}
int hipPointerGetAttributes(void *attributes, const void *p) {
    (void)attributes, (void)p;
    return last_error = INVALID_VALUE; /* ordinary memory */
}

int hipGetDeviceCount(int *n) {
    *n = 1;
    return SUCCESS;
}
int hipSetDevice(int device) {
    (void)device;
    return SUCCESS;
}
int hipDeviceGetAttribute(int *v, int attribute, int device) {
    (void)attribute, (void)device;
    *v = 160 * 1024;
    return SUCCESS;
}
int hipFuncSetAttribute(const void *f, int attribute, int v) {
    (void)f, (void)attribute, (void)v;
    return SUCCESS;
}
const char *hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : e ? "invalid value" : "success"; }
int hipGetLastError(void) {
    const int e = last_error;
    last_error = SUCCESS;
    return e;
}

int hipStreamCreateWithFlags(void **s, unsigned flags) {
    (void)flags;
    return (*s = malloc(1)) ? SUCCESS : OUT_OF_MEMORY;
}
int hipStreamDestroy(void *s) {
    free(s);
    return SUCCESS;
}
int hipStreamSynchronize(void *s) {
    (void)s;
    return SUCCESS;
}
int hipStreamWaitEvent(void *s, void *e, unsigned flags) {
    (void)s, (void)e, (void)flags;
    return SUCCESS;
}
int hipEventCreateWithFlags(void **e, unsigned flags) { return hipStreamCreateWithFlags(e, flags); }
int hipEventDestroy(void *e) { return hipStreamDestroy(e); }
int hipEventRecord(void *e, void *s) {
    (void)e, (void)s;
    return SUCCESS;
}
int hipEventElapsedTime(float *ms, void *a, void *b) {
    (void)a, (void)b;
    *ms = 1.0f;
    return SUCCESS;
}

/* Kernels: what the compiler's launch stubs and module initialisers call. */
typedef struct {
    uint32_t x, y, z;
} dim3_t;
static dim3_t push_grid, push_block;
static size_t push_lds;
static void *push_stream;
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void *stream) {
    push_grid = grid, push_block = block, push_lds = lds, push_stream = stream;
    return SUCCESS;
}
int __hipPopCallConfiguration(dim3_t *grid, dim3_t *block, size_t *lds, void **stream) {
    *grid = push_grid, *block = push_block, *lds = push_lds, *stream = push_stream;
    return SUCCESS;
}
int hipLaunchKernel(const void *f, dim3_t grid, dim3_t block, void **args, size_t lds, void *stream) {
    (void)args, (void)lds, (void)stream;
    if (!grid.x || !grid.y || !grid.z || !block.x) return last_error = INVALID_VALUE;
    for (int i = 0; i < nkernels; i++)
        if (kernels[i].host == f) kernels[i].launches++;
    return result("hipLaunchKernel");
}
void **__hipRegisterFatBinary(const void *data) {
    static void *module;
    (void)data;
    return &module;
}
void __hipUnregisterFatBinary(void **module) { (void)module; }
void __hipRegisterFunction(void **module, const void *host, char *device, const char *name, unsigned threads, void *tid,
                           void *bid, void *block, void *grid, int *wave) {
    (void)module, (void)device, (void)threads, (void)tid, (void)bid, (void)block, (void)grid, (void)wave;
    if (nkernels == MAX_KERNELS) abort();
    kernels[nkernels].host = host;
    kernels[nkernels++].name = strdup(name);
}
void __hipRegisterVar(void **module, void *var, char *host, char *device, int ext, size_t size, int constant, int global) {
    (void)module, (void)var, (void)host, (void)device, (void)ext, (void)size, (void)constant, (void)global;
}

/* rocFFT: the fused transforms only set it up. */
int rocfft_setup(void) { return 0; }
