/* The HIP runtime calls of the library on the host, for tests of its host code without a GPU:
 * device memory is host memory, kernels do nothing, and any allocation can be made to fail.
 * Copies and fills that leave a live device allocation are counted, not done. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;
#define MAX 4096
static struct { char* p; size_t n; } block[MAX];
static long allocs, fail_at = -1, outside, live;

static void* add(size_t n)
{
    for (int i = 0; i < MAX; ++i)
        if (!block[i].p) {
            block[i].n = n;
            ++live;
            return block[i].p = calloc(1, n ? n : 1);
        }
    abort();
}
static int inside(const void* q, size_t n)
{
    const char* p = q;
    for (int i = 0; i < MAX; ++i)
        if (block[i].p && p >= block[i].p && p + n <= block[i].p + block[i].n) return 1;
    ++outside;
    return 0;
}
static int drop(void* p)
{
    for (int i = 0; p && i < MAX; ++i)
        if (block[i].p == p) { free(p); block[i].p = 0; --live; return 0; }
    if (p) ++outside;
    return 0;
}

void stub_fail(long k) { fail_at = k < 0 ? -1 : allocs + k; }   /* the k-th hipMalloc from here */
long stub_outside(void) { return outside; }
long stub_live(void) { return live; }

int hipMalloc(void** p, size_t n)
{
    if (allocs++ == fail_at) { *p = 0; return 2; }
    *p = add(n);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; *p = add(n); return 0; }
int hipFree(void* p) { return drop(p); }
int hipHostFree(void* p) { return drop(p); }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st)
{
    (void)st;
    if (n == 0) return 0;
    const int ok = (kind == 2 || inside(d, n)) & (kind == 1 || inside(s, n));   /* 1: to, 2: from the device */
    if (ok) memmove(d, s, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* st)
{
    (void)st;
    if (inside(d, n)) memset(d, v, n);
    return 0;
}
int hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** a, size_t s, void* st)
{
    (void)f; (void)g; (void)b; (void)a; (void)s; (void)st;
    return 0;
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t s, void* st) { (void)g; (void)b; (void)s; (void)st; return 0; }
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* s, void** st)
{
    const dim3_t one = {1, 1, 1};
    *g = one; *b = one; *s = 0; *st = 0;
    return 0;
}
int hipSetDevice(int d) { (void)d; return 0; }
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { (void)e; return "stub"; }
int hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; *s = add(1); return 0; }
int hipStreamSynchronize(void* s) { (void)s; return 0; }
int hipStreamDestroy(void* s) { return drop(s); }
int hipEventCreate(void** e) { *e = add(1); return 0; }
int hipEventDestroy(void* e) { return drop(e); }
int hipEventRecord(void* e, void* s) { (void)e; (void)s; return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 1.f; return 0; }
