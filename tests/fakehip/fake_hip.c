/* A HIP runtime without a device, for CPU tests of the host library: memory is
 * host memory, copies and clears are done at once, kernels do nothing.  It
 * records every launch (kernel name, grid, first argument) and can refuse the
 * n-th allocation from now.  Loaded with RTLD_GLOBAL before libamrgpu.so, whose
 * runtime calls then come here (tests/fake_hip.py).
 */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef int err_t;                       /* hipError_t */
enum { OK = 0, OUT_OF_MEMORY = 2 };
typedef struct { unsigned x, y, z; } dim3;

/* ---- what the tests read and set ---- */
enum { MAXK = 4096, MAXL = 65536 };
static struct { const void* f; const char* name; } kern[MAXK];
static struct { const char* name; unsigned grid; uint64_t arg0; } rec[MAXL];
static int nkern, nrec, nalloc[2], nfail[2], live[2];

void fake_clear(void) { nrec = 0; }
int fake_launches(void) { return nrec; }
const char* fake_name(int i) { return rec[i].name; }
unsigned fake_grid(int i) { return rec[i].grid; }
uint64_t fake_arg0(int i) { return rec[i].arg0; }
/* kind 0: device, 1: pinned; refuse the n-th allocation from now (0: none) */
void fake_refuse(int kind, int n) { nfail[kind] = n; }
int fake_allocs(int kind) { return nalloc[kind]; }
int fake_live(int kind) { return live[kind]; }

/* ---- memory ---- */
static err_t get(int kind, void** p, size_t n) {
    nalloc[kind]++;
    if (nfail[kind] > 0 && --nfail[kind] == 0) { *p = NULL; return OUT_OF_MEMORY; }
    *p = calloc(1, n ? n : 1);
    live[kind]++;
    return OK;
}
static err_t put(int kind, void* p) {
    if (p) live[kind]--;
    free(p);
    return OK;
}
err_t hipMalloc(void** p, size_t n) { return get(0, p, n); }
err_t hipHostMalloc(void** p, size_t n, unsigned flags) { (void)flags; return get(1, p, n); }
err_t hipFree(void* p) { return put(0, p); }
err_t hipHostFree(void* p) { return put(1, p); }
err_t hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) {
    (void)kind; (void)st;
    if (n) memcpy(d, s, n);
    return OK;
}
err_t hipMemsetAsync(void* d, int v, size_t n, void* st) {
    (void)st;
    if (n) memset(d, v, n);
    return OK;
}
err_t hipGetSymbolAddress(void** p, const void* sym) {
    static void* m;
    (void)sym;
    if (!m) m = calloc(1, 1 << 20);
    *p = m;
    return OK;
}

/* ---- launches ---- */
static struct { dim3 g, b; size_t sh; void* st; } conf;
void** __hipRegisterFatBinary(const void* d) { static void* h; (void)d; return &h; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterVar(void** m, void* v, char* h, char* n, int e, size_t s, int c, int g) {
    (void)m; (void)v; (void)h; (void)n; (void)e; (void)s; (void)c; (void)g;
}
void __hipRegisterFunction(void** m, const void* f, char* dn, const char* name, unsigned t, void* a,
                           void* b, void* c, void* d, int* w) {
    (void)m; (void)dn; (void)t; (void)a; (void)b; (void)c; (void)d; (void)w;
    if (nkern < MAXK) { kern[nkern].f = f; kern[nkern++].name = name; }
}
err_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, void* st) {
    conf.g = g; conf.b = b; conf.sh = sh; conf.st = st;
    return OK;
}
err_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, void** st) {
    *g = conf.g; *b = conf.b; *sh = conf.sh; *st = conf.st;
    return OK;
}
err_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t sh, void* st) {
    (void)b; (void)sh; (void)st;
    if (nrec < MAXL) {
        int k = 0;
        while (k < nkern && kern[k].f != f) k++;
        rec[nrec].name = k < nkern ? kern[k].name : "?";
        rec[nrec].grid = g.x;
        rec[nrec].arg0 = 0;
        memcpy(&rec[nrec].arg0, args[0], 8);
        nrec++;
    }
    return OK;
}
err_t hipFuncSetAttribute(const void* f, int a, int v) { (void)f; (void)a; (void)v; return OK; }
err_t hipFuncGetAttributes(void* at, const void* f) { (void)f; memset(at, 0, 56); return OK; }
err_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int b, size_t sh) {
    (void)f; (void)b; (void)sh;
    *n = 1;
    return OK;
}

/* ---- device, streams, events, graphs ---- */
err_t hipGetDevice(int* d) { *d = 0; return OK; }
err_t hipDeviceGetAttribute(int* v, int a, int d) { (void)a; (void)d; *v = 256; return OK; }
err_t hipGetLastError(void) { return OK; }
const char* hipGetErrorString(err_t e) { return e == OUT_OF_MEMORY ? "out of memory" : "error"; }
static err_t handle(void** h) { static int x; *h = &x; return OK; }
err_t hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; return handle(s); }
err_t hipStreamDestroy(void* s) { (void)s; return OK; }
err_t hipStreamSynchronize(void* s) { (void)s; return OK; }
err_t hipEventCreate(void** e) { return handle(e); }
err_t hipEventCreateWithFlags(void** e, unsigned f) { (void)f; return handle(e); }
err_t hipEventDestroy(void* e) { (void)e; return OK; }
err_t hipEventRecord(void* e, void* s) { (void)e; (void)s; return OK; }
err_t hipEventSynchronize(void* e) { (void)e; return OK; }
err_t hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 0; return OK; }
err_t hipStreamBeginCapture(void* s, int m) { (void)s; (void)m; return OK; }
err_t hipStreamEndCapture(void* s, void** g) { (void)s; return handle(g); }
err_t hipGraphInstantiate(void** x, void* g, void** n, char* l, size_t s) {
    (void)g; (void)n; (void)l; (void)s;
    return handle(x);
}
err_t hipGraphLaunch(void* x, void* s) { (void)x; (void)s; return OK; }
err_t hipGraphDestroy(void* g) { (void)g; return OK; }
err_t hipGraphExecDestroy(void* x) { (void)x; return OK; }
