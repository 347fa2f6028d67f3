/*
 * handle_check.c -- what a handle asks of the device, checked without one.
 * The HIP calls of libparties_vof.so resolve to the functions below: device
 * memory is host memory, kernels are counted and not run.  Modes:
 *   layout NX NY    offsets of the arrays the kernels read in pairs of doubles
 *   lds NX NY       launches of the FFT solves with more than 64 KiB of dynamic
 *                   LDS, and those of them whose kernel was not allowed it
 *   transfers NX NY work still queued when a transfer of a field returns, for a
 *                   host array and for a device array; what the latter carried;
 *                   bytes of host memory pinned for them
 */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "../../parties-vof-ibm_amd/host/pv_host.h"

/* ---- the runtime's part ---- */
#define NBLOCK 256
static struct { char *p; size_t n; } block[NBLOCK];
static int nblock;

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d)
{
    (void)d;
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { (void)e; return "none"; }

hipError_t hipMalloc(void **p, size_t n)
{
    if (nblock == NBLOCK || posix_memalign(p, 4096, n ? n : 1)) return hipErrorOutOfMemory;
    block[nblock].p = (char *)*p;
    block[nblock++].n = n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    int k;
    for (k = 0; k < nblock; k++)
        if (block[k].p == (char *)p) block[k] = block[--nblock];
    free(p);
    return hipSuccess;
}
static size_t pinned;
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags)
{
    (void)flags;
    pinned += n;
    *p = malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { (void)k; memcpy(d, s, n); return hipSuccess; }
/* work queued on the one stream and work known to be finished */
static long queued, finished;
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind k, hipStream_t st)
{
    size_t j;
    (void)k; (void)st;
    for (j = 0; j < h; j++) memcpy((char *)d + j * dp, (const char *)s + j * sp, w);
    queued++;
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    int k;
    memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeUnregistered;
    for (k = 0; k < nblock; k++)
        if ((char *)p >= block[k].p && (char *)p < block[k].p + block[k].n) a->type = hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags) { (void)flags; *e = (hipEvent_t)calloc(1, sizeof(long)); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)s; *(long *)e = queued; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (*(long *)e > finished) finished = *(long *)e;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)st;
    return hipMemcpy(d, s, n, k);
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned flags) { (void)flags; *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; finished = queued; return hipSuccess; }

static struct { dim3 g, b; size_t lds; hipStream_t s; } cfg;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    cfg.g = g; cfg.b = b; cfg.lds = lds; cfg.s = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = cfg.g; *b = cfg.b; *lds = cfg.lds; *s = cfg.s;
    return hipSuccess;
}
static struct { const void *f; size_t lds; } allowed[NBLOCK];
static int nallowed, nlarge, nrefused;
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v)
{
    if (a != hipFuncAttributeMaxDynamicSharedMemorySize || nallowed == NBLOCK) return hipErrorInvalidValue;
    allowed[nallowed].f = f;
    allowed[nallowed++].lds = (size_t)v;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds, hipStream_t s)
{
    (void)g; (void)b; (void)args; (void)s;
    if (lds > 65536) {
        int k, ok = 0;
        for (k = 0; k < nallowed; k++) ok |= allowed[k].f == f && allowed[k].lds >= lds;
        nlarge++;
        nrefused += !ok;
    }
    queued++;
    return hipSuccess;
}

/* ---- the checks ---- */
static pv_bag *create(int nx, int ny)
{
    pv_params p;
    pv_bag *b;
    pv_params_default(&p);
    p.NXM = nx;
    p.NYM = ny;
    p.ymax = (double)ny / nx;
    p.p_max_iter = 2;
    if (pv_create(&p, 0, &b)) { fprintf(stderr, "%s\n", pv_last_error()); exit(1); }
    return b;
}

static unsigned past(const void *p, unsigned n) { return (unsigned)((size_t)p % n); }

static int layout(int nx, int ny)
{
    pv_bag *b = create(nx, ny);
    unsigned worst = 0;
    int k;
    for (k = 0; k < PV_FI_END; k++)
        if (past(b->f[k], 128) > worst) worst = past(b->f[k], 128);
    printf("field %u\n", worst);
    if (b->fft.ok) printf("rtx %u\nwx %u\n", past(b->fft.rtx, 16), past(b->fft.wx, 16));
    if (b->mg_ok) {
        /* both hierarchies: the smoothing levels' arrays, the bottom matrix (read in pairs where its
         * size is even), the other residual */
        unsigned lev = 0, h = 0;
        for (k = 0; k < 2; k++) {
            const pvk_mg *m = k ? &b->mgf : &b->mg;
            const unsigned n = k ? 8 : 16;
            const pvk_mglev *e = &m->L[m->nlev - 1];
            int l, q;
            for (l = 0; l + 1 < m->nlev; l++) {
                const void *a[5] = { m->L[l].x, m->L[l].f, m->L[l].bx, m->L[l].by, m->L[l].xp };
                for (q = 0; q < 5; q++) lev += past(a[q], n);
                lev += (m->L[l].pitch & 1) + (m->L[l].nx & 1);
            }
            if (e->nx * e->ny % 2 == 0) h += past(m->H, n);
        }
        printf("level %u\nH %u\nr2 %u\n", lev, h, past(b->mgw.r2, 16));
    }
    pv_destroy(b);
    return 0;
}

static int lds(int nx, int ny)
{
    pv_bag *b = create(nx, ny);
    if (pv_Pressure_solve_fft(b, PV_F_SCRATCH0, PV_F_SCRATCH1)) { fprintf(stderr, "%s\n", pv_last_error()); return 1; }
    pv_set_pressure_solver(b, PV_PSOLVE_FFT_PCG);
    pv_Pressure_solve_cg(b, NULL);       /* start and two iterations; no kernel ran, so it did not stop */
    printf("large %d\nrefused %d\n", nlarge, nrefused);
    pv_destroy(b);
    return 0;
}

static int transfers(int nx, int ny)
{
    pv_bag *b = create(nx, ny);
    const size_t n = (size_t)(nx + 7) * (ny + 7);
    double *h = (double *)calloc(n, sizeof(double)), *d, *e;
    const size_t pinned0 = pinned;
    size_t k, wrong = 0;
    hipMalloc((void **)&d, n * sizeof(double));
    hipMalloc((void **)&e, n * sizeof(double));
    for (k = 0; k < n; k++) { d[k] = (double)k; e[k] = -1.0; }
    if (pv_set_field(b, PV_F_U, h)) return 1;
    printf("set %ld\n", queued - finished);
    if (pv_get_field(b, PV_F_U, h)) return 1;
    printf("get %ld\n", queued - finished);
    printf("pinned %zu\n", pinned - pinned0);
    if (pv_set_field(b, PV_F_V, d)) return 1;
    printf("device_set %ld\n", queued - finished);
    if (pv_get_field(b, PV_F_V, e)) return 1;
    printf("device_get %ld\n", queued - finished);
    for (k = 0; k < n; k++) wrong += e[k] != d[k];
    printf("wrong %zu\n", wrong);
    pv_destroy(b);
    return 0;
}

int main(int argc, char **argv)
{
    if (argc == 4 && !strcmp(argv[1], "layout")) return layout(atoi(argv[2]), atoi(argv[3]));
    if (argc == 4 && !strcmp(argv[1], "lds")) return lds(atoi(argv[2]), atoi(argv[3]));
    if (argc == 4 && !strcmp(argv[1], "transfers")) return transfers(atoi(argv[2]), atoi(argv[3]));
    return 2;
}
