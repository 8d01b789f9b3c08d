/* Set-up and launch of a batch of small templates over a HIP runtime of host memory that fails one call on request.
 *
 * The HIP functions that libfastfft_amd.so imports are defined here and exported by the program, which the dynamic
 * linker prefers to the runtime's: allocations are host memory, kernel launches do nothing, and, as the runtime does,
 * a failed call leaves its error to be returned (and cleared) by hipGetLastError.
 *
 * usage: batch_without_memory <libfastfft_amd.so> <malloc|memcpy> <k> <error code>
 * The k-th call of that kind from fastfft_set_batch on fails with the code (k = 0: none does).  Prints the status of
 * fastfft_set_batch, then of fastfft_fwd_image_inv_batch if the batch was set, and the batch's description.
 */
#include <dlfcn.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

#include "fastfft/fastfft.h"

static hipError_t  last_error = hipSuccess;
static const char* fail_what  = "";
static int         fail_at = 0, fail_code = 0, calls = 0, armed = 0;

static hipError_t result(const char* what) {
    if ( armed && strcmp(what, fail_what) == 0 && ++calls == fail_at )
        return last_error = (hipError_t)fail_code;
    return hipSuccess;
}

hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int d) {
    (void)d;
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    const hipError_t e = result("malloc");
    *p                 = e == hipSuccess ? aligned_alloc(256, (n + 255) / 256 * 256) : NULL;
    return e;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
    (void)k;
    const hipError_t e = result("memcpy");
    if ( e == hipSuccess )
        memcpy(d, s, n);
    return e;
}
hipError_t  hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t  hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t  hipGetLastError(void) { const hipError_t e = last_error; last_error = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t e) { (void)e; return "an error"; }
hipError_t  hipFuncSetAttribute(const void* f, hipFuncAttribute a, int v) { (void)f; (void)a; (void)v; return hipSuccess; }
hipError_t  hipGetSymbolAddress(void** p, const void* s) {
    static char table[1 << 20];
    (void)s;
    *p = table;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t m, hipStream_t s) {
    (void)f; (void)g; (void)b; (void)a; (void)m; (void)s;
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) { (void)g; (void)b; (void)m; (void)s; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    g->x = g->y = g->z = b->x = b->y = b->z = 1;
    *m = 0;
    *s = NULL;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) { (void)s; *c = hipStreamCaptureStatusNone; return hipSuccess; }

enum { N_TEMPLATES = 6, SIZE = 60, WINDOW = 81, NX = 2048, NY = 1024 };

#define CHECK(call) do { const int rc_ = (int)(call); if ( rc_ ) { printf("%s: %d %s\n", #call, rc_, error_string( )); return 1; } } while ( 0 )
#define SYM(ret, name, ...) ret (*name)(__VA_ARGS__) = (ret (*)(__VA_ARGS__))dlsym(lib, "fastfft_" #name)

int main(int argc, char** argv) {
    if ( argc != 5 )
        return 2;
    void* lib = dlopen(argv[1], RTLD_NOW);
    if ( ! lib ) {
        printf("%s\n", dlerror( ));
        return 2;
    }
    fail_what = argv[2];
    fail_at   = atoi(argv[3]);
    fail_code = atoi(argv[4]);
    SYM(const char*, last_error_string, void);
    const char* (*error_string)(void) = last_error_string;
    SYM(int, create, fastfft_plan*, int, int, int);
    SYM(int, set_fwd_plan, fastfft_plan, size_t, size_t, size_t, size_t, size_t, size_t, int);
    SYM(int, set_inv_plan, fastfft_plan, size_t, size_t, size_t, size_t, size_t, size_t, int);
    SYM(int, set_output_window, fastfft_plan, int, int, int);
    SYM(int, set_batch, fastfft_plan, int, const void* const*, const int*, void* const*, int*, float*);
    SYM(int, fwd_image_inv_batch, fastfft_plan, const void*, fastfft_op, fastfft_op, fastfft_op);
    SYM(int, describe, fastfft_plan, const char*, char*, size_t);
    fastfft_plan p = NULL;
    CHECK(create(&p, FASTFFT_INPUT_F32, FASTFFT_IMAGE_C64, 2));
    CHECK(set_fwd_plan(p, SIZE, SIZE, 1, NX, NY, 1, 1));
    CHECK(set_inv_plan(p, NX, NY, 1, WINDOW, WINDOW, 1, 1));
    CHECK(set_output_window(p, -(WINDOW / 2), -(WINDOW / 2), 0));
    const void* in[N_TEMPLATES];
    void*       out[N_TEMPLATES];
    int         sizes[2 * N_TEMPLATES];
    for ( int i = 0; i < N_TEMPLATES; i++ ) {
        in[i]        = calloc(SIZE * (SIZE + 2), sizeof(float));
        out[i]       = calloc(WINDOW * (WINDOW + 2), sizeof(float));
        sizes[2 * i] = sizes[2 * i + 1] = SIZE;
    }
    void* image = aligned_alloc(256, (size_t)(NX / 2 + 1) * NY * 8);
    setenv("FASTFFT_NO_BATCH_GRAPH", "1", 1);
    armed        = 1;
    const int rc = set_batch(p, N_TEMPLATES, in, sizes, out, NULL, NULL);
    armed        = 0;
    printf("set_batch %d\n", rc);
    if ( rc )
        return 0;
    const fastfft_op noop = {FASTFFT_OP_NOOP, 1.f}, mul = {FASTFFT_OP_CONJ_MUL, 1.f};
    printf("batch %d\n", fwd_image_inv_batch(p, image, noop, mul, noop));
    char text[4096];
    CHECK(describe(p, "batch", text, sizeof(text)));
    *strchr(text, '\n') = 0;
    printf("%s\n", text);
    return 0;
}
