/* A host-memory stand-in for the HIP calls that plsqr_cnn_conv_forward and
 * plsqr_cnn_conv_backward make, preloaded in front of the runtime so that their
 * host code runs without a GPU.  Kernels do nothing; a launch reports the code
 * in HIP_STUB_LAUNCH (0: success) as hipGetLastError does.  Every allocation's
 * size goes to stdout as "alloc <bytes>". */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
    unsigned x, y, z;
} dim3_t;

static int last;

int hipMalloc(void **p, size_t n) {
    printf("alloc %zu\n", n);
    fflush(stdout);
    *p = calloc(n, 1);
    return *p ? 0 : 2;
}

int hipFree(void *p) {
    free(p);
    return 0;
}

int hipMemcpy(void *d, const void *s, size_t n, int kind) {
    (void)kind;
    memcpy(d, s, n);
    return 0;
}

int hipDeviceSynchronize(void) { return 0; }

int hipGetDevice(int *d) {
    *d = 0;
    return 0;
}

int hipDeviceGetAttribute(int *v, int attr, int dev) {
    (void)attr;
    (void)dev;
    *v = 256;
    return 0;
}

int hipGetLastError(void) {
    const int e = last;
    last = 0;
    return e;
}

int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void *stream) {
    (void)grid;
    (void)block;
    (void)lds;
    (void)stream;
    return 0;
}

int __hipPopCallConfiguration(dim3_t *grid, dim3_t *block, size_t *lds, void **stream) {
    grid->x = grid->y = grid->z = block->x = block->y = block->z = 1;
    *lds = 0;
    *stream = NULL;
    return 0;
}

int hipLaunchKernel(const void *f, dim3_t grid, dim3_t block, void **args, size_t lds, void *stream) {
    (void)f;
    (void)grid;
    (void)block;
    (void)args;
    (void)lds;
    (void)stream;
    const char *e = getenv("HIP_STUB_LAUNCH");
    last = e ? atoi(e) : 0;
    return last;
}
