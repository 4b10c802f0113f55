/* Stands in for the HIP runtime's launch entry points in a process without a
   GPU: loaded with global visibility before libcc1d_amd.so, its definitions
   are the ones that the library's calls reach. Every launch goes to a callback
   with the kernel's name, grid and arguments, and nothing is enqueued. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned x, y, z; } dim3_t;
typedef void (*launch_cb)(const char* kernel, unsigned gx, unsigned gy, unsigned bx, void** args);

static struct { const void* host; const char* name; } *kernels;
static size_t n_kernels, room;
static launch_cb callback;

void spy_callback(launch_cb cb) { callback = cb; }

void __hipRegisterFunction(void** modules, const void* host, char* device, const char* name, unsigned limit, void* tid,
                           void* bid, void* block, void* grid, int* wsize) {
    (void)modules, (void)device, (void)limit, (void)tid, (void)bid, (void)block, (void)grid, (void)wsize;
    if (n_kernels == room) {
        room = room ? 2 * room : 1024;
        kernels = realloc(kernels, room * sizeof *kernels);
        if (!kernels) abort();
    }
    kernels[n_kernels].host = host;
    kernels[n_kernels++].name = name;
}

int hipLaunchKernel(const void* host, dim3_t grid, dim3_t block, void** args, size_t shared, void* stream) {
    (void)shared, (void)stream;
    for (size_t i = 0; i < n_kernels; ++i)
        if (kernels[i].host == host) {
            if (callback) callback(kernels[i].name, grid.x, grid.y, block.x, args);
            return 0;
        }
    return 98; /* hipErrorInvalidDeviceFunction */
}

/* the static scratch of cc1d_bwd_typed_noalloc: device 0, an address nobody reads */
int hipGetDevice(int* device) { *device = 0; return 0; }
int hipGetSymbolAddress(void** address, const void* symbol) {
    (void)symbol;
    *address = (void*)(size_t)(1 << 20);
    return 0;
}
