/* Stands in for the HIP runtime where libtlq.so's choice of kernels is tested without a GPU: loaded ahead of the library with its symbols global, it
 * takes the library's runtime calls and reports success, so that the library's launch log names what would run -- or refuses the LDS of kernels whose
 * name holds a given text. */
#include <stdint.h>
#include <stdio.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;
enum { kFunctions = 8192 };
static struct { const void* f; const char* name; } functions[kFunctions];
static int n_functions = 0;
static char refused[256] = "";
static dim3_t grid_, block_;
static size_t lds_;
static void* stream_;

void** __hipRegisterFatBinary(const void* data) { static void* handle; return (void)data, &handle; }
void __hipUnregisterFatBinary(void** handle) { (void)handle; }
void __hipRegisterFunction(void** handle, const void* f, char* device, const char* name, unsigned limit, void* tid, void* bid, void* bdim, void* gdim, int* wsize) {
  (void)handle, (void)device, (void)limit, (void)tid, (void)bid, (void)bdim, (void)gdim, (void)wsize;
  if (n_functions < kFunctions) functions[n_functions].f = f, functions[n_functions++].name = name;
}
void __hipRegisterVar(void** handle, void* var, char* host, char* device, int ext, size_t size, int constant, int global) {
  (void)handle, (void)var, (void)host, (void)device, (void)ext, (void)size, (void)constant, (void)global;
}
int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void* stream) { return grid_ = grid, block_ = block, lds_ = lds, stream_ = stream, 0; }
int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* lds, void** stream) { return *grid = grid_, *block = block_, *lds = lds_, *stream = stream_, 0; }
int hipGetDevice(int* device) { return *device = 0, 0; }
int hipDeviceGetAttribute(int* value, int attribute, int device) { return (void)attribute, (void)device, *value = 256, 0; } /* compute units: all that is asked for */
int hipGetLastError(void) { return 0; }
const char* hipGetErrorString(int e) { return e ? "refused" : "no error"; }
int hipGetSymbolAddress(void** address, const void* symbol) { return *address = (void*)symbol, 0; }
int hipLaunchKernel(const void* f, dim3_t grid, dim3_t block, void** args, size_t lds, void* stream) {
  return (void)f, (void)grid, (void)block, (void)args, (void)lds, (void)stream, 0;
}
int hipFuncSetAttribute(const void* f, int attribute, int value) {
  (void)attribute, (void)value;
  for (int i = 0; refused[0] && i < n_functions; ++i)
    if (functions[i].f == f && strstr(functions[i].name, refused)) return 1;
  return 0;
}

void recorder_refuse(const char* text) { snprintf(refused, sizeof(refused), "%s", text); }
