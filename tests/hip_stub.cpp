// A HIP runtime without a device, for tests of the library's host side: memory is the host's, modules and functions are names,
// nothing runs.  Every launch is handed to the callback a test registers; the allocation a test names fails.
#include <cstdlib>
#include <cstring>
#include <string>

typedef void (*launch_fn)(const char* name, const unsigned* shape, void** params);   // shape: grid, block, shared bytes
static launch_fn on_launch = nullptr;
static size_t fail_over = ~(size_t) 0;   // hipMalloc of more than this many bytes fails
static long fail_copy = -1;              // copies to the device until one fails (-1: none)
static long graph_launches = 0;

extern "C" {
void stub_on_launch(launch_fn f) { on_launch = f; }
void stub_fail_allocations_over(size_t bytes) { fail_over = bytes; }
void stub_fail_copy_after(long n) { fail_copy = n; }
long stub_graph_launches() { return graph_launches; }

int hipInit(unsigned) { return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceGetName(char* s, int n, int) { std::strncpy(s, "stub", (size_t) n); return 0; }
int hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t) 1 << 38; return 0; }
int hipMalloc(void** p, size_t n) { *p = n > fail_over ? nullptr : std::malloc(n); return *p ? 0 : 2; }
int hipFree(void* p) { std::free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n); return *p ? 0 : 2; }
int hipHostFree(void* p) { std::free(p); return 0; }
int hipMemcpyHtoD(void* d, const void* s, size_t n) {
    if (fail_copy == 0) return 1;
    if (fail_copy > 0) fail_copy--;
    std::memcpy(d, s, n);
    return 0;
}
int hipMemcpyDtoH(void* d, const void* s, size_t n) { std::memcpy(d, s, n); return 0; }
int hipMemcpyDtoHAsync(void* d, const void* s, size_t n, void*) { std::memcpy(d, s, n); return 0; }
int hipMemcpyHtoDAsync(void* d, const void* s, size_t n, void*) { std::memcpy(d, s, n); return 0; }
int hipMemsetD8Async(void* d, unsigned char v, size_t n, void*) { std::memset(d, v, n); return 0; }
int hipModuleLoadData(void** m, const void*) { *m = (void*) 1; return 0; }
int hipModuleUnload(void*) { return 0; }
int hipModuleGetFunction(void** f, void*, const char* name) { *f = strdup(name); return 0; }
int hipModuleLaunchKernel(void* f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, unsigned shared, void*, void** params, void**) {
    const unsigned shape[] = {gx, gy, gz, bx, by, bz, shared};
    if (on_launch) on_launch((const char*) f, shape, params);
    return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) { *s = (void*) 16; return 0; }
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipDeviceSynchronize() { return 0; }
int hipEventCreate(void** e) { *e = (void*) 16; return 0; }
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0.0f; return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) { *g = (void*) 16; return 0; }
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) { *x = (void*) 16; return 0; }
int hipGraphLaunch(void*, void*) { graph_launches++; return 0; }
int hipGraphExecDestroy(void*) { return 0; }
int hipGraphDestroy(void*) { return 0; }
const char* hipGetErrorName(int) { return "stub"; }
const char* hipGetErrorString(int) { return "stub"; }
int hipGetSymbolAddress(void** p, const void*) { static char ws[16]; *p = ws; return 0; }
}
