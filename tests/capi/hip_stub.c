/* A HIP runtime that does nothing, for the host library's choices on the CPU: it counts the bytes of device memory asked
 * for and the launches, and keeps the names of the first 16 kernels. Built by tests/test_host_choice.py as libamdhip64.so.7. */
#include <stddef.h>
#include <stdlib.h>

size_t stub_bytes;
unsigned stub_launches;
const char *stub_name[16];
static char dev[128u << 10] __attribute__((aligned(256)));

int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { return (void)a, (void)d, *v = 256, 0; }
int hipModuleLoad(void **m, const char *p) { return (void)p, *m = dev, 0; }
int hipModuleGetFunction(void **f, void *m, const char *n) { return (void)m, *f = (void *)n, 0; }
int hipModuleGetGlobal(void **p, size_t *n, void *m, const char *s) { return (void)m, (void)s, *p = dev, *n = (size_t)64 << 20, 0; }
int hipModuleLaunchKernel(void *f) { return stub_launches < 16u ? (void)(stub_name[stub_launches] = f) : (void)0, stub_launches++, 0; }
int hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int *n) { return *n = 2, 0; }
int hipMalloc(void **p, size_t n) { return stub_bytes += n, *p = dev, 0; }
const char *hipGetErrorString(int e) { return (void)e, "stub"; }
#define NOTHING(f) \
  int f(void) { return 0; }
NOTHING(hipSetDevice) NOTHING(hipModuleUnload) NOTHING(hipFree) NOTHING(hipMemcpy) NOTHING(hipMemset) NOTHING(hipDeviceSynchronize)
NOTHING(hipEventCreate) NOTHING(hipEventDestroy) NOTHING(hipEventRecord) NOTHING(hipEventSynchronize) NOTHING(hipEventElapsedTime)
NOTHING(hipStreamCreate) NOTHING(hipStreamDestroy) NOTHING(hipStreamSynchronize) NOTHING(hipStreamWaitEvent)
NOTHING(hipStreamBeginCapture) NOTHING(hipStreamEndCapture) NOTHING(hipGraphInstantiate) NOTHING(hipGraphDestroy)
NOTHING(hipGraphLaunch) NOTHING(hipGraphExecDestroy) NOTHING(hipHostMalloc) NOTHING(hipHostFree) NOTHING(hipMemcpyAsync)
