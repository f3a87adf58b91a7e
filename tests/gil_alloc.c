/* A torch allocator (CUDAPluggableAllocator) that counts the allocations made while the calling thread holds the
 * Python GIL. */
#include <Python.h>
#include <hip/hip_runtime_api.h>

static int held, all;
int gil_held(void) { return held; }
int gil_all(void) { return all; }

void *gil_alloc(ssize_t size, int device, hipStream_t stream) {
  (void)device, (void)stream;
  void *p = 0;
  held += PyGILState_Check();
  ++all;
  return hipMalloc(&p, (size_t)size) == hipSuccess ? p : 0;
}

void gil_free(void *p, ssize_t size, int device, hipStream_t stream) {
  (void)size, (void)device, (void)stream;
  (void)hipFree(p);
}
