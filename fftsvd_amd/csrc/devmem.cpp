// Device memory of the library's buffers (DBuf): freed blocks are kept and
// handed out again (devcache.h).  hipFree waits for everything the device has
// in flight, so the temporaries of a setup, which runs on up to a dozen host
// threads and streams, made every thread wait for all the others' kernels, and
// a destroyed problem took 0.1 ms a buffer.  A 31 000-panel FP64 problem waited
// 320 ms in hipFree, summed over the threads of its setup; kept blocks take
// its setup from 90 to 52 ms and its destruction from 18 to 2 ms.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <stdexcept>

#include "devcache.h"
#include "internal.h"

namespace fsvd {
namespace {

struct HipMemory {
   static int device() {
      int dev = 0;
      FSVD_CHECK(hipGetDevice(&dev));
      return dev;
   }
   static size_t total() {
      size_t fr = 0, all = 0;
      return hipMemGetInfo(&fr, &all) == hipSuccess ? all : 0;
   }
   static void* alloc(size_t bytes) {
      void* p = nullptr;
      why = hipMalloc(&p, bytes);
      if (why == hipSuccess) return p;
      (void)hipGetLastError();
      return nullptr;
   }
   static thread_local hipError_t why;   // the last allocation's result
   static void free(void* p) { (void)hipFree(p); }
};

thread_local hipError_t HipMemory::why = hipSuccess;

// Never destroyed: buffers may be released by other static destructors; the
// process's end returns the memory.
DeviceCache<HipMemory>& cache() {
   static auto* c = new DeviceCache<HipMemory>;
   return *c;
}

// FFTSVD_FILL_MEMORY=1: NaN in every block that is handed out, on a stream of
// its own that waits for no other, so that a block in use shows at once.
void fill(void* p, size_t bytes) {
   hipStream_t s = nullptr;
   FSVD_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
   FSVD_CHECK(hipMemsetAsync(p, 0xff, bytes, s));
   FSVD_CHECK(hipStreamSynchronize(s));
   (void)hipStreamDestroy(s);
}

}  // namespace

void* dev_take(size_t bytes) {
   void* p = cache().take(bytes);
   if (!p) FSVD_CHECK(HipMemory::why);
   if (const char* e = std::getenv("FFTSVD_FILL_MEMORY"); e && e[0] == '1') fill(p, bytes);
   return p;
}
void dev_give(void* p) { cache().give(p); }
void dev_built() { cache().built(); }
size_t dev_trim() { return cache().trim(); }

}  // namespace fsvd
