// Device memory of the library's buffers (DBuf): freed blocks are kept and
// handed out again.  hipFree waits for everything the device has in flight,
// so the temporaries of a setup, which runs on up to a dozen host threads and
// streams, made every thread wait for all the others' kernels, and a
// destroyed problem took 0.1 ms a buffer.  A 31 000-panel FP64 problem waited
// 320 ms in hipFree, summed over the threads of its setup; kept blocks take
// its setup from 90 to 52 ms and its destruction from 18 to 2 ms.
//
// A block is handed out again at once, on any thread and stream, so it must
// be idle when it is released: every owner waits for the stream its buffers
// were used on before they go out of scope.  Where an exception unwinds past
// that wait, the block goes to hipFree, which waits by itself.
#include <hip/hip_runtime.h>

#include <exception>
#include <map>
#include <mutex>
#include <stdexcept>
#include <unordered_map>
#include <vector>

#include "internal.h"

namespace fsvd {
namespace {

struct Live {
   size_t bytes;
   int dev;
};
struct Free {
   void* p;
   unsigned long long gen;   // the build count when it was released
};

class DeviceCache {
 public:
   void* take(size_t bytes) {
      int dev = 0;
      FSVD_CHECK(hipGetDevice(&dev));
      const size_t want = rounded(bytes);
      std::lock_guard<std::mutex> g(mu_);
      // the smallest kept block of this device that wastes at most a quarter
      auto it = free_.lower_bound({dev, want});
      if (it != free_.end() && it->first.first == dev && it->first.second <= want + want / 4) {
         void* p = it->second.p;
         const size_t have = it->first.second;
         held_ -= have;
         free_.erase(it);
         live_[p] = {have, dev};
         return p;
      }
      void* p = nullptr;
      hipError_t e = hipMalloc(&p, want);
      if (e != hipSuccess && !free_.empty()) {
         // give everything kept back and try again
         (void)hipGetLastError();
         drop([](unsigned long long) { return true; });
         e = hipMalloc(&p, want);
      }
      FSVD_CHECK(e);
      live_[p] = {want, dev};
      if (!limit_) {
         size_t fr = 0, total = 0;
         limit_ = hipMemGetInfo(&fr, &total) == hipSuccess && total ? total / 24 : (size_t)1 << 30;
      }
      return p;
   }
   void give(void* p) {
      std::lock_guard<std::mutex> g(mu_);
      auto it = live_.find(p);
      if (it == live_.end()) return;
      const Live l = it->second;
      live_.erase(it);
      if (std::uncaught_exceptions() > 0 || l.bytes > limit_) {
         (void)hipFree(p);
         return;
      }
      free_.insert({{l.dev, l.bytes}, {p, gen_}});
      held_ += l.bytes;
      while (held_ > limit_) {
         // the block kept longest
         auto old = free_.begin();
         for (auto f = free_.begin(); f != free_.end(); ++f)
            if (f->second.gen < old->second.gen) old = f;
         (void)hipFree(old->second.p);
         held_ -= old->first.second;
         free_.erase(old);
      }
   }
   // A problem has been built: what was released before the last two builds
   // began and not taken since goes back to the device.
   void built() {
      std::lock_guard<std::mutex> g(mu_);
      gen_++;
      drop([this](unsigned long long gen) { return gen + 2 < gen_; });
   }

 private:
   // multiples of an eighth of the leading power of two (at least 512 bytes)
   static size_t rounded(size_t b) {
      size_t step = 512;
      while (step * 16 <= b) step <<= 1;
      return (b + step - 1) / step * step;
   }
   template <typename F>
   void drop(F&& gone) {
      for (auto f = free_.begin(); f != free_.end();)
         if (gone(f->second.gen)) {
            (void)hipFree(f->second.p);
            held_ -= f->first.second;
            f = free_.erase(f);
         } else {
            ++f;
         }
   }
   std::mutex mu_;
   std::unordered_map<void*, Live> live_;
   std::multimap<std::pair<int, size_t>, Free> free_;   // by device and size
   size_t held_ = 0, limit_ = 0;                        // kept bytes: at most 1/24 of the device's memory
   unsigned long long gen_ = 0;
};

// Never destroyed: buffers may be released by other static destructors; the
// process's end returns the memory.
DeviceCache& cache() {
   static DeviceCache* c = new DeviceCache;
   return *c;
}

}  // namespace

void* dev_take(size_t bytes) { return cache().take(bytes); }
void dev_give(void* p) { cache().give(p); }
void dev_built() { cache().built(); }

}  // namespace fsvd
