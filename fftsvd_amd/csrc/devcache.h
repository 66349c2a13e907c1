// Freed blocks of device memory, kept and handed out again (DeviceCache).
// Independent of HIP: Api gives
//    static int device();                      the calling thread's device
//    static size_t total();                    its memory, 0 if unknown
//    static void* alloc(size_t bytes);         nullptr if there is none
//    static void free(void* p);                waits until p's device is idle
//
// A block is handed out again at once, on any thread and stream, so it must
// be idle when it is released: every owner waits for the stream its buffers
// were used on before they go out of scope.  Where an exception unwinds past
// that wait, the block is freed, which waits by itself.
//
// Kept bytes are bounded per device (1/24 of its memory).  A block is freed
// when the bound asks for it (the longest kept first), when two later builds
// have not taken it, when an allocation fails, or on trim().  Sizes are
// rounded up by at most 1/8 and a block is reused for requests of at least
// 4/5 of it, so a buffer holds at most 1.41 times what was asked for.
// Api::free waits for the whole device: it is called without the lock, so
// that other threads' requests do not wait behind it.
#pragma once

#include <cstddef>
#include <exception>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

namespace fsvd {

template <typename Api>
class DeviceCache {
 public:
   // nullptr if the device has no memory left, kept blocks given back included
   void* take(size_t bytes) {
      const int dev = Api::device();
      const size_t want = rounded(bytes);
      bool bounded = false;
      {
         std::lock_guard<std::mutex> g(mu_);
         Device& d = devices_[dev];
         bounded = d.limit > 0;
         // the smallest kept block that wastes at most a quarter of the request
         auto it = d.kept.lower_bound(want);
         if (it != d.kept.end() && it->first <= want + want / 4) {
            void* p = it->second.p;
            live_[p] = {it->first, dev};
            d.held -= it->first;
            d.kept.erase(it);
            return p;
         }
      }
      void* p = Api::alloc(want);
      if (!p) {
         // one thread at a time, so that none gives up while another frees
         std::lock_guard<std::mutex> r(retry_);
         trim();
         p = Api::alloc(want);
         if (!p) return nullptr;
      }
      const size_t total = bounded ? 0 : Api::total();
      std::lock_guard<std::mutex> g(mu_);
      live_[p] = {want, dev};
      if (!bounded) devices_[dev].limit = total ? total / 24 : (size_t)1 << 30;
      return p;
   }

   void give(void* p) {
      std::vector<void*> gone;
      {
         std::lock_guard<std::mutex> g(mu_);
         auto it = live_.find(p);
         if (it == live_.end()) return;
         const Live l = it->second;
         live_.erase(it);
         Device& d = devices_[l.dev];
         if (std::uncaught_exceptions() > 0 || l.bytes > d.limit) {
            gone.push_back(p);
         } else {
            d.kept.insert({l.bytes, {p, gen_}});
            d.held += l.bytes;
            while (d.held > d.limit) {
               auto old = d.kept.begin();
               for (auto f = d.kept.begin(); f != d.kept.end(); ++f)
                  if (f->second.gen < old->second.gen) old = f;
               gone.push_back(old->second.p);
               d.held -= old->first;
               d.kept.erase(old);
            }
         }
      }
      for (void* q : gone) Api::free(q);
   }

   // A problem has been built: what was released before the last two builds
   // began and not taken since goes back to the device.
   void built() {
      drop([this](unsigned long long gen) { return gen + 2 < gen_; }, true);
   }

   // Everything kept goes back to the devices; the bytes.
   size_t trim() {
      return drop([](unsigned long long) { return true; }, false);
   }

 private:
   struct Live {
      size_t bytes;
      int dev;
   };
   struct Kept {
      void* p;
      unsigned long long gen;   // the build count when it was released
   };
   struct Device {
      std::multimap<size_t, Kept> kept;
      size_t held = 0, limit = 0;   // bytes kept, and how many at most
   };

   // multiples of an eighth of the leading power of two (at least 512 bytes)
   static size_t rounded(size_t b) {
      size_t step = 512;
      while (step * 16 <= b) step <<= 1;
      return (b + step - 1) / step * step;
   }

   template <typename F>
   size_t drop(F&& goes, bool count) {
      std::vector<void*> gone;
      size_t bytes = 0;
      {
         std::lock_guard<std::mutex> g(mu_);
         if (count) gen_++;
         for (auto& e : devices_) {
            Device& d = e.second;
            for (auto f = d.kept.begin(); f != d.kept.end();)
               if (goes(f->second.gen)) {
                  gone.push_back(f->second.p);
                  bytes += f->first;
                  d.held -= f->first;
                  f = d.kept.erase(f);
               } else {
                  ++f;
               }
         }
      }
      for (void* p : gone) Api::free(p);
      return bytes;
   }

   std::mutex mu_, retry_;
   std::unordered_map<void*, Live> live_;
   std::map<int, Device> devices_;
   unsigned long long gen_ = 0;
};

}  // namespace fsvd
