"""The cache of freed device blocks (csrc/devcache.h) over a pretended memory of
two devices: reuse and its waste, the bound per device and the order in which
blocks leave it, builds, failing allocations, unwinding, and that no block is
freed while the cache is locked (CPU only, compiled with g++)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <stdexcept>
#include <thread>
#include <vector>
#include "devcache.h"

struct Memory {
   static int dev;
   static size_t room[2];                       // bytes left per device
   static std::map<char*, std::pair<size_t, int>> out;
   static std::vector<void*> freed;
   static std::function<void()> hook;
   static int device() { return dev; }
   static size_t total() { return 24 * 16384; }   // the cache keeps 16384
   static void* alloc(size_t n) {
      if (n > room[dev]) return nullptr;
      static size_t at = 4096;
      char* p = (char*)(at += 1 << 20);
      room[dev] -= n;
      out[p] = {n, dev};
      return p;
   }
   static void free(void* p) {
      auto it = out.find((char*)p);
      if (it == out.end()) std::abort();
      room[it->second.second] += it->second.first;
      out.erase(it);
      freed.push_back(p);
      if (hook) hook();
   }
};
int Memory::dev = 0;
size_t Memory::room[2] = {1 << 20, 1 << 20};
std::map<char*, std::pair<size_t, int>> Memory::out;
std::vector<void*> Memory::freed;
std::function<void()> Memory::hook;

using Cache = fsvd::DeviceCache<Memory>;
#define CHECK(x) if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }

int main() {
   {  // reuse: same size, up to a quarter of waste, not more; sizes rounded up by at most 1/8
      Cache c;
      for (size_t n = 1; n < 200000; n += 37) {
         void* p = c.take(n);
         const size_t have = Memory::out[(char*)p].first;
         CHECK(have >= n && (n < 4096 ? have < n + 512 : have <= n + n / 8));
         c.give(p);
         c.trim();
      }
      void* p = c.take(5000);
      c.give(p);
      CHECK(c.take(3000) != p);
      CHECK(c.take(4200) == p);
      c.give(p);
      Memory::dev = 1;
      CHECK(c.take(5000) != p);   // another device's
      Memory::dev = 0;
      CHECK(c.take(5000) == p);
   }
   {  // the bound, per device, the longest kept first; a block above it is freed at once
      Cache c;
      std::vector<void*> p, q;
      for (int i = 0; i < 6; i++) p.push_back(c.take(4096));
      Memory::dev = 1;
      for (int i = 0; i < 4; i++) q.push_back(c.take(4096));
      void* big = c.take(20000);
      Memory::freed.clear();
      c.give(big);
      CHECK(Memory::freed == std::vector<void*>{big});
      Memory::freed.clear();
      c.give(p[3]);
      c.built();
      c.give(p[0]);
      c.give(p[1]);
      c.give(p[2]);
      for (void* x : q) c.give(x);
      CHECK(Memory::freed.empty());      // 16384 kept on each
      c.give(p[4]);
      CHECK(Memory::freed == std::vector<void*>{p[3]});
      Memory::dev = 0;
      CHECK(c.trim() == 8 * 4096 && Memory::freed.size() == 9);
      c.give(p[5]);
      CHECK(c.trim() == 4096);
   }
   {  // two builds that leave a block unused give it back at the third
      Cache c;
      void* p = c.take(4096);
      c.give(p);
      Memory::freed.clear();
      c.built();
      c.built();
      CHECK(Memory::freed.empty());
      c.built();
      CHECK(Memory::freed == std::vector<void*>{p});
   }
   {  // a failing allocation gives everything kept back and is tried again
      Cache c;
      std::vector<void*> p;
      for (int i = 0; i < 4; i++) p.push_back(c.take(4096));
      Memory::room[0] = 4096;
      for (void* x : p) c.give(x);
      Memory::freed.clear();
      void* r = c.take(16384);
      CHECK(r && Memory::freed.size() == 4);
      CHECK(!c.take(16384));
      Memory::room[0] = 1 << 20;
      c.give(r);
   }
   {  // unwinding: freed, not kept
      Cache c;
      struct Owner { Cache& c; void* p; ~Owner() { c.give(p); } };
      Memory::freed.clear();
      void* p = c.take(4096);
      try {
         Owner o{c, p};
         throw std::runtime_error("x");
      } catch (const std::exception&) {
      }
      CHECK(Memory::freed == std::vector<void*>{p});
      c.give(p);   // unknown by now: nothing happens
      CHECK(Memory::freed.size() == 1);
   }
   {  // another thread takes and gives while a block is being freed
      Cache c;
      void* p = c.take(4096);
      bool ran = false;
      Memory::hook = [&] {
         Memory::hook = nullptr;
         std::thread([&] { c.give(c.take(512)); ran = true; }).join();
      };
      c.give(p);
      c.trim();
      CHECK(ran);
   }
   std::puts("ok");
   return 0;
}
"""


def test_device_cache(tmp_path):
    src = tmp_path / "cache.cpp"
    src.write_text(SOURCE)
    exe = str(tmp_path / "cache")
    r = subprocess.run(["g++", "-std=c++17", "-g", "-Wall", "-Werror", "-I",
                        os.path.join(ROOT, "fftsvd_amd", "csrc"), str(src), "-o", exe, "-lpthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
