// The per-device value cache of the launchers, filled by several threads at
// once (built with -fsanitize=thread).
#include <cstdio>
#include <thread>
#include <vector>

#include "ocfd_device_cache.h"

static int looked_up(int dev) {
  static ocfd::DeviceCache cache;
  return cache.get(dev, [&] { return 100 + dev; });
}

int main() {
  std::vector<std::thread> t;
  std::vector<int> bad(8, 0);
  for (int i = 0; i < 8; i++)
    t.emplace_back([i, &bad] {
      for (int r = 0; r < 2000; r++)
        for (int dev = 0; dev < ocfd::DeviceCache::DEVICES; dev++) bad[i] += looked_up(dev) != 100 + dev;
    });
  for (auto &x : t) x.join();
  int n = 0;
  for (int x : bad) n += x;
  std::printf("wrong %d\n", n);
  return n != 0;
}
