// Host check of plh::capacity_key, built against the library and run by tests/test_capacity_key.py: two geometries
// with one key must be served by the same kernels, since the co-residency looked up for the first one asked
// (recurrent_capacity) sizes the launches of both.
#include <cstdio>
#include <map>
#include <string>
#include <vector>

#include "plh_internal.h"

using namespace plh;

// The variants a launch of this geometry may run (with and without lengths, each tile count, with and without the
// in-kernel layer-0 projection).
static std::vector<const void*> kernels(const Geometry& g, int tile_rows) {
  if (g.rec) {
    std::vector<const void*> k = {rec_kernel(g.HP, false)};
    if (g.rec_x0) k.push_back(rec_kernel(g.HP, true));
    return k;
  }
  if (g.slices > 1) {
    std::vector<const void*> k;
    for (int t = 1; t <= g.max_wg_tiles; ++t) k.push_back(sliced_kernel(g.HP, t));
    return k;
  }
  return {wavefront_kernel(g.HP, tile_rows, false, g.wide_ok != 0),
          wavefront_kernel(g.HP, tile_rows, true, g.wide_ok != 0)};
}

int main() {
  std::map<long long, std::vector<const void*>> seen;
  long bad = 0, n = 0;
  const int Is[] = {1, 5, 32, 33, 64, 100, 128, 129, 200, 256, 300, 512, 600, 1100};
  const int Hs[] = {1, 32, 33, 64, 65, 100, 128, 129, 200, 256, 257, 400, 512, 513, 800, 1024};
  for (int I : Is)
    for (int H : Hs)
      for (int rec = 0; rec < 2; ++rec)
        for (int rows = 8; rows <= 16; rows += 8) {
          Geometry g;
          std::string why;
          if (!make_geometry(I, H, 2, 3, &g, &why)) return std::printf("%s\n", why.c_str()), 1;
          if (rec ? !g.rec_ok : !(g.wave_ok || g.wide_ok)) continue;
          if (rec) g = as_layer_sequential(g);
          if (rows == 8 && (g.rec || g.slices > 1)) continue;
          const std::vector<const void*> k = kernels(g, rows);
          ++n;
          for (const void* f : k)
            if (!f) ++bad;
          const auto it = seen.emplace(capacity_key(0, g, rows), k).first;
          if (it->second != k || capacity_key(1, g, rows) == capacity_key(0, g, rows)) {
            ++bad;
            std::printf("I=%d H=%d rec=%d rows=%d shares a key with other kernels\n", I, H, rec, rows);
          }
        }
  std::printf("%ld geometries, %zu keys, %ld mismatches\n", n, seen.size(), bad);
  return bad != 0;
}
