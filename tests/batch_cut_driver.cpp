// The device's work list of a batch: every target's rays once, items of each
// kind's length, sphere-traced tiles in few items (host build of
// host/batch_plan.cpp).  Prints what is wrong.
#include <algorithm>
#include <cstdio>

#include "../rayengine_amd/csrc/host/batch_plan.hpp"

using namespace re;

static int bad = 0;
static void check(bool ok, const char* what, long a, long b) {
  if (!ok) std::printf("%s (%ld, %ld)\n", what, a, b);
  bad += !ok;
}

int main() {
  for (int32_t item : {1, 63, 64, 65, 256, 4096})
    for (long n : {1l, 63l, 65l, 65536l, 65537l, 131072l, 131073l, 1000003l, 30000000l}) {
      const int32_t per = plain_item_rays(n, item);
      check(per >= 1 && per <= item && per >= std::min(item, 64), "length", item, n);
      // never finer than the counter is read in good time, as far as item_rays lets it
      check(per == item || (n + per - 1) / per <= 1024, "items", item, n);
    }
  const long n = 400000;
  re_batch_scene scene{};
  scene.ray_begin = 0;
  scene.ray_count = 70001;
  re_batch_tile tiles[3] = {};
  const long begin[3] = {70001, 150000, 250007}, count[3] = {79999, 100007, 149993};
  const int mode[3] = {0, 1, 1};
  for (int k = 0; k < 3; ++k) {
    tiles[k].mode = mode[k];
    tiles[k].ray_begin = begin[k];
    tiles[k].ray_count = count[k];
  }
  const int32_t cut = 64, plain = plain_item_rays(count[1] + count[2], 256);
  BatchPlan p;
  check(plan_batch(&scene, 1, tiles, 3, n, cut, p, plain) == RE_OK, "plan", 0, 0);
  std::vector<char> seen(n, 0);
  std::vector<int32_t> items(4, 0);
  for (const BatchItem& it : p.items) {
    const int32_t per = it.kind == kItemPlain ? plain : cut;
    const int32_t s = it.slot;
    const long b = s == 0 ? 0 : begin[s - 1], c = s == 0 ? 70001 : count[s - 1];
    check(it.count == per || it.begin + it.count == b + c, "count", it.count, s);
    check(it.begin >= b && it.begin + it.count <= b + c, "range", it.begin, s);
    for (long r = it.begin; r < it.begin + it.count; ++r) ++seen[r];
    ++items[s];
  }
  for (long r = 0; r < n; ++r)
    if (seen[r] != 1) check(false, "ray taken other than once", r, seen[r]);
  check(items == p.remaining, "remaining", 0, 0);
  return bad != 0;
}
