// Sums of what a level of the device kd build adds to the next one, at and
// beyond the 31 bits its references are indexed with (host build of
// kdbuild.hpp).  Prints what is wrong.
#include <cstddef>
#include <cstdio>
#include <initializer_list>

#include "../rayengine_amd/csrc/kdbuild.hpp"

using namespace re::kdb;

static int bad = 0;
static void check(bool ok, const char* what) {
  if (!ok) std::printf("%s\n", what);
  bad += !ok;
}

static const Params P{8, 64, 32, 1, 1.0f, 1.0f, 0.0f};

static LNode node(bool split, int32_t n, int32_t cl, int32_t cr) {
  LNode nd{};
  nd.n = n;
  nd.depth = 5;
  nd.split = split;
  nd.cl = cl;
  nd.cr = cr;
  return nd;
}

// The nodes' sum as a scan may take it: one by one, or both halves first.
static Adds sum(const LNode* v, int n, bool halves) {
  if (n == 1) return node_adds(v[0], P);
  const int m = halves ? n / 2 : n - 1;
  return AddsSum{}(sum(v, m, halves), sum(v + m, n - m, halves));
}

int main() {
  const int32_t top = 0x7fffffff;
  for (bool halves : {false, true}) {
    const LNode one[1] = {node(true, top, top, top)};  // every reference on both sides
    check(sum(one, 1, halves).refs == 2 * (int64_t)top && !level_fits(1, 0, sum(one, 1, halves)), "one node, all twice");
    const LNode four[4] = {node(true, 1 << 29, 1 << 29, 1 << 29), node(true, 1 << 29, 1 << 29, 1 << 29),
                           node(true, 1 << 29, 1 << 29, 1 << 29), node(true, 1 << 29, 1 << 29, 1 << 29)};
    check(sum(four, 4, halves).refs == (int64_t)1 << 32, "2^32 references");  // 0 in 32 bits
    check(!level_fits(7, 0, sum(four, 4, halves)), "2^32 references refused");
    check(!level_fits(7, 0, sum(four, 2, halves)), "2^31 references refused");
    const LNode fit[2] = {node(true, 1 << 30, 1 << 29, 1 << 29), node(true, top - (1 << 30), top - (1 << 30), 0)};
    check(sum(fit, 2, halves).refs == top && level_fits(3, 0, sum(fit, 2, halves)), "2^31 - 1 references accepted");
    check(level_fits(0x3fffffff - 4, 0, sum(fit, 2, halves)) && !level_fits(0x3fffffff - 3, 0, sum(fit, 2, halves)),
          "2^30 - 1 nodes");
    const LNode leaves[3] = {node(false, 1 << 30, 0, 0), node(false, 7, 0, 0), node(true, 2000, 1100, 1000)};
    const Adds a = sum(leaves, 3, halves);
    check(a.leaf == (1 << 30) + 7 && a.kids == 2 && a.refs == 2100, "mixed level");
    check(a.last == (kBigBit | (1u << 30)), "largest leaf and the bit of a big child");
    check(level_fits(3, top - a.leaf, a) && !level_fits(3, top - a.leaf + 1, a), "2^31 - 1 triangle records");
  }
  return bad != 0;
}
