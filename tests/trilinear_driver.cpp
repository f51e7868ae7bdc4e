// Compares the trilinear sample's fast paths with its plain form bit for bit
// on the host: quotients by reciprocal against IEEE division, 32-bit brick
// offsets against the general addresses.  Prints the number of mismatches.
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "../rayengine_amd/csrc/terrain_math.hpp"

using namespace re;

static uint32_t bits(float x) {
  uint32_t u;
  std::memcpy(&u, &x, 4);
  return u;
}

int main() {
  std::mt19937 rng(7);
  auto uni = [&](float lo, float hi) { return lo + (hi - lo) * (float)(rng() >> 8) * (1.0f / 16777216.0f); };
  long bad_div = 0, bad_cell = 0, n_div = 0, n_cell = 0;
  // quotients: spacings 1 / n, awkward mantissas, the ends of the exponent range
  std::vector<float> spacings;
  for (int n = 2; n <= 300; ++n) spacings.push_back(1.0f / (float)n);
  for (int k = 0; k < 200; ++k) spacings.push_back(std::ldexp(1.0f + (float)(rng() >> 9) * 0x1p-23f, (int)(rng() % 79) - 39));
  for (float m : {1.0f - 0x1p-24f, 1.0f + 0x1p-23f, 1.5f, 2.0f - 0x1p-23f})
    for (int e : {-38, -8, 0, 38}) spacings.push_back(std::ldexp(m, e));
  for (float s : spacings) {
    const float r = 1.0f / s;
    for (int k = 0; k < 4000; ++k) {
      // quotients over the guarded range, half of them next to whole numbers
      float q = std::ldexp(1.0f + (float)(rng() >> 9) * 0x1p-23f, (int)(rng() % 118) - 59);
      if (k & 1) q = (float)(rng() % 4096) + 1.0f;
      float p = q * s;
      if (k & 2) p = std::nextafter(p, (k & 4) ? INFINITY : -INFINITY);
      const float want = p / s;
      if (!(std::fabs(want) >= 0x1p-60f && std::fabs(want) <= 0x1p60f)) continue;
      ++n_div;
      if (bits(div_by(p, s, r)) != bits(want)) ++bad_div;
    }
  }
  // cells: volumes of every remainder of the brick size, points inside,
  // on the faces and outside
  struct Shape {
    int d[3];
    float sp[3];
  };
  std::vector<Shape> shapes = {{{2, 2, 2}, {0.5f, 0.5f, 0.5f}}, {{256, 16, 9}, {1.0f / 256, 1.0f / 256, 1.0f / 256}}};
  for (int k = 0; k < 40; ++k) {
    Shape sh;
    for (int a = 0; a < 3; ++a) {
      sh.d[a] = 2 + (int)(rng() % 40);
      sh.sp[a] = k % 3 == 0 ? 0.03125f : (k % 3 == 1 ? 1.0f / (float)sh.d[a] : uni(0.001f, 3.0f));
    }
    shapes.push_back(sh);
  }
  for (const Shape& sh : shapes) {
    int32_t bd[3];
    for (int a = 0; a < 3; ++a) bd[a] = (sh.d[a] + 7) / 8;
    std::vector<float> data((size_t)bd[0] * bd[1] * bd[2] * kBrickVox);
    for (float& v : data) v = uni(-1.0f, 1.0f);
    const VolView fast = make_view(data.data(), sh.d, bd, sh.sp);
    VolView plain = fast;
    plain.by_inv = 0;
    if (!fast.narrow) ++bad_cell;
    for (int k = 0; k < 20000; ++k) {
      float c[3];
      for (int a = 0; a < 3; ++a) {
        c[a] = uni(-0.5f, (float)sh.d[a] + 0.5f) * sh.sp[a];
        if (k % 5 == 1) c[a] = (float)(rng() % (unsigned)(sh.d[a] + 1)) * sh.sp[a];
        if (k % 7 == 2) c[a] = std::nextafter(c[a], -1.0f);
        if (k % 97 == 3 && a == k % 3) c[a] = (k & 1) ? 0.0f : -0.0f;
      }
      const f3 p{c[0], c[1], c[2]};
      ++n_cell;
      if (bits(trilinear<true>(fast, p)) != bits(trilinear<false>(plain, p))) ++bad_cell;
    }
  }
  std::printf("quotients %ld mismatches %ld\ncells %ld mismatches %ld\n", n_div, bad_div, n_cell, bad_cell);
  return bad_div || bad_cell ? 1 : 0;
}
