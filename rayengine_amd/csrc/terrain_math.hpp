// Gradient noise, fBm terrain field, bricked volume addressing and trilinear
// sampling, shared by the noise-fill and sphere-tracing kernels.
//
// The noise primitive follows eval / gradientDotV / quintic
// (RayEngine/src/cuda-src/sdf_functions.cuh:25-135) with its exact operation
// order.  The reference hashes through a 2D texture whose contents are
// undefined (a 2 KB table copied as 256 rows of 1 KB); this build defines the
// hash as P[P[P[x] + y] + z] on the doubled 512-entry permutation table that
// RPerlinNoise prepares (RayEngine/src/World/PerlinNoise.h:48-51).
#pragma once

#include "re_math.hpp"

namespace re {

// Volumes are stored in blocks of 4x4x4 voxels, x fastest inside a block and
// blocks x fastest: one 128-byte cache line holds a 4x4x2 block, so the 8
// corners of a trilinear cell usually share 1-2 lines, and a voxel's address
// is a sum of one short expression per axis.  (Morton order inside 8x8x8
// bricks shares its lines alike but takes twice the instructions to address.)
// The padded dimensions are multiples of kBrick, the unit of the kernels that
// go over whole volumes.
constexpr int kBlock = 4;
constexpr int kBlockVox = kBlock * kBlock * kBlock;
constexpr int kBrick = 8;
constexpr int kBrickVox = kBrick * kBrick * kBrick;

// Voxel l (0..63) of a block, and block b (0..7) of a brick: x, y, z.
RE_HD void block_voxel(uint32_t l, int& x, int& y, int& z) {
  x = (int)(l & 3u);
  y = (int)((l >> 2) & 3u);
  z = (int)(l >> 4);
}
RE_HD void brick_block(uint32_t b, int& x, int& y, int& z) {
  x = (int)(b & 1u);
  y = (int)((b >> 1) & 1u);
  z = (int)(b >> 2);
}

struct VolView {
  const float* data;
  int32_t dim[3];   // voxels per axis
  int32_t bdim[3];  // bricks per axis
  float spacing[3];
  // Set by make_view, for trilinear's grid coordinates and addresses.
  float inv[3];      // 1 / spacing, correctly rounded
  int32_t by_inv;    // 2: spacings are powers of two, p * inv is p / spacing; 1: quotients by div_by; 0: divide
  int32_t narrow;    // voxel offsets fit 30 bits and the block strides 24: 32-bit addresses
};

inline VolView make_view(const float* data, const int32_t* dim, const int32_t* bdim, const float* spacing) {
  VolView v;
  v.data = data;
  v.by_inv = 2;
  for (int a = 0; a < 3; ++a) {
    v.dim[a] = dim[a];
    v.bdim[a] = bdim[a];
    v.spacing[a] = spacing[a];
    v.inv[a] = 1.0f / spacing[a];
    int e = 0;
    const float m = frexpf(spacing[a], &e);
    // div_by's remainders are exact for spacings well inside the exponent range
    if (!(spacing[a] > 0.0f) || e < -40 || e > 40) v.by_inv = 0;
    else if (m != 0.5f && v.by_inv == 2) v.by_inv = 1;
  }
  const int64_t slab = (int64_t)bdim[0] * bdim[1] * (kBrickVox / 2);  // one layer of blocks
  v.narrow = slab < (1 << 24) && 2 * slab * bdim[2] <= (1 << 30);
  return v;
}

RE_HD int64_t vox_index(const int32_t* bdim, int x, int y, int z) {
  const int64_t b = ((int64_t)(z >> 2) * (2 * bdim[1]) + (y >> 2)) * (2 * bdim[0]) + (x >> 2);
  return b * kBlockVox + ((z & 3) << 4) + ((y & 3) << 2) + (x & 3);
}

// 16-case gradient dot product (sdf_functions.cuh:25-48) as s1*A + s2*B with
// A, B in {x, y, z} and s1, s2 = +-1, which rounds identically to each case
// (x - y == x + (-y) and multiplying by +-1 is exact).
RE_HD float grad_dot(uint32_t h, float x, float y, float z) {
  switch (h & 15u) {
    case 0: return x + y;
    case 1: return -x + y;
    case 2: return x - y;
    case 3: return -x - y;
    case 4: return x + z;
    case 5: return -x + z;
    case 6: return x - z;
    case 7: return -x - z;
    case 8: return y + z;
    case 9: return -y + z;
    case 10: return y - z;
    case 11: return -y - z;
    case 12: return y + x;
    case 13: return -x + y;
    case 14: return -y + z;
    default: return -y - z;
  }
}

// grad_dot's two coefficients as three, one of them zero: s1 A + s2 B =
// fma(gx, x, fma(gy, y, gz z)) to the bit for finite x, y, z (the products
// with 0 and +-1 are exact, so one rounding is left; a zero sum may differ in
// its sign, which the blend's later sums, all ending in 0 + amp * noise, do
// not show).
RE_HD f3 grad_coeffs(uint32_t h) {
  h &= 15u;
  const float s0 = (h & 1u) ? -1.0f : 1.0f, s1 = (h & 2u) ? -1.0f : 1.0f;
  if (h < 4u) return f3{s0, s1, 0.0f};
  if (h < 8u) return f3{s0, 0.0f, s1};
  if (h < 12u) return f3{0.0f, s0, s1};
  if (h == 12u) return f3{1.0f, 1.0f, 0.0f};
  if (h == 13u) return f3{-1.0f, 1.0f, 0.0f};
  return f3{0.0f, -1.0f, h == 14u ? 1.0f : -1.0f};
}

RE_HD float quintic(float t) { return t * t * t * (t * (t * 6 - 15) + 10); }

// One octave of noise_eval split in two: the cell-relative coordinates and
// fades of p in its lattice cell (fx, fy, fz = floor of p), and the blend of
// the eight corner gradients given the corners' hashes h[0..7] (corner order
// 000, 100, 010, 110, 001, 101, 011, 111 in x, y, z).
struct NoiseCell {
  float x0, x1, y0, y1, z0, z1, u, v, w;
};

RE_HD NoiseCell noise_cell(f3 p, int fx, int fy, int fz) {
  NoiseCell c;
  const float tx = p.x - (float)fx, ty = p.y - (float)fy, tz = p.z - (float)fz;
  c.u = quintic(tx);
  c.v = quintic(ty);
  c.w = quintic(tz);
  c.x0 = tx;
  c.x1 = tx - 1;
  c.y0 = ty;
  c.y1 = ty - 1;
  c.z0 = tz;
  c.z1 = tz - 1;
  return c;
}

// The blend of the corner gradients a, b, cc, d (z0), e, f, g, hh (z1).
RE_HD float noise_mix(float a, float b, float cc, float d, float e, float f, float g, float hh, float u, float v,
                      float w) {
  float k0 = a;
  float k1 = (b - a);
  float k2 = (cc - a);
  float k3 = (e - a);
  float k4 = (a + d - b - cc);
  float k5 = (a + f - b - e);
  float k6 = (a + g - cc - e);
  float k7 = (b + cc + e + hh - a - d - f - g);
  return k0 + k1 * u + k2 * v + k3 * w + k4 * u * v + k5 * u * w + k6 * v * w + k7 * u * v * w;
}

RE_HD float noise_blend(const uint32_t* h, const NoiseCell& c) {
  return noise_mix(grad_dot(h[0], c.x0, c.y0, c.z0), grad_dot(h[1], c.x1, c.y0, c.z0),
                   grad_dot(h[2], c.x0, c.y1, c.z0), grad_dot(h[3], c.x1, c.y1, c.z0),
                   grad_dot(h[4], c.x0, c.y0, c.z1), grad_dot(h[5], c.x1, c.y0, c.z1),
                   grad_dot(h[6], c.x0, c.y1, c.z1), grad_dot(h[7], c.x1, c.y1, c.z1), c.u, c.v, c.w);
}

// The corners' hashes of lattice cell (fx, fy, fz).
template <typename Table>
RE_HD void noise_hashes(const Table& P, int fx, int fy, int fz, uint32_t* h) {
  const int xi0 = fx & 255, yi0 = fy & 255, zi0 = fz & 255;
  const int xi1 = (xi0 + 1) & 255, yi1 = (yi0 + 1) & 255, zi1 = (zi0 + 1) & 255;
  const uint32_t px0 = P[xi0], px1 = P[xi1];
  const uint32_t p00 = P[px0 + yi0], p10 = P[px1 + yi0], p01 = P[px0 + yi1], p11 = P[px1 + yi1];
  h[0] = P[p00 + zi0];
  h[1] = P[p10 + zi0];
  h[2] = P[p01 + zi0];
  h[3] = P[p11 + zi0];
  h[4] = P[p00 + zi1];
  h[5] = P[p10 + zi1];
  h[6] = P[p01 + zi1];
  h[7] = P[p11 + zi1];
}

// P is the doubled table (512 entries, values 0..255).
template <typename Table>
RE_HD float noise_eval(const Table& P, f3 p) {
  const int fx = (int)floorf(p.x), fy = (int)floorf(p.y), fz = (int)floorf(p.z);
  uint32_t h[8];
  noise_hashes(P, fx, fy, fz, h);
  return noise_blend(h, noise_cell(p, fx, fy, fz));
}

struct FbmParams {
  int32_t octaves;
  float lacunarity, gain, base_freq, y_offset;
};

// Terrain field value: (p.y - y_offset) - sum_o gain^o * noise(p * base_freq *
// lacunarity^o), i.e. minus the density fBm(p) - (p.y - y_offset).  Positive
// above the surface, like the reference's terrain distance
// (RayEngine/src/cuda-src/sdf_functions.cuh:476-503).
// noise(q) is one octave of the noise at q (noise_eval, or an equivalent
// evaluation of it).
template <typename Noise>
RE_HD float fbm_field(const FbmParams& fp, f3 p, const Noise& noise) {
  float sum = 0.0f, amp = 1.0f, freq = fp.base_freq;
  for (int o = 0; o < fp.octaves; ++o) {
    sum = sum + amp * noise(f3{p.x * freq, p.y * freq, p.z * freq});
    freq = freq * fp.lacunarity;
    amp = amp * fp.gain;
  }
  return (p.y - fp.y_offset) - sum;
}

template <typename Table>
RE_HD float terrain_field(const Table& P, const FbmParams& fp, f3 p) {
  return fbm_field(fp, p, [&](f3 q) { return noise_eval(P, q); });
}

// p / s from the correctly rounded reciprocal r of s: two corrections by the
// exact remainder.  p * r lies within 2 ulp of the quotient, the first
// correction within 1, and from there the second gives the correctly rounded
// quotient (P. Markstein, "Computation of elementary functions on the IBM
// RISC System/6000 processor", 1990), as long as the remainders are exact:
// |p / s| in [2^-60, 2^60] and s in [2^-40, 2^40].  Five operations where the
// device's IEEE division takes eleven, one of them at a quarter of the rate.
RE_HD float div_by(float p, float s, float r) {
  const float q0 = p * r;
  const float q1 = fmaf(fmaf(-q0, s, p), r, q0);
  return fmaf(fmaf(-q1, s, p), r, q1);
}

// Grid coordinates p / spacing.
RE_HD f3 grid_coord(const VolView& V, f3 p) {
  if (V.by_inv == 2) return f3{p.x * V.inv[0], p.y * V.inv[1], p.z * V.inv[2]};
  if (V.by_inv == 1) {
    const f3 g{div_by(p.x, V.spacing[0], V.inv[0]), div_by(p.y, V.spacing[1], V.inv[1]),
               div_by(p.z, V.spacing[2], V.inv[2])};
    const float ax = fabsf(g.x), ay = fabsf(g.y), az = fabsf(g.z);
    // (a NaN in one coordinate comes from a NaN or infinite p and stays one)
    if (fminf(fminf(ax, ay), az) >= 0x1p-60f && fmaxf(fmaxf(ax, ay), az) <= 0x1p60f && !(ax != ax) && !(ay != ay) &&
        !(az != az))
      return g;
  }
  return f3{p.x / V.spacing[0], p.y / V.spacing[1], p.z / V.spacing[2]};
}

RE_HD int imin(int a, int b) { return a < b ? a : b; }
RE_HD int imax(int a, int b) { return a > b ? a : b; }

#if defined(__HIP_DEVICE_COMPILE__)
RE_HD uint32_t mul24(uint32_t a, uint32_t b) { return __umul24(a, b); }
#else
RE_HD uint32_t mul24(uint32_t a, uint32_t b) { return a * b; }
#endif

RE_HD float trilerp(const float* c, float tx, float ty, float tz) {
  float a0 = c[0] * (1.f - tx) + c[1] * tx;
  float b0 = c[2] * (1.f - tx) + c[3] * tx;
  float e = a0 * (1.f - ty) + b0 * ty;
  float a1 = c[4] * (1.f - tx) + c[5] * tx;
  float b1 = c[6] * (1.f - tx) + c[7] * tx;
  float f = a1 * (1.f - ty) + b1 * ty;
  return e * (1 - tz) + f * tz;
}

// The cell of a trilinear sample: the eight corner values (x fastest, then
// y, then z) and the position inside the cell.
struct TriCell {
  float c[8];
  float tx, ty, tz;
};

// Loads the cell of world point p: grid coordinate c = p / spacing, cell
// index clamped to [0, dim-2].  The marching kernels are bound by the vector
// instructions of this routine more than by its loads: 212 per sample with
// IEEE divisions and eight 64-bit Morton brick addresses, about 80 now.  An
// address is a sum of one part per axis, so a cell needs two parts per axis,
// and with NARROW (V.narrow: up to 4 GiB, which is every volume up to 1024^3)
// the parts are 32-bit offsets from a scalar base.  NARROW is a template
// parameter because the compiler merges the loads of a run-time branch's two
// sides into one set with 64-bit addresses.
template <bool NARROW>
RE_HD TriCell tri_load(const VolView& V, f3 p) {
  const f3 g = grid_coord(V, p);
  int ix = (int)g.x, iy = (int)g.y, iz = (int)g.z;
  ix = imax(imin(ix, V.dim[0] - 2), 0);
  iy = imax(imin(iy, V.dim[1] - 2), 0);
  iz = imax(imin(iz, V.dim[2] - 2), 0);
  TriCell t;
  t.tx = g.x - (float)ix;
  t.ty = g.y - (float)iy;
  t.tz = g.z - (float)iz;
  if (NARROW) {
    // (x >> 2) 64 + (x & 3) = x + 15 (x & ~3), and likewise 4 y + (y >> 2) (row - 16), 16 z + (z >> 2) (slab - 64)
    const uint32_t row = (uint32_t)V.bdim[0] * (2 * kBlockVox), slab = row * 2u * (uint32_t)V.bdim[1];
    uint32_t X[2], Y[2], Z[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t x = (uint32_t)(ix + k), y = (uint32_t)(iy + k), z = (uint32_t)(iz + k);
      X[k] = mul24(x & ~3u, 15u) + x;
      Y[k] = mul24(y >> 2, row - 16u) + (y << 2);
      Z[k] = mul24(z >> 2, slab - 64u) + (z << 4);
    }
    const char* const D = reinterpret_cast<const char*>(V.data);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t off = (X[k & 1] + Y[(k >> 1) & 1] + Z[k >> 2]) << 2;
      t.c[k] = *reinterpret_cast<const float*>(D + off);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) t.c[k] = V.data[vox_index(V.bdim, ix + (k & 1), iy + ((k >> 1) & 1), iz + (k >> 2))];
  }
  return t;
}

// Trilinear sample at world point p, lerps in x then y then z
// (interpolate / bilinear, RayEngine/src/cuda-src/sdf_functions.cuh:209-265).
template <bool NARROW>
RE_HD float trilinear(const VolView& V, f3 p) {
  const TriCell t = tri_load<NARROW>(V, p);
  return trilerp(t.c, t.tx, t.ty, t.tz);
}

}  // namespace re
