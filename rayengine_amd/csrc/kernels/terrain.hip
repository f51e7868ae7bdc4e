// Noise-volume generation and sphere tracing of the terrain field on gfx950.
//
// noise_fill_kernel: a wave per brick, the permutation table and its gradients
// staged in LDS, every wave store one block's contiguous 256 bytes.  Replaces
// generate_noise (RayEngine/src/cuda-src/renderer.cu:105-126), which used
// 8-thread blocks and a linear float2 grid.
//
// sdf_trace_kernel: one ray per lane.  Clip to the volume box, then the
// reference march (single_ray_sphere_trace,
// RayEngine/src/cuda-src/sphere_tracing.cuh:182-216): sample, step
// t += d * scale, then test d <= eps * t on the stepped t, at most max_steps
// samples.  Normals by forward differences of the sampled field with
// delta = min(0.001 t, 0.002) (compute_sdf_normal,
// RayEngine/src/cuda-src/sdf_functions.cuh:506-516).
#include <cmath>

#include "../device_paths.hpp"
#include "../terrain_math.hpp"

namespace re {
namespace {

// One octave's terms of one coordinate of a voxel: the lattice cell, the
// position in it and its fade.
struct AxisTerm {
  int cell;
  float t, fade;
  __device__ __forceinline__ void set(float q) {
    cell = (int)floorf(q);
    t = q - (float)cell;
    fade = quintic(t);
  }
};

// The permutation table doubled and scaled to byte offsets (4 P), and the
// gradients of the doubled table: the corner hash P[P[P[x] + y] + z] and its
// gradient are three reads, each address one add from the read before.
struct NoiseLds {
  uint32_t p4[512];
  float4 grad[512];
};

__device__ __forceinline__ uint32_t lds_p4(const NoiseLds& S, uint32_t byte) {
  return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(S.p4) + byte);
}

// The gradient of the corner with p = 4 P[P[x] + y] and lattice z.
__device__ __forceinline__ float4 lds_grad(const NoiseLds& S, uint32_t p, uint32_t z) {
  return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(S.grad) + ((p << 2) + (z << 4)));
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane));
}

// From this many 8^3 bricks on a wave takes a whole brick; below, a 4^3 block,
// since waves of whole bricks would leave SIMDs (1,024) without work: 128^3
// (4,096 bricks) 27 us against 43 in blocks, 96^3 (1,728) 22 either way, 64^3
// (512) 18 against 11.5, 40^3 (125) 22 against 8.4.
constexpr int64_t kNoiseWideBricks = 2048;

// Fills the volume with the terrain field, a wave per brick of (4 N)^3 voxels
// (N = 2 or 1), each lane N^3 voxels that lie 4 apart.  Bound by vector
// instructions.  The terms of an octave that depend on one coordinate only
// (cell, position, fade) are computed for the N coordinates a lane meets per
// axis instead of for its N^3 voxels, and a gradient's dot product is three
// multiply-adds with coefficients from LDS.  When the whole brick lies in one
// lattice cell (four of the five octaves of the 256^3 unit-cube terrain,
// aligned with it), eight lanes look the cell's corners up, the coefficients
// move to scalar registers and the voxels of a lane share the y and z parts;
// otherwise every lane looks its own up.
// The kernel before gave a lane two voxels of a 4^3 block with scalar branches
// where the block was in one cell and a divergent 16-case switch elsewhere:
// 256^3 in 368 us, now 138; 203 x 165 x 187, whose cells are not aligned with
// the blocks, 235 us, now 81.
template <int N>
__global__ void __launch_bounds__(256) noise_fill_kernel(float* __restrict__ out, const uint32_t* __restrict__ perm,
                                                         int32_t dx, int32_t dy, int32_t dz, int32_t bx, int32_t by,
                                                         uint32_t n_bricks, float sx, float sy, float sz, float ox,
                                                         float oy, float oz, FbmParams fp) {
  __shared__ NoiseLds S;
  for (int i = threadIdx.x; i < 512; i += 256) {
    const uint32_t h = perm[i];
    S.p4[i] = 4u * h;
    const f3 g = grad_coeffs(h);
    S.grad[i] = make_float4(g.x, g.y, g.z, 0.0f);
  }
  __syncthreads();
  // bricks of 4 N voxels: bx and by are 8-voxel bricks per axis
  // (at most 2^30 of them: dimensions go up to 4096)
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  if (w >= n_bricks) return;
  const int lane = threadIdx.x & 63;
  const uint32_t nx = (uint32_t)bx * (2 / N), ny = (uint32_t)by * (2 / N);
  const int gx = (int)(w % nx), gy = (int)((w / nx) % ny), gz = (int)(w / nx / ny);
  int lx, ly, lz;
  block_voxel((uint32_t)lane, lx, ly, lz);
  const int x0 = gx * (kBlock * N) + lx, y0 = gy * (kBlock * N) + ly, z0 = gz * (kBlock * N) + lz;
  float px[N], py[N], pz[N], sum[N * N * N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    px[k] = ox + (float)(x0 + kBlock * k) * sx;
    py[k] = oy + (float)(y0 + kBlock * k) * sy;
    pz[k] = oz + (float)(z0 + kBlock * k) * sz;
  }
#pragma unroll
  for (int k = 0; k < N * N * N; ++k) sum[k] = 0.0f;
  float amp = 1.0f, freq = fp.base_freq;
  for (int oct = 0; oct < fp.octaves; ++oct) {
    AxisTerm X[N], Y[N], Z[N];
    bool split = false;
    const int fx = __builtin_amdgcn_readfirstlane((int)floorf(px[0] * freq)),
              fy = __builtin_amdgcn_readfirstlane((int)floorf(py[0] * freq)),
              fz = __builtin_amdgcn_readfirstlane((int)floorf(pz[0] * freq));
#pragma unroll
    for (int k = 0; k < N; ++k) {
      X[k].set(px[k] * freq);
      Y[k].set(py[k] * freq);
      Z[k].set(pz[k] * freq);
      split = split || X[k].cell != fx || Y[k].cell != fy || Z[k].cell != fz;
    }
    if (__ballot(split) == 0ull) {
      const uint32_t xi = (uint32_t)(fx + (lane & 1)) & 255u, yi = (uint32_t)(fy + ((lane >> 1) & 1)) & 255u,
                     zi = (uint32_t)(fz + ((lane >> 2) & 1)) & 255u;
      const float4 e = lds_grad(S, lds_p4(S, lds_p4(S, 4u * xi) + 4u * yi), zi);
      float ex[8], ey[8], ez[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        ex[c] = lane_value(e.x, c);
        ey[c] = lane_value(e.y, c);
        ez[c] = lane_value(e.z, c);
      }
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const float zs[2] = {Z[k].t, Z[k].t - 1};
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const float ys[2] = {Y[j].t, Y[j].t - 1};
          float yz[8];
#pragma unroll
          for (int c = 0; c < 8; ++c) yz[c] = fmaf(ey[c], ys[(c >> 1) & 1], ez[c] * zs[c >> 2]);
#pragma unroll
          for (int i = 0; i < N; ++i) {
            const float xs[2] = {X[i].t, X[i].t - 1};
            float g[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) g[c] = fmaf(ex[c], xs[c & 1], yz[c]);
            const float v = noise_mix(g[0], g[1], g[2], g[3], g[4], g[5], g[6], g[7], X[i].fade, Y[j].fade, Z[k].fade);
            sum[(k * N + j) * N + i] = sum[(k * N + j) * N + i] + amp * v;
          }
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < N * N; ++q) {
        const AxisTerm A = X[q % N], B = Y[q / N];
        uint32_t p[4];  // 4 P[P[x] + y] of the four (x, y) corners
        {
          const uint32_t px0 = lds_p4(S, 4u * ((uint32_t)A.cell & 255u)),
                         px1 = lds_p4(S, 4u * ((uint32_t)(A.cell + 1) & 255u));
          const uint32_t yi0 = 4u * ((uint32_t)B.cell & 255u), yi1 = 4u * ((uint32_t)(B.cell + 1) & 255u);
          p[0] = lds_p4(S, px0 + yi0);
          p[1] = lds_p4(S, px1 + yi0);
          p[2] = lds_p4(S, px0 + yi1);
          p[3] = lds_p4(S, px1 + yi1);
        }
        const float xs[2] = {A.t, A.t - 1}, ys[2] = {B.t, B.t - 1};
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const uint32_t zi[2] = {(uint32_t)Z[k].cell & 255u, (uint32_t)(Z[k].cell + 1) & 255u};
          const float zs[2] = {Z[k].t, Z[k].t - 1};
          float g[8];
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const float4 e = lds_grad(S, p[c & 3], zi[c >> 2]);
            g[c] = fmaf(e.x, xs[c & 1], fmaf(e.y, ys[(c >> 1) & 1], e.z * zs[c >> 2]));
          }
          const float v = noise_mix(g[0], g[1], g[2], g[3], g[4], g[5], g[6], g[7], A.fade, B.fade, Z[k].fade);
          sum[k * N * N + q] = sum[k * N * N + q] + amp * v;
        }
      }
    }
    freq = freq * fp.lacunarity;
    amp = amp * fp.gain;
  }
  const int32_t bdim[3] = {bx, by, 0};  // (vox_index needs no z count)
#pragma unroll
  for (int q = 0; q < N * N * N; ++q) {
    const int x = x0 + kBlock * (q % N), y = y0 + kBlock * ((q / N) % N), z = z0 + kBlock * (q / (N * N));
    const bool in = x < dx && y < dy && z < dz;
    out[vox_index(bdim, x, y, z)] = in ? (py[(q / N) % N] - fp.y_offset) - sum[q] : 0.0f;
  }
}

// The field for any parameters, one voxel per thread: coordinates or
// frequencies that leave the range in which noise_fill_kernel's products with
// zero coefficients are exact.
struct LdsTable {
  const uint32_t* t;
  __device__ uint32_t operator[](uint32_t i) const { return t[i]; }
};

__global__ void __launch_bounds__(256) noise_fill_any_kernel(float* __restrict__ out,
                                                             const uint32_t* __restrict__ perm, int32_t dx, int32_t dy,
                                                             int32_t dz, int32_t bx, int32_t by, float sx, float sy,
                                                             float sz, float ox, float oy, float oz, FbmParams fp) {
  const int64_t brick = blockIdx.x;
  const int32_t bdim[3] = {bx, by, 0};
  const int gx = (int)(brick % bx), gy = (int)((brick / bx) % by), gz = (int)(brick / ((int64_t)bx * by));
  for (int m = threadIdx.x; m < kBrickVox; m += blockDim.x) {
    int qx, qy, qz, lx, ly, lz;
    brick_block((uint32_t)m >> 6, qx, qy, qz);
    block_voxel((uint32_t)m & 63u, lx, ly, lz);
    const int x = gx * kBrick + qx * kBlock + lx, y = gy * kBrick + qy * kBlock + ly, z = gz * kBrick + qz * kBlock + lz;
    float v = 0.0f;
    if (x < dx && y < dy && z < dz)
      v = terrain_field(LdsTable{perm}, fp, f3{ox + (float)x * sx, oy + (float)y * sy, oz + (float)z * sz});
    out[vox_index(bdim, x, y, z)] = v;
  }
}

template <bool NORMALS, bool NARROW>
__global__ void __launch_bounds__(256) sdf_trace_kernel(VolView V, float bx0, float by0, float bz0, float bx1,
                                                        float by1, float bz1, const float* __restrict__ ray_o,
                                                        const float* __restrict__ ray_d, int64_t n, int32_t max_steps,
                                                        float eps, float step_scale, int32_t step_rule,
                                                        float* __restrict__ t_out, uint8_t* __restrict__ hit_out,
                                                        int32_t* __restrict__ steps_out, float* __restrict__ nrm_out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const f3 o{ray_o[3 * i], ray_o[3 * i + 1], ray_o[3 * i + 2]};
  const f3 d{ray_d[3 * i], ray_d[3 * i + 1], ray_d[3 * i + 2]};
  const float bmin[3] = {bx0, by0, bz0}, bmax[3] = {bx1, by1, bz1};
  int32_t steps = 0;
  float t = kInf;
  const bool hit = plain_march<NARROW>(V, bmin, bmax, o, d, max_steps, eps, step_scale, step_rule, t, steps);
  t_out[i] = hit ? t : kInf;
  hit_out[i] = hit ? 1 : 0;
  if (steps_out) steps_out[i] = steps;
  if (NORMALS) {
    f3 nrm{0.0f, 0.0f, 0.0f};
    if (hit) {
      const float delta = fminf((float)(0.001 * (double)t), 0.002f);
      const f3 p = add(o, smul(t, d));
      const float c = trilinear<NARROW>(V, p);
      nrm = normalize(f3{trilinear<NARROW>(V, add(p, f3{delta, 0.0f, 0.0f})) - c,
                         trilinear<NARROW>(V, add(p, f3{0.0f, delta, 0.0f})) - c,
                         trilinear<NARROW>(V, add(p, f3{0.0f, 0.0f, delta})) - c});
    }
    nrm_out[3 * i] = nrm.x;
    nrm_out[3 * i + 1] = nrm.y;
    nrm_out[3 * i + 2] = nrm.z;
  }
}

// Brush distances (sphere_distance / aabb_distance,
// RayEngine/src/cuda-src/sdf_functions.cuh:422-437): |p| - r, and the box
// distance |max(|p| - s, 0)| + min(max(d.x, d.y, d.z), 0).
__device__ __forceinline__ float vlen(float x, float y, float z) { return sqrtf(x * x + y * y + z * z); }

__device__ __forceinline__ float box_distance(float px, float py, float pz, const float* s) {
  const float dx = fabsf(px) - s[0], dy = fabsf(py) - s[1], dz = fabsf(pz) - s[2];
  return vlen(fmaxf(dx, 0.0f), fmaxf(dy, 0.0f), fmaxf(dz, 0.0f)) + fminf(fmaxf(dx, fmaxf(dy, dz)), 0.0f);
}

// One brush applied to every voxel (insert_sphere_to_texture,
// RayEngine/src/cuda-src/renderer.cu:30-92): offset p = voxel point - brush
// point, optionally snapped in x and z; then, on (distance, material) pairs,
// SPHERE_ADD: sdf_smin (h = max(k - |a - b|, 0) / k, the pair of the smaller
// distance with h^2 k / 4 taken off its distance), SPHERE_SUBTRACT and
// CUBE_SUBTRACT: the pair of the larger distance against the negated brush
// distance (sdf_fmaxf), CUBE_ADD: the componentwise minimum (fminf on
// float2) -- sdf_functions.cuh:270-289.  A work-group takes eight consecutive
// 4^3 blocks, a wave per block, so that the kernel streams the volume once in
// the order of memory (8 bytes in and out per voxel).
__global__ void __launch_bounds__(256) volume_edit_kernel(EditLaunch L) {
  const uint32_t nx = 2u * (uint32_t)L.bdim[0], ny = 2u * (uint32_t)L.bdim[1];
  int lx, ly, lz;
  block_voxel((uint32_t)threadIdx.x & 63u, lx, ly, lz);
  for (uint32_t k = threadIdx.x >> 6; k < 8u; k += blockDim.x >> 6) {
    // (at most 2^30 blocks: dimensions go up to 4096)
    const uint32_t b = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 8u + k));
    const int x = (int)(b % nx) * kBlock + lx, y = (int)(b / nx % ny) * kBlock + ly, z = (int)(b / nx / ny) * kBlock + lz;
    if (x >= L.dim[0] || y >= L.dim[1] || z >= L.dim[2]) continue;
    const int64_t i = (int64_t)b * kBlockVox + (threadIdx.x & 63);
    float px = (float)x * L.spacing[0] - L.center[0];
    const float py = (float)y * L.spacing[1] - L.center[1];
    float pz = (float)z * L.spacing[2] - L.center[2];
    if (L.snap) {
      const float snap = L.extent[0];
      px = floorf(px - fabsf(fmodf(px, snap)));
      pz = floorf(pz - fabsf(fmodf(pz, snap)));
    }
    const float ad = L.data[i], am = L.mat[i];
    float rd = ad, rm = am;
    if (L.type == 0) {
      const float bd = vlen(px, py, pz) - L.extent[0];
      const float h = fmaxf(L.k - fabsf(ad - bd), 0.0f) / L.k;
      const bool a_min = ad < bd ? true : false;
      rd = (a_min ? ad : bd) - h * h * L.k * 0.25f;
      rm = a_min ? am : L.material;
    } else if (L.type == 1) {
      const float bd = -(vlen(px, py, pz) - L.extent[0]);
      if (!(ad > bd)) {
        rd = bd;
        rm = L.material;
      }
    } else if (L.type == 2) {
      const float bd = box_distance(px, py, pz, L.extent);
      rd = fminf(ad, bd);
      rm = fminf(am, L.material);
    } else {
      const float bd = -box_distance(px, py, pz, L.extent);
      if (!(ad > bd)) {
        rd = bd;
        rm = L.material;
      }
    }
    L.data[i] = rd;
    L.mat[i] = rm;
  }
}

}  // namespace

hipError_t launch_volume_edit(const EditLaunch& L, hipStream_t s) {
  const int64_t bricks = (int64_t)L.bdim[0] * L.bdim[1] * L.bdim[2];
  if (bricks <= 0) return hipSuccess;
  hipLaunchKernelGGL(volume_edit_kernel, dim3((unsigned)bricks), dim3(256), 0, s, L);
  return hipGetLastError();
}

hipError_t launch_noise_fill(const NoiseLaunch& L, hipStream_t s) {
  const int64_t bricks = (int64_t)L.bdim[0] * L.bdim[1] * L.bdim[2];
  // The largest coordinate any octave meets, in lattice cells.
  double reach = 0.0, freq = std::fabs((double)L.fbm.base_freq), most = freq;
  for (int o = 1; o < L.fbm.octaves; ++o) {
    freq *= std::fabs((double)L.fbm.lacunarity);
    most = freq > most ? freq : most;
  }
  for (int a = 0; a < 3; ++a) {
    const double r = std::fabs((double)L.origin[a]) + (double)L.bdim[a] * kBrick * (double)L.spacing[a];
    reach = r > reach ? r : reach;
  }
  if (!(reach * most < 1e30)) {
    hipLaunchKernelGGL(noise_fill_any_kernel, dim3((unsigned)bricks), dim3(256), 0, s, L.out, L.perm, L.dim[0],
                       L.dim[1], L.dim[2], L.bdim[0], L.bdim[1], L.spacing[0], L.spacing[1], L.spacing[2], L.origin[0],
                       L.origin[1], L.origin[2], L.fbm);
    return hipGetLastError();
  }
#define RE_LAUNCH(N, COUNT)                                                                                           \
  hipLaunchKernelGGL(noise_fill_kernel<N>, dim3((unsigned)(((COUNT) + 3) / 4)), dim3(256), 0, s, L.out, L.perm,       \
                     L.dim[0], L.dim[1], L.dim[2], L.bdim[0], L.bdim[1], (uint32_t)(COUNT), L.spacing[0], L.spacing[1],         \
                     L.spacing[2], L.origin[0], L.origin[1], L.origin[2], L.fbm)
  if (bricks >= kNoiseWideBricks) RE_LAUNCH(2, bricks);
  else RE_LAUNCH(1, 8 * bricks);
#undef RE_LAUNCH
  return hipGetLastError();
}

hipError_t launch_sdf_trace(const SdfLaunch& L, hipStream_t s) {
  if (L.n <= 0) return hipSuccess;
  const int block = L.block > 0 ? L.block : 64;  // one wave (with normals 74 us against 76 at 256, 2,073,600 rays)
  const int64_t grid = (L.n + block - 1) / block;
#define RE_LAUNCH(NRM, NARROW)                                                                                \
  hipLaunchKernelGGL((sdf_trace_kernel<NRM, NARROW>), dim3((unsigned)grid), dim3(block), 0, s, L.vol, L.box_min[0],  \
                     L.box_min[1], L.box_min[2], L.box_max[0], L.box_max[1], L.box_max[2], L.ray_o, L.ray_d, \
                     L.n, L.max_steps, L.eps, L.step_scale, L.step_rule, L.t, L.hit, L.steps, L.nrm)
  if (L.vol.narrow) {
    if (L.nrm) RE_LAUNCH(true, true); else RE_LAUNCH(false, true);
  } else {
    if (L.nrm) RE_LAUNCH(true, false); else RE_LAUNCH(false, false);
  }
#undef RE_LAUNCH
  return hipGetLastError();
}

}  // namespace re
