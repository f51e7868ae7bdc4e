// Rope kd-tree construction on the device, breadth first: every level's
// nodes choose their split planes in parallel (one wave per node), their
// triangle references are partitioned (straddlers clipped in double
// precision) and scattered, in parent order, into the next level; then the
// preorder numbering, the ropes and the flat arrays are computed from the
// finished node set.  Each decision is the host builder's (host/kdtree.cpp)
// with the same floating-point operations in the same order, so the result
// is the host tree, entry for entry; the host build stays the reference the
// device build is tested against.  Replaces the host build of RKDTreeCPU
// (RayEngine/src/Primitives/KDTree.cpp:335-834) and its flattening
// (KDThreeGPU.cpp:155-194), which the reference runs on the CPU before every
// upload (timed at RTScene.cpp:186-198).
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../capi_util.hpp"
#include "../device_paths.hpp"
#include "../kdbuild.hpp"

namespace re {
namespace kdb {
namespace {

// ---------------------------------------------------------------- helpers

__device__ __forceinline__ float area_of(float dx, float dy, float dz) { return 2.0f * (dx * dy + dx * dz + dy * dz); }

// Surface-area cost of splitting box [lo, hi] on `axis` at `pos` with nl
// references below and nr above (host: Builder::cost_of).
__device__ __forceinline__ float split_cost(const Params& P, const float* lo, const float* hi, int axis, float pos,
                                            int64_t nl, int64_t nr, float inv_sa) {
  const float ex = hi[0] - lo[0], ey = hi[1] - lo[1], ez = hi[2] - lo[2];
  float al, ar;
  if (axis == 0) {
    al = area_of(pos - lo[0], ey, ez);
    ar = area_of(hi[0] - pos, ey, ez);
  } else if (axis == 1) {
    al = area_of(ex, pos - lo[1], ez);
    ar = area_of(ex, hi[1] - pos, ez);
  } else {
    al = area_of(ex, ey, pos - lo[2]);
    ar = area_of(ex, ey, hi[2] - pos);
  }
  float c = P.ct + P.ci * (al * (float)nl + ar * (float)nr) * inv_sa;
  if (nl == 0 || nr == 0) c *= P.eb;
  return c;
}

// nextafter(x, +inf) and nextafter(x, -inf) for finite or infinite x.
__device__ __forceinline__ float next_up(float x) {
  if (x != x || x == kInf) return x;
  if (x == 0.0f) return __uint_as_float(1u);
  const uint32_t u = __float_as_uint(x);
  return __uint_as_float(x > 0.0f ? u + 1u : u - 1u);
}
__device__ __forceinline__ float next_down(float x) {
  if (x != x || x == -kInf) return x;
  if (x == 0.0f) return __uint_as_float(0x80000001u);
  const uint32_t u = __float_as_uint(x);
  return __uint_as_float(x > 0.0f ? u - 1u : u + 1u);
}

__device__ __forceinline__ float get3(const float* v, int a) { return a == 0 ? v[0] : (a == 1 ? v[1] : v[2]); }

// std::min / std::max as the host builder uses them (the first argument
// unless the second compares strictly smaller / larger), so equal values of
// opposite zero sign are picked as on the host.
template <typename T>
__device__ __forceinline__ T smin(T a, T b) { return b < a ? b : a; }
template <typename T>
__device__ __forceinline__ T smax(T a, T b) { return a < b ? b : a; }

// Is (c, a, p) a better split than (bc, ba, bp)?  The host scans axes in
// order and candidates in ascending position and keeps a candidate only if
// its cost is strictly lower, so the winner is the lowest cost, then the
// lowest axis, then the lowest position; costs that are not below +inf
// (including NaN) never win.
__device__ __forceinline__ bool better(float c, int a, float p, float bc, int ba, float bp) {
  if (!(c < kInf)) return false;
  if (c < bc) return true;
  return c == bc && (a < ba || (a == ba && p < bp));
}

// Bounding box of triangle `prim` clipped to [lo, hi] grown by a relative
// tolerance (Sutherland-Hodgman in double precision), intersected with
// [lo, hi] (host: Builder::clip_box).  A triangle clipped by six planes has
// at most 9 vertices.  poly2 holds the lane's two polygons, read and written
// in turn, in LDS with a column per lane (no bank conflicts); a vertex is read
// once and its distance kept for the next edge.  With the polygons in scratch
// memory, copied back after each plane and each vertex read twice, the kernel
// was the build's largest: 2^20 triangles 8.4 ms of device time and 5.7 now,
// 2^18 3.20 and 2.57 (one read a vertex but in scratch: 6.6 and 2.75).
constexpr int kMaxV = 10;
__device__ bool clip_box(const float* __restrict__ tv, int32_t prim, const float* lo, const float* hi, Ref& out,
                         double (*poly2)[64]) {
  const int lane = threadIdx.x;
  int np = 3, cur = 0;
  const float* t = tv + 9 * (int64_t)prim;
  for (int v = 0; v < 3; ++v)
    for (int a = 0; a < 3; ++a) poly2[3 * v + a][lane] = t[3 * v + a];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double tol = 1e-6 * (fabs((double)lo[a]) + fabs((double)hi[a]) + 1e-3);
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      if (np == 0) continue;
      const double plane = side == 0 ? (double)lo[a] - tol : (double)hi[a] + tol;
      const double sgn = side == 0 ? 1.0 : -1.0;
      double(*const in)[64] = poly2 + cur * 3 * kMaxV;
      double(*const to)[64] = poly2 + (cur ^ 1) * 3 * kMaxV;
      double P[3] = {in[0][lane], in[1][lane], in[2][lane]};
      const double first[3] = {P[0], P[1], P[2]};
      double dp = sgn * (P[a] - plane);
      const double dfirst = dp;
      int nq = 0;
      for (int v = 0; v < np; ++v) {
        // the next vertex, and after the last one the first
        double Q[3] = {first[0], first[1], first[2]}, dq = dfirst;
        if (v + 1 < np) {
          for (int k = 0; k < 3; ++k) Q[k] = in[3 * (v + 1) + k][lane];
          dq = sgn * (Q[a] - plane);
        }
        if (dp >= 0.0 && nq < kMaxV) {
          for (int k = 0; k < 3; ++k) to[3 * nq + k][lane] = P[k];
          ++nq;
        }
        if ((dp >= 0.0) != (dq >= 0.0) && nq < kMaxV) {
          const double s = dp / (dp - dq);
          for (int k = 0; k < 3; ++k) to[3 * nq + k][lane] = P[k] + s * (Q[k] - P[k]);
          ++nq;
        }
        for (int k = 0; k < 3; ++k) P[k] = Q[k];
        dp = dq;
      }
      np = nq;
      cur ^= 1;
    }
  }
  double(*const poly)[64] = poly2 + cur * 3 * kMaxV;
  if (np == 0) return false;
  out.prim = prim;
  for (int a = 0; a < 3; ++a) {
    double mn = poly[a][lane], mx = poly[a][lane];
    for (int v = 1; v < np; ++v) {
      mn = smin(mn, poly[3 * v + a][lane]);
      mx = smax(mx, poly[3 * v + a][lane]);
    }
    const float fl = next_down((float)mn), fh = next_up((float)mx);
    out.lo[a] = smax(fl, lo[a]);
    out.hi[a] = smin(fh, hi[a]);
    if (out.lo[a] > out.hi[a]) out.lo[a] = out.hi[a] = smin(smax((float)mn, lo[a]), hi[a]);
  }
  return true;
}

// ---------------------------------------------------------------- per level

// What the host keeps of the soup: per axis the vertex that gives the root
// box its minimum and its maximum, as keys (value in unsigned order, vertex
// index) whose minimum is taken, and whether any coordinate is not finite.
// The host scans vertices in order and replaces a bound only by a strictly
// lower (higher) value, so among equal values, +0 and -0 included, the first
// vertex wins: the key's low word.
struct SoupBounds {
  unsigned long long lo[3], hi[3];
  uint32_t bad;
};

__device__ __forceinline__ uint32_t ordered(float x) {
  const uint32_t u = __float_as_uint(x == 0.0f ? 0.0f : x);
  return (u & 0x80000000u) ? ~u : u | 0x80000000u;
}

__global__ void clear_bounds_kernel(SoupBounds* __restrict__ b) {
  if (threadIdx.x < 3) b->lo[threadIdx.x] = b->hi[threadIdx.x] = ~0ull;
  if (threadIdx.x == 0) b->bad = 0;
}

// The root's references, and the bounds of the soup on the way (a pass of their
// own on the host before: a build of 2^18 triangles 5.52 ms, now 5.25).  At
// most kInitBlocks blocks, so that few blocks add to the bounds.
constexpr int kInitBlocks = 512;

__global__ void __launch_bounds__(256) init_refs_kernel(const float* __restrict__ tv, int64_t n,
                                                        Ref* __restrict__ refs, int32_t* __restrict__ ref_node,
                                                        SoupBounds* __restrict__ bounds) {
  __shared__ unsigned long long sh[6];
  __shared__ int any_bad;
  if (threadIdx.x < 6) sh[threadIdx.x] = ~0ull;
  if (threadIdx.x == 0) any_bad = 0;
  __syncthreads();
  unsigned long long kl[3] = {~0ull, ~0ull, ~0ull}, kh[3] = {~0ull, ~0ull, ~0ull};
  bool bad = false;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float* t = tv + 9 * i;
    Ref r;
    r.prim = (int32_t)i;
    for (int a = 0; a < 3; ++a) {
      const float v[3] = {t[a], t[3 + a], t[6 + a]};
      r.lo[a] = smin(smin(v[0], v[1]), v[2]);
      r.hi[a] = smax(smax(v[0], v[1]), v[2]);
      for (int k = 0; k < 3; ++k) {
        bad = bad || !isfinite(v[k]);
        const uint32_t o = ordered(v[k]);
        const unsigned long long at = (unsigned long long)(3 * i + k);
        kl[a] = min(kl[a], ((unsigned long long)o << 32) | at);
        kh[a] = min(kh[a], ((unsigned long long)(~o) << 32) | at);
      }
    }
    refs[i] = r;
    ref_node[i] = 0;
  }
  for (int a = 0; a < 3; ++a) {
    for (int off = 32; off >= 1; off >>= 1) {
      kl[a] = min(kl[a], (unsigned long long)__shfl_xor((unsigned long long)kl[a], off));
      kh[a] = min(kh[a], (unsigned long long)__shfl_xor((unsigned long long)kh[a], off));
    }
    if ((threadIdx.x & 63) == 0) {
      atomicMin(&sh[a], kl[a]);
      atomicMin(&sh[3 + a], kh[a]);
    }
  }
  if (bad) any_bad = 1;
  __syncthreads();
  if (threadIdx.x < 3) atomicMin(&bounds->lo[threadIdx.x], sh[threadIdx.x]);
  else if (threadIdx.x < 6) atomicMin(&bounds->hi[threadIdx.x - 3], sh[threadIdx.x]);
  if (threadIdx.x == 6 && any_bad) atomicOr(&bounds->bad, 1u);
}

__device__ __forceinline__ int bin_of(float v, float lo, float hi, float scale, int nb) {
  const float pc = smin(smax(v, lo), hi);
  return min(nb - 1, max(0, (int)((pc - lo) * scale)));
}

// Adds a reference to its node's bin counts: per axis a, the bin of its
// clamped minimum (row 2 a) and of its clamped maximum (row 2 a + 1).
__device__ __forceinline__ void bin_ref(const Ref& r, const LNode& nd, int nb, int32_t* h) {
  for (int a = 0; a < 3; ++a) {
    const float lo = get3(nd.lo, a), hi = get3(nd.hi, a), ext = hi - lo;
    if (!(ext > 0.0f)) continue;
    const float scale = (float)nb / ext;
    atomicAdd(&h[(2 * a) * nb + bin_of(get3(r.lo, a), lo, hi, scale, nb)], 1);
    atomicAdd(&h[(2 * a + 1) * nb + bin_of(get3(r.hi, a), lo, hi, scale, nb)], 1);
  }
}

// Bin counts of the nodes too large for one wave (host: find_split, binned
// branch).  A chunk of kBinChunk references belongs to at most two of them,
// its first reference's node and its last's: both are counted in LDS and
// added to the node's histogram once per chunk.  (Counting the references of
// mixed chunks, most of them once nodes are a few thousand references large,
// with global atomics took 26 us per level on a 2^18-triangle soup; 10 us
// now, in the two thirds of the levels that have such nodes.)
__global__ void __launch_bounds__(256) bin_count_kernel(const Ref* __restrict__ refs,
                                                        const int32_t* __restrict__ ref_node, int64_t nref,
                                                        const LNode* __restrict__ nodes, int32_t* __restrict__ hist,
                                                        Params P) {
  __shared__ int32_t sh[2][6 * kMaxBins];
  const int nb = max(4, P.n_bins);
  const int64_t c0 = (int64_t)blockIdx.x * kBinChunk;
  const int64_t c1 = min(c0 + (int64_t)kBinChunk, nref);
  const int32_t first = ref_node[c0], last = ref_node[c1 - 1];
  const bool big0 = nodes[first].mode == kModeBig, big1 = last != first && nodes[last].mode == kModeBig;
  if (!big0 && !big1) return;
  for (int k = threadIdx.x; k < 6 * nb; k += blockDim.x) sh[0][k] = sh[1][k] = 0;
  __syncthreads();
  for (int64_t i = c0 + threadIdx.x; i < c1; i += blockDim.x) {
    const int32_t node = ref_node[i];
    if (node == first ? big0 : (node == last && big1)) bin_ref(refs[i], nodes[node], nb, sh[node == first ? 0 : 1]);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < 6 * nb; k += blockDim.x) {
    if (sh[0][k]) atomicAdd(&hist[nodes[first].rbegin / kBinChunk * (6 * nb) + k], sh[0][k]);
    if (sh[1][k]) atomicAdd(&hist[nodes[last].rbegin / kBinChunk * (6 * nb) + k], sh[1][k]);
  }
}

struct Plane {
  float cost, pos;
  int axis, nl, nr;
};

// The best bin plane of a node from its bin counts h (LDS): lane k costs the
// plane between bins k - 1 and k.
__device__ __forceinline__ Plane binned_plane(const float* nlo, const float* nhi, int n, const int32_t* h, int nb,
                                              float inv_sa, const Params& P) {
  const int k = threadIdx.x & 63;
  Plane best{kInf, 0.0f, -1, 0, 0};
  for (int a = 0; a < 3; ++a) {
    const float lo = nlo[a], hi = nhi[a];
    const float ext = hi - lo;
    if (!(ext > 0.0f)) continue;
    // references with their minimum below the plane, and all but those with
    // their maximum below it
    const uint32_t cmin = k < nb ? (uint32_t)h[(2 * a) * nb + k] : 0u;
    const uint32_t cmax = k < nb ? (uint32_t)h[(2 * a + 1) * nb + k] : 0u;
    const int nl = (int)(wave_incl_scan(cmin) - cmin), nr = n - (int)(wave_incl_scan(cmax) - cmax);
    float c = kInf, pos = 0.0f;
    if (k >= 1 && k < nb) {
      pos = lo + ext * (float)k / (float)nb;
      if (pos > lo && pos < hi) c = split_cost(P, nlo, nhi, a, pos, nl, nr, inv_sa);
      if (!(c < kInf)) c = kInf;  // NaN never wins; keep the reduction's order total
    }
    // lowest cost, then lowest k, across the wave
    float wc = c;
    int wk = (c < kInf) ? k : 1 << 20;
    for (int off = 32; off >= 1; off >>= 1) {
      const float oc = __shfl_xor(wc, off);
      const int ok = __shfl_xor(wk, off);
      if (oc < wc || (oc == wc && ok < wk)) {
        wc = oc;
        wk = ok;
      }
    }
    if (wk < (1 << 20)) {
      const float wpos = __shfl(pos, wk);
      const int wnl = __shfl(nl, wk), wnr = __shfl(nr, wk);
      if (better(wc, a, wpos, best.cost, best.axis, best.pos)) best = Plane{wc, wpos, a, wnl, wnr};
    }
  }
  return best;
}

struct ExactLds {
  float2 iv[3][kExactMax + 1];  // per axis: {lo, hi} of each reference; the pad spreads the axes over the banks
};

// The best plane of a node with at most 64 references: every reference's
// minimum and the float just past its maximum are candidate planes (host:
// find_split, exact branch).  The node's 6 n candidates (axis, reference,
// side) are dealt to the lanes; each lane counts the references below and
// above its own plane by walking the n reference intervals of its axis in LDS
// (the lanes of an axis read one address, a broadcast) and costs the plane
// once, and the wave then reduces to the winner.  Bound by vector-instruction
// issue.  The form before took the candidates one at a time with every lane
// costing the same plane, 6 n rounds of two ballots, a cross-lane read and
// the cost: 109 us per level on a 2^18-triangle soup against 14 us.
__device__ __forceinline__ Plane exact_plane(const float* nlo, const float* nhi, int n, const Ref* __restrict__ refs,
                                             ExactLds& S, float inv_sa, const Params& P) {
  const int lane = threadIdx.x & 63;
  if (lane < n) {
    const Ref r = refs[lane];
    for (int a = 0; a < 3; ++a) S.iv[a][lane] = make_float2(r.lo[a], r.hi[a]);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float bc = kInf, bp = 0.0f;
  int ba = 3, bq = 0, bnl = 0, bnr = 0;  // axis 3: none
  for (int e = lane; e < 6 * n; e += 64) {
    const int a = e >= 4 * n ? 2 : (e >= 2 * n ? 1 : 0);
    const int q = e - 2 * n * a;
    const float2 own = S.iv[a][q >> 1];
    const float pos = (q & 1) ? next_up(own.y) : own.x;
    const float lo = get3(nlo, a), hi = get3(nhi, a);
    if (!(hi - lo > 0.0f) || !(pos > lo && pos < hi)) continue;
    int nl = 0, nr = 0;
    for (int k = 0; k < n; ++k) {
      const float2 r = S.iv[a][k];
      nl += r.x < pos ? 1 : 0;
      nr += r.y >= pos ? 1 : 0;
    }
    const float c = split_cost(P, nlo, nhi, a, pos, nl, nr, inv_sa);
    if (better(c, a, pos, bc, ba, bp)) {
      bc = c;
      ba = a;
      bp = pos;
      bq = q;
      bnl = nl;
      bnr = nr;
    }
  }
  // The winner over the lanes.  Planes at +0 and -0 compare equal (and have
  // equal counts): the lower candidate index q of the axis is taken, as when
  // the candidates are scanned in order.
  for (int off = 32; off >= 1; off >>= 1) {
    const float oc = __shfl_xor(bc, off), op = __shfl_xor(bp, off);
    const int oa = __shfl_xor(ba, off), oq = __shfl_xor(bq, off), ol = __shfl_xor(bnl, off),
              orr = __shfl_xor(bnr, off);
    if (better(oc, oa, op, bc, ba, bp) || (oc < kInf && oc == bc && oa == ba && op == bp && oq < bq)) {
      bc = oc;
      ba = oa;
      bp = op;
      bq = oq;
      bnl = ol;
      bnr = orr;
    }
  }
  return Plane{bc, bp, ba == 3 ? -1 : ba, bnl, bnr};
}

// One wave per node: its split plane, by every candidate or by bins.  A node
// of 65 to kWaveBinMax references is binned here, in the wave's own LDS
// histogram, a larger one's counts come from bin_count_kernel.
union SplitLds {
  ExactLds exact;
  int32_t hist[6 * kMaxBins];
};

__global__ void __launch_bounds__(256) split_kernel(LNode* __restrict__ nodes, int32_t nn,
                                                    const Ref* __restrict__ refs, const int32_t* __restrict__ hist,
                                                    Params P) {
  __shared__ SplitLds lds[4];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  if (w >= nn) return;
  LNode& nd = nodes[w];
  const int mode = nd.mode;
  if (mode == kModeLeaf) return;
  SplitLds& S = lds[threadIdx.x >> 6];
  const int n = nd.n;
  const float nlo[3] = {nd.lo[0], nd.lo[1], nd.lo[2]}, nhi[3] = {nd.hi[0], nd.hi[1], nd.hi[2]};
  const float sa = area_of(nhi[0] - nlo[0], nhi[1] - nlo[1], nhi[2] - nlo[2]);
  const float inv_sa = sa > 0.0f ? 1.0f / sa : 0.0f;
  Plane best;
  if (mode == kModeExact) {
    best = exact_plane(nlo, nhi, n, refs + nd.rbegin, S.exact, inv_sa, P);
  } else {
    const int nb = max(4, P.n_bins);
    const int32_t* g = hist + nd.rbegin / kBinChunk * (6 * nb);
    for (int k = lane; k < 6 * nb; k += 64) S.hist[k] = mode == kModeBig ? g[k] : 0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (mode == kModeBinned) {
      for (int i = lane; i < n; i += 64) bin_ref(refs[nd.rbegin + i], nd, nb, S.hist);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    best = binned_plane(nlo, nhi, n, S.hist, nb, inv_sa, P);
  }
  if (lane == 0) {
    nd.axis = best.axis;
    nd.pos = best.pos;
    nd.nl = best.nl;
    nd.nr = best.nr;
  }
}

__device__ __forceinline__ bool will_try(const LNode& nd) {
  return nd.mode != kModeLeaf && nd.axis >= 0 && !(nd.nl == nd.n && nd.nr == nd.n);
}

// Which side(s) each reference goes to (host: build, partition loop): the
// flags word holds the below side in bit 0 and the above side in bit 32, so
// that one scan ranks both.  References that straddle the plane while
// clipping is on are listed for part_clip_kernel, which clips them with full
// waves.  A block covers kFlagChunk references and takes its part of the list
// with one atomic: with one per wave (and two more per wave on the node's
// counts, which now come from the scan) the top levels, where every wave adds
// to one address, took 289 us per launch on 2^20 triangles.
constexpr int kFlagChunk = 1024;
constexpr uint64_t kBelow = 1ull, kAbove = 1ull << 32;

__global__ void __launch_bounds__(256) part_flags_kernel(const Ref* __restrict__ refs,
                                                         const int32_t* __restrict__ ref_node, int64_t nref,
                                                         const LNode* __restrict__ nodes, Params P,
                                                         uint64_t* __restrict__ flags, int32_t* __restrict__ strad,
                                                         int32_t* __restrict__ n_strad) {
  __shared__ int32_t list[kFlagChunk];
  __shared__ int32_t n_list, base;
  if (threadIdx.x == 0) n_list = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int64_t c0 = (int64_t)blockIdx.x * kFlagChunk;
  for (int k = 0; k < kFlagChunk; k += 256) {
    const int64_t i = c0 + k + threadIdx.x;
    bool st = false;
    if (i < nref) {
      uint64_t f = 0;
      const LNode& nd = nodes[ref_node[i]];
      if (will_try(nd)) {
        const bool to_l = refs[i].lo[nd.axis] < nd.pos, to_r = refs[i].hi[nd.axis] >= nd.pos;
        st = to_l && to_r && P.clip;
        if (!st) f = (to_l ? kBelow : 0) | (to_r ? kAbove : 0);
      }
      flags[i] = f;
    }
    const unsigned long long sm = __ballot(st);
    if (sm) {
      int at = 0;
      if (lane == 0) at = atomicAdd(&n_list, __popcll(sm));
      at = __builtin_amdgcn_readfirstlane(at);
      if (st) list[at + __popcll(sm & ((1ull << lane) - 1ull))] = (int32_t)i;
    }
  }
  __syncthreads();
  const int m = n_list;
  if (threadIdx.x == 0 && m > 0) base = atomicAdd(n_strad, m);
  __syncthreads();
  for (int k = threadIdx.x; k < m; k += 256) strad[base + k] = list[k];
}

// Thread 2s + side clips straddler s against the below (side 0) or above
// (side 1) child box (host: Builder::clip_box on both children).  The two
// threads of a straddler are neighbouring lanes; the even one writes its
// flags.
__global__ void __launch_bounds__(64) part_clip_kernel(const float* __restrict__ tv, const Ref* __restrict__ refs,
                                                        const int32_t* __restrict__ ref_node,
                                                        const LNode* __restrict__ nodes,
                                                        const int32_t* __restrict__ strad,
                                                        const int32_t* __restrict__ n_strad,
                                                        uint64_t* __restrict__ flags, Ref* __restrict__ box_l,
                                                        Ref* __restrict__ box_r) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  __shared__ double poly2[2 * 3 * kMaxV][64];
  const int64_t ns = *n_strad;
  if ((t - (threadIdx.x & 63)) >= 2 * ns) return;  // whole waves past the list leave together
  int ok = 0;
  const int side = (int)(t & 1);
  int64_t i = 0;
  if (t < 2 * ns) {
    i = strad[t >> 1];
    const LNode& nd = nodes[ref_node[i]];
    float lo[3] = {nd.lo[0], nd.lo[1], nd.lo[2]}, hi[3] = {nd.hi[0], nd.hi[1], nd.hi[2]};
    if (side == 0) {
      if (nd.axis == 0) hi[0] = nd.pos;
      else if (nd.axis == 1) hi[1] = nd.pos;
      else hi[2] = nd.pos;
    } else {
      if (nd.axis == 0) lo[0] = nd.pos;
      else if (nd.axis == 1) lo[1] = nd.pos;
      else lo[2] = nd.pos;
    }
    Ref c;
    ok = clip_box(tv, refs[i].prim, lo, hi, c, poly2) ? 1 : 0;
    if (ok) (side == 0 ? box_l : box_r)[i] = c;
  }
  const unsigned long long m = __ballot(ok);
  if (t < 2 * ns && side == 0) {
    const unsigned long long two = m >> (threadIdx.x & 63);
    flags[i] = ((two & 1ull) ? kBelow : 0) | ((two & 2ull) ? kAbove : 0);
  }
}

// The split decision of every node, its below and above counts taken from
// the scan of its references' flags (flags_x exclusive; a node's references
// are contiguous).
__global__ void decide_kernel(LNode* __restrict__ nodes, int32_t nn, const uint64_t* __restrict__ flags,
                              const uint64_t* __restrict__ flags_x, Params P, Adds* __restrict__ adds) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nn) return;
  LNode& nd = nodes[i];
  if (nd.n > 0) {
    const int64_t last = nd.rbegin + nd.n - 1;
    const uint64_t c = flags_x[last] + flags[last] - flags_x[nd.rbegin];
    nd.cl = (int32_t)(uint32_t)c;
    nd.cr = (int32_t)(c >> 32);
  }
  nd.split = (will_try(nd) && !(nd.cl == nd.n && nd.cr == nd.n)) ? 1 : 0;
  adds[i] = node_adds(nd, P);
}

// Totals of the scan over a level's nodes, to pinned host memory (read after
// the stream's synchronisation); the straddler list starts empty again for
// the next level.
__global__ void totals_kernel(const Adds* adds, const Adds* adds_x, int64_t nn, Adds* out, int32_t* n_strad) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    *out = AddsSum{}(adds_x[nn - 1], adds[nn - 1]);
    *n_strad = 0;
  }
}

__global__ void emit_kernel(LNode* __restrict__ nodes, int32_t nn, const Adds* __restrict__ adds_x,
                            LNode* __restrict__ next, int32_t next_gid, int64_t pool_base, GNode* __restrict__ gn,
                            Params P) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nn) return;
  LNode& nd = nodes[i];
  GNode g;
  for (int a = 0; a < 3; ++a) {
    g.lo[a] = nd.lo[a];
    g.hi[a] = nd.hi[a];
  }
  g.depth = nd.depth;
  if (nd.split) {
    const int c = adds_x[i].kids;
    nd.child = c;
    nd.crbegin = adds_x[i].refs;
    LNode b{}, u{};
    for (int a = 0; a < 3; ++a) {
      b.lo[a] = u.lo[a] = nd.lo[a];
      b.hi[a] = u.hi[a] = nd.hi[a];
    }
    if (nd.axis == 0) { b.hi[0] = nd.pos; u.lo[0] = nd.pos; }
    else if (nd.axis == 1) { b.hi[1] = nd.pos; u.lo[1] = nd.pos; }
    else { b.hi[2] = nd.pos; u.lo[2] = nd.pos; }
    b.rbegin = nd.crbegin;
    b.n = nd.cl;
    u.rbegin = nd.crbegin + nd.cl;
    u.n = nd.cr;
    b.depth = u.depth = nd.depth + 1;
    b.mode = mode_of(b.n, b.depth, P);
    u.mode = mode_of(u.n, u.depth, P);
    b.gid = next_gid + c;
    u.gid = next_gid + c + 1;
    next[c] = b;
    next[c + 1] = u;
    g.axis = nd.axis;
    g.split = nd.pos;
    g.child0 = b.gid;
    g.child1 = u.gid;
    g.pool_n = 0;
    g.pool = 0;
  } else {
    nd.pool = pool_base + adds_x[i].leaf;
    g.axis = -1;
    g.split = 0.0f;
    g.child0 = g.child1 = -1;
    g.pool_n = nd.n;
    g.pool = nd.pool;
  }
  gn[nd.gid] = g;
}

// Each reference to its place in the children (the clipped boxes are those
// of the straddlers only; every other reference keeps its box) or, in a leaf,
// to the pool.
__global__ void scatter_kernel(const Ref* __restrict__ refs, const int32_t* __restrict__ ref_node, int64_t nref,
                               const LNode* __restrict__ nodes, const uint64_t* __restrict__ flags,
                               const uint64_t* __restrict__ flags_x, const Ref* __restrict__ box_l,
                               const Ref* __restrict__ box_r, Params P, Ref* __restrict__ next_refs,
                               int32_t* __restrict__ next_node, int32_t* __restrict__ pool) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nref) return;
  const LNode& nd = nodes[ref_node[i]];
  if (nd.split) {
    const uint64_t f = flags[i], rank = flags_x[i] - flags_x[nd.rbegin];
    const Ref r = refs[i];
    const bool clipped = P.clip && get3(r.lo, nd.axis) < nd.pos && get3(r.hi, nd.axis) >= nd.pos;
    if (f & kBelow) {
      const int64_t k = nd.crbegin + (int64_t)(uint32_t)rank;
      next_refs[k] = clipped ? box_l[i] : r;
      next_node[k] = nd.child;
    }
    if (f & kAbove) {
      const int64_t k = nd.crbegin + nd.cl + (int64_t)(rank >> 32);
      next_refs[k] = clipped ? box_r[i] : r;
      next_node[k] = nd.child + 1;
    }
  } else {
    pool[nd.pool + (i - nd.rbegin)] = refs[i].prim;
  }
}

// ---------------------------------------------------------------- finishing

__global__ void sizes_kernel(const GNode* __restrict__ gn, int32_t g0, int32_t cnt, int32_t* __restrict__ size,
                             int32_t* __restrict__ nleaf) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt) return;
  const int g = g0 + i;
  const GNode& n = gn[g];
  if (n.axis < 0) {
    size[g] = 1;
    nleaf[g] = 1;
  } else {
    size[g] = 1 + size[n.child0] + size[n.child1];
    nleaf[g] = nleaf[n.child0] + nleaf[n.child1];
  }
}

// Preorder entry index and leaf id (host: the iterative preorder of
// re_kd_build), and the ropes handed down (host: Builder::link).
__global__ void preorder_kernel(const GNode* __restrict__ gn, int32_t g0, int32_t cnt,
                                const int32_t* __restrict__ size, const int32_t* __restrict__ nleaf,
                                int32_t* __restrict__ entry, int32_t* __restrict__ lbase,
                                int32_t* __restrict__ ropes) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt) return;
  const int g = g0 + i;
  const GNode& n = gn[g];
  if (n.axis < 0) return;
  const int c0 = n.child0, c1 = n.child1;
  entry[c0] = entry[g] + 1;
  entry[c1] = entry[g] + 1 + size[c0];
  lbase[c0] = lbase[g];
  lbase[c1] = lbase[g] + nleaf[c0];
  // faces: LEFT 0, FRONT 1, RIGHT 2, BACK 3, TOP 4, BOTTOM 5
  int sl, sr;
  if (n.axis == 0) { sl = 0; sr = 2; }
  else if (n.axis == 1) { sl = 5; sr = 4; }
  else { sl = 3; sr = 1; }
  for (int f = 0; f < 6; ++f) {
    const int r = ropes[6 * (int64_t)g + f];
    ropes[6 * (int64_t)c0 + f] = f == sr ? c1 : r;
    ropes[6 * (int64_t)c1 + f] = f == sl ? c0 : r;
  }
}

__constant__ int kFaceAxisD[6] = {0, 2, 0, 2, 1, 1};
__constant__ int kFaceHighD[6] = {0, 1, 1, 0, 1, 0};

// Leaf records: box, ropes pushed down to the deepest node covering the whole
// face (host: Builder::push_down), and the per-leaf reference counts.  Eight
// threads per node: thread f < 6 of a leaf's eight walks down face f's rope,
// the last writes the rest of the record.  Bound by the walks' chains of
// dependent loads; with one thread per leaf, its six walks one after another
// and an atomic maximum of the depth and leaf size at the end, it took 110 us
// on a 2^18-triangle soup, and 465 us with eight threads and those atomics;
// 48 us in this form.
__global__ void __launch_bounds__(256) leaves_kernel(const GNode* __restrict__ gn, int32_t total,
                                                     const int32_t* __restrict__ entry,
                                                     const int32_t* __restrict__ lbase,
                                                     const int32_t* __restrict__ ropes, LeafRec* __restrict__ leaves,
                                                     int32_t* __restrict__ leaf_cnt,
                                                     int32_t* __restrict__ leaf_gid) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 8 * (int64_t)total) return;
  const int g = (int)(i >> 3), f = (int)(i & 7);
  const GNode& n = gn[g];
  if (n.axis >= 0 || f == 6) return;
  const int lid = lbase[g];
  LeafRec& lr = leaves[lid];
  if (f == 7) {
    for (int a = 0; a < 3; ++a) {
      lr.bmin[a] = n.lo[a];
      lr.bmax[a] = n.hi[a];
    }
    lr.first = 0;
    lr.count = (uint32_t)n.pool_n;
    lr.pad[0] = lr.pad[1] = 0;
    leaf_cnt[lid] = n.pool_n;
    leaf_gid[lid] = g;
    return;
  }
  const int axis = kFaceAxisD[f];
  const bool high = kFaceHighD[f] != 0;
  int r = ropes[6 * (int64_t)g + f];
  while (r >= 0 && gn[r].axis >= 0) {
    const GNode& t = gn[r];
    if (t.axis == axis) {
      r = high ? t.child0 : t.child1;
    } else if (t.split <= get3(n.lo, t.axis)) {
      r = t.child1;
    } else if (t.split >= get3(n.hi, t.axis)) {
      r = t.child0;
    } else {
      break;
    }
  }
  lr.rope[f] = r < 0 ? kNoRope : (gn[r].axis < 0 ? leaf_ref((uint32_t)lbase[r]) : entry[r]);
}

__global__ void entries_kernel(const GNode* __restrict__ gn, int32_t total, const int32_t* __restrict__ entry,
                               const int32_t* __restrict__ lbase, NodeEntry* __restrict__ out) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= total) return;
  const GNode& n = gn[g];
  NodeEntry e;
  if (n.axis < 0) {
    e.split = 0.0f;
    e.meta = kLeafMeta | (uint32_t)lbase[g];
  } else {
    e.split = n.split;
    e.meta = ((uint32_t)n.axis << 30) | (uint32_t)entry[n.child1];
  }
  out[entry[g]] = e;
}

// Triangle records in leaf order: v0, e1 = v1 - v0, e2 = v2 - v0, prim
// (RayEngine/src/World/RTScene.cpp:228-248).
__global__ void tris_kernel(const GNode* __restrict__ gn, int32_t n_leaves, const int32_t* __restrict__ leaf_gid,
                            const int32_t* __restrict__ first, const int32_t* __restrict__ pool,
                            const float* __restrict__ tv, LeafRec* __restrict__ leaves, TriRec* __restrict__ tris) {
  const int w = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  if (w >= n_leaves) return;
  const GNode& n = gn[leaf_gid[w]];
  const int64_t f = first[w];
  if (lane == 0) leaves[w].first = (uint32_t)f;
  for (int j = lane; j < n.pool_n; j += 64) {
    const int32_t pi = pool[n.pool + j];
    const float* t = tv + 9 * (int64_t)pi;
    TriRec tr;
    for (int a = 0; a < 3; ++a) {
      tr.v0[a] = t[a];
      tr.e1[a] = t[3 + a] - t[a];
      tr.e2[a] = t[6 + a] - t[a];
    }
    tr.prim = pi;
    tris[f + j] = tr;
  }
}

// ---------------------------------------------------------------- host side

unsigned blocks(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// Device buffers of one build.  Those below kOwnBytes are carved from chunks,
// first the one the context keeps, and are reused only by the next build (a
// level's hipMalloc and hipFree calls, 157 of each on a 2^18-triangle soup,
// took longer than its kernels); larger ones are allocated one by one, so
// that a large build holds no more than its live arrays.  release() only
// marks such a buffer; it is freed by flush(), which the caller calls after
// synchronizing the stream, so no buffer is freed while queued work may still
// use it.
struct Bufs {
  static constexpr size_t kOwnBytes = (size_t)64 << 20, kMinChunk = (size_t)8 << 20;
  Workspace& ws;
  hipStream_t s;
  std::vector<void*> chunks, ptrs, dead;  // allocated here; ptrs: one buffer each
  char* at = nullptr;
  size_t left = 0, carved = 0;    // of the current chunk; of all chunks
  Bufs(Workspace& w, hipStream_t st) : ws(w), s(st), at(w.chunk), left(w.bytes) {}
  ~Bufs() {
    // The end of the build, or an error on the way: nothing may use the
    // buffers any more.  The kept chunk becomes one of what was carved.
    (void)hipStreamSynchronize(s);
    for (void* p : chunks) (void)hipFree(p);
    for (void* p : ptrs) (void)hipFree(p);
    if (carved > ws.bytes && ws.bytes < kKeepBytes) {
      if (ws.chunk) (void)hipFree(ws.chunk);
      ws.chunk = nullptr;
      ws.bytes = 0;
      const size_t want = std::min(carved + carved / 8, kKeepBytes);
      if (hipMalloc((void**)&ws.chunk, want) == hipSuccess) ws.bytes = want;
      else (void)hipGetLastError();  // the next build allocates its own
    }
  }
  hipError_t take(void** p, size_t bytes) {
    *p = nullptr;
    bytes = (bytes + 255) & ~(size_t)255;
    if (bytes >= kOwnBytes) {
      const hipError_t e = hipMalloc(p, bytes);
      if (e == hipSuccess) ptrs.push_back(*p);
      return e;
    }
    if (bytes > left) {
      const size_t chunk = std::max(bytes, std::min(std::max(kMinChunk, carved), kOwnBytes));
      void* q = nullptr;
      const hipError_t e = hipMalloc(&q, chunk);
      if (e != hipSuccess) return e;
      chunks.push_back(q);
      at = (char*)q;
      left = chunk;
    }
    *p = at;
    at += bytes;
    left -= bytes;
    carved += bytes;
    return hipSuccess;
  }
  template <typename T>
  hipError_t alloc(T** p, size_t count) {
    return take((void**)p, std::max<size_t>(count, 1) * sizeof(T));
  }
  void release(void* p) {
    if (p && std::find(ptrs.begin(), ptrs.end(), p) != ptrs.end()) dead.push_back(p);
  }
  void flush() {
    for (void* p : dead) {
      auto it = std::find(ptrs.begin(), ptrs.end(), p);
      if (it != ptrs.end()) {
        (void)hipFree(p);
        ptrs.erase(it);
      }
    }
    dead.clear();
  }
};

// A device array that only grows; `keep` elements are copied on growth.
template <typename T>
struct Arr {
  T* p = nullptr;
  int64_t cap = 0;
  hipError_t ensure(Bufs& B, int64_t need, hipStream_t s, int64_t keep = 0) {
    if (need <= cap) return hipSuccess;
    const int64_t nc = std::max<int64_t>(need + need / 2, 64);
    T* q = nullptr;
    hipError_t e = B.alloc(&q, (size_t)nc);
    if (e != hipSuccess) return e;
    if (keep > 0) e = hipMemcpyAsync(q, p, (size_t)keep * sizeof(T), hipMemcpyDeviceToDevice, s);
    B.release(p);
    p = q;
    cap = nc;
    return e;
  }
};

// Writes a word of every page of an array about to be copied to, where the
// allocator gives it fresh pages (32 MB on): the runtime's copy faults them in
// at a third of the rate.  Build of 10^6 triangles into 14.1 M records 198 ms
// without and 159 with it, into 122 M records 1,310 and 1,040; with the arrays
// zeroed whole 241 and 1,170.  Smaller arrays come from pages in use before.
template <typename T>
void touch_pages(RecVec<T>& v) {
  const size_t bytes = v.size() * sizeof(T);
  if (bytes < ((size_t)32 << 20)) return;
  for (size_t at = 0; at < bytes; at += 4096) reinterpret_cast<volatile char*>(v.data())[at] = 0;
}

// Exclusive prefix sum with a reusable temporary buffer.
struct Scanner {
  Arr<char> tmp;
  template <typename T, typename Op = hipcub::Sum>
  hipError_t run(Bufs& B, const T* in, T* out, int64_t n, hipStream_t s, Op op = Op{}, T zero = T{}) {
    if (n <= 0) return hipSuccess;
    size_t bytes = 0;
    hipError_t e = hipcub::DeviceScan::ExclusiveScan(nullptr, bytes, in, out, op, zero, (int)n, s);
    if (e == hipSuccess) e = tmp.ensure(B, (int64_t)bytes, s);
    if (e == hipSuccess) e = hipcub::DeviceScan::ExclusiveScan(tmp.p, bytes, in, out, op, zero, (int)n, s);
    return e;
  }
};

}  // namespace

#define KDB_TRY(expr)                     \
  do {                                    \
    hipError_t e_ = (expr);               \
    if (e_ != hipSuccess) return e_;      \
  } while (0)

// Builds the tree of n (> 0) triangles; the outputs are host vectors.
// device_ms gets the device time of the build (events around all of it).
// root_min and root_max receive the root box; with a coordinate that is not
// finite, finite is set to false and nothing is built.
hipError_t build_device(const float* tri_v, int64_t n, float* root_min, float* root_max, bool& finite,
                        const Params& P, Workspace& ws, hipStream_t s, RecVec<NodeEntry>& out_nodes,
                        RecVec<LeafRec>& out_leaves, RecVec<TriRec>& out_tris, int32_t& depth,
                        int32_t& max_leaf, float& device_ms) {
  if (!ws.totals) KDB_TRY(hipHostMalloc((void**)&ws.totals, sizeof(Adds), hipHostMallocDefault));
  Bufs B(ws, s);
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  KDB_TRY(hipEventCreate(&ev0));
  KDB_TRY(hipEventCreate(&ev1));
  struct EvGuard {
    hipEvent_t a, b;
    ~EvGuard() {
      (void)hipEventDestroy(a);
      (void)hipEventDestroy(b);
    }
  } evg{ev0, ev1};
  const int nb = std::max(4, P.n_bins);
  float* tv = nullptr;
  KDB_TRY(B.alloc(&tv, (size_t)(9 * n)));
  KDB_TRY(hipMemcpyAsync(tv, tri_v, (size_t)(9 * n) * sizeof(float), hipMemcpyHostToDevice, s));
  KDB_TRY(hipEventRecord(ev0, s));

  // Level arrays: current and next references / nodes swap every level.
  Arr<Ref> refs, nrefs, box_l, box_r;
  Arr<int32_t> ref_node, nnode, strad;
  Arr<uint64_t> flags, flags_x;
  Arr<LNode> lv, next;
  Arr<int32_t> hist;
  Arr<Adds> adds, adds_x;
  Arr<GNode> gn;
  Arr<int32_t> pool;
  Scanner scan;
  int32_t* n_strad = nullptr;
  KDB_TRY(B.alloc(&n_strad, 1));
  KDB_TRY(refs.ensure(B, n, s));
  KDB_TRY(ref_node.ensure(B, n, s));
  SoupBounds* bounds = nullptr;
  KDB_TRY(B.alloc(&bounds, 1));
  hipLaunchKernelGGL(clear_bounds_kernel, dim3(1), dim3(64), 0, s, bounds);
  hipLaunchKernelGGL(init_refs_kernel, dim3(std::min(blocks(n, 256), (unsigned)kInitBlocks)), dim3(256), 0, s, tv, n,
                     refs.p, ref_node.p, bounds);
  KDB_TRY(hipGetLastError());
  SoupBounds sb;
  KDB_TRY(hipMemcpyAsync(&sb, bounds, sizeof(sb), hipMemcpyDeviceToHost, s));
  KDB_TRY(hipStreamSynchronize(s));
  finite = sb.bad == 0;
  if (!finite) return hipSuccess;
  for (int a = 0; a < 3; ++a) {
    root_min[a] = std::min(kInf, tri_v[3 * (int64_t)(uint32_t)sb.lo[a] + a]);
    root_max[a] = std::max(-kInf, tri_v[3 * (int64_t)(uint32_t)sb.hi[a] + a]);
  }
  KDB_TRY(lv.ensure(B, 1, s));
  bool any_big = false;  // the level holds a node that many blocks bin
  max_leaf = 0;
  KDB_TRY(hipMemsetAsync(n_strad, 0, sizeof(int32_t), s));
  {
    LNode root{};
    for (int a = 0; a < 3; ++a) {
      root.lo[a] = root_min[a];
      root.hi[a] = root_max[a];
    }
    root.rbegin = 0;
    root.n = (int32_t)n;
    root.depth = 1;
    root.gid = 0;
    root.mode = mode_of(root.n, root.depth, P);
    any_big = root.mode == kModeBig;
    KDB_TRY(hipMemcpyAsync(lv.p, &root, sizeof(root), hipMemcpyHostToDevice, s));
  }
  int64_t nn = 1, nref = n, gused = 1, pused = 0;
  KDB_TRY(gn.ensure(B, 1024, s));
  KDB_TRY(pool.ensure(B, n + 1024, s));
  std::vector<std::pair<int32_t, int32_t>> levels;  // (first gid, count)
  int32_t gbase = 0;

  while (nn > 0) {
    levels.emplace_back(gbase, (int32_t)nn);
    KDB_TRY(hist.ensure(B, (nref / kBinChunk + 1) * 6 * nb, s));
    if (any_big) {
      KDB_TRY(hipMemsetAsync(hist.p, 0, (size_t)((nref / kBinChunk + 1) * 6 * nb) * sizeof(int32_t), s));
      hipLaunchKernelGGL(bin_count_kernel, dim3(blocks(nref, kBinChunk)), dim3(256), 0, s, refs.p, ref_node.p, nref,
                         lv.p, hist.p, P);
    }
    hipLaunchKernelGGL(split_kernel, dim3(blocks(nn * 64, 256)), dim3(256), 0, s, lv.p, (int32_t)nn, refs.p, hist.p,
                       P);
    KDB_TRY(hipGetLastError());

    KDB_TRY(strad.ensure(B, nref, s));
    KDB_TRY(flags.ensure(B, nref, s));
    KDB_TRY(flags_x.ensure(B, nref, s));
    KDB_TRY(box_l.ensure(B, nref, s));
    KDB_TRY(box_r.ensure(B, nref, s));
    hipLaunchKernelGGL(part_flags_kernel, dim3(blocks(nref, kFlagChunk)), dim3(256), 0, s, refs.p, ref_node.p, nref,
                       lv.p, P, flags.p, strad.p, n_strad);
    if (P.clip)
      hipLaunchKernelGGL(part_clip_kernel, dim3(blocks(2 * nref, 64)), dim3(64), 0, s, tv, refs.p, ref_node.p,
                         lv.p, strad.p, n_strad, flags.p, box_l.p, box_r.p);
    KDB_TRY(hipGetLastError());
    KDB_TRY(scan.run(B, flags.p, flags_x.p, nref, s));

    KDB_TRY(adds.ensure(B, nn, s));
    KDB_TRY(adds_x.ensure(B, nn, s));
    hipLaunchKernelGGL(decide_kernel, dim3(blocks(nn, 256)), dim3(256), 0, s, lv.p, (int32_t)nn, flags.p, flags_x.p,
                       P, adds.p);
    KDB_TRY(hipGetLastError());
    KDB_TRY(scan.run(B, adds.p, adds_x.p, nn, s, AddsSum{}, Adds{0, 0, 0, 0u}));
    hipLaunchKernelGGL(totals_kernel, dim3(1), dim3(64), 0, s, adds.p, adds_x.p, nn, ws.totals, n_strad);
    KDB_TRY(hipGetLastError());
    KDB_TRY(hipStreamSynchronize(s));
    const Adds sum = *ws.totals;
    const int64_t n_next = sum.kids, r_next = sum.refs, l_now = sum.leaf;
    any_big = (sum.last & kBigBit) != 0;
    max_leaf = std::max(max_leaf, (int32_t)(sum.last & ~kBigBit));
    if (!level_fits(gbase + nn, pused, sum)) return hipErrorInvalidValue;

    KDB_TRY(gn.ensure(B, gused + n_next, s, gused));
    KDB_TRY(pool.ensure(B, pused + l_now, s, pused));
    KDB_TRY(next.ensure(B, n_next, s));
    KDB_TRY(nrefs.ensure(B, r_next, s));
    KDB_TRY(nnode.ensure(B, r_next, s));
    const int32_t next_gid = gbase + (int32_t)nn;
    hipLaunchKernelGGL(emit_kernel, dim3(blocks(nn, 256)), dim3(256), 0, s, lv.p, (int32_t)nn, adds_x.p, next.p, next_gid,
                       pused, gn.p, P);
    hipLaunchKernelGGL(scatter_kernel, dim3(blocks(nref, 256)), dim3(256), 0, s, refs.p, ref_node.p, nref, lv.p,
                       flags.p, flags_x.p, box_l.p, box_r.p, P, nrefs.p, nnode.p, pool.p);
    KDB_TRY(hipGetLastError());
    std::swap(lv, next);
    std::swap(refs, nrefs);
    std::swap(ref_node, nnode);
    gused += n_next;
    pused += l_now;
    gbase = next_gid;
    nn = n_next;
    nref = r_next;
    if (!B.dead.empty()) {
      KDB_TRY(hipStreamSynchronize(s));
      B.flush();
    }
  }

  const int32_t total = (int32_t)gused;
  int32_t *size = nullptr, *nleaf = nullptr, *entry = nullptr, *lbase = nullptr, *ropes = nullptr;
  KDB_TRY(B.alloc(&size, (size_t)total));
  KDB_TRY(B.alloc(&nleaf, (size_t)total));
  KDB_TRY(B.alloc(&entry, (size_t)total));
  KDB_TRY(B.alloc(&lbase, (size_t)total));
  KDB_TRY(B.alloc(&ropes, 6 * (size_t)total));
  for (auto it = levels.rbegin(); it != levels.rend(); ++it)
    hipLaunchKernelGGL(sizes_kernel, dim3(blocks(it->second, 256)), dim3(256), 0, s, gn.p, it->first, it->second,
                       size, nleaf);
  KDB_TRY(hipGetLastError());
  KDB_TRY(hipMemsetAsync(entry, 0, sizeof(int32_t), s));
  KDB_TRY(hipMemsetAsync(lbase, 0, sizeof(int32_t), s));
  KDB_TRY(hipMemsetAsync(ropes, 0xff, 6 * sizeof(int32_t), s));
  for (auto& lvl : levels)
    hipLaunchKernelGGL(preorder_kernel, dim3(blocks(lvl.second, 256)), dim3(256), 0, s, gn.p, lvl.first, lvl.second,
                       size, nleaf, entry, lbase, ropes);
  KDB_TRY(hipGetLastError());
  int32_t n_leaves = 0;
  KDB_TRY(hipMemcpyAsync(&n_leaves, nleaf, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  KDB_TRY(hipStreamSynchronize(s));

  LeafRec* leaves = nullptr;
  NodeEntry* entries = nullptr;
  int32_t *leaf_cnt = nullptr, *leaf_gid = nullptr, *first = nullptr;
  KDB_TRY(B.alloc(&leaves, (size_t)n_leaves));
  KDB_TRY(B.alloc(&entries, (size_t)total));
  KDB_TRY(B.alloc(&leaf_cnt, (size_t)n_leaves));
  KDB_TRY(B.alloc(&leaf_gid, (size_t)n_leaves));
  KDB_TRY(B.alloc(&first, (size_t)n_leaves + 1));
  hipLaunchKernelGGL(leaves_kernel, dim3(blocks(8 * (int64_t)total, 256)), dim3(256), 0, s, gn.p, total, entry, lbase, ropes,
                     leaves, leaf_cnt, leaf_gid);
  hipLaunchKernelGGL(entries_kernel, dim3(blocks(total, 256)), dim3(256), 0, s, gn.p, total, entry, lbase, entries);
  KDB_TRY(hipGetLastError());
  KDB_TRY(scan.run(B, leaf_cnt, first, n_leaves, s));
  int64_t n_tris = pused;  // every leaf reference becomes one triangle record
  TriRec* tris = nullptr;
  KDB_TRY(B.alloc(&tris, (size_t)n_tris));
  hipLaunchKernelGGL(tris_kernel, dim3(blocks((int64_t)n_leaves * 64, 256)), dim3(256), 0, s, gn.p, n_leaves,
                     leaf_gid, first, pool.p, tv, leaves, tris);
  KDB_TRY(hipGetLastError());
  KDB_TRY(hipEventRecord(ev1, s));

  out_nodes.resize((size_t)total);
  out_leaves.resize((size_t)n_leaves);
  out_tris.resize((size_t)n_tris);
  touch_pages(out_nodes);
  touch_pages(out_leaves);
  touch_pages(out_tris);
  KDB_TRY(hipMemcpyAsync(out_nodes.data(), entries, (size_t)total * sizeof(NodeEntry), hipMemcpyDeviceToHost, s));
  KDB_TRY(hipMemcpyAsync(out_leaves.data(), leaves, (size_t)n_leaves * sizeof(LeafRec), hipMemcpyDeviceToHost, s));
  KDB_TRY(hipMemcpyAsync(out_tris.data(), tris, (size_t)n_tris * sizeof(TriRec), hipMemcpyDeviceToHost, s));
  KDB_TRY(hipStreamSynchronize(s));
  KDB_TRY(hipEventElapsedTime(&device_ms, ev0, ev1));
  depth = (int32_t)levels.size();  // the last level holds leaves only
  return hipSuccess;
}

}  // namespace kdb
}  // namespace re
