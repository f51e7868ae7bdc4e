// The surrogate's training kernel on the CPU, its waves run in chosen orders.
//
// kernels/surrogate.hip is compiled as host code, with the device's vector and
// wave operations defined below.  Every lane is a fiber; the lanes of a wave
// run up to their next wave operation, which is computed when all 64 have
// come, and a wave runs as far as it can before the next one in the order gets
// its turn: up to a block barrier that others have not reached.  Barriers are
// all that orders waves on the device, so a result that depends on the order
// is one the device may also give.
//
// Usage: mlp_train_waves_driver CHUNKS...   (one block; exit status 1 when a
// batch of that many 64-point chunks gives other bits in some order)
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(...) ((void)0)

#include <ucontext.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

namespace emu {

constexpr int kThreads = 512, kLanes = 64, kWaves = kThreads / kLanes;
enum State { kReady, kWaveOp, kBarrier, kDone };

struct Fiber {
  ucontext_t ctx;
  std::vector<char> stack;
  State state;
};
Fiber fibers[kThreads];
ucontext_t main_ctx;
int cur = 0;
std::function<void()> body;
struct Idx { unsigned x, y; };

void yield(State s) {
  fibers[cur].state = s;
  const int me = cur;
  swapcontext(&fibers[me].ctx, &main_ctx);
}

void entry() {
  body();
  yield(kDone);
}

// Operands of the wave operation at hand, and its results.
float wa[kLanes][8], wb[kLanes][8], wc[kLanes][4];
std::function<void()> wave_op;

void run_block(const int* order) {
  for (int i = 0; i < kThreads; ++i) {
    Fiber& f = fibers[i];
    f.stack.resize(1 << 17);
    getcontext(&f.ctx);
    f.ctx.uc_stack.ss_sp = f.stack.data();
    f.ctx.uc_stack.ss_size = f.stack.size();
    f.ctx.uc_link = nullptr;
    makecontext(&f.ctx, entry, 0);
    f.state = kReady;
  }
  for (;;) {
    int done = 0, waiting = 0;
    for (int k = 0; k < kWaves; ++k) {
      const int w = order[k];
      for (;;) {  // the wave, as far as it goes
        int n_op = 0, n_bar = 0, n_done = 0;
        for (int l = 0; l < kLanes; ++l) {
          cur = w * kLanes + l;
          if (fibers[cur].state == kReady) swapcontext(&main_ctx, &fibers[cur].ctx);
          n_op += fibers[cur].state == kWaveOp;
          n_bar += fibers[cur].state == kBarrier;
          n_done += fibers[cur].state == kDone;
        }
        if (n_op == kLanes) {
          wave_op();
          for (int l = 0; l < kLanes; ++l) fibers[w * kLanes + l].state = kReady;
          continue;
        }
        if (n_op != 0 || (n_bar != 0 && n_done != 0)) {
          std::fprintf(stderr, "wave %d: lanes apart\n", w);
          std::exit(2);
        }
        done += n_done == kLanes;
        waiting += n_bar == kLanes;
        break;
      }
    }
    if (done == kWaves) return;
    if (waiting != kWaves) {
      std::fprintf(stderr, "a barrier that %d of %d waves reach\n", waiting, kWaves);
      std::exit(2);
    }
    for (Fiber& f : fibers) f.state = kReady;
  }
}

}  // namespace emu

// --- what the kernel uses of the device
#undef __launch_bounds__
#define __launch_bounds__(...)
#define __align__(n)
#define threadIdx (emu::Idx{(unsigned)emu::cur, 0u})
static const emu::Idx blockIdx{0, 0}, gridDim{1, 1}, blockDim{emu::kThreads, 1};

static void __syncthreads() { emu::yield(emu::kBarrier); }
static float __shfl_xor(float v, int mask) {
  const int l = emu::cur & 63;
  emu::wa[l][0] = v;
  emu::wave_op = [] {};
  emu::yield(emu::kWaveOp);
  const float r = emu::wa[l ^ mask][0];
  emu::wave_op = [] {};  // read before any lane writes its next operand
  emu::yield(emu::kWaveOp);
  return r;
}
typedef __bf16 emu_bf16x8 __attribute__((ext_vector_type(8)));
typedef float emu_f32x4 __attribute__((ext_vector_type(4)));
static emu_f32x4 emu_mfma(emu_bf16x8 a, emu_bf16x8 b, emu_f32x4 c) {
  using namespace emu;
  const int l = cur & 63;
  for (int s = 0; s < 8; ++s) {
    wa[l][s] = (float)a[s];
    wb[l][s] = (float)b[s];
  }
  for (int r = 0; r < 4; ++r) wc[l][r] = c[r];
  wave_op = [] {
    for (int o = 0; o < kLanes; ++o)
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * (o >> 4) + r, col = o & 15;
        float v = wc[o][r];
        for (int k = 0; k < 32; ++k) v += wa[16 * (k >> 3) + row][k & 7] * wb[16 * (k >> 3) + col][k & 7];
        wc[o][r] = v;
      }
  };
  yield(kWaveOp);
  return emu_f32x4{wc[l][0], wc[l][1], wc[l][2], wc[l][3]};
}
#define __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, x, y, z) emu_mfma(a, b, c)
static int emu_uniform(int v) { return v; }
#define __builtin_amdgcn_readfirstlane emu_uniform
#define __builtin_amdgcn_fractf(x) ((x) - std::floor(x))
#define __builtin_amdgcn_sinf(x) std::sin(6.28318530718f * (x))
#define __builtin_amdgcn_cosf(x) std::cos(6.28318530718f * (x))
#define __builtin_amdgcn_exp2f(x) std::exp2(x)
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))

// --- what the file's other code names; not run here
hipError_t hipGetLastError() { return hipSuccess; }
template <typename... A>
static unsigned emu_unused(A...) { std::abort(); }
static float __shfl(float, int) { std::abort(); }
static float __uint_as_float(unsigned u) { float f; std::memcpy(&f, &u, 4); return f; }
static unsigned __float_as_uint(float f) { unsigned u; std::memcpy(&u, &f, 4); return u; }
#define __builtin_amdgcn_mbcnt_lo emu_unused
#define __builtin_amdgcn_mbcnt_hi emu_unused
#define __builtin_amdgcn_update_dpp emu_unused
#define __builtin_amdgcn_readlane emu_unused
#define __builtin_amdgcn_ds_bpermute emu_unused
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_wave_barrier() ((void)0)
#define __ballot emu_unused
#define __any emu_unused
#define __ffsll __builtin_ffsll
#define __popcll __builtin_popcountll
#define atomicMin emu_unused
#define atomicAdd emu_unused

#include "../rayengine_amd/csrc/kernels/surrogate.hip"

namespace re {
namespace {

alignas(16) unsigned char lds_raw[sizeof(TrainLds)];

int run(int chunks) {
  const int batch = 64 * chunks;
  uint64_t seed = 0x9e3779b97f4a7c15ull * (uint64_t)(chunks + 1);
  auto uni = [&seed]() {
    seed = seed * 6364136223846793005ull + 1442695040888963407ull;
    return (float)(seed >> 40) * (1.0f / 16777216.0f);
  };
  std::vector<bf16x8> pack(mlp::kPack / 8);
  for (bf16x8& v : pack)
    for (int s = 0; s < 8; ++s) v[s] = (__bf16)(0.4f * uni() - 0.2f);
  std::vector<float> small(mlp::kSmall);
  for (float& v : small) v = uni() - 0.5f;
  std::vector<float4> samples(batch);
  for (float4& v : samples) v = make_float4(uni(), uni(), uni(), 4.0f * uni() - 2.0f);

  const int orders[][emu::kWaves] = {{0, 1, 2, 3, 4, 5, 6, 7}, {7, 6, 5, 4, 3, 2, 1, 0},
                                     {0, 2, 4, 6, 1, 3, 5, 7}, {1, 3, 5, 7, 0, 2, 4, 6},
                                     {4, 5, 6, 7, 0, 1, 2, 3}, {3, 6, 0, 5, 2, 7, 1, 4}};
  std::vector<float> first;
  int bad = 0;
  for (const auto& order : orders) {
    std::memset(lds_raw, 0, sizeof(lds_raw));
    std::vector<float> partial(mlp::kParams + 1, NAN);
    emu::body = [&] {
      mlp_train_kernel(pack.data(), small.data(), samples.data(), batch, 0, batch, 4.0f, partial.data());
    };
    emu::run_block(order);
    if (first.empty()) first = partial;
    int n = 0;
    for (int p = 0; p <= mlp::kParams; ++p)
      n += std::memcmp(&partial[p], &first[p], 4) != 0 || !std::isfinite(partial[p]);
    if (n) {
      std::printf("%d chunks, waves in order %d %d %d %d %d %d %d %d: %d of %d values differ\n", chunks, order[0],
                  order[1], order[2], order[3], order[4], order[5], order[6], order[7], n, mlp::kParams + 1);
      bad = 1;
    }
  }
  return bad;
}

}  // namespace
}  // namespace re

int main(int argc, char** argv) {
  int bad = 0;
  for (int i = 1; i < argc; ++i) bad |= re::run(std::atoi(argv[i]));
  return bad;
}
