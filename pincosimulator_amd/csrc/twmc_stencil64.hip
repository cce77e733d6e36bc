// twmc_stencil64.hip -- register-resident TWMC step kernel for a 64 x 64
// periodic lattice in FP32 with the hopping applied as its exact real-space
// form.
//
// The reference applies the hopping in k-space (TWMCBaseSolver.cpp:80-88,
// :235-242): h = IDFT(K . DFT(beta)) / N with
// K = -2iJ([nx != 1] cos(2 pi kx / nx) + [ny != 1] cos(2 pi ky / ny)).
// Because e^{ik} + e^{-ik} = 2 cos k, that product is, term by term, the
// nearest-neighbour sum
//     h(x, y) = -iJ (beta(x-1, y) + beta(x+1, y) + beta(x, y-1) + beta(x, y+1))
// with periodic wrap -- the same linear map, without the FFT round trip (the
// two agree to rounding, ~1e-16 relative in FP64).  This kernel evaluates that
// form: one 1024-thread workgroup owns one trajectory, two site pairs per
// thread in registers, the neighbours from an LDS copy of the state.  Per step
// and site: the 4-term sum, the local drift, one Philox4x32-10 call per site
// pair with Box-Muller, the update.  Frames are captured by separate launches
// (the register-FFT capture kernel for the per-trajectory means and the k-space
// sums, the site-major kernel for the per-site sums), so this loop carries no
// capture code.
#include <type_traits>

#include "twmc_cplx.h"
#include "twmc_internal.h"
#include "twmc_rng.h"

namespace twmc {

namespace {

constexpr int kL = 64;

// Thread t owns the site pairs t and t + 1024 (rows of 32 pairs).  Even and odd
// sites lie in separate LDS halves, 8 bytes from lane to lane (no bank
// conflicts); a step reads one copy of the state and writes the other, so one
// barrier per step, and two steps per loop pass make every LDS address a
// register plus a constant.  UI0: Im U = 0 (a real interaction), so the real part
// of the drift factor is the constant A0 and its per-site FMA drops out.
//
// What bounds it: VALU issue, 44.5 instructions per site-step of which the four
// transcendental ones run on their own unit beside the others when other waves
// have work: 64 registers for eight waves per SIMD (two values spill with a real U),
// two workgroups per CU.  The
// two do not advance evenly (the older one is served first), so in launches of more
// than a few steps (queue_pays) trajectories are taken from a queue: dealt out by
// workgroup, one of the two finished early and left the other to a half-filled CU.  16384 trajectories, 500-step launches:
// 60.9 us per step = 1.10e12 site-steps/s; dealt out 69.6; one wave per trajectory
// with its rows in registers (128 VGPRs, four waves per SIMD), the form before
// both, 80.2; this form at four waves per SIMD 75.8; raised priority around the
// samples, as in the banded kernel, 61.8.  Few trajectories have a whole CU each
// instead of one SIMD: 64 of them 5.85 -> 1.27 us per step, 1024 6.23 -> 4.5.  Each
// site's operations and their order are those of the one-wave form: the same
// bits.
constexpr int kBlock = 1024;
constexpr int kPairs = kL * kL / 2;

// clears the launch's work queue
__global__ void queue_reset_kernel(unsigned int* queue) {
  if (threadIdx.x == 0) *queue = 0u;
}

template <bool UI0>
__global__ void __launch_bounds__(kBlock, 8) stencil64_step_kernel(StepArgs g) {
  __shared__ cpx<float> st[2][2][kPairs];  // [copy][even, odd site][pair]
  const cpx<float> r0 = reinterpret_cast<const cpx<float>*>(g.rsl)[0];
  const cpx<float> u0 = reinterpret_cast<const cpx<float>*>(g.U)[0];
  const cpx<float> f0 = reinterpret_cast<const cpx<float>*>(g.F)[0];
  const float dtf = float(g.dt);
  const float Ur = dtf * u0.re, Ui = dtf * u0.im;
  const float A0 = fmaf(dtf, r0.re, Ui), B0 = fmaf(dtf, r0.im, -Ur);
  const float fr = -dtf * f0.im, fi = dtf * f0.re;
  const float sig = float(g.dt4);
  const float nl = -1.3862943611198906f * sig * sig;
  const float jdt = float(-0.5 * g.kscale * g.dt);

  // pair p0 = t, p1 = t + 1024; x-neighbours p0 + 32 and p1 - 32 never wrap
  const int p0 = threadIdx.x, row = p0 & ~31;
  const int lft = row + ((p0 - 1) & 31), rgt = row + ((p0 + 1) & 31);
  const int dn0 = (p0 - 32) & (kPairs - 1), up1 = (p0 + kBlock + 32) & (kPairs - 1);

  // the first trajectory by workgroup, the next ones as the launch says
  for (int b = blockIdx.x; b < g.n_traj;) {
    const uint64_t traj = g.traj_ids[b];
    float4* gb = reinterpret_cast<float4*>(reinterpret_cast<cpx<float>*>(g.beta) + (size_t)b * kL * kL);
    cpx<float> beta[4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int p = p0 + kBlock * j;
      const float4 v = gb[p];
      st[0][0][p] = beta[2 * j] = mk(v.x, v.y);
      st[0][1][p] = beta[2 * j + 1] = mk(v.z, v.w);
    }
    __syncthreads();
    // one step from copy C to copy 1 - C of the state
    auto step_from = [&](auto copy, uint32_t step) __attribute__((always_inline)) {
      constexpr int C = decltype(copy)::value;
      const cpx<float>(*cur)[kPairs] = st[C];
      cpx<float>(*nxt)[kPairs] = st[1 - C];
      // opaque per step, so that no Philox round is hoisted out of the loop
      uint32_t pair = (uint32_t)p0;
      asm volatile("" : "+v"(pair));
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        // the neighbours' old values: read together, under the Philox rounds
        const int up = j ? up1 : p0 + 32, dn = j ? p0 + kBlock - 32 : dn0;
        const cpx<float> left = cur[1][lft + kBlock * j], right = cur[0][rgt + kBlock * j];
        const cpx<float> xu[2] = {cur[0][up], cur[1][up]}, xd[2] = {cur[0][dn], cur[1][dn]};
        const u32x4 w = philox4x32_10_wave(make_counter(traj, TAG_WIENER, step, pair + (uint32_t)(kBlock * j)),
                                           g.key0, g.key1);
        float rs[2], cs[2], sn[2];
        box_muller_f32_scaled(w.x, w.y, nl, rs[0], cs[0], sn[0]);
        box_muller_f32_scaled(w.z, w.w, nl, rs[1], cs[1], sn[1]);
        const cpx<float> z0 = beta[2 * j], z1 = beta[2 * j + 1];
        const cpx<float> ym[2] = {left, z0}, yp[2] = {z1, right};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const cpx<float> v = h ? z1 : z0;
          const float sr = xd[h].re + (xu[h].re + (ym[h].re + yp[h].re));
          const float si = xd[h].im + (xu[h].im + (ym[h].im + yp[h].im));
          const float m = fmaf(v.im, v.im, v.re * v.re);
          const float cr = UI0 ? A0 : fmaf(-Ui, m, A0), ci = fmaf(Ur, m, B0);
          float dr = fmaf(rs[h], cs[h], fr);
          dr = fmaf(cr, v.re, dr);
          dr = fmaf(-ci, v.im, dr);
          dr = fmaf(jdt, si, dr);
          float di = fmaf(rs[h], sn[h], fi);
          di = fmaf(cr, v.im, di);
          di = fmaf(ci, v.re, di);
          di = fmaf(-jdt, sr, di);
          beta[2 * j + h] = mk(v.re + dr, v.im + di);
          nxt[h][p0 + kBlock * j] = beta[2 * j + h];
        }
      }
      __syncthreads();
    };
    int s = 0;
    for (; s + 2 <= g.n_steps; s += 2) {
      step_from(std::integral_constant<int, 0>{}, uint32_t(g.step0 + (uint64_t)s));
      step_from(std::integral_constant<int, 1>{}, uint32_t(g.step0 + (uint64_t)s + 1));
    }
    if (s < g.n_steps) step_from(std::integral_constant<int, 0>{}, uint32_t(g.step0 + (uint64_t)s));
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const cpx<float> v0 = beta[2 * j], v1 = beta[2 * j + 1];
      gb[p0 + kBlock * j] = make_float4(v0.re, v0.im, v1.re, v1.im);
    }
    // the next trajectory: of this workgroup's share, or from the queue; through a word of
    // copy 1 (its load writes copy 0)
    int* next = reinterpret_cast<int*>(&st[1][0][0]);
    __syncthreads();
    if (threadIdx.x == 0) *next = (int)(gridDim.x + (g.queue ? atomicAdd(g.queue, 1u) : (unsigned int)b));
    __syncthreads();
    b = __builtin_amdgcn_readfirstlane(*next);
  }
}

}  // namespace

bool stencil64_supported(int nx, int ny, int hopping, int precision, int param_stride) {
  return nx == 64 && ny == 64 && hopping == 0 && precision == 32 && param_stride == 0;
}

hipError_t launch_stencil64(const StepArgs& a, int grid, hipStream_t s) {
  StepArgs q = a;
  if (!queue_pays(a, grid, 32)) q.queue = nullptr;
  else hipLaunchKernelGGL(queue_reset_kernel, dim3(1), dim3(64), 0, s, q.queue);
  if (a.u_real)
    hipLaunchKernelGGL(stencil64_step_kernel<true>, dim3(grid), dim3(kBlock), 0, s, q);
  else
    hipLaunchKernelGGL(stencil64_step_kernel<false>, dim3(grid), dim3(kBlock), 0, s, q);
  return hipGetLastError();
}

int stencil64_block() { return kBlock; }

hipError_t stencil64_occupancy(int* blocks_per_cu) {
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, (const void*)stencil64_step_kernel<false>, kBlock, 0);
}

}  // namespace twmc
