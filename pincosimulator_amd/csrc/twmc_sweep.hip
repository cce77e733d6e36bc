// twmc_sweep.hip -- a parameter sweep of many uneven lattices (1D chains and
// 2D squares of different sizes, each point with its own F, detuning, ...)
// advanced by ONE persistent launch per frame.
//
// Work items are (point, block of trajectories).  Workgroups take items from a
// global counter in decreasing order of cost (largest lattices first), so the
// uneven items balance across the chip.  A step item holds tb trajectories of
// one point stacked as the rows of one array (a chain's trajectory is one
// row, a 2D point's nx rows), so small lattices still fill a workgroup; the
// frame capture takes 2D points one trajectory per item (its FFT runs along
// both dimensions) and chains as stacked rows, transformed along the rows
// only.  tb per lattice shape is chosen by twmc_sweep_autotune, which times
// the candidates on the device.  A step applies the hopping as the exact
// nearest-neighbour form of the reference's FFT product (the x- and
// y-neighbours read from the LDS copy of the state), then the same Philox
// increments and Euler update as the single-system kernels, so every
// trajectory of a sweep equals the same trajectory run alone (to FP32
// rounding); the Stockham FFT runs only in the frame capture, for the
// k-space bins.
// The frame loop (counter reset + step kernel per frame) can be captured once
// into a hipGraph and launched as one graph.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <map>
#include <type_traits>
#include <string>
#include <vector>

#include "../../include/twmc_hip.h"
#include "twmc_cplx.h"
#include "twmc_internal.h"
#include "twmc_rng.h"
#include "twmc_stockham.h"

namespace twmc {

namespace {

constexpr int kSweepBlock = 256;  // the capture launch
constexpr int kSweepMaxSites = 4096;  // sites per work item (LDS and registers)
constexpr int kPPT = kSweepMaxSites / 2 / kSweepBlock;
constexpr int kStepBlock = 1024;  // the step launch
constexpr int kStepPairs = kSweepMaxSites / 2;
constexpr int kStepPPT = kStepPairs / kStepBlock;
constexpr int kBins = 32;  // radial |k| bins: 0 is k = 0, 1..31 split (0, pi sqrt 2]
constexpr int kMaxRows = 256;  // stacked trajectories per work item
constexpr int kMaxNx = 64;     // rows of a 2D point
constexpr int kMaxNy = 512;    // row length (chain length or 2D row)

struct SweepPointDev {
  int nx, ny, tb, fft_x;  // fft_x = 1: 2D point (rows are lattice rows), 0: stacked 1D trajectories
  RadixPlan px, py;
  int tw_x, tw_y;  // offsets into the twiddle pool
  float rsl_re, rsl_im, u_re, u_im, f_re, f_im;
  float dt4, kscale;
  int n_traj;
  uint64_t traj_id0;
  uint64_t state_off;  // complex elements
  uint64_t m_off;      // offset of [n_traj][n_frames] per-trajectory means
  int bin_off;         // offset of the mode -> radial bin table (one entry per mode of one trajectory)
  int index;           // point index (offset of its [n_frames][kBins + 2] k-space / mean-field sums)
};

struct SweepItemDev {
  int point, t0;
};

struct SweepArgs {
  const SweepPointDev* points;
  const SweepItemDev* items;
  int n_items;
  unsigned int* counter;
  const cpx<float>* tw_pool;
  cpx<float>* beta;
  double* traj_m2;
  double* traj_m4;
  const unsigned char* bin_pool;  // mode -> bin
  double* ksum;                   // [points][n_frames][kBins + 2]: sum of |DFT beta|^2 per bin, sum of beta
  float dt;
  uint32_t key0, key1;
  uint64_t step0;
  int n_steps, capture, frame, n_frames;
  const uint64_t* traj_ids;  // one-point batches of the main API: ids by index (else traj_id0 + index)
};

// clears the work-queue counters of the capture and the step launch
__global__ void sweep_reset_kernel(unsigned int* counter) {
  if (threadIdx.x < 2 && blockIdx.x == 0) counter[threadIdx.x] = 0u;
}

// One work item advanced g.n_steps Euler-Maruyama steps (the step launch).
// The item is ntr trajectories of nxt rows each, stacked: 2D points have
// nxt = nx lattice rows and x-hopping (XHOP), chains one row each and no
// x-hopping; MULTI = false is the single-trajectory case (one trajectory id
// for the whole item).  Thread t owns the site pairs p = t + 1024 j, sites 2p
// and 2p + 1 of one row (rows have even length), so the pair's two values are
// each other's y-neighbours; the other y-neighbours and the x-neighbours come
// from the LDS copy of the state: even and odd sites in separate halves, 8 bytes
// from lane to lane, one copy read and the other written per step (one
// barrier), two steps per loop pass so that both copies' addresses are a
// register plus a constant.  The hopping h = -i J S, S the sum over the
// periodic nearest neighbours, is the exact real-space form of the reference's
// IDFT(K DFT(beta)) / N (TWMCBaseSolver.cpp:80-88, :235-242); a length-2
// dimension gives the one neighbour twice, as the FFT form does.
// UI0: Im U = 0 in every point, so the per-site FMA of the drift's real part
// drops out.
template <bool UI0, bool XHOP, bool MULTI>
__device__ __forceinline__ void step_item(const SweepArgs& g, const SweepPointDev& P, const SweepItemDev& item,
                                          cpx<float>* st, float4* gbeta, int nxt, int ny, int npairs) {
  // neighbour offsets and Philox counters of the owned pairs, fixed for the item
  int lft[kStepPPT], rgt[kStepPPT], up[kStepPPT], dn[kStepPPT];
  uint32_t pid[kStepPPT];
  uint64_t trj[kStepPPT];
  cpx<float> beta[2 * kStepPPT];
  const uint64_t traj0 = g.traj_ids ? g.traj_ids[item.t0] : P.traj_id0 + (uint64_t)item.t0;  // wave-uniform
  const int yh = ny / 2;
  const int wave_p = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63);  // first pair of the wave
#pragma unroll
  for (int j = 0; j < kStepPPT; ++j) {
    const int p = threadIdx.x + kStepBlock * j;
    const int row = p / yh, q = p - row * yh;
    const int tr = MULTI ? row / nxt : 0, r0 = tr * nxt, r = row - r0;
    lft[j] = kStepPairs + row * yh + (q == 0 ? yh - 1 : q - 1);  // an odd site
    rgt[j] = row * yh + (q + 1 == yh ? 0 : q + 1);               // an even site
    up[j] = (r0 + (r == 0 ? nxt - 1 : r - 1)) * yh + q;
    dn[j] = (r0 + (r + 1 == nxt ? 0 : r + 1)) * yh + q;
    pid[j] = (uint32_t)(p - tr * (nxt * yh));
    trj[j] = traj0;
    if (p < npairs) {
      if (MULTI) trj[j] = g.traj_ids ? g.traj_ids[item.t0 + tr] : traj0 + (uint64_t)tr;
      const float4 v = gbeta[p];
      st[p] = beta[2 * j] = mk(v.x, v.y);
      st[kStepPairs + p] = beta[2 * j + 1] = mk(v.z, v.w);
    } else {
      // lanes past the item's end compute along in a wave that has some of it, on
      // slot 0, and store nothing
      lft[j] = rgt[j] = up[j] = dn[j] = 0;
      beta[2 * j] = beta[2 * j + 1] = mk(0.f, 0.f);
    }
  }
  // step constants: dt (rsl + i U (|b|^2 - 1)) = (A0 - Ui |b|^2) + i (B0 + Ur |b|^2),
  // dt iF = (fr, fi), dt h = -i jdt S, sigma^2 folded into the Box-Muller log multiplier
  const float dt = g.dt;
  const float Ur = dt * P.u_re, Ui = dt * P.u_im;
  const float A0 = fmaf(dt, P.rsl_re, Ui), B0 = fmaf(dt, P.rsl_im, -Ur);
  const float fr = -dt * P.f_im, fi = dt * P.f_re;
  const float jdt = dt * (-0.5f * P.kscale);  // dt J
  const float nl = -1.3862943611198906f * P.dt4 * P.dt4;
  __syncthreads();

  // one step from copy C of the state to the other
  auto step_from = [&](auto copy, uint32_t step) __attribute__((always_inline)) {
    constexpr int C = decltype(copy)::value;
    const cpx<float>* cur = st + 2 * kStepPairs * C;
    cpx<float>* nxt_st = st + 2 * kStepPairs * (1 - C);
#pragma unroll
    for (int j = 0; j < kStepPPT; ++j) {
      const int p = threadIdx.x + kStepBlock * j;
      if (wave_p + kStepBlock * j < npairs) {
        const cpx<float> L = cur[lft[j]], R = cur[rgt[j]];
        cpx<float> u[2], d[2];
        if (XHOP) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            u[h] = cur[kStepPairs * h + up[j]];
            d[h] = cur[kStepPairs * h + dn[j]];
          }
        }
        // opaque per step, so that no Philox round is hoisted out of the loop
        uint32_t pair = pid[j];
        asm volatile("" : "+v"(pair));
        const u32x4 w = MULTI ? philox4x32_10(make_counter(trj[j], TAG_WIENER, step, pair), g.key0, g.key1)
                              : philox4x32_10_wave(make_counter(traj0, TAG_WIENER, step, pair), g.key0, g.key1);
        float rs[2], cs[2], sn[2];
        // a wave forming its samples goes first, so that the waves do not bunch up
        // before the transcendental unit (48x48 x 1999: 5.17 -> 4.92 us per step;
        // stacked 2D items lose by it: 30x30 x 2500 2.6 -> 3.0)
        if constexpr (!MULTI) __builtin_amdgcn_s_setprio(2);
        box_muller_f32_scaled(w.x, w.y, nl, rs[0], cs[0], sn[0]);
        box_muller_f32_scaled(w.z, w.w, nl, rs[1], cs[1], sn[1]);
        if constexpr (!MULTI) __builtin_amdgcn_s_setprio(0);
        const cpx<float> z0 = beta[2 * j], z1 = beta[2 * j + 1];
        float sr[2], si[2];
        sr[0] = z1.re + L.re;
        si[0] = z1.im + L.im;
        sr[1] = R.re + z0.re;
        si[1] = R.im + z0.im;
        if (XHOP) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            sr[h] += d[h].re + u[h].re;
            si[h] += d[h].im + u[h].im;
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const cpx<float> z = h ? z1 : z0;
          const float mq = fmaf(z.im, z.im, z.re * z.re);
          const float cr = UI0 ? A0 : fmaf(-Ui, mq, A0), ci = fmaf(Ur, mq, B0);
          // increment = noise + dt iF + drift + hopping, all small, added to beta once
          float dr = fmaf(rs[h], cs[h], fr);
          dr = fmaf(cr, z.re, dr);
          dr = fmaf(-ci, z.im, dr);
          dr = fmaf(jdt, si[h], dr);
          float di = fmaf(rs[h], sn[h], fi);
          di = fmaf(cr, z.im, di);
          di = fmaf(ci, z.re, di);
          di = fmaf(-jdt, sr[h], di);
          beta[2 * j + h] = mk(z.re + dr, z.im + di);
        }
        if (p < npairs) {
          nxt_st[p] = beta[2 * j];
          nxt_st[kStepPairs + p] = beta[2 * j + 1];
        }
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
  for (int j = 0; j < kStepPPT; ++j) {
    const int p = threadIdx.x + kStepBlock * j;
    if (p < npairs) gbeta[p] = make_float4(beta[2 * j].re, beta[2 * j].im, beta[2 * j + 1].re, beta[2 * j + 1].im);
  }
}

// The step launch: 1024-thread workgroups, up to two site pairs per thread, 64
// registers for eight waves per SIMD (the transcendental instructions then run
// beside the others, as in the 64x64 kernel); ten values spill, thirteen with a
// complex U.
// Bound by VALU issue: 45.6 instructions per site-step (2D; chains 43.5), four of
// them transcendental.  A 512-point sweep frame 35.8 -> 32.3 ms against 256-thread
// workgroups of up to eight pairs per thread (168 registers, three waves per
// SIMD); one-system batches of 16384 trajectories, us per step: 16x16 6.55 -> 5.15,
// 36x50 39.2 -> 33.1, 48x48 45.7 -> 41.1, 1x512 10.2 -> 8.8 (9.5e11 site-steps/s),
// and of 32: 16x16 1.27 -> 0.41, 48x48 1.70 -> 0.84.
template <bool UI0>
__global__ void __launch_bounds__(kStepBlock, 8) sweep_step_kernel(SweepArgs g) {
  extern __shared__ __align__(16) unsigned char smem[];
  int& s_item = *reinterpret_cast<int*>(smem);
  cpx<float>* st = reinterpret_cast<cpx<float>*>(smem + 64);  // [2 copies][even, odd][pairs]
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_item = (int)atomicAdd(g.counter, 1u);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(s_item);
    if (it >= g.n_items) break;  // every workgroup reaches this once the queue is drained
    const SweepItemDev item = g.items[it];
    const SweepPointDev& P = g.points[item.point];
    const int ntr = min(P.tb, P.n_traj - item.t0);
    const int nxt = P.fft_x ? P.nx : 1, ny = P.ny;  // rows per trajectory
    const int npairs = ntr * nxt * ny / 2;          // ny is even for every supported size
    float4* gbeta = reinterpret_cast<float4*>(g.beta + P.state_off + (size_t)item.t0 * nxt * ny);
    if (!P.fft_x)
      step_item<UI0, false, true>(g, P, item, st, gbeta, 1, ny, npairs);
    else if (ntr == 1)
      step_item<UI0, true, false>(g, P, item, st, gbeta, nxt, ny, npairs);
    else
      step_item<UI0, true, true>(g, P, item, st, gbeta, nxt, ny, npairs);
  }
}

// The frame's capture launch: per-trajectory means, mean field and k-space bins.
__global__ void __launch_bounds__(kSweepBlock) sweep_capture_kernel(SweepArgs g) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* red = reinterpret_cast<double*>(smem);  // [8]
  cpx<float>* bufA = reinterpret_cast<cpx<float>*>(smem + 64);
  cpx<float>* bufB = bufA + kSweepMaxSites;
  cpx<float>* twx = bufB + kSweepMaxSites;    // [kMaxNx]
  cpx<float>* twy = twx + kMaxNx;             // [kMaxNy]
  __shared__ int s_item;
  __shared__ double s_bins[kBins + 2];

  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_item = (int)atomicAdd(g.counter, 1u);
    __syncthreads();
    const int it = s_item;
    if (it >= g.n_items) break;  // every workgroup reaches this once the queue is drained
    const SweepItemDev item = g.items[it];
    const SweepPointDev P = g.points[item.point];
    // trajectories in the item: 2D points one at a time, chains stacked as rows
    const int ntr = P.fft_x ? 1 : min(P.tb, P.n_traj - item.t0);
    const int nxt = P.fft_x ? P.nx : 1;        // rows per trajectory
    const int rows_traj = P.fft_x ? 1 : ntr;  // chains: one trajectory per row
    const int nx = nxt * ntr;                  // rows of the item array
    const int ny = P.ny;
    const int m = nx * ny;
    const int npairs = m / 2;  // ny is even for every supported size
    for (int i = threadIdx.x; i < ny; i += blockDim.x) twy[i] = g.tw_pool[P.tw_y + i];
    if (P.fft_x)
      for (int i = threadIdx.x; i < P.nx; i += blockDim.x) twx[i] = g.tw_pool[P.tw_x + i];
    __syncthreads();

    // the item's state: this thread's pairs p = t + 256 j in registers
    cpx<float>* gbeta = g.beta + P.state_off + (size_t)item.t0 * nxt * ny;
    auto load_state = [&](cpx<float> (&beta)[2 * kPPT]) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < kPPT; ++j) {
        const int p = threadIdx.x + kSweepBlock * j;
        if (p < npairs) {
          beta[2 * j] = gbeta[2 * p];
          beta[2 * j + 1] = gbeta[2 * p + 1];
        }
      }
    };

    {
      cpx<float> beta[2 * kPPT];
      load_state(beta);
      // the capture launch records the frame: per-trajectory means, mean
      // field and k-space bins of the state
#pragma unroll
      for (int j = 0; j < kPPT; ++j) {
        const int p = threadIdx.x + kSweepBlock * j;
        if (p < npairs) {
          bufA[2 * p] = beta[2 * j];
          bufA[2 * p + 1] = beta[2 * j + 1];
        }
      }
      __syncthreads();
      {
        // per-trajectory site means of |beta|^2 and |beta|^4 (FP64), summed
        // in a fixed order so that repeated runs agree bit for bit; for
        // stacked chains every row of the item is a trajectory
        if (threadIdx.x < kBins + 2) s_bins[threadIdx.x] = 0.0;
        if (P.fft_x) {
          double a2 = 0.0, a4 = 0.0;
#pragma unroll
          for (int j = 0; j < kPPT; ++j) {
            const int p = threadIdx.x + kSweepBlock * j;
            if (p < npairs)
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const cpx<float> z = beta[2 * j + h];
                const double nn = double(z.re) * double(z.re) + double(z.im) * double(z.im);
                a2 += nn;
                a4 += nn * nn;
              }
          }
#pragma unroll
          for (int o = 32; o > 0; o >>= 1) {
            a2 += __shfl_xor(a2, o, 64);
            a4 += __shfl_xor(a4, o, 64);
          }
          if ((threadIdx.x & 63) == 0) {
            red[2 * (threadIdx.x >> 6)] = a2;
            red[2 * (threadIdx.x >> 6) + 1] = a4;
          }
          __syncthreads();
          if (threadIdx.x == 0) {
            double s2 = 0, s4 = 0;
            for (int w = 0; w < kSweepBlock / 64; ++w) {
              s2 += red[2 * w];
              s4 += red[2 * w + 1];
            }
            const size_t o = P.m_off + (size_t)item.t0 * g.n_frames + g.frame;
            g.traj_m2[o] = s2 / double(m);
            g.traj_m4[o] = s4 / double(m);
          }
        } else {
          for (int r = threadIdx.x; r < rows_traj; r += blockDim.x) {
            double s2 = 0, s4 = 0;
            for (int c = 0; c < ny; ++c) {
              const cpx<float> z = bufA[r * ny + c];
              const double nn = double(z.re) * double(z.re) + double(z.im) * double(z.im);
              s2 += nn;
              s4 += nn * nn;
            }
            const size_t o = P.m_off + (size_t)(item.t0 + r) * g.n_frames + g.frame;
            g.traj_m2[o] = s2 / double(ny);
            g.traj_m4[o] = s4 / double(ny);
          }
        }
        // ensemble sum of beta over all sites (mean field)
        double br = 0.0, bi = 0.0;
#pragma unroll
        for (int j = 0; j < kPPT; ++j) {
          const int p = threadIdx.x + kSweepBlock * j;
          if (p < npairs)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              br += double(beta[2 * j + h].re);
              bi += double(beta[2 * j + h].im);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          br += __shfl_xor(br, o, 64);
          bi += __shfl_xor(bi, o, 64);
        }
        __syncthreads();  // s_bins cleared, bufA reads done before the FFT overwrites it
        if ((threadIdx.x & 63) == 0) {
          atomicAdd(&s_bins[kBins], br);
          atomicAdd(&s_bins[kBins + 1], bi);
        }
      }

      {
        // k-space populations: forward FFT, rows (length ny) then columns
        // (length nx) for 2D points; |DFT beta|^2 per radial bin, summed over
        // this item's trajectories
        // the radix plans are read where they lie in global memory: indexing
        // the local copy's plan arrays would put the whole copy in scratch
        const SweepPointDev& Pg = g.points[item.point];
        cpx<float>* cur = fft_dim<-1>(bufA, bufB, Pg.py, nx, ny, 1, twy);
        if (P.fft_x) {
          cpx<float>* other = (cur == bufA) ? bufB : bufA;
          cur = fft_dim<-1>(cur, other, Pg.px, ny, 1, ny, twx);
        }
        for (int i = threadIdx.x; i < m; i += blockDim.x) {
          const cpx<float> f = cur[i];
          const int mode = P.fft_x ? i : i % ny;
          atomicAdd(&s_bins[g.bin_pool[P.bin_off + mode]], double(f.re) * double(f.re) + double(f.im) * double(f.im));
        }
        __syncthreads();
        if (threadIdx.x < kBins + 2)
          atomicAdd(&g.ksum[((size_t)P.index * g.n_frames + g.frame) * (kBins + 2) + threadIdx.x], s_bins[threadIdx.x]);
      }
    }
  }
}

// vacuum-type start beta_0 = beta_init + sigma xi (TWMCBaseSolver.cpp:126-134)
// a site pair per thread and pass: one Philox draw per pair and, while a point's pairs
// fit 32 bits, no 64-bit division (512 points, 63M sites: 1.31 -> 0.90 ms)
__global__ void sweep_init_kernel(const SweepPointDev* points, int n_points, const double* binit, cpx<float>* beta,
                                  uint32_t key0, uint32_t key1) {
  for (int p = 0; p < n_points; ++p) {
    const SweepPointDev P = points[p];
    const int n = P.nx * P.ny, np = n / 2;  // ny is even for every supported size
    const uint64_t total = (uint64_t)P.n_traj * np;
    const double br = binit[4 * p], bi = binit[4 * p + 1], sr = binit[4 * p + 2], si = binit[4 * p + 3];
    for (uint64_t idx = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; idx < total;
         idx += (uint64_t)gridDim.x * blockDim.x) {
      const int t = total >> 32 ? (int)(idx / (uint32_t)np) : (int)((uint32_t)idx / (uint32_t)np);
      const int q = (int)(idx - (uint64_t)t * (uint32_t)np);
      const u32x4 w = philox4x32_10(make_counter(P.traj_id0 + t, TAG_INIT, 0u, (uint32_t)q), key0, key1);
      cpx<float>* out = beta + P.state_off + 2 * idx;
      for (int h = 0; h < 2; ++h) {
        double zr, zi;
        box_muller_f64(h ? w.z : w.x, h ? w.w : w.y, zr, zi);
        out[h] = mk(float(br + (sr * zr - si * zi)), float(bi + (sr * zi + si * zr)));
      }
    }
  }
}

const void* step_kernel(bool u_real) {
  return u_real ? (const void*)sweep_step_kernel<true> : (const void*)sweep_step_kernel<false>;
}

// dynamic LDS: two copies of an item's state, the capture launch the FFT tables too
size_t sweep_lds_bytes(bool capture) { return 64 + 2 * kSweepMaxSites * 8 + (capture ? (kMaxNx + kMaxNy) * 8 : 0); }

// a step launch's LDS limit (above the default 64 KB) and its workgroups per CU
hipError_t step_occupancy(bool u_real, int* per_cu) {
  const int lds = (int)sweep_lds_bytes(false);
  hipError_t e = hipFuncSetAttribute(step_kernel(u_real), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, step_kernel(u_real), kStepBlock, lds);
  return e;
}

hipError_t launch_step(const SweepArgs& a, bool u_real, int grid, hipStream_t s) {
  void* args[] = {const_cast<SweepArgs*>(&a)};
  return hipLaunchKernel(step_kernel(u_real), dim3(grid), dim3(kStepBlock), args, sweep_lds_bytes(false), s);
}

}  // namespace
}  // namespace twmc

using namespace twmc;

namespace {

thread_local std::string g_sweep_error;

struct SweepCtx {
  std::string err;
  int device = 0;
  hipStream_t stream = nullptr;
  double dt = 0.0;
  uint64_t frame_steps = 1, seed = 0;
  std::vector<twmc_sweep_point> pts;
  std::vector<SweepPointDev> dev_pts;
  std::vector<int> tb;  // trajectories per work item, per point
  bool u_real = true;   // Im U = 0 in every point
  std::vector<cpx<float>> tw_pool;
  std::vector<unsigned char> bin_pool;
  uint64_t total_traj = 0, total_sites = 0;
  void *d_points = nullptr, *d_items = nullptr, *d_counter = nullptr, *d_tw = nullptr,
       *d_beta = nullptr, *d_m2 = nullptr, *d_m4 = nullptr, *d_binit = nullptr, *d_bins = nullptr,
       *d_ksum = nullptr;
  size_t ksum_cap = 0;
  size_t m_cap = 0;
  int n_items = 0, n_items_cap = 0, grid = 0, grid_cap = 0;
  void* d_items_cap = nullptr;  // the capture launch's items: 2D points one trajectory each
  twmc_stats stats{};
};

// (a HIP error is cleared: the next call's hipGetLastError would report it again)
int sfail(SweepCtx* c, int code, const std::string& m) {
  if (code == TWMC_ERR_HIP) (void)hipGetLastError();
  if (c) c->err = m;
  g_sweep_error = m;
  return code;
}

#define SCHK(c, expr)                                                                  \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess) return sfail(c, TWMC_ERR_HIP, std::string(#expr ": ") + hipGetErrorString(e_)); \
  } while (0)

// the twiddle factors of length L; returns their offset
int add_twiddles(SweepCtx* c, int L) {
  const int off = (int)c->tw_pool.size();
  for (int m = 0; m < L; ++m) {
    long double a = -2.0L * 3.14159265358979323846264338327950288L * m / L;
    c->tw_pool.push_back(mk(float(cosl(a)), float(sinl(a))));
  }
  return off;
}

// radial bin of every mode of an nx x ny lattice: bin 0 is k = 0; the other
// modes go to 1 + floor(|k| / w) (at most 31) with w = pi sqrt 2 / 31 and
// |k| = 2 pi sqrt((kx'/nx)^2 + (ky'/ny)^2), kx' = min(kx, nx - kx)
int add_bins(SweepCtx* c, int nx, int ny) {
  int off = (int)c->bin_pool.size();
  const double w = M_PI * std::sqrt(2.0) / 31.0;
  for (int kx = 0; kx < nx; ++kx)
    for (int ky = 0; ky < ny; ++ky) {
      int ax = std::min(kx, nx - kx), ay = std::min(ky, ny - ky);
      if (ax == 0 && ay == 0) {
        c->bin_pool.push_back(0);
        continue;
      }
      double k = 2.0 * M_PI * std::sqrt(double(ax) * ax / (double(nx) * nx) + double(ay) * ay / (double(ny) * ny));
      int b = 1 + std::min(30, (int)std::floor(k / w));
      c->bin_pool.push_back((unsigned char)b);
    }
  return off;
}

// lays out points and the two work-item lists (largest first) for tb: the step
// launch stacks tb trajectories of every point per item, the capture launch takes
// 2D points one trajectory per item (chains as in the step launch).  The lists in
// use are replaced only when everything is there.
int build_items(SweepCtx* c, const std::vector<int>& tb) {
  struct List {
    void* d = nullptr;
    int n = 0;
    ~List() {
      if (d) (void)hipFree(d);
    }
  } list[2];
  for (int pass = 0; pass < 2; ++pass) {
    const bool cap = pass == 1;
    std::vector<std::pair<double, SweepItemDev>> items;
    for (size_t p = 0; p < c->pts.size(); ++p) {
      const SweepPointDev& P = c->dev_pts[p];
      const int step = (cap && P.fft_x) ? 1 : tb[p];
      for (int t0 = 0; t0 < P.n_traj; t0 += step) {
        const int rows = std::min(step, P.n_traj - t0);
        const double cost = double(rows) * P.nx * P.ny * std::log2(double(P.nx * P.ny) + 1.0);
        items.push_back({cost, SweepItemDev{(int)p, t0}});
      }
    }
    std::stable_sort(items.begin(), items.end(), [](auto& a, auto& b) { return a.first > b.first; });
    std::vector<SweepItemDev> flat;
    for (auto& it : items) flat.push_back(it.second);
    list[pass].n = (int)flat.size();
    SCHK(c, hipMalloc(&list[pass].d, flat.size() * sizeof(SweepItemDev)));
    SCHK(c, hipMemcpy(list[pass].d, flat.data(), flat.size() * sizeof(SweepItemDev), hipMemcpyHostToDevice));
  }
  std::vector<SweepPointDev> pts = c->dev_pts;
  for (size_t p = 0; p < pts.size(); ++p) pts[p].tb = tb[p];
  SCHK(c, hipMemcpy(c->d_points, pts.data(), pts.size() * sizeof(SweepPointDev), hipMemcpyHostToDevice));
  std::swap(c->d_items, list[0].d);
  std::swap(c->d_items_cap, list[1].d);
  c->n_items = list[0].n;
  c->n_items_cap = list[1].n;
  c->dev_pts = pts;
  c->tb = tb;
  return TWMC_OK;
}

// one segment: reset the queues, the frame capture (if any), then the steps;
// each persistent launch drains its own queue counter
hipError_t launch_segment(SweepCtx* c, const SweepArgs& a) {
  hipLaunchKernelGGL(sweep_reset_kernel, dim3(1), dim3(64), 0, c->stream, (unsigned int*)c->d_counter);
  if (a.capture) {
    SweepArgs ca = a;
    ca.n_steps = 0;
    ca.counter = (unsigned int*)c->d_counter;
    ca.items = (const SweepItemDev*)c->d_items_cap;
    ca.n_items = c->n_items_cap;
    hipLaunchKernelGGL(sweep_capture_kernel, dim3(c->grid_cap), dim3(kSweepBlock), sweep_lds_bytes(true), c->stream,
                       ca);
  }
  if (a.n_steps > 0) {
    SweepArgs sa = a;
    sa.capture = 0;
    sa.counter = (unsigned int*)c->d_counter + 1;
    hipError_t e = launch_step(sa, c->u_real, c->grid, c->stream);
    if (e != hipSuccess) return e;
  }
  return hipGetLastError();
}

SweepArgs base_args(SweepCtx* c) {
  SweepArgs a{};
  a.points = (const SweepPointDev*)c->d_points;
  a.items = (const SweepItemDev*)c->d_items;
  a.n_items = c->n_items;
  a.counter = (unsigned int*)c->d_counter;
  a.tw_pool = (const cpx<float>*)c->d_tw;
  a.beta = (cpx<float>*)c->d_beta;
  a.traj_m2 = (double*)c->d_m2;
  a.traj_m4 = (double*)c->d_m4;
  a.bin_pool = (const unsigned char*)c->d_bins;
  a.ksum = (double*)c->d_ksum;
  a.dt = (float)c->dt;
  a.key0 = uint32_t(c->seed & 0xffffffffu);
  a.key1 = uint32_t(c->seed >> 32);
  return a;
}

int init_state(SweepCtx* c) {
  hipLaunchKernelGGL(sweep_init_kernel, dim3(1024), dim3(256), 0, c->stream, (const SweepPointDev*)c->d_points,
                     (int)c->pts.size(), (const double*)c->d_binit, (cpx<float>*)c->d_beta,
                     uint32_t(c->seed & 0xffffffffu), uint32_t(c->seed >> 32));
  SCHK(c, hipGetLastError());
  return TWMC_OK;
}

}  // namespace

namespace twmc {

// The main API's FP32 FFT-hopping batches of one site-uniform system run
// their steps on this kernel as a single point: the state layout is the
// same (trajectories contiguous, each row-major), each step item stacks tb
// trajectories, and the trajectory ids come from the batch's id array.  The
// batch's frames stay with the LDS kernel (its capture-only launch), which
// forms the per-site and per-mode sums of that API.
bool stack_supported(int nx, int ny) {
  return ny % 2 == 0 && ny <= kMaxNy && nx <= kMaxNx && nx * ny <= kSweepMaxSites && (nx == 1 || ny > 1);
}

hipError_t stack_prepare(StackPlan& sp, int nx, int ny, int n_traj, const double rsl[2], const double u[2],
                         const double f[2], double dt4, double kscale) {
  stack_release(sp);
  SweepPointDev P{};
  P.nx = nx;
  P.ny = ny;
  P.fft_x = nx > 1 ? 1 : 0;
  P.rsl_re = float(rsl[0]);
  P.rsl_im = float(rsl[1]);
  P.u_re = float(u[0]);
  P.u_im = float(u[1]);
  P.f_re = float(f[0]);
  P.f_im = float(f[1]);
  P.dt4 = float(dt4);
  P.kscale = float(kscale);
  P.n_traj = n_traj;
  int dev = 0, cus = 0, per_cu = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  sp.u_real = u[1] == 0.0;
  if (e == hipSuccess) e = step_occupancy(sp.u_real, &per_cu);
  if (e != hipSuccess) return e;
  // Trajectories per item: about 2048 sites, one pair per thread, when the batch
  // fills every workgroup slot of the chip (16x16 x 128 sweep points: 6.5e11
  // site-steps/s with 2048 sites, 6.1e11 with 1024 and 6.2e11 with 4096), and no
  // more than it takes to give every slot an item: a few trajectories then run
  // side by side on as many CUs (8x16 x 32: 0.37 us per step one to an item,
  // 0.70 stacked sixteen to an item).
  const int slots = std::max(1, per_cu) * cus;
  P.tb = std::max(1, std::min({(n_traj + slots - 1) / slots, 2048 / (nx * ny), kMaxRows}));
  std::vector<SweepItemDev> items;
  for (int t0 = 0; t0 < n_traj; t0 += P.tb) items.push_back(SweepItemDev{0, t0});
  sp.n_items = (int)items.size();
  sp.tb = P.tb;
  sp.step = {std::min(sp.n_items, slots), kStepBlock, sweep_lds_bytes(false)};
  if (e == hipSuccess) e = hipMalloc(&sp.d_point, sizeof(SweepPointDev));
  if (e == hipSuccess) e = hipMalloc(&sp.d_items, items.size() * sizeof(SweepItemDev));
  if (e == hipSuccess) e = hipMalloc(&sp.d_counter, 2 * sizeof(unsigned int));
  if (e == hipSuccess) e = hipMemcpy(sp.d_point, &P, sizeof(SweepPointDev), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(sp.d_items, items.data(), items.size() * sizeof(SweepItemDev), hipMemcpyHostToDevice);
  if (e != hipSuccess) stack_release(sp);
  return e;
}

hipError_t stack_launch(const StackPlan& sp, const StepArgs& a, hipStream_t s) {
  SweepArgs g{};
  g.points = (const SweepPointDev*)sp.d_point;
  g.items = (const SweepItemDev*)sp.d_items;
  g.n_items = sp.n_items;
  g.counter = (unsigned int*)sp.d_counter;
  g.beta = (cpx<float>*)a.beta;
  g.dt = float(a.dt);
  g.key0 = a.key0;
  g.key1 = a.key1;
  g.step0 = a.step0;
  g.n_steps = a.n_steps;
  g.traj_ids = a.traj_ids;
  hipLaunchKernelGGL(sweep_reset_kernel, dim3(1), dim3(64), 0, s, (unsigned int*)sp.d_counter);
  return launch_step(g, sp.u_real, sp.step.grid, s);
}

void stack_release(StackPlan& sp) {
  void* bufs[] = {sp.d_point, sp.d_items, sp.d_counter};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  sp.d_point = sp.d_items = sp.d_counter = nullptr;
  sp.n_items = 0;
}

}  // namespace twmc

extern "C" {

const char* twmc_sweep_last_error(const twmc_sweep_ctx* ctx) {
  return ctx ? reinterpret_cast<const SweepCtx*>(ctx)->err.c_str() : g_sweep_error.c_str();
}

int twmc_sweep_create(const twmc_sweep_point* pts, uint64_t n_points, double dt, uint64_t frame_steps,
                      uint64_t seed, int device, twmc_sweep_ctx** ctx_out) {
  if (!pts || !ctx_out || n_points == 0) return sfail(nullptr, TWMC_ERR_INVALID, "empty sweep");
  if (!(dt > 0.0) || frame_steps < 1) return sfail(nullptr, TWMC_ERR_INVALID, "dt and frame_steps must be positive");
  // one launch advances one frame; its step count is an int kernel argument
  if (frame_steps > (uint64_t(1) << 30)) return sfail(nullptr, TWMC_ERR_INVALID, "frame_steps above 2^30");
  *ctx_out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return sfail(nullptr, TWMC_ERR_HIP, "no HIP device available");
  if (device < 0 || device >= ndev) return sfail(nullptr, TWMC_ERR_INVALID, "device index out of range");
  SweepCtx* c = new SweepCtx();
  c->device = device;
  c->dt = dt;
  c->frame_steps = frame_steps;
  c->seed = seed;
  c->pts.assign(pts, pts + n_points);
  std::map<int, int> twiddles;                    // length -> offset
  std::map<std::pair<int, int>, int> bin_tables;  // shape -> bin table offset
  auto twiddles_of = [&](int L) {
    auto it = twiddles.find(L);
    if (it == twiddles.end()) it = twiddles.emplace(L, add_twiddles(c, L)).first;
    return it->second;
  };
  uint64_t state_off = 0, m_off = 0;
  for (uint64_t p = 0; p < n_points; ++p) {
    const twmc_sweep_point& q = pts[p];
    int nx = q.nx, ny = q.ny;
    if (nx > 1 && ny == 1) std::swap(nx, ny);  // chains are 1 x N
    SweepPointDev P{};
    P.nx = nx;
    P.ny = ny;
    P.fft_x = nx > 1 ? 1 : 0;
    if (nx * ny > kSweepMaxSites || ny > kMaxNy || nx > kMaxNx || (ny % 2) != 0 || q.n_traj == 0 ||
        q.n_traj > (uint64_t)INT32_MAX || !make_radix_plan(ny, P.py) || !make_radix_plan(nx, P.px)) {
      delete c;
      return sfail(nullptr, TWMC_ERR_UNSUPPORTED,
                   "sweep point " + std::to_string(p) + ": up to 4096 sites, 64 rows, rows of even length <= 512");
    }
    P.tw_y = twiddles_of(ny);
    P.tw_x = twiddles_of(nx);
    // rsl = -i omega - gamma/2 (TWMCBaseSolver.cpp:74)
    P.rsl_re = float(q.omega[1] - q.gamma / 2.0);
    P.rsl_im = float(-q.omega[0]);
    P.u_re = float(q.U[0]);
    P.u_im = float(q.U[1]);
    if (q.U[1] != 0.0) c->u_real = false;
    P.f_re = float(q.F[0]);
    P.f_im = float(q.F[1]);
    P.dt4 = float(std::sqrt(q.gamma * dt / 4.0));
    P.kscale = float(-2.0 * q.J);
    P.n_traj = (int)q.n_traj;
    P.traj_id0 = q.traj_id0;
    P.state_off = state_off;
    P.m_off = m_off;
    P.index = (int)p;
    {
      auto bt = bin_tables.find({nx, ny});
      if (bt == bin_tables.end()) bt = bin_tables.emplace(std::make_pair(nx, ny), add_bins(c, nx, ny)).first;
      P.bin_off = bt->second;
    }
    state_off += (uint64_t)q.n_traj * nx * ny;
    m_off += q.n_traj;  // times n_frames at run time
    c->dev_pts.push_back(P);
    // default stacking: fill a workgroup with about 2048 sites
    c->tb.push_back(std::max(1, std::min({(int)q.n_traj, 2048 / (nx * ny), kMaxRows})));
  }
  c->total_traj = m_off;
  c->total_sites = state_off;
  hipError_t e = hipSetDevice(device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipMalloc(&c->d_points, c->dev_pts.size() * sizeof(SweepPointDev));
  if (e == hipSuccess) e = hipMalloc(&c->d_counter, 256);
  if (e == hipSuccess) e = hipMalloc(&c->d_tw, c->tw_pool.size() * sizeof(cpx<float>));
  if (e == hipSuccess) e = hipMalloc(&c->d_beta, state_off * sizeof(cpx<float>));
  std::vector<double> binit(4 * n_points);
  for (uint64_t p = 0; p < n_points; ++p) {
    binit[4 * p] = pts[p].beta_init[0];
    binit[4 * p + 1] = pts[p].beta_init[1];
    binit[4 * p + 2] = pts[p].beta_sigma[0];
    binit[4 * p + 3] = pts[p].beta_sigma[1];
  }
  if (e == hipSuccess) e = hipMalloc(&c->d_binit, binit.size() * 8);
  if (e == hipSuccess) e = hipMalloc(&c->d_bins, c->bin_pool.size());
  if (e == hipSuccess) e = hipMemcpy(c->d_bins, c->bin_pool.data(), c->bin_pool.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(c->d_tw, c->tw_pool.data(), c->tw_pool.size() * sizeof(cpx<float>), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(c->d_binit, binit.data(), binit.size() * 8, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipFuncSetAttribute((const void*)sweep_capture_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sweep_lds_bytes(true));
  int per_cu = 0, per_cu_cap = 0, cus = 0;
  if (e == hipSuccess) e = step_occupancy(c->u_real, &per_cu);
  if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu_cap, (const void*)sweep_capture_kernel, kSweepBlock, sweep_lds_bytes(true));
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
  if (e != hipSuccess) {
    std::string m = std::string("sweep setup: ") + hipGetErrorString(e);
    twmc_sweep_destroy(reinterpret_cast<twmc_sweep_ctx*>(c));
    return sfail(nullptr, TWMC_ERR_HIP, m);
  }
  c->grid = std::max(1, per_cu) * cus;
  c->grid_cap = std::max(1, per_cu_cap) * cus;
  int rc = build_items(c, c->tb);
  if (rc) {
    std::string m = c->err;
    twmc_sweep_destroy(reinterpret_cast<twmc_sweep_ctx*>(c));
    return sfail(nullptr, rc, m);
  }
  *ctx_out = reinterpret_cast<twmc_sweep_ctx*>(c);
  return TWMC_OK;
}

void twmc_sweep_destroy(twmc_sweep_ctx* ctx) {
  if (!ctx) return;
  SweepCtx* c = reinterpret_cast<SweepCtx*>(ctx);
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  void* bufs[] = {c->d_points, c->d_items, c->d_items_cap, c->d_counter, c->d_tw, c->d_beta, c->d_m2, c->d_m4, c->d_binit,
                  c->d_bins, c->d_ksum};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

int twmc_sweep_set_batching(twmc_sweep_ctx* ctx, const int32_t* tb) {
  if (!ctx || !tb) return sfail(nullptr, TWMC_ERR_INVALID, "null argument");
  SweepCtx* c = reinterpret_cast<SweepCtx*>(ctx);
  std::vector<int> next(c->pts.size());
  for (size_t p = 0; p < c->pts.size(); ++p) {
    const SweepPointDev& P = c->dev_pts[p];
    const int v = tb[p];
    if (v < 1 || v > kMaxRows || (int64_t)v * P.nx * P.ny > kSweepMaxSites)
      return sfail(c, TWMC_ERR_INVALID, "stacking exceeds 4096 sites or 256 trajectories");
    next[p] = std::min(v, P.n_traj);
  }
  return build_items(c, next);
}

int twmc_sweep_get_batching(twmc_sweep_ctx* ctx, int32_t* tb) {
  if (!ctx || !tb) return sfail(nullptr, TWMC_ERR_INVALID, "null argument");
  SweepCtx* c = reinterpret_cast<SweepCtx*>(ctx);
  for (size_t p = 0; p < c->tb.size(); ++p) tb[p] = c->tb[p];
  return TWMC_OK;
}

// Runs the sweep from the vacuum start; frames follow the reference loop with
// store_initial.  use_graph captures the frame loop into one hipGraph.
int twmc_sweep_run(twmc_sweep_ctx* ctx, double t_start, double t_end, int32_t use_graph, double* traj_m2, double* traj_m4,
                   double* ksum, uint64_t* n_frames_out, double* kernel_ms) {
  if (!ctx) return sfail(nullptr, TWMC_ERR_INVALID, "null argument");
  SweepCtx* c = reinterpret_cast<SweepCtx*>(ctx);
  SCHK(c, hipSetDevice(c->device));
  // frame schedule (TWMCBaseSolver.cpp:221-266), store_initial = true
  double dt_obs = c->dt * (double)c->frame_steps;
  uint64_t nf = (uint64_t)(size_t)nearbyint((t_end - t_start) / dt_obs) + 1;
  std::vector<uint64_t> cap{0};
  uint64_t i_frame = 1, i_step = 0;
  double t = t_start;
  while (t <= t_end) {
    t += c->dt;
    i_step++;
    if ((i_step % c->frame_steps == 0) && i_frame < nf) {
      cap.push_back(i_step);
      i_frame++;
      if (i_frame == nf) break;
    }
  }
  const uint64_t frames = i_frame;
  size_t need = (size_t)c->total_traj * frames;
  if (need > c->m_cap) {
    if (c->d_m2) (void)hipFree(c->d_m2);
    if (c->d_m4) (void)hipFree(c->d_m4);
    c->d_m2 = c->d_m4 = nullptr;
    c->m_cap = 0;
    SCHK(c, hipMalloc(&c->d_m2, need * 8));
    SCHK(c, hipMalloc(&c->d_m4, need * 8));
    c->m_cap = need;
  }
  const size_t kneed = c->pts.size() * frames * (kBins + 2);
  if (kneed > c->ksum_cap) {
    if (c->d_ksum) (void)hipFree(c->d_ksum);
    c->d_ksum = nullptr;
    c->ksum_cap = 0;
    SCHK(c, hipMalloc(&c->d_ksum, kneed * 8));
    c->ksum_cap = kneed;
  }
  SCHK(c, hipMemsetAsync(c->d_ksum, 0, kneed * 8, c->stream));  // before any graph capture
  // per-trajectory means are laid out [point block][traj][frame]
  std::vector<SweepPointDev> pts = c->dev_pts;
  for (auto& P : pts) P.m_off *= frames;
  SCHK(c, hipMemcpyAsync(c->d_points, pts.data(), pts.size() * sizeof(SweepPointDev), hipMemcpyHostToDevice, c->stream));
  int rc = init_state(c);
  if (rc) return rc;
  SCHK(c, hipStreamSynchronize(c->stream));

  // events and graph of this run, released on every return path
  struct RunResources {
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    ~RunResources() {
      if (exec) (void)hipGraphExecDestroy(exec);
      if (graph) (void)hipGraphDestroy(graph);
      if (e1) (void)hipEventDestroy(e1);
      if (e0) (void)hipEventDestroy(e0);
    }
  } res;
  SCHK(c, hipEventCreate(&res.e0));
  SCHK(c, hipEventCreate(&res.e1));
  hipEvent_t e0 = res.e0, e1 = res.e1;
  if (use_graph) SCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  else SCHK(c, hipEventRecord(e0, c->stream));
  for (size_t k = 0; k < cap.size(); ++k) {
    uint64_t end = (k + 1 < cap.size()) ? cap[k + 1] : i_step;
    SweepArgs a = base_args(c);
    a.step0 = cap[k];
    a.n_steps = (int)(end - cap[k]);
    a.capture = 1;
    a.frame = (int)k;
    a.n_frames = (int)frames;
    hipError_t le = launch_segment(c, a);
    if (le != hipSuccess) {
      if (use_graph) {
        hipGraph_t g2;
        (void)hipStreamEndCapture(c->stream, &g2);
        if (g2) (void)hipGraphDestroy(g2);
      }
      return sfail(c, TWMC_ERR_HIP, std::string("sweep launch: ") + hipGetErrorString(le));
    }
  }
  if (use_graph) {
    SCHK(c, hipStreamEndCapture(c->stream, &res.graph));
    SCHK(c, hipGraphInstantiate(&res.exec, res.graph, nullptr, nullptr, 0));
    SCHK(c, hipEventRecord(e0, c->stream));
    SCHK(c, hipGraphLaunch(res.exec, c->stream));
  }
  SCHK(c, hipEventRecord(e1, c->stream));
  SCHK(c, hipStreamSynchronize(c->stream));
  float ms = 0.f;
  SCHK(c, hipEventElapsedTime(&ms, e0, e1));
  c->stats.step_kernel_ms += ms;
  c->stats.step_launches += cap.size();
  c->stats.site_steps += 0;
  for (size_t p = 0; p < c->pts.size(); ++p)
    c->stats.site_steps += (uint64_t)c->dev_pts[p].n_traj * c->dev_pts[p].nx * c->dev_pts[p].ny * i_step;
  c->stats.grid = c->grid;
  c->stats.block = kStepBlock;
  c->stats.lds_bytes = (int)sweep_lds_bytes(false);
  if (kernel_ms) *kernel_ms = ms;
  if (n_frames_out) *n_frames_out = frames;
  if (traj_m2) SCHK(c, hipMemcpy(traj_m2, c->d_m2, need * 8, hipMemcpyDeviceToHost));
  if (traj_m4) SCHK(c, hipMemcpy(traj_m4, c->d_m4, need * 8, hipMemcpyDeviceToHost));
  if (ksum) SCHK(c, hipMemcpy(ksum, c->d_ksum, kneed * 8, hipMemcpyDeviceToHost));
  return TWMC_OK;
}

int twmc_sweep_mode_bins(twmc_sweep_ctx* ctx, uint64_t point, uint8_t* bins) {
  if (!ctx || !bins) return sfail(nullptr, TWMC_ERR_INVALID, "null argument");
  SweepCtx* c = reinterpret_cast<SweepCtx*>(ctx);
  if (point >= c->pts.size()) return sfail(c, TWMC_ERR_INVALID, "point index out of range");
  const SweepPointDev& P = c->dev_pts[point];
  std::memcpy(bins, &c->bin_pool[P.bin_off], (size_t)P.nx * P.ny);
  return TWMC_OK;
}

// Times each candidate stacking per lattice shape on a short run (steps steps
// of every point of that shape) and keeps the fastest per site-step.
int twmc_sweep_autotune(twmc_sweep_ctx* ctx, int32_t steps, int32_t* tb_out) {
  if (!ctx) return sfail(nullptr, TWMC_ERR_INVALID, "null argument");
  SweepCtx* c = reinterpret_cast<SweepCtx*>(ctx);
  if (steps < 1) steps = 20;
  std::map<std::pair<int, int>, std::vector<size_t>> by_shape;  // (rows, row length) -> points
  for (size_t p = 0; p < c->pts.size(); ++p) by_shape[{c->dev_pts[p].nx, c->dev_pts[p].ny}].push_back(p);
  std::vector<int32_t> best = c->tb;
  for (auto& kv : by_shape) {
    const int sites = kv.first.first * kv.first.second;
    if (2 * sites > kSweepMaxSites) {  // one trajectory per item is the only choice
      for (size_t p : kv.second) best[p] = 1;
      continue;
    }
    double best_rate = -1.0;
    for (int cand = 1; cand * sites <= kSweepMaxSites && cand <= kMaxRows; cand *= 2) {
      if (cand > c->dev_pts[kv.second[0]].n_traj && cand > 1) break;
      std::vector<int32_t> tb = c->tb;
      for (size_t p : kv.second) tb[p] = cand;
      // time only this shape: a context holding just these points
      std::vector<twmc_sweep_point> sub;
      for (size_t p : kv.second) sub.push_back(c->pts[p]);
      twmc_sweep_ctx* tctx = nullptr;
      int rc = twmc_sweep_create(sub.data(), sub.size(), c->dt, (uint64_t)steps, c->seed, c->device, &tctx);
      if (rc) return sfail(c, rc, twmc_sweep_last_error(nullptr));
      std::vector<int32_t> subtb(sub.size(), cand);
      rc = twmc_sweep_set_batching(tctx, subtb.data());
      double ms = 0.0;
      if (!rc) rc = twmc_sweep_run(tctx, 0.0, c->dt * steps, 0, nullptr, nullptr, nullptr, nullptr, &ms);
      uint64_t ss = reinterpret_cast<SweepCtx*>(tctx)->stats.site_steps;
      twmc_sweep_destroy(tctx);
      if (rc) return sfail(c, rc, "autotune run failed");
      double rate = ms > 0 ? double(ss) / ms : 0.0;
      if (rate > best_rate) {
        best_rate = rate;
        for (size_t p : kv.second) best[p] = cand;
      }
    }
  }
  int rc = twmc_sweep_set_batching(ctx, best.data());
  if (rc) return rc;
  if (tb_out)
    for (size_t p = 0; p < best.size(); ++p) tb_out[p] = best[p];
  return TWMC_OK;
}

int twmc_sweep_query(twmc_sweep_ctx* ctx, twmc_stats* st) {
  if (!ctx || !st) return sfail(nullptr, TWMC_ERR_INVALID, "null argument");
  *st = reinterpret_cast<SweepCtx*>(ctx)->stats;
  return TWMC_OK;
}

}  // extern "C"
