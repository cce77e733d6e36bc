// twmc_sparse.hip -- step kernel for matrix hopping with few nonzeros per column
// (the Lieb chain open or periodic, disordered chains, ladders and square
// lattices) of up to 512 sites, in FP64, or in FP32 with parameters drawn per
// trajectory: the cases the FP32 banded kernel does not take (twmc_ahead.hip steps
// small batches of them).
//
// The reference's Lieb solver applies h_j = -i sum_i beta_i C_ij with a sparse
// product per step (TWMCLiebSolver.cpp:259-267).  Here a wave holds one or more
// whole trajectories: S sites per lane (one to four Philox pairs), their
// states, site parameters and up to M coefficients C_ij in registers for the
// whole launch.  A step writes the state to the wave's LDS slice, reads each
// site's M neighbours by precomputed address (entries without a bond read a
// slot that holds zero, so no value of an uncoupled site enters), and updates.
// All of it stays inside one wave: no barrier, the four waves of a workgroup
// share only the Box-Muller tables.
//
// What bounds it: with fewer waves than SIMDs the latency of one step's chain,
// else VALU issue (about 95 instructions per FP64 site-step).  The noise does
// not depend on the state, so with two sites per lane the next step's draw is
// formed beside this step's LDS round trip and update.
// Measured, us per step of the whole batch, against the LDS kernel's product (256
// threads per trajectory, columns through global index tables): FP64 Lieb chain
// of 72 sites x 2500 trajectories 6.85 -> 1.09, x 16384 37.9 -> 5.3, 384 sites x 4096
// 16.2 -> 6.2 (2.6e11 site-steps/s); FP32 with drawn energies, 384 sites x 4096 9.8 ->
// 2.25 (7.0e11).
#include <algorithm>
#include <cmath>

#include "twmc_cplx.h"
#include "twmc_f64math.h"
#include "twmc_internal.h"
#include "twmc_rng.h"

namespace twmc {

namespace {

constexpr int kWaves = 4;  // waves per workgroup, each on its own trajectories

// the FP64 Box-Muller's ln and sin / cos tables (twmc_f64math.h)
alignas(16) __device__ const double kF64TabDev[f64::kTabSize] = TWMC_F64_TABLES;

// increments sqrt(gamma dt / 4) xi of a site pair
template <typename T, bool PRIO>
__device__ __forceinline__ void pair_noise(const u32x4& x, T sig, T (&re)[2], T (&im)[2], const f64::Series& k,
                                           const double* ltab) {
  // rounded products: fused into the update in some forms of the step and not in
  // others, they would make a trajectory's bits depend on the batch
  TWMC_NO_CONTRACT
  if constexpr (sizeof(T) == 8) {
    const uint32_t a[2] = {x.x, x.z}, b[2] = {x.y, x.w};
    f64::box_muller<2>(a, b, re, im, k, ltab);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      re[h] *= sig;
      im[h] *= sig;
    }
  } else {
    const float nl = -1.3862943611198906f * sig * sig;
    float r[2], c[2], s[2];
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(2);
    box_muller_f32_scaled(x.x, x.y, nl, r[0], c[0], s[0]);
    box_muller_f32_scaled(x.z, x.w, nl, r[1], c[1], s[1]);
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      re[h] = r[h] * c[h];
      im[h] = r[h] * s[h];
    }
  }
}

// order of the wave's own LDS accesses (the hardware runs them in order)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// PRIO (FP32, more than two waves per SIMD): a wave forming its Box-Muller samples
// goes first, so that the waves do not bunch up before the transcendental unit
// (384 sites x 4096 2.42 -> 2.22 us per step; 72 x 1000, one wave, 0.33 -> 0.37).
// FT: the drive is F(t), read per step instead of held: after the hopping sums, whose
// neighbours' registers are free by then, and under the draw (400 sites of six
// neighbours, FP64, 64 trajectories: 3.80 -> 3.44 us per step, the LDS kernel's product
// 3.61; three neighbours 3.23 -> 2.92, 3.04).  The eight-site form of six neighbours
// still spills five registers.
template <typename T, int S, int M, bool PRIO, bool FT>
__global__ void __launch_bounds__(64 * kWaves, S == 2 ? 2 : 1) sparse_step_kernel(StepArgs g) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int n = g.n, lp = (n + S - 1) / S, tpw = 64 / lp;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double* ltab = reinterpret_cast<const double*>(smem);
  constexpr int kTab = sizeof(T) == 8 ? f64::kTabSize * (int)sizeof(double) : 0;
  // the tables' loads run beside those of the coefficients below
  constexpr int kTabLoads = f64::kTabSize / (64 * kWaves);
  static_assert(kTabLoads * 64 * kWaves == f64::kTabSize, "whole rounds of the workgroup");
  double tab[kTabLoads];
  if constexpr (sizeof(T) == 8)
#pragma unroll
    for (int k = 0; k < kTabLoads; ++k) tab[k] = kF64TabDev[threadIdx.x + 64 * kWaves * k];
  f64::Series bmk = f64::kSeries;
  if constexpr (sizeof(T) == 8) f64::pin(bmk);

  // this lane: trajectory tr of the wave, sites S q .. S q + S - 1 (lanes past
  // the last trajectory repeat lane 0 and write nothing).  Site S q + s lies
  // at slot s lp + q, so that neighbouring lanes read neighbouring slots; slot
  // S lp holds zero.
  const bool act = lane < tpw * lp;
  const int tr = act ? lane / lp : 0, q = act ? lane - tr * lp : 0;
  const int slots = S * lp + 1;
  cpx<T>* const ring = reinterpret_cast<cpx<T>*>(smem + kTab) + (size_t)(wave * tpw + tr) * slots;
  if (act && q == 0) ring[S * lp] = mk(T(0), T(0));

  // FP32 forms the increment from constants scaled by dt, FP64 scales the drift
  // once at the end (one more fma per component; dt C_ij rounded would be a
  // systematic 1e-16 of the bond over the whole run)
  constexpr bool kScaled = sizeof(T) == 4;
  const T dt = T(g.dt), sig = T(g.dt4), cdt = kScaled ? dt : T(1);
  T cf[S][M];
  int at[S][M];
  const T* coef = reinterpret_cast<const T*>(g.ell_coef);
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int j = q * S + s, e = min(j, n - 1) * M + m;
      const int row = g.ell_row[e];
      const T c = coef[e];
      const bool bond = j < n && row >= 0;
      cf[s][m] = bond ? c : T(0);
      at[s][m] = bond ? (row % S) * lp + row / S : S * lp;
    }
  if constexpr (sizeof(T) == 8) {
#pragma unroll
    for (int k = 0; k < kTabLoads; ++k) reinterpret_cast<double*>(smem)[threadIdx.x + 64 * kWaves * k] = tab[k];
    __syncthreads();
  }

  const int n_waves = gridDim.x * kWaves;
  for (int b0 = (blockIdx.x * kWaves + wave) * tpw; b0 < g.n_traj; b0 += n_waves * tpw) {
    // a trajectory past the batch's end: the last one again, not stored
    const bool live = act && b0 + tr < g.n_traj;
    const int b = min(b0 + tr, g.n_traj - 1);
    const uint64_t traj = g.traj_ids[b];
    cpx<T>* gb = reinterpret_cast<cpx<T>*>(g.beta) + (size_t)b * n;
    const size_t poff = (size_t)(g.param_stride ? b : 0) * n;
    // c (rsl + i U (|b|^2 - 1)) = (A0 - Ui |b|^2) + i (B0 + Ur |b|^2), c i F = (fr, fi), c = cdt
    constexpr int SF = FT ? 1 : S, SG = FT ? S : 1;
    T zr[S], zi[S], A0[S], B0[S], Ur[S], Ui[S], fr[SF], fi[SF];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int j = q * S + s;
      const bool in = j < n;
      const cpx<T> zero = mk(T(0), T(0));
      const cpx<T> z = in ? gb[j] : zero;
      const cpx<T> r = in ? reinterpret_cast<const cpx<T>*>(g.rsl)[poff + j] : zero;
      const cpx<T> u = in ? reinterpret_cast<const cpx<T>*>(g.U)[poff + j] : zero;
      const cpx<T> f = in ? reinterpret_cast<const cpx<T>*>(g.F)[poff + j] : zero;
      zr[s] = z.re;
      zi[s] = z.im;
      A0[s] = cdt * (r.re + u.im);
      B0[s] = cdt * (r.im - u.re);
      Ur[s] = cdt * u.re;
      Ui[s] = cdt * u.im;
      if constexpr (!FT) {
        fr[s] = -cdt * f.im;
        fi[s] = cdt * f.re;
      }
    }
    T wr[S], wi[S];
    auto draw = [&](uint32_t step) __attribute__((always_inline)) {
      // opaque, so that no Philox round is hoisted out of the step loop
      uint32_t pair = (uint32_t)(q * (S / 2));
      asm volatile("" : "+v"(pair));
#pragma unroll
      for (int p = 0; p < S / 2; ++p) {
        const u32x4 x = philox4x32_10(make_counter(traj, TAG_WIENER, step, pair + (uint32_t)p), g.key0, g.key1);
        T re[2], im[2];
        pair_noise<T, PRIO>(x, sig, re, im, bmk, ltab);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          wr[2 * p + h] = re[h];
          wi[2 * p + h] = im[h];
        }
      }
    };
    constexpr bool kAhead = S == 2;  // the next step's noise beside this step's update
    if constexpr (kAhead) draw(uint32_t(g.step0));
    // F(t): the interval of the step before and its ends, so that a step reads only the drive
    int ft_id = 0;
    const double ft0 = FT ? g.ft_times[0] : 0.0;
    double ft_lo = ft0, ft_hi = FT && g.ft_n > 1 ? g.ft_times[1] : HUGE_VAL;
    int due = 0, frame = 0;  // steps to the next stored frame, frames stored
    auto store_frame = [&] {
      cpx<T>* out = reinterpret_cast<cpx<T>*>(g.frames) + ((size_t)b * g.frames_stride + g.frame0 + frame) * n;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int j = q * S + s;
        if (live && j < n) out[j] = mk(zr[s], zi[s]);
      }
      ++frame;
      due = g.group_steps;
    };
    for (int st = 0; st < g.n_steps; ++st) {
      if (due-- == 0 && frame < g.group) {
        store_frame();
        --due;
      }
      if (act) {
#pragma unroll
        for (int s = 0; s < S; ++s) ring[s * lp + q] = mk(zr[s], zi[s]);
      }
      wave_sync();
      cpx<T> v[S][M];
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int m = 0; m < M; ++m) v[s][m] = ring[at[s][m]];
      wave_sync();
      T dr[S], di[S];
      // F(t) before this step (TWMCLiebSolver.cpp:252-256), as c i F
      T gr[SG], gi[SG];
      auto drive = [&]() __attribute__((always_inline)) {
        const double t = g.t0 + double(st) * g.dt;
        while (ft_hi < t) {
          ++ft_id;
          ft_lo = ft_hi;
          ft_hi = ft_id + 1 < g.ft_n ? g.ft_times[ft_id + 1] : HUGE_VAL;
        }
        const T fdt = T(t <= ft0 ? 0.0 : t - ft_lo);
        const cpx<T>* fv = reinterpret_cast<const cpx<T>*>(g.ft_vals) + (size_t)ft_id * n;
        const cpx<T>* fs = reinterpret_cast<const cpx<T>*>(g.ft_slopes) + (size_t)ft_id * n;
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const int j = min(q * S + s, n - 1);
          gr[s] = -cdt * fma(fdt, fs[j].im, fv[j].im);
          gi[s] = cdt * fma(fdt, fs[j].re, fv[j].re);
        }
      };
#pragma unroll
      for (int s = 0; s < S; ++s) {
        dr[s] = FT ? T(0) : fr[FT ? 0 : s];
        di[s] = FT ? T(0) : fi[FT ? 0 : s];
      }
      if constexpr (FT && kAhead) drive();
      T nr[S], ni[S];  // this step's noise
      if constexpr (kAhead) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
          nr[s] = wr[s];
          ni[s] = wi[s];
        }
        draw(uint32_t(g.step0 + (uint64_t)st + 1));
      }
      // c h_j = -i sum c C_ij beta_i
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int s = 0; s < S; ++s) {
          dr[s] = fma(cf[s][m], v[s][m].im, dr[s]);
          di[s] = fma(-cf[s][m], v[s][m].re, di[s]);
        }
      // read here, beside the draw: the neighbours' registers are free by now
      if constexpr (FT && !kAhead) drive();
      if constexpr (!kAhead) {
        draw(uint32_t(g.step0 + (uint64_t)st));
#pragma unroll
        for (int s = 0; s < S; ++s) {
          nr[s] = wr[s];
          ni[s] = wi[s];
        }
      }
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const T x = zr[s], y = zi[s], mq = fma(y, y, x * x);
        const T cr = fma(-Ui[s], mq, A0[s]), ci = fma(Ur[s], mq, B0[s]);
        if constexpr (FT) {
          dr[s] += gr[s];
          di[s] += gi[s];
        }
        // increment = noise + dt iF + dt h + drift, all small, added to beta once
        const T ur = fma(-ci, y, fma(cr, x, dr[s])), ui = fma(ci, x, fma(cr, y, di[s]));
        zr[s] = x + (kScaled ? nr[s] + ur : fma(dt, ur, nr[s]));
        zi[s] = y + (kScaled ? ni[s] + ui : fma(dt, ui, ni[s]));
      }
    }
    if (frame < g.group) store_frame();  // the state after the last step
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int j = q * S + s;
      if (live && j < n) gb[j] = mk(zr[s], zi[s]);
    }
  }
}

template <typename T, int S, bool PRIO, bool FT>
const void* kernel_m(int m) {
  return m <= 3 ? (const void*)sparse_step_kernel<T, S, 3, PRIO, FT> : (const void*)sparse_step_kernel<T, S, 6, PRIO, FT>;
}

template <typename T, bool PRIO, bool FT>
const void* kernel_s(int s, int m) {
  return s == 2   ? kernel_m<T, 2, PRIO, FT>(m)
         : s == 4 ? kernel_m<T, 4, PRIO, FT>(m)
         : s == 6 ? kernel_m<T, 6, PRIO, FT>(m)
                  : kernel_m<T, 8, PRIO, FT>(m);
}

template <bool FT>
const void* kernel_ft(int precision, int s, int m, bool prio) {
  return precision == 64 ? kernel_s<double, false, FT>(s, m)
         : prio          ? kernel_s<float, true, FT>(s, m)
                         : kernel_s<float, false, FT>(s, m);
}

const void* kernel_for(int precision, int s, int m, bool prio, bool ft) {
  return ft ? kernel_ft<true>(precision, s, m, prio) : kernel_ft<false>(precision, s, m, prio);
}

size_t lds_bytes(int n, int precision, int s) {
  const int lp = (n + s - 1) / s, tpw = 64 / lp;
  return (precision == 64 ? sizeof(double) * f64::kTabSize : 0) +
         (size_t)kWaves * tpw * (s * lp + 1) * (precision == 64 ? 16 : 8);
}

}  // namespace

int sparse_entries(int most) { return most <= 3 ? 3 : most <= 6 ? 6 : 0; }

bool sparse_supported(int n, int hopping, int most) {
  return hopping == 1 && n >= 1 && n <= kSparseMaxSites && sparse_entries(most) > 0;
}

// Sites per lane and grid: the smallest estimated time of a step.  A SIMD with w
// waves takes w times a wave's issue time, but not less than one wave's chain;
// waves beyond the grid follow in rounds.  Measured per site pair: FP64 0.38 us
// of issue, a chain of 0.48 us; FP32 0.20 us, 0.08 + 0.23 us.  Few trajectories
// give two sites per lane (the shortest chain), many the S that leaves the
// fewest lanes and SIMDs without work.
hipError_t sparse_plan(int n, int precision, int most, bool ft, size_t n_traj, int cus, SparsePlan* plan) {
  double best = 0.0;
  plan->s = 0;
  for (int s : {2, 4, 6, 8}) {
    const int lp = (n + s - 1) / s;
    if (lp > 64) continue;
    const size_t per_block = (size_t)kWaves * (64 / lp);
    const size_t blocks = (n_traj + per_block - 1) / per_block;
    const bool prio = blocks > 2 * (size_t)cus;
    const void* f = kernel_for(precision, s, most, prio, ft);
    const size_t lds = lds_bytes(n, precision, s);
    if (lds > 65536) {
      hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    int per_cu = 0;  // workgroups of kWaves waves, one per SIMD
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, 64 * kWaves, lds);
    if (e != hipSuccess) return e;
    const double issue = (precision == 64 ? 0.38 : 0.20) * (s / 2);
    const double chain = precision == 64 ? 0.48 * (s / 2) : 0.08 + 0.23 * (s / 2);
    auto round = [&](size_t w) { return std::max(chain, issue * double(w)); };
    for (int w = 1; w <= std::max(1, per_cu); ++w) {
      const size_t grid = (size_t)w * cus;
      const size_t full = blocks / grid, rest = blocks - full * grid;
      const double cost = double(full) * round(w) + (rest ? round((rest + cus - 1) / cus) : 0.0);
      if (plan->s == 0 || cost < best || (cost == best && s == plan->s)) {  // ties: more waves per SIMD
        best = cost;
        plan->s = s;
        plan->prio = prio;
        plan->step = {(int)std::min(blocks, grid), 64 * kWaves, lds};
      }
    }
  }
  return hipSuccess;
}

hipError_t launch_sparse(const StepArgs& a, int precision, const SparsePlan& plan, hipStream_t s) {
  const void* f = kernel_for(precision, plan.s, a.ell_m, plan.prio, a.ft_n > 0);
  if (plan.step.lds > 65536) {
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)plan.step.lds);
    if (e != hipSuccess) return e;
  }
  void* args[] = {const_cast<StepArgs*>(&a)};
  return hipLaunchKernel(f, dim3(plan.step.grid), dim3(plan.step.block), args, plan.step.lds, s);
}

}  // namespace twmc
