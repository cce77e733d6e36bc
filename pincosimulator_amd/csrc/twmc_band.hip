// twmc_band.hip -- register-resident TWMC step kernel for matrix hopping with
// a banded coupling matrix (chains, ladders, the Lieb chain) in FP32.
//
// The reference's Lieb solver applies h_j = -i sum_i beta_i C_ij with a sparse
// product (TWMCLiebSolver.cpp:259-267).  When every nonzero C_ij has
// |i - j| <= W (cyclically, when N = 64 S), that product is a (2W+1)-point
// stencil along the site index, and a dense or LDS-staged product only moves
// zeros.  One wavefront owns one trajectory: lane l holds sites l S .. l S + S - 1
// in registers (S even; N padded to 64 S, the padding sites have zero
// coefficients, stay finite and are never stored), together with the coefficients
// dt C_(j+d) j of its sites and its dt-scaled site parameters.  The W sites on
// either side of a lane's block come from lanes l - 1 and l + 1 by whole-wave
// DPP rotations.  Per step: the hopping sums of all owned sites from the old
// state, then per site pair one Philox4x32-10 call with Box-Muller and the
// update, the same FMA chain as the other FP32 kernels.
#include "twmc_cplx.h"
#include "twmc_internal.h"
#include "twmc_rng.h"

namespace twmc {

namespace {

// lane l reads lane l - 1 (DPP wave_ror:1) / lane l + 1 (wave_rol:1), wrapping at 64
__device__ __forceinline__ float from_prev_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x13c, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_next_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x134, 0xf, 0xf, true));
}

// The W sites at either end of every lane's block, in the wave's LDS.
template <int W>
struct alignas(W == 2 ? 16 : 8) Edge {
  cpx<float> v[W];
};

// order of the wave's own LDS accesses (the hardware runs them in order)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// the Lieb chain's bonds as offsets d of the coupled site j + d, by the site
// index mod 3 (A_i = 3i, B_i = 3i + 1, C_i = 3i + 2; TWMCLiebSolver.cpp:52-85):
// A-B (+1); B-A (-1), B-C (+1), B-C of the previous cell (-2); C-B (-1),
// C-B of the next cell (+2)
__host__ __device__ constexpr bool lieb_bond(int r, int d) {
  return r == 0 ? d == 1 : r == 1 ? (d == -1 || d == 1 || d == -2) : (d == -1 || d == 2);
}

// LIEB (S = 6, W = 2): each lane's six sites are two whole cells, so the
// offsets without a bond are known per register and their multiplications
// by zero are left out (6 of the 10 complex products per cell remain)
// UNI: Re rsl, F and a real U are the same at every site, so of the site tables
// only Im rsl (the on-site energies) takes registers, and 64 of them hold the
// kernel at eight waves per SIMD.
// PAD (UNI and DENSE): n < 64 S.  Tables per site are zero on the padding, but a uniform
// one drives it, without the energies that may keep the real sites off resonance: it can
// overflow, and 0 times infinity reach the first and last sites.  Each step sets it back
// to zero (8192 trajectories, us per step, not reset / reset / parameters per site in the
// form before: 72 sites 1.38 / 1.42 / 1.53, 210 2.36 / 2.45 / 3.18, 330 3.12 / 3.30 / 3.74,
// 495 4.86 / 5.05 / 5.54).
// DENSE: more than two waves per SIMD.  Bound by VALU issue: 41 instructions per
// site-step of the 384-site Lieb chain, 37 beside the transcendental ones, which
// have a unit of their own.  Free-running waves bunch up before that unit and
// leave the VALU idle; raising a wave's priority while it forms its Box-Muller
// samples keeps the unit fed (384 sites x 8192 trajectories, us per step: 3.55
// without, 3.20 with; two sites per lane, one pair per step, do not bunch and
// take no priority: 126 sites x 16384 2.63 without, 2.65 with).  The lanes' edge
// sites go through LDS, two writes and two reads instead of 4 W DPP moves (x
// 16384: 6.20 -> 6.13, 126 sites 2.77 -> 2.63).  Otherwise, bound by the latency
// of a step: DPP and no priority (384 sites x 1000: 0.57 against 0.68 us).
// Before, 99 registers and the latency form for all: 384 sites x 8192 3.69, x
// 16384 7.16 us per step (8.8e11 -> 1.03e12 site-steps/s).
// waves per SIMD that the uniform form's registers allow with at most three spilled (six
// sites per lane and DENSE: two in the Lieb form and W = 1, three in W = 3)
constexpr int uni_waves(int s, int w, bool lieb) {
  return s == 2 || lieb ? 8 : s == 4 ? (w <= 2 ? 7 : 6) : s == 6 ? (w == 1 ? 7 : 5) : w == 1 ? 5 : 4;
}
template <int S, int W, bool FT, bool LIEB, bool UNI, bool DENSE, bool PAD>
__global__ void __launch_bounds__(64, UNI ? uni_waves(S, W, LIEB) : 1) band_step_kernel(StepArgs g) {
  static_assert(!LIEB || (S == 6 && W == 2), "the Lieb pattern needs two cells per lane");
  static_assert(!UNI || !FT, "F(t) is per site");
  static_assert(!DENSE || !FT, "F(t) runs the latency form");
  static_assert(!PAD || (UNI && DENSE), "parameters per site are zero on the padding");
  constexpr bool LDSX = DENSE, PRIO = DENSE && S >= 4;
  constexpr int D = 2 * W + 1;
  constexpr int SP = UNI ? 1 : S;  // entries of a uniform table
  __shared__ Edge<W> first[64], last[64];
  const int lane = threadIdx.x;
  const int n = g.n;
  const int base = lane * S;
  const float dt = float(g.dt), sig = float(g.dt4);
  const float nl = -1.3862943611198906f * sig * sig;  // -2 ln2 sigma^2 (Box-Muller)

  // this lane's coefficients and site tables; the site parameters are shared
  // by all trajectories (the kernel is chosen only then):
  //   dt (rsl + i U (|b|^2 - 1)) = (A0 - Ui |b|^2) + i (B0 + Ur |b|^2), dt i F = (fr, fi)
  float cf[S][D], A0[SP], B0[S], Ur[SP], Ui[SP], fr[SP], fi[SP];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int j = base + s;
#pragma unroll
    for (int d = 0; d < D; ++d) cf[s][d] = g.band_coef[(size_t)j * D + d];
    const bool live = j < n;
    const cpx<float> r = live ? reinterpret_cast<const cpx<float>*>(g.rsl)[j] : mk(0.f, 0.f);
    const cpx<float> u = live ? reinterpret_cast<const cpx<float>*>(g.U)[j] : mk(0.f, 0.f);
    const cpx<float> f = live ? reinterpret_cast<const cpx<float>*>(g.F)[j] : mk(0.f, 0.f);
    B0[s] = dt * (r.im - u.re);
    if constexpr (!UNI) {
      A0[s] = dt * (r.re + u.im);
      Ur[s] = dt * u.re;
      Ui[s] = dt * u.im;
      fr[s] = -dt * f.im;
      fi[s] = dt * f.re;
    }
  }
  if constexpr (UNI) {
    const cpx<float> r = reinterpret_cast<const cpx<float>*>(g.rsl)[0], u = reinterpret_cast<const cpx<float>*>(g.U)[0],
                     f = reinterpret_cast<const cpx<float>*>(g.F)[0];
    A0[0] = dt * (r.re + u.im);
    Ur[0] = dt * u.re;
    Ui[0] = 0.f;
    fr[0] = -dt * f.im;
    fi[0] = dt * f.re;
  }

  for (int b = blockIdx.x; b < g.n_traj; b += gridDim.x) {
    const uint64_t traj = g.traj_ids[b];
    cpx<float>* gb = reinterpret_cast<cpx<float>*>(g.beta) + (size_t)b * n;
    float br[S], bi[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int j = base + s;
      const cpx<float> v = j < n ? gb[j] : mk(0.f, 0.f);
      br[s] = v.re;
      bi[s] = v.im;
    }

    if (g.capture) {
      // per-trajectory site means and the optional frame dump; the per-site
      // ensemble sums come from the site-major kernel launched before this one
      double m2 = 0.0, m4 = 0.0;
      cpx<float>* out =
          g.dump ? reinterpret_cast<cpx<float>*>(g.traj_out) + ((size_t)b * g.n_frames + g.frame) * n : nullptr;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int j = base + s;
        if (j < n) {
          const double nn = double(br[s]) * double(br[s]) + double(bi[s]) * double(bi[s]);
          m2 += nn;
          m4 += nn * nn;
          if (out) out[j] = mk(br[s], bi[s]);
        }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        m2 += __shfl_xor(m2, o, 64);
        m4 += __shfl_xor(m4, o, 64);
      }
      if (lane == 0) {
        g.traj_m2[(size_t)b * g.n_frames + g.frame] = m2 / double(n);
        g.traj_m4[(size_t)b * g.n_frames + g.frame] = m4 / double(n);
      }
    }

    int ft_id = 0;
    for (int st = 0; st < g.n_steps; ++st) {
      const uint32_t step = uint32_t(g.step0 + (uint64_t)st);
      // site-pair base of this lane, opaque so the Philox rounds stay in the loop
      uint32_t pbase = (uint32_t)(base / 2);
      asm volatile("" : "+v"(pbase));
      float dr[S], di[S];
      if constexpr (FT) {
        // F(t) before this step (TWMCLiebSolver.cpp:252-256), as dt i F
        const float fdt = float(drive_interval(g.ft_times, g.ft_n, g.t0 + double(st) * g.dt, ft_id));
        const cpx<float>* fv = reinterpret_cast<const cpx<float>*>(g.ft_vals) + (size_t)ft_id * n;
        const cpx<float>* fs = reinterpret_cast<const cpx<float>*>(g.ft_slopes) + (size_t)ft_id * n;
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const int j = base + s;
          const cpx<float> v = j < n ? fv[j] : mk(0.f, 0.f), sl = j < n ? fs[j] : mk(0.f, 0.f);
          dr[s] = -dt * fmaf(fdt, sl.im, v.im);
          di[s] = dt * fmaf(fdt, sl.re, v.re);
        }
      } else {
#pragma unroll
        for (int s = 0; s < S; ++s) {
          dr[s] = fr[UNI ? 0 : s];
          di[s] = fi[UNI ? 0 : s];
        }
      }
      // old values of the W sites before and after this lane's block
      Edge<W> el, er;
      if constexpr (LDSX) {
        Edge<W> e0, e1;
#pragma unroll
        for (int k = 0; k < W; ++k) {
          e0.v[k] = mk(br[k], bi[k]);
          e1.v[k] = mk(br[S - W + k], bi[S - W + k]);
        }
        first[lane] = e0;
        last[lane] = e1;
        wave_sync();
        el = last[(lane - 1) & 63];
        er = first[(lane + 1) & 63];
        wave_sync();
      } else {
#pragma unroll
        for (int k = 0; k < W; ++k) {
          el.v[k] = mk(from_prev_lane(br[S - W + k]), from_prev_lane(bi[S - W + k]));
          er.v[k] = mk(from_next_lane(br[k]), from_next_lane(bi[k]));
        }
      }
      // dt h_j = -i sum_d dt C_(j+d) j beta_(j+d): (sum c Im beta, -sum c Re beta)
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int d = -W; d <= W; ++d) {
          if (LIEB && !lieb_bond(s % 3, d)) continue;
          const int t = s + d;
          const float vre = t < 0 ? el.v[(t + 2 * W) % W].re : t >= S ? er.v[(t - S) % W].re : br[t < 0 || t >= S ? 0 : t];
          const float vim = t < 0 ? el.v[(t + 2 * W) % W].im : t >= S ? er.v[(t - S) % W].im : bi[t < 0 || t >= S ? 0 : t];
          dr[s] = fmaf(cf[s][d + W], vim, dr[s]);
          di[s] = fmaf(-cf[s][d + W], vre, di[s]);
        }
      // noise and update
#pragma unroll
      for (int p = 0; p < S / 2; ++p) {
        const u32x4 ctr = make_counter(traj, TAG_WIENER, step, pbase + (uint32_t)p);
        const u32x4 w = DENSE || UNI ? philox4x32_10_wave(ctr, g.key0, g.key1) : philox4x32_10(ctr, g.key0, g.key1);
        float rn[2], cs[2], sn[2];
        if constexpr (PRIO) __builtin_amdgcn_s_setprio(2);
        box_muller_f32_scaled(w.x, w.y, nl, rn[0], cs[0], sn[0]);
        box_muller_f32_scaled(w.z, w.w, nl, rn[1], cs[1], sn[1]);
        if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int s = 2 * p + h;
          const float x = br[s], y = bi[s];
          const float mq = fmaf(y, y, x * x);
          const int t = UNI ? 0 : s;
          const float cr = UNI ? A0[0] : fmaf(-Ui[t], mq, A0[t]), ci = fmaf(Ur[t], mq, B0[s]);
          // increment = noise + dt iF + dt h + drift, all small, added to beta once
          float ur = fmaf(rn[h], cs[h], dr[s]);
          ur = fmaf(cr, x, ur);
          ur = fmaf(-ci, y, ur);
          float ui = fmaf(rn[h], sn[h], di[s]);
          ui = fmaf(cr, y, ui);
          ui = fmaf(ci, x, ui);
          const bool live = !PAD || base + s < n;
          br[s] = live ? x + ur : 0.f;
          bi[s] = live ? y + ui : 0.f;
        }
      }
    }

#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int j = base + s;
      if (j < n) gb[j] = mk(br[s], bi[s]);
    }
  }
}

// Bound by latency the uniform form gains where it saves most registers, four and more
// sites per lane without padding (512 sites, W = 2, x 1000: 0.91 -> 0.88 us per step, the
// Philox rounds with the trajectory's words in scalar registers; with parameters per site
// those lengthen the chain, 384 x 64 0.60 -> 0.63); for
// the Lieb chain and with padding to reset it loses (384 x 1500 0.98 / 1.05, 210 x 64
// 0.42 / 0.45, 495 x 1000 0.90 / 0.94): those take the parameters per site.
template <int S, int W, bool LIEB>
const void* kernel_swl(bool ft, bool uni, bool dense, bool pad) {
  if (ft) return (const void*)band_step_kernel<S, W, true, LIEB, false, false, false>;
  if (uni && dense)
    return pad ? (const void*)band_step_kernel<S, W, false, LIEB, true, true, true>
               : (const void*)band_step_kernel<S, W, false, LIEB, true, true, false>;
  if constexpr (S >= 4 && !LIEB)
    if (uni && !pad) return (const void*)band_step_kernel<S, W, false, LIEB, true, false, false>;
  return dense ? (const void*)band_step_kernel<S, W, false, LIEB, false, true, false>
               : (const void*)band_step_kernel<S, W, false, LIEB, false, false, false>;
}

template <int S>
const void* kernel_s(int w, bool lieb, bool ft, bool uni, bool dense, bool pad) {
  if constexpr (S == 6)
    if (lieb && w == 2) return kernel_swl<6, 2, true>(ft, uni, dense, pad);
  switch (w) {
    case 1: return kernel_swl<S, 1, false>(ft, uni, dense, pad);
    case 2: return kernel_swl<S, 2, false>(ft, uni, dense, pad);
    default: return kernel_swl<S, 3, false>(ft, uni, dense, pad);
  }
}

const void* kernel_for(int n, int w, bool lieb, bool ft, bool uni, bool dense) {
  const bool pad = 64 * band_sites_per_lane(n) != n;
  switch (band_sites_per_lane(n)) {
    case 2: return kernel_s<2>(w, lieb, ft, uni, dense, pad);
    case 4: return kernel_s<4>(w, lieb, ft, uni, dense, pad);
    case 6: return kernel_s<6>(w, lieb, ft, uni, dense, pad);
    default: return kernel_s<8>(w, lieb, ft, uni, dense, pad);
  }
}

}  // namespace

int band_sites_per_lane(int n) { return 2 * ((n + 127) / 128); }

int band_width(const double* coupling, int n) {
  if (n < 1 || n > kBandMaxSites) return -1;
  const int S = band_sites_per_lane(n);
  const bool cyclic = 64 * S == n;
  int w = 0;
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) {
      if (coupling[(size_t)i * n + j] == 0.0) continue;
      int d = i > j ? i - j : j - i;
      if (cyclic) d = d < n - d ? d : n - d;
      w = d > w ? d : w;
    }
  return w;
}

bool band_supported(int n, int hopping, int precision, int param_stride, int width) {
  return hopping == 1 && precision == 32 && param_stride == 0 && n >= 1 && n <= kBandMaxSites && width >= 0 &&
         width <= kBandMaxWidth && width <= band_sites_per_lane(n);
}

void band_coefficients(const double* coupling, int n, int w, double dt, float* out) {
  const int S = band_sites_per_lane(n), D = 2 * w + 1;
  const bool cyclic = 64 * S == n;
  for (int j = 0; j < 64 * S; ++j)
    for (int d = -w; d <= w; ++d) {
      int i = j + d;
      double c = 0.0;
      if (j < n) {
        if (cyclic) i = (i % n + n) % n;
        if (i >= 0 && i < n) c = coupling[(size_t)i * n + j];
      }
      out[(size_t)j * D + d + w] = float(dt * c);
    }
}

bool band_lieb_pattern(const float* coef, int n, int w) {
  const int S = band_sites_per_lane(n);
  if (S != 6 || w != 2) return false;
  for (int j = 0; j < 64 * S; ++j)
    for (int d = -w; d <= w; ++d)
      if (!lieb_bond(j % 3, d) && coef[(size_t)j * (2 * w + 1) + d + w] != 0.f) return false;
  return true;
}

hipError_t launch_band(const StepArgs& a, int grid, hipStream_t s) {
  const void* f = kernel_for(a.n, a.band_w, a.band_lieb != 0, a.ft_n > 0, a.band_uni != 0, a.band_dense != 0);
  void* args[] = {const_cast<StepArgs*>(&a)};
  return hipLaunchKernel(f, dim3(grid), dim3(64), args, 0, s);
}

// the batch gives every SIMD more than two waves
bool band_dense(size_t n_traj, int cus) { return n_traj > 2 * 4 * (size_t)cus; }

// occupancy of the instantiation launch_band runs (for F(t) that of a static
// drive, the larger of the two)
hipError_t band_occupancy(int n, int w, int lieb, int uni, int dense, int* blocks_per_cu) {
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(
      blocks_per_cu, kernel_for(n, w, lieb != 0, false, uni != 0, dense != 0), 64, 0);
}

}  // namespace twmc
