// twmc_ahead.hip -- step kernel for small batches of small systems: periodic lattices of
// up to 256 sites, the hopping in its nearest-neighbour form (the exact real-space form
// of the reference's FFT product, TWMCBaseSolver.cpp:80-88, :235-242), and matrix
// hopping with few nonzeros per column (TWMCLiebSolver.cpp:259-267), up to 256 sites with
// six, 512 with three (above 256, FP64, 16 values spill).
//
// What bounds it: the latency of one step after the other; the chip is mostly idle.
// In the LDS kernel (twmc_generic.hip) and the sparse kernel (twmc_sparse.hip) a wave's
// step is the whole chain of ten Philox rounds, Box-Muller and update.  But the noise does not depend on the state, so here
// a workgroup of four waves (eight above 128 sites) owns a trajectory: one wave steps
// it, one to eight sites per lane, and the others write the next steps' noise into
// LDS, a chunk ahead, every lane a pair of some step.  The chain is then one LDS
// exchange and the update.  Every operation is that kernel's, so the bits are the same
// for either.  us per step, before -> now: 256 trajectories of 64 sites, FP64,
// 0.54 -> 0.17 (0.15 us is 360 clocks); 100 of 4x4 with a drawn drive, FP64, 0.74 ->
// 0.16; 256 of 5x13, FP32, 0.65 -> 0.21; Lieb chain of 72 sites, FP64, 256 trajectories
// 0.52 -> 0.19, 1000 0.58 -> 0.44.
#include <algorithm>

#include "twmc_cplx.h"
#include "twmc_f64math.h"
#include "twmc_internal.h"
#include "twmc_rng.h"

namespace twmc {

namespace {

// the FP64 Box-Muller's ln and sin / cos tables (twmc_f64math.h)
alignas(16) __device__ const double kF64TabDev[f64::kTabSize] = TWMC_F64_TABLES;

constexpr int waves_of(int spl) { return spl >= 4 ? 8 : 4; }
// noise of a chunk: steps x sites (rounded up to even).  512: the LDS then holds six
// workgroups per CU, with 1024 three (1000 trajectories of 72 sites, FP64: 0.46 ->
// 0.40 us per step; up to 768 the same)
constexpr int chunk_sites(int spl) { return spl == 8 ? 3072 : spl == 4 ? 2048 : 512; }
constexpr int kChunkSteps = 64;    // at most

template <typename T>
constexpr int kTab = sizeof(T) == 8 ? f64::kTabSize : 0;

template <typename T, int SPL>
struct Lds {
  double tab[kTab<T> + 2];
  cpx<T> st[64 * SPL + 1];  // the last one zero
  // lanes past the lattice read, and drop, up to 64 SPL entries past a step's row
  cpx<T> noise[2][chunk_sites(SPL) + 64 * SPL];
};

// what a lane wrote is seen by the wave's other lanes (LDS operations of a wave are
// in order; this keeps the compiler's)
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// SPL: sites per lane of the stepping wave.  M = 0: the periodic lattice, UNIF:
// StepArgs::site_uniform, XN: it has x neighbours (nx > 1).  M > 0: matrix hopping with
// up to M nonzeros per column.
template <typename T, int SPL, int M, bool UNIF, bool XN>
__global__ void __launch_bounds__(64 * waves_of(SPL)) ahead_step_kernel(StepArgs g) {
  constexpr int kWaves = waves_of(SPL);
  constexpr bool kF64 = sizeof(T) == 8;
  constexpr bool kOnePlus = kF64 && UNIF;  // (1 + c) z with 1 + dt Re rsl formed once
  extern __shared__ __align__(16) unsigned char smem[];
  Lds<T, SPL>& lds = *reinterpret_cast<Lds<T, SPL>*>(smem);
  if constexpr (kF64)
    for (int i = threadIdx.x; i < f64::kTabSize; i += 64 * kWaves) lds.tab[i] = kF64TabDev[i];
  __syncthreads();

  const int n = g.n, np = (n + 1) / 2, stride = 2 * np, b = blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint64_t traj = g.traj_ids[b];
  const int ksteps = min(kChunkSteps, chunk_sites(SPL) / stride);
  // item / np as umulhi (items below 2^16)
  const uint32_t magic = np > 1 ? (uint32_t)((0x100000000ull + (uint32_t)np - 1) / (uint32_t)np) : 0u;
  auto produce = [&](int buf, int s0, int first, int waves) {
    const int items = min(ksteps, g.n_steps - s0) * np;
    for (int q = 64 * first + lane; q < items; q += 64 * waves) {
      const int k = np > 1 ? (int)__umulhi((uint32_t)q, magic) : q, p = q - k * np;
      const u32x4 x = philox4x32_10(make_counter(traj, TAG_WIENER, uint32_t(g.step0 + (uint64_t)(s0 + k)), (uint32_t)p),
                                    g.key0, g.key1);
      T re[2], im[2];
      if constexpr (kF64) {
        const uint32_t wa[2] = {x.x, x.z}, wb[2] = {x.y, x.w};
        f64::box_muller<2>(wa, wb, re, im, f64::kSeries, lds.tab);
        if constexpr (M > 0) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            re[h] *= g.dt4;
            im[h] *= g.dt4;
          }
        }
      } else if constexpr (M > 0) {
        const float sig = float(g.dt4), nl = -1.3862943611198906f * sig * sig;
        float r[2], cs[2], sn[2];
        box_muller_f32_scaled(x.x, x.y, nl, r[0], cs[0], sn[0]);
        box_muller_f32_scaled(x.z, x.w, nl, r[1], cs[1], sn[1]);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          re[h] = r[h] * cs[h];
          im[h] = r[h] * sn[h];
        }
      } else {
        box_muller_f32(x.x, x.y, re[0], im[0]);
        box_muller_f32(x.z, x.w, re[1], im[1]);
      }
      cpx<T>* out = lds.noise[buf] + 2 * q;  // row k, sites 2p and 2p + 1
      out[0] = mk(re[0], im[0]);
      out[1] = mk(re[1], im[1]);
    }
  };

  // the stepping wave's sites lane + 64 j: state, constants scaled by dt (matrix hopping
  // in FP64: not scaled, as in the sparse kernel), neighbours
  constexpr int kNb = M > 0 ? M : XN ? 4 : 2;
  cpx<T> z[SPL], rd[SPL], ud[SPL], fd[SPL];
  T cf[SPL][M > 0 ? M : 1];
  int nb[SPL][kNb];
  const T dt = T(g.dt), dt4 = T(g.dt4), djv = T(-0.5 * g.kscale * g.dt), cdt = M > 0 && kF64 ? T(1) : dt;
  cpx<T>* const gb = reinterpret_cast<cpx<T>*>(g.beta) + (size_t)b * n;
  const size_t poff = g.param_stride ? (size_t)b * n : 0;
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const int i = lane + 64 * j, x = i / g.ny, y = i - x * g.ny;
    const bool in = wave == 0 && i < n;
    const size_t ip = UNIF ? 0 : poff + (in ? i : 0);
    const cpx<T> r = reinterpret_cast<const cpx<T>*>(g.rsl)[ip], u = reinterpret_cast<const cpx<T>*>(g.U)[ip],
                 f = reinterpret_cast<const cpx<T>*>(g.F)[ip];
    z[j] = in ? gb[i] : mk(T(0), T(0));
    ud[j] = mk(cdt * u.re, cdt * u.im);
    fd[j] = mk(-cdt * f.im, cdt * f.re);
    if constexpr (M > 0) {
      // c (rsl + i U (|b|^2 - 1)) = (rd.re - ud.im |b|^2) + i (rd.im + ud.re |b|^2), c = cdt
      rd[j] = mk(cdt * (r.re + u.im), cdt * (r.im - u.re));
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int row = in ? g.ell_row[i * M + m] : -1;
        cf[j][m] = row >= 0 ? reinterpret_cast<const T*>(g.ell_coef)[i * M + m] : T(0);
        nb[j][m] = row >= 0 ? row : 64 * SPL;
      }
    } else {
      rd[j] = mk(kOnePlus ? T(1) + dt * r.re : dt * r.re, dt * r.im);
      nb[j][0] = y + 1 == g.ny ? i + 1 - g.ny : i + 1;
      nb[j][1] = y == 0 ? i + g.ny - 1 : i - 1;
      if constexpr (XN) {
        nb[j][2] = i + g.ny >= n ? i + g.ny - n : i + g.ny;
        nb[j][3] = i < g.ny ? i - g.ny + n : i - g.ny;
      }
#pragma unroll
      for (int h = 0; h < kNb; ++h) nb[j][h] = in ? nb[j][h] : 0;
    }
  }
  if (M > 0 && threadIdx.x == 0) lds.st[64 * SPL] = mk(T(0), T(0));

  int due = 0, frame = 0;  // steps to the next stored frame, frames stored
  auto store_frame = [&] {
    cpx<T>* out = reinterpret_cast<cpx<T>*>(g.frames) + ((size_t)b * g.frames_stride + g.frame0 + frame) * n;
#pragma unroll
    for (int j = 0; j < SPL; ++j)
      if (lane + 64 * j < n) out[lane + 64 * j] = z[j];
    ++frame;
    due = g.group_steps;
  };

  produce(0, 0, wave, kWaves);
  __syncthreads();
  for (int s0 = 0, c = 0; s0 < g.n_steps; s0 += ksteps, c ^= 1) {
    if (wave == 0) {
      const int steps = min(ksteps, g.n_steps - s0);
      const cpx<T>* row = lds.noise[c] + lane;
      cpx<T> xi[SPL];
#pragma unroll
      for (int j = 0; j < SPL; ++j) xi[j] = row[64 * j];
      for (int k = 0; k < steps; ++k) {
        if (due-- == 0 && frame < g.group) {
          store_frame();
          --due;
        }
#pragma unroll
        for (int j = 0; j < SPL; ++j) lds.st[lane + 64 * j] = z[j];
        lds_order();
        cpx<T> a[SPL][kNb];
#pragma unroll
        for (int j = 0; j < SPL; ++j)
#pragma unroll
          for (int h = 0; h < kNb; ++h) a[j][h] = lds.st[nb[j][h]];
        lds_order();
        row += k + 1 < steps ? stride : 0;
        cpx<T> next[SPL];
#pragma unroll
        for (int j = 0; j < SPL; ++j) next[j] = row[64 * j];
#pragma unroll
        for (int j = 0; j < SPL; ++j) {
          const cpx<T> w = z[j];
          if constexpr (M > 0) {
            // c h = -i sum c C_ij beta_i; increment = noise + dt iF + dt h + drift
            T dr = fd[j].re, di = fd[j].im;
#pragma unroll
            for (int m = 0; m < M; ++m) {
              dr = fma(cf[j][m], a[j][m].im, dr);
              di = fma(-cf[j][m], a[j][m].re, di);
            }
            const T mq = fma(w.im, w.im, w.re * w.re);
            const T cr = fma(-ud[j].im, mq, rd[j].re), ci = fma(ud[j].re, mq, rd[j].im);
            const T ur = fma(-ci, w.im, fma(cr, w.re, dr)), ui = fma(ci, w.re, fma(cr, w.im, di));
            z[j] = mk(w.re + (kF64 ? fma(dt, ur, xi[j].re) : xi[j].re + ur),
                      w.im + (kF64 ? fma(dt, ui, xi[j].im) : xi[j].im + ui));
          } else {
            // y + 1 and y - 1 neighbours, then x + 1 and x - 1
            T sr = a[j][0].re + a[j][1].re, si = a[j][0].im + a[j][1].im;
            if constexpr (XN) {
              sr += a[j][2].re + a[j][3].re;
              si += a[j][2].im + a[j][3].im;
            }
            // increment dt (c z + h + i F) + dt4 xi as one FMA chain per component;
            // dt h = dt J (S_im, -S_re)
            const T q = fma(w.re, w.re, fma(w.im, w.im, T(-1)));
            const T ci = fma(ud[j].re, q, rd[j].im), cr = fma(-ud[j].im, q, rd[j].re);
            T dr = fma(dt4, xi[j].re, fd[j].re);
            dr = fma(djv, si, dr);
            T di = fma(dt4, xi[j].im, fd[j].im);
            di = fma(-djv, sr, di);
            if constexpr (kOnePlus) {
              dr = fma(-ci, w.im, dr);
              di = fma(ci, w.re, di);
              z[j] = mk(fma(cr, w.re, dr), fma(cr, w.im, di));
            } else {
              dr = fma(cr, w.re, dr);
              dr = fma(-ci, w.im, dr);
              di = fma(cr, w.im, di);
              di = fma(ci, w.re, di);
              z[j] = mk(w.re + dr, w.im + di);
            }
          }
          xi[j] = next[j];
        }
      }
    } else if (s0 + ksteps < g.n_steps) {
      produce(c ^ 1, s0 + ksteps, wave - 1, kWaves - 1);
    }
    __syncthreads();
  }
  if (wave == 0 && frame < g.group) store_frame();  // the state after the last step
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const int i = lane + 64 * j;
    if (wave == 0 && i < n) gb[i] = z[j];
  }
}

struct Launch {
  const void* f;
  int block;
  size_t lds;
};

template <typename T, int SPL>
Launch launch_s(int m, bool unif, bool xn) {
  const void* f = nullptr;
  if constexpr (SPL <= 4)
    f = m > 3 ? (const void*)ahead_step_kernel<T, SPL, 6, false, false>
        : m > 0 ? nullptr
        : unif ? (xn ? (const void*)ahead_step_kernel<T, SPL, 0, true, true> : (const void*)ahead_step_kernel<T, SPL, 0, true, false>)
               : (xn ? (const void*)ahead_step_kernel<T, SPL, 0, false, true> : (const void*)ahead_step_kernel<T, SPL, 0, false, false>);
  if (m == 3) f = (const void*)ahead_step_kernel<T, SPL, 3, false, false>;
  return {f, 64 * waves_of(SPL), sizeof(Lds<T, SPL>)};
}

template <typename T>
Launch launch_t(int n, int m, bool unif, bool xn) {
  return n <= 64    ? launch_s<T, 1>(m, unif, xn)
         : n <= 128 ? launch_s<T, 2>(m, unif, xn)
         : n <= 256 ? launch_s<T, 4>(m, unif, xn)
                    : launch_s<T, 8>(m, unif, xn);
}

Launch launch_of(int precision, int n, int m, bool unif, bool xn) {
  return precision == 64 ? launch_t<double>(n, m, unif, xn) : launch_t<float>(n, m, unif, xn);
}

}  // namespace

// The lines below are those of long launches.  A workgroup first fills its tables and a
// chunk of noise, one trajectory each, so where several share a CU a launch of few steps
// costs more than the LDS and sparse kernels' (us of a launch, those kernels / this one:
// FP64, 1x64, 2048 trajectories, 4 steps 9.7 / 12.4, 32 steps 23.4 / 22.8; FP32, 4096, 8
// steps 9.5 / 14.3; FP64, 16x16, 512, 4 steps 10.3 / 13.4, 256 9.8 / 10.4, 16 steps 16.0 /
// 13.9): half the batch below 64 steps, a quarter below 8.  Batches with frames gain by
// several in a launch whatever their steps (350 trajectories of 3x57, 4 frames of 5: 0.54
// ms, with the LDS kernel 0.66).
namespace {
size_t batch_limit(int per_cu, uint64_t n_steps, int cus) {
  return (size_t)per_cu * cus / (n_steps < 8 ? 4 : n_steps < 64 ? 2 : 1);
}
}  // namespace

// A step costs the same for any batch until the CUs hold several workgroups; from
// then on the LDS and nn kernels, whose waves are full, overtake it.  Measured, us per
// step, those kernels against this one:
//   FP64, 1x64   256 trajectories 0.54 / 0.17, 1000 0.58 / 0.36, 2000 0.63 / 0.62, 4000 0.96 / 1.14
//   FP64, 4x4, drawn F   100 trajectories 0.74 / 0.16, 2000 0.73 / 0.50, 4000 0.75 / 0.91
//   FP64, 1x128  256 trajectories 0.55 / 0.23, 1000 0.63 / 0.60, 2000 0.96 / 1.10
//   FP32, 1x64   256 trajectories 0.34 / 0.13, 2000 0.39 / 0.30, 4000 0.51 / 0.50, 8000 0.85 / 0.90
//   FP32, 1x128, drawn F   256 trajectories 0.47 / 0.19, 4000 1.00 / 0.84
//   FP64, 16x16  256 trajectories 0.67 / 0.42, 512 1.00 / 0.81, 1000 1.13 / 1.58
//   FP32, 9x21   256 trajectories 0.50 / 0.36, 512 0.57 / 0.43, 2000 0.96 / 1.04
bool ahead_pays(int nx, int ny, int precision, size_t n_traj, uint64_t n_steps, int cus) {
  const int n = nx * ny;
  const int per_cu = n > 128 ? 2 : precision == 32 ? 16 : n > 64 ? 4 : 8;
  return ny > 1 && n <= 256 && n_traj <= batch_limit(per_cu, n_steps, cus);
}

// The sparse kernel against this one, us per step, Lieb chains with drawn energies:
//   FP64, 72 sites   256 trajectories 0.52 / 0.19, 1000 0.58 / 0.44, 2000 0.92 / 0.79
//   FP64, 144 sites  256 trajectories 0.98 / 0.33, 512 1.01 / 0.65, 1000 1.10 / 1.23
//   FP64, 384 sites  256 trajectories 1.49 / 0.70, 512 1.55 / 1.39, 1000 1.70 / 2.76
//   FP32, 72 sites   256 trajectories 0.33 / 0.18, 2000 0.47 / 0.35
//   FP32, 144 sites  256 trajectories 0.54 / 0.31, 512 0.55 / 0.37, 1000 0.58 / 0.69
//   FP32, 384 sites  256 trajectories 0.79 / 0.52, 512 0.80 / 1.00
bool ahead_pays_sparse(int n, int most, int precision, size_t n_traj, uint64_t n_steps, int cus) {
  const int per_cu = n <= 128 ? 8 : n <= 256 || precision == 64 ? 2 : 1;
  return (n <= 256 || (n <= 512 && most <= 3)) && n_traj <= batch_limit(per_cu, n_steps, cus);
}

LaunchShape ahead_shape(int n, int ell_m, int precision, size_t n_traj) {
  const Launch l = launch_of(precision, n, ell_m, false, false);  // the same for all forms
  return {(int)n_traj, l.block, l.lds};
}

hipError_t launch_ahead(const StepArgs& a, int precision, hipStream_t s) {
  const Launch l = launch_of(precision, a.n, a.hopping == 1 ? a.ell_m : 0, a.site_uniform != 0, a.nx > 1);
  if (l.lds > 65536) {
    hipError_t e = hipFuncSetAttribute(l.f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l.lds);
    if (e != hipSuccess) return e;
  }
  void* args[] = {const_cast<StepArgs*>(&a)};
  return hipLaunchKernel(l.f, dim3(a.n_traj), dim3(l.block), args, l.lds, s);
}

}  // namespace twmc
