// twmc_nn.hip -- step kernel for periodic lattices of 65 to 4096 sites, the hopping
// in its nearest-neighbour form (the exact real-space form of the reference's FFT
// product, TWMCBaseSolver.cpp:80-88, :235-242): FP64, and the FP32 lattices that the
// stacked kernel does not take (rows of odd length, an energy or a drive that varies
// from site to site or is drawn per trajectory).  One workgroup owns one trajectory:
// a pair per thread (two for 2049 to 4096 sites), the state in registers, the
// neighbours from one LDS copy of it; in launches of more than a few steps
// (queue_pays) trajectories come from a work queue.
//
// What bounds it: VALU issue, at eight waves per SIMD.
//  * FP64, uniform: the LDS kernel (twmc_generic.hip) keeps the Box-Muller
//    coefficients, both sites' intermediates and six neighbours in 128 registers,
//    four waves per SIMD; here 64 registers hold eight: the coefficients lie in scalar
//    registers, the sites' samples are formed one after the other, the neighbours read
//    at their use.  Every operation and its order are that kernel's, so are the bits.
//    us per step before -> now: 4096 trajectories of 32x32 14.76 -> 13.1, of 36x50
//    30.1 -> 24.7, of 48x48 32.6 -> 29.0, of 64x64 51.5 -> 48.0; 256 trajectories of
//    36x50 2.50 -> 1.99.  Left: the table rows are read at random, 16 bytes a lane, four
//    per pair, and conflict about threefold in the LDS banks (up to 2048 sites a copy of
//    the kernel reading one row was 11% faster).
//  * Odd rows: the LDS kernel forms each site's neighbour places, a division among
//    them, in every step; here they are formed once and held (uniform, FP64, above 2048
//    sites, eleven values spill).  8192 trajectories, FP32
//    40x41 35.3 -> 19.6, 63x63 73.9 -> 42.7; FP64 40x41 75.0 -> 50.3, 63x63 136 -> 103.
//  * A varying parameter: the LDS kernel reads rsl, U and F of every site from memory
//    in every step (64x64, FP32: 98 KB a step and trajectory, 7.4 TB/s); here the one
//    that varies is scaled once and lies in LDS.  8192 trajectories, drawn F, FP32
//    16x16 4.29 -> 2.99, 36x50 41.6 -> 22.1, 64x64 109 -> 43; 64 trajectories of 64x64
//    3.33 -> 1.64; FP64 32x32 37.2 -> 27.0, 64x64 215 -> 106.
#include <algorithm>

#include "twmc_cplx.h"
#include "twmc_f64math.h"
#include "twmc_internal.h"
#include "twmc_rng.h"

namespace twmc {

namespace {

// the FP64 Box-Muller's ln and sin / cos tables (twmc_f64math.h)
alignas(16) __device__ const double kF64TabDev[f64::kTabSize] = TWMC_F64_TABLES;

template <typename T>
constexpr int kTabBytes = sizeof(T) == 8 ? f64::kTabSize * (int)sizeof(double) : 0;

// eight waves per SIMD, except where the LDS holds one workgroup of 16 waves per CU:
// FP64, 2049 to 4096 sites with a parameter beside the state
constexpr int waves_per_simd(int es, int ppt, int v) { return es == 8 && ppt == 2 && v != kVaryNone ? 4 : 8; }

__global__ void queue_reset_kernel(unsigned int* queue) {
  if (threadIdx.x == 0) *queue = 0u;
}

__device__ __forceinline__ float scalar(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double scalar(double v) {
  const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v)), hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
  return __hiloint2double(hi, lo);
}
template <typename T>
__device__ __forceinline__ cpx<T> scalar(cpx<T> z) {
  return mk(scalar(z.re), scalar(z.im));
}

// V: what varies from site to site (and from trajectory to trajectory, if drawn):
// nothing, rsl, or F, whose values scaled by dt are then in LDS beside the state.
// ODD: the row length is odd, so a pair may lie across two rows and each site has
// its own four neighbours; else the pair's sites are each other's neighbours and
// share the rest of their places.  XN: the lattice has x neighbours (nx > 1).
// UI0 (FP64): Im U = 0, so the factor of z in the new value is a constant.
template <typename T, int BLOCK, int PPT, int V, bool ODD, bool XN, bool UI0>
__global__ void __launch_bounds__(BLOCK, waves_per_simd(sizeof(T), PPT, V)) nn_step_kernel(StepArgs g) {
  constexpr bool kF64 = sizeof(T) == 8;
  // FP64, uniform: the LDS kernel's form, z + c z = (1 + c) z with 1 + dt Re rsl
  // formed once.  Its rounding (2^-53, 1e-13 of dt Re rsl) is no larger than that
  // kernel's, but would be where that kernel adds c z to z, with varying parameters
  constexpr bool kOnePlus = kF64 && V == kVaryNone;
  constexpr int kPairs = BLOCK * PPT;
  extern __shared__ __align__(16) unsigned char smem[];
  double* const ltab = reinterpret_cast<double*>(smem);
  int* const s_next = reinterpret_cast<int*>(smem + kTabBytes<T>);
  cpx<T>* const st = reinterpret_cast<cpx<T>*>(smem + kTabBytes<T> + 16);  // [even, odd][pair]
  cpx<T>* const par = st + 2 * kPairs;                                     // V: the same order
  f64::Series bmk = f64::kSeries;
  if constexpr (kF64) {
    for (int i = threadIdx.x; i < f64::kTabSize; i += BLOCK) ltab[i] = kF64TabDev[i];
    f64::pin_scalar(bmk);
  }

  const int n = g.n, npairs = (n + 1) / 2;
  const int wave_p = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63);
  // the neighbours' places in st: even rows [left of 2p, right of 2p + 1, up, down],
  // the last two in either half; odd rows [left, right, up, down] of each site
  int nb[PPT][ODD ? 8 : 4];
#pragma unroll
  for (int j = 0; j < PPT; ++j) {
    const int p = threadIdx.x + BLOCK * j;
    if constexpr (ODD) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = 2 * p + h, x = i / g.ny, y = i - x * g.ny;
        const int site[4] = {y == 0 ? i + g.ny - 1 : i - 1, y + 1 == g.ny ? i + 1 - g.ny : i + 1,
                             i + g.ny >= n ? i + g.ny - n : i + g.ny, i < g.ny ? i - g.ny + n : i - g.ny};
#pragma unroll
        for (int k = 0; k < 4; ++k)  // a site past the lattice is computed along and not stored
          nb[j][4 * h + k] = i < n ? kPairs * (site[k] & 1) + (site[k] >> 1) : 0;
      }
    } else {
      const int yh = g.ny / 2, row = p / yh, q = p - row * yh;
      nb[j][0] = kPairs + (q == 0 ? p + yh - 1 : p - 1);
      nb[j][1] = q + 1 == yh ? p + 1 - yh : p + 1;
      nb[j][2] = p + yh >= npairs ? p + yh - npairs : p + yh;
      nb[j][3] = p < yh ? p - yh + npairs : p - yh;
      if (p >= npairs) nb[j][0] = nb[j][1] = nb[j][2] = nb[j][3] = 0;
    }
  }
  // dt rsl (or 1 + dt Re rsl, kOnePlus), dt U, dt i F, dt J
  const T dt = T(g.dt), dt4 = T(g.dt4);
  const cpx<T>* const r_all = reinterpret_cast<const cpx<T>*>(g.rsl);
  const cpx<T>* const f_all = reinterpret_cast<const cpx<T>*>(g.F);
  const cpx<T> u0 = reinterpret_cast<const cpx<T>*>(g.U)[0];
  const cpx<T> ud = scalar(mk(dt * u0.re, dt * u0.im));
  auto drift = [dt](cpx<T> r) { return mk(kOnePlus ? T(1) + dt * r.re : dt * r.re, dt * r.im); };
  auto drive = [dt](cpx<T> f) { return mk(-dt * f.im, dt * f.re); };
  const cpx<T> r0 = drift(r_all[0]), f0 = drive(f_all[0]);  // in vector registers: an FMA reads one scalar
  const T djv = scalar(T(-0.5 * g.kscale * g.dt));

  for (int b = blockIdx.x; b < g.n_traj;) {
    const uint64_t traj = g.traj_ids[b];
    cpx<T>* gb = reinterpret_cast<cpx<T>*>(g.beta) + (size_t)b * n;
    const size_t poff = g.param_stride ? (size_t)b * n : 0;
    cpx<T> beta[2 * PPT];
#pragma unroll
    for (int j = 0; j < PPT; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int p = threadIdx.x + BLOCK * j, i = 2 * p + h;
        beta[2 * j + h] = mk(T(0), T(0));
        if (i < n) {
          beta[2 * j + h] = gb[i];
          if constexpr (V == kVaryRsl) par[kPairs * h + p] = drift(r_all[poff + i]);  // read by this thread only
          if constexpr (V == kVaryF) par[kPairs * h + p] = drive(f_all[poff + i]);
        }
      }
    for (int s = 0; s < g.n_steps; ++s) {
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        const int p = threadIdx.x + BLOCK * j;
        if (p < npairs) {
          st[p] = beta[2 * j];
          st[kPairs + p] = beta[2 * j + 1];
        }
      }
      __syncthreads();
      const uint32_t step = uint32_t(g.step0 + (uint64_t)s);
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        if (wave_p + BLOCK * j < npairs) {
          uint32_t pair = threadIdx.x + BLOCK * j;
          asm volatile("" : "+v"(pair));  // keeps the Philox rounds inside the loop
          const u32x4 x = philox4x32_10_wave(make_counter(traj, TAG_WIENER, step, pair), g.key0, g.key1);
          const cpx<T> z0 = beta[2 * j], z1 = beta[2 * j + 1];
          cpx<T> nz[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            T xr[1], xi[1];
            if constexpr (kF64) {
              const uint32_t wa[1] = {h ? x.z : x.x}, wb[1] = {h ? x.w : x.y};
              f64::box_muller<1, true>(wa, wb, xr, xi, bmk, ltab);
            } else {
              box_muller_f32(h ? x.z : x.x, h ? x.w : x.y, xr[0], xi[0]);
            }
            const cpx<T> z = h ? z1 : z0;
            // y + 1 and y - 1 neighbours, then x + 1 and x - 1
            cpx<T> a, c, d, e;
            if constexpr (ODD) {
              a = st[nb[j][4 * h + 1]], c = st[nb[j][4 * h]];
              if constexpr (XN) d = st[nb[j][4 * h + 2]], e = st[nb[j][4 * h + 3]];
            } else {
              a = h ? st[nb[j][1]] : z1, c = h ? z0 : st[nb[j][0]];
              if constexpr (XN) d = st[kPairs * h + nb[j][2]], e = st[kPairs * h + nb[j][3]];
            }
            T sr = a.re + c.re, si = a.im + c.im;
            if constexpr (XN) {
              sr += d.re + e.re;
              si += d.im + e.im;
            }
            const cpx<T> rd = V == kVaryRsl ? par[kPairs * h + threadIdx.x + BLOCK * j] : r0;
            const cpx<T> fd = V == kVaryF ? par[kPairs * h + threadIdx.x + BLOCK * j] : f0;
            // increment dt (c z + h + i F) + dt4 xi as one FMA chain per component;
            // dt h = dt J (S_im, -S_re)
            const T q = fma(z.re, z.re, fma(z.im, z.im, T(-1)));
            const T ci = fma(ud.re, q, rd.im), cr = UI0 ? rd.re : fma(-ud.im, q, rd.re);
            T dr = fma(dt4, xr[0], fd.re);
            dr = fma(djv, si, dr);
            T di = fma(dt4, xi[0], fd.im);
            di = fma(-djv, sr, di);
            if constexpr (kOnePlus) {  // (1 + c) z last
              dr = fma(-ci, z.im, dr);
              di = fma(ci, z.re, di);
              nz[h] = mk(fma(cr, z.re, dr), fma(cr, z.im, di));
            } else {
              dr = fma(cr, z.re, dr);
              dr = fma(-ci, z.im, dr);
              di = fma(cr, z.im, di);
              di = fma(ci, z.re, di);
              nz[h] = mk(z.re + dr, z.im + di);
            }
          }
          beta[2 * j] = nz[0];
          beta[2 * j + 1] = nz[1];
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < PPT; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = 2 * (threadIdx.x + BLOCK * j) + h;
        if (i < n) gb[i] = beta[2 * j + h];
      }
    // the next trajectory: of this workgroup's share, or from the queue (the barriers of
    // the steps separate this word's uses)
    if (!g.queue) {
      b += gridDim.x;
      continue;
    }
    if (threadIdx.x == 0) *s_next = (int)(gridDim.x + atomicAdd(g.queue, 1u));
    __syncthreads();
    b = __builtin_amdgcn_readfirstlane(*s_next);
    __syncthreads();
  }
}

struct Launch {
  const void* f;
  int block;
  size_t lds;
};

// FP32, 513 to 1024 pairs: only the waves that have pairs, so that three workgroups of 9
// or 10 waves share a CU (27x41, us per step: 1500 trajectories 2.96 -> 2.62, 8192 15.8 ->
// 13.7; 30x36 with a drawn F, 1500: 3.44 -> 2.60).  Fewer pairs and FP64 gain and lose
// by batch, -10 to +8%: full workgroups.
template <typename T, int BLOCK, int PPT, int V, bool ODD, bool UI0>
Launch launch_x(int np, bool xn) {
  return {xn ? (const void*)nn_step_kernel<T, BLOCK, PPT, V, ODD, true, UI0>
             : (const void*)nn_step_kernel<T, BLOCK, PPT, V, ODD, false, UI0>,
          sizeof(T) == 4 && BLOCK == 1024 && PPT == 1 ? (np + 63) / 64 * 64 : BLOCK, kTabBytes<T> + 16 + (size_t)BLOCK * PPT * 2 * sizeof(cpx<T>) * (V == kVaryNone ? 1 : 2)};
}

template <typename T, int V, bool ODD, bool UI0>
Launch launch_s(int n, bool xn) {
  const int np = (n + 1) / 2;
  return np <= 64     ? launch_x<T, 64, 1, V, ODD, UI0>(np, xn)
         : np <= 128  ? launch_x<T, 128, 1, V, ODD, UI0>(np, xn)
         : np <= 256  ? launch_x<T, 256, 1, V, ODD, UI0>(np, xn)
         : np <= 512  ? launch_x<T, 512, 1, V, ODD, UI0>(np, xn)
         : np <= 1024 ? launch_x<T, 1024, 1, V, ODD, UI0>(np, xn)
                      : launch_x<T, 1024, 2, V, ODD, UI0>(np, xn);
}

template <typename T, int V>
Launch launch_v(int nx, int ny, bool ui0) {
  const int n = nx * ny;
  const bool xn = nx > 1;
  if (ny % 2) return launch_s<T, V, true, false>(n, xn);
  if constexpr (V == kVaryNone) {
    if constexpr (sizeof(T) == 4) return {nullptr, 0, 0};  // the stacked kernel's
    else if (ui0) return launch_s<T, V, false, true>(n, xn);
  }
  if constexpr (V != kVaryNone || sizeof(T) == 8) return launch_s<T, V, false, false>(n, xn);
}

template <typename T>
Launch launch_t(int nx, int ny, int vary, bool ui0) {
  return vary == kVaryNone  ? launch_v<T, kVaryNone>(nx, ny, ui0)
         : vary == kVaryRsl ? launch_v<T, kVaryRsl>(nx, ny, ui0)
                            : launch_v<T, kVaryF>(nx, ny, ui0);
}

Launch launch_of(int nx, int ny, int precision, int vary, bool ui0) {
  return precision == 64 ? launch_t<double>(nx, ny, vary, ui0) : launch_t<float>(nx, ny, vary, ui0);
}

hipError_t allow_lds(const Launch& l) {
  if (l.lds <= 65536) return hipSuccess;
  return hipFuncSetAttribute(l.f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l.lds);
}

}  // namespace

// From 65 sites on (below, the LDS kernel packs two or four trajectories into a wave),
// FP64 with even rows from 129 on: there the LDS kernel's two waves of one trajectory
// are as fast.  us per step, LDS kernel against this one, 4500 / 10000 trajectories:
// FP32 5x13 1.43, 2.55 to 1.01, 1.80, 8x16 with a drawn F 1.30, 2.44 to 1.04, 1.88; FP64 5x13
// 2.60, 5.11 to 2.26, 4.69, 8x16 with a drawn F 2.56, 5.9 to 2.72, 4.81 (4x8 and 7x9,
// FP64, 4500: 1.60, 1.72 to 2.52, 2.17).
bool nn_supported(int nx, int ny, int precision, int vary) {
  const int n = nx * ny;
  return (vary == kVaryNone || vary == kVaryRsl || vary == kVaryF) && ny > 1 && n <= 4096 &&
         n > (precision == 64 && ny % 2 == 0 ? 128 : 64) && (precision == 64 || vary != kVaryNone || ny % 2);
}

// FP64 with even rows: where the LDS kernel's own launch is as fast or faster it stays.
// Its 128 registers give each wave more to overlap, which tells until the CUs hold more
// than four waves per SIMD.  us per step there against here:
//   up to 256 sites, uniform: the same at every batch (16x16, 8192: 7.7, 7.4);
//     one parameter varying (held in registers there): 16x16, 1500 trajectories
//     1.59 / 1.81, 3000 3.14 / 3.29, 6000 6.08 / 5.65, 20000 20.1 / 16.7;
//   257 to 512, uniform: 1x512, 130 trajectories 0.64 / 0.72, 700 1.36 / 1.42, 3000
//     5.11 / 4.67;
//   2049 to 4096, uniform: 64x64, 32 trajectories 2.97 / 3.29, 512 6.38 / 6.62, 768
//     10.24 / 9.52.
// Between, and with odd rows, this kernel wins at every batch (32x32, 32 trajectories,
// 1.19 / 1.03).
bool nn_pays(int nx, int ny, int precision, int vary, size_t n_traj, int cus) {
  const int n = nx * ny;
  const size_t per_cu = n_traj / (size_t)cus;
  if (precision != 64 || ny % 2) return true;
  if (n <= 256) return vary != kVaryNone && per_cu >= 12;
  if (vary != kVaryNone) return true;
  return n <= 512 ? per_cu >= 4 : n <= 2048 || n_traj > 2 * (size_t)cus;
}

hipError_t nn_occupancy(int nx, int ny, int precision, int vary, bool u_real, int* blocks_per_cu, LaunchShape* shape) {
  const Launch l = launch_of(nx, ny, precision, vary, u_real);
  shape->block = l.block;
  shape->lds = l.lds;
  hipError_t e = allow_lds(l);
  if (e != hipSuccess) return e;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, l.f, l.block, l.lds);
}

hipError_t launch_nn(const StepArgs& a, int precision, int grid, hipStream_t s) {
  const Launch l = launch_of(a.nx, a.ny, precision, a.vary, a.u_real != 0);
  hipError_t e = allow_lds(l);
  if (e != hipSuccess) return e;
  StepArgs q = a;
  if (!queue_pays(a, grid, precision)) q.queue = nullptr;
  else hipLaunchKernelGGL(queue_reset_kernel, dim3(1), dim3(64), 0, s, q.queue);
  void* args[] = {&q};
  return hipLaunchKernel(l.f, dim3(grid), dim3(l.block), args, l.lds, s);
}

}  // namespace twmc
