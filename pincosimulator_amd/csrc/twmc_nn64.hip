// twmc_nn64.hip -- FP64 step kernel for site-uniform periodic lattices with an even
// row length, 257 to 4096 sites, the hopping in its nearest-neighbour form (the
// exact real-space form of the reference's FFT product,
// TWMCBaseSolver.cpp:80-88, :235-242).  One workgroup owns one trajectory: a
// pair per thread (two for 2049 to 4096 sites), the state in registers, the
// neighbours from one LDS copy of it; trajectories come from a work queue.
//
// What bounds it: VALU issue.  The LDS kernel's FP64 step
// (twmc_generic.hip) keeps the Box-Muller coefficients, both sites' intermediates
// and six neighbours in 128 registers, four waves per SIMD; here 64 registers
// hold eight: the coefficients lie in scalar registers, the sites' samples are
// formed one after the other, the neighbours read at their use.  Every operation
// and its order are that kernel's, so are the bits.  us per step before (that
// kernel) -> now: 4096 trajectories of 32x32 14.76 -> 13.10, of 36x50 30.1 -> 24.7, of
// 48x48 32.6 -> 29.0, of 64x64 51.5 -> 48.0; 256 trajectories of 36x50 2.50 -> 1.99.
// Left: the table rows are read at random, 16 bytes a lane, four per pair, and
// conflict about threefold in the LDS banks (up to 2048 sites a copy of the kernel
// reading one row was 11% faster).
#include <algorithm>

#include "twmc_cplx.h"
#include "twmc_f64math.h"
#include "twmc_internal.h"
#include "twmc_rng.h"

namespace twmc {

namespace {

// the FP64 Box-Muller's ln and sin / cos tables (twmc_f64math.h)
alignas(16) __device__ const double kF64TabDev[f64::kTabSize] = TWMC_F64_TABLES;

__global__ void queue_reset_kernel(unsigned int* queue) {
  if (threadIdx.x == 0) *queue = 0u;
}

// XN: the lattice has x neighbours (nx > 1).  UI0: Im U = 0, so the factor of z in
// the new value is a constant.
template <int BLOCK, int PPT, bool XN, bool UI0>
__global__ void __launch_bounds__(BLOCK, 8) nn64_step_kernel(StepArgs g) {
  constexpr int kPairs = BLOCK * PPT;
  extern __shared__ __align__(16) unsigned char smem[];
  double* const ltab = reinterpret_cast<double*>(smem);
  int* const s_next = reinterpret_cast<int*>(smem + sizeof(double) * f64::kTabSize);
  cpx<double>* const st = reinterpret_cast<cpx<double>*>(smem + sizeof(double) * f64::kTabSize + 16);  // [even, odd][pair]
  for (int i = threadIdx.x; i < f64::kTabSize; i += BLOCK) ltab[i] = kF64TabDev[i];
  f64::Series bmk = f64::kSeries;
  f64::pin_scalar(bmk);

  const int npairs = g.n / 2, yh = g.ny / 2;
  const int wave_p = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63);
  int lft[PPT], rgt[PPT], up[PPT], dn[PPT];
#pragma unroll
  for (int j = 0; j < PPT; ++j) {
    const int p = threadIdx.x + BLOCK * j;
    const int row = p / yh, q = p - row * yh;
    lft[j] = kPairs + (q == 0 ? p + yh - 1 : p - 1);
    rgt[j] = q + 1 == yh ? p + 1 - yh : p + 1;
    up[j] = p + yh >= npairs ? p + yh - npairs : p + yh;
    dn[j] = p < yh ? p - yh + npairs : p - yh;
    if (p >= npairs) lft[j] = rgt[j] = up[j] = dn[j] = 0;  // computed along in a partly filled wave, not stored
  }
  // dt rsl, dt U, dt i F, dt J as the LDS kernel forms them
  const double dt = g.dt, dt4 = g.dt4;
  const cpx<double> r0 = reinterpret_cast<const cpx<double>*>(g.rsl)[0];
  const cpx<double> u0 = reinterpret_cast<const cpx<double>*>(g.U)[0];
  const cpx<double> f0 = reinterpret_cast<const cpx<double>*>(g.F)[0];
  const cpx<double> rd = mk(dt * r0.re, dt * r0.im), ud = mk(dt * u0.re, dt * u0.im), fd = mk(-dt * f0.im, dt * f0.re);
  const double rd1 = 1.0 + rd.re;
  const double djv = -0.5 * g.kscale * g.dt;

  for (int b = blockIdx.x; b < g.n_traj;) {
    const uint64_t traj = g.traj_ids[b];
    cpx<double>* gb = reinterpret_cast<cpx<double>*>(g.beta) + (size_t)b * g.n;
    cpx<double> beta[2 * PPT];
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
      const int p = threadIdx.x + BLOCK * j;
      beta[2 * j] = beta[2 * j + 1] = mk(0.0, 0.0);
      if (p < npairs) {
        beta[2 * j] = gb[2 * p];
        beta[2 * j + 1] = gb[2 * p + 1];
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
          const cpx<double> z0 = beta[2 * j], z1 = beta[2 * j + 1];
          cpx<double> nz[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint32_t wa[1] = {h ? x.z : x.x}, wb[1] = {h ? x.w : x.y};
            double xr[1], xi[1];
            f64::box_muller<1, true>(wa, wb, xr, xi, bmk, ltab);
            const cpx<double> z = h ? z1 : z0;
            // y + 1 and y - 1 neighbours, then x + 1 and x - 1
            const cpx<double> a = h ? st[rgt[j]] : z1, c = h ? z0 : st[lft[j]];
            double sr = a.re + c.re, si = a.im + c.im;
            if constexpr (XN) {
              const cpx<double> d = st[kPairs * h + up[j]], e = st[kPairs * h + dn[j]];
              sr += d.re + e.re;
              si += d.im + e.im;
            }
            // increment dt (c z + h + i F) + dt4 xi as one FMA chain per component,
            // the (1 + c) z term last; dt h = dt J (S_im, -S_re)
            const double q = fma(z.re, z.re, fma(z.im, z.im, -1.0));
            const double ci = fma(ud.re, q, rd.im), cr1 = UI0 ? rd1 : fma(-ud.im, q, rd1);
            double dr = fma(dt4, xr[0], fd.re);
            dr = fma(djv, si, dr);
            dr = fma(-ci, z.im, dr);
            double di = fma(dt4, xi[0], fd.im);
            di = fma(-djv, sr, di);
            di = fma(ci, z.re, di);
            nz[h] = mk(fma(cr1, z.re, dr), fma(cr1, z.im, di));
          }
          beta[2 * j] = nz[0];
          beta[2 * j + 1] = nz[1];
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
      const int p = threadIdx.x + BLOCK * j;
      if (p < npairs) {
        gb[2 * p] = beta[2 * j];
        gb[2 * p + 1] = beta[2 * j + 1];
      }
    }
    // the next trajectory, from the queue (the barriers of the steps separate this
    // word's uses)
    if (threadIdx.x == 0) *s_next = (int)(gridDim.x + atomicAdd(g.queue, 1u));
    __syncthreads();
    b = __builtin_amdgcn_readfirstlane(*s_next);
    __syncthreads();
  }
}

template <int BLOCK, int PPT>
const void* kernel_b(bool xn, bool ui0) {
  return xn ? (ui0 ? (const void*)nn64_step_kernel<BLOCK, PPT, true, true> : (const void*)nn64_step_kernel<BLOCK, PPT, true, false>)
            : (ui0 ? (const void*)nn64_step_kernel<BLOCK, PPT, false, true> : (const void*)nn64_step_kernel<BLOCK, PPT, false, false>);
}

struct Shape {
  int block, ppt;
};

Shape shape_of(int n) {
  const int np = n / 2;
  return np <= 256 ? Shape{256, 1} : np <= 512 ? Shape{512, 1} : np <= 1024 ? Shape{1024, 1} : Shape{1024, 2};
}

const void* kernel_for(int nx, int n, bool ui0) {
  const Shape s = shape_of(n);
  const bool xn = nx > 1;
  return s.block == 256 ? kernel_b<256, 1>(xn, ui0) : s.block == 512 ? kernel_b<512, 1>(xn, ui0)
         : s.ppt == 1   ? kernel_b<1024, 1>(xn, ui0) : kernel_b<1024, 2>(xn, ui0);
}

size_t lds_bytes(int n) {
  const Shape s = shape_of(n);
  return sizeof(double) * f64::kTabSize + 16 + (size_t)s.block * s.ppt * 32;
}

}  // namespace

bool nn64_supported(int nx, int ny, int precision, bool site_uniform) {
  const int n = nx * ny;
  return precision == 64 && site_uniform && ny % 2 == 0 && n > 256 && n <= 4096;
}

// Two pairs per thread (above 2048 sites) and at most two trajectories per CU: the LDS
// kernel's own launch there (1024 threads too, 128 registers, one barrier per step)
// gives each wave more to overlap, and the eight waves per SIMD have no third
// trajectory to take up: 64x64, us per step there against here, 32 trajectories 2.97
// to 3.29, 512 6.38 to 6.62 (48x48: 1.96 to 2.10, 4.21 to 4.08).  From the third on
// this kernel wins (64x64: 513 trajectories 9.28 to 8.92, 768 10.24 to 9.52); up to
// 2048 sites it wins at every batch (32 trajectories of 32x32 1.19 to 1.03).
bool nn64_pays(int n, size_t n_traj, int cus) { return n <= 2048 || n_traj > 2 * (size_t)cus; }

int nn64_block(int n) { return shape_of(n).block; }

hipError_t nn64_occupancy(int nx, int ny, bool u_real, int* blocks_per_cu) {
  const void* f = kernel_for(nx, nx * ny, u_real);
  const size_t lds = lds_bytes(nx * ny);
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, f, nn64_block(nx * ny), lds);
}

hipError_t launch_nn64(const StepArgs& a, int grid, hipStream_t s) {
  const void* f = kernel_for(a.nx, a.n, a.u_real != 0);
  const size_t lds = lds_bytes(a.n);
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(queue_reset_kernel, dim3(1), dim3(64), 0, s, a.queue);
  void* args[] = {const_cast<StepArgs*>(&a)};
  return hipLaunchKernel(f, dim3(grid), dim3(nn64_block(a.n)), args, lds, s);
}

}  // namespace twmc
