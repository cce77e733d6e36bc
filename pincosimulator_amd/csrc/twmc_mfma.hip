// twmc_mfma.hip -- matrix-hopping TWMC step on the matrix cores.
//
// For general (disordered, Lieb, long-range) hopping the reference computes
// h = -i (beta . C) per trajectory with a sparse product
// (src/TWMC/Solvers/TWMCLiebSolver.cpp:259-267).  Here the hopping of a block
// of 16 or 32 trajectories is one GEMM per step,
//     Y = C^T [Re beta_1 .. Re beta_32 | Im beta_1 .. Im beta_32]   (N x 64),
// on v_mfma_f32_16x16x32_bf16 with FP32 accumulation.  FP32 operands are
// split as x = x_hi + x_lo (both BF16) and the product is
//     A_hi X_hi + A_hi X_lo + A_lo X_hi,
// which keeps about 16 significant bits (the dropped A_lo X_lo term and the
// BF16 rounding of the low parts are ~2^-16 relative).
//
// One workgroup (8 waves) owns its trajectories for a whole segment: the
// accumulators of a lane hold Y for Re and Im of the same (site, trajectory), and
// the Euler update runs in registers, on the FP32 state that never leaves the lane.
// Each step the state is re-staged in LDS as the BF16 hi/lo B operand; A = C^T (hi/lo,
// zero-padded to np = 128, 256, 384 or 512 and in fragment order, mfma_swizzle, so
// that a fragment load is one contiguous 1 KiB read) comes from L2, shared by every
// workgroup.
//
// What bounds it: at 8192 trajectories of 384 sites the matrix cores (5.8 of 14.5 us
// a step at their peak), A from L2 (590 KB a step and workgroup) and 3.2 us of VALU
// work beside them; at small batches the latency of a workgroup's step on the few CUs
// that have one.  us per step before (32 trajectories, 32-row tiles of 4 waves for np not
// 128, 256 or 384, every padded row and column computed) -> now: 2048 trajectories of
// 48 sites 4.16 -> 1.30, 200 11.4 -> 3.85, 256 6.30 -> 3.93, 300 16.5 -> 6.45, 384 11.2 ->
// 7.0, 500 27.6 -> 10.9; 8192 of 48 4.32 -> 1.73, 200 12.4 -> 7.3, 300 18.9 -> 12.7, 500
// 33.9 -> 28.8.
#include <cstring>

#include "twmc_cplx.h"
#include "twmc_internal.h"
#include "twmc_rng.h"

namespace twmc {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// two FP32 values -> packed BF16 high parts (round to nearest even, one
// v_cvt_pk_bf16_f32) and packed BF16 parts of the remainders, so that
// x = hi + lo to ~2^-16 relative
__device__ __forceinline__ void split_bf16(float x0, float x1, uint32_t& hi, uint32_t& lo) {
  const f32x2 v = {x0, x1};
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  const f32x2 d = {x0 - __uint_as_float(hi << 16), x1 - __uint_as_float(hi & 0xffff0000u)};
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(d, bf16x2));
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// The step on v_mfma_f32_16x16x32_bf16 for np = 128 TPW: 8 waves (two per SIMD, so one
// wave's MFMAs run while the other waits for operands or at a barrier), 16 QG
// trajectories per workgroup.  Wave w owns the TPW 16-site row tiles w TPW .. w TPW +
// TPW - 1 and all 2 QG 16-column tiles: Re and Im of trajectories 0-15 (ct = 0, 1) and,
// QG = 2, 16-31 (ct = 2, 3).  Lane l holds column l % 16 and rows 4 (l / 16) + r, r < 4,
// of each result tile, so Re and Im of the same (site, trajectory) meet in one lane.  A
// (16-row tiles, 32-wide k blocks, fragment order) streams from L2 one k block
// ahead; B (the state as BF16 hi/lo) is staged in LDS every step.  A lane owns
// 2 QG TPW site pairs per step, one for every 2 / QG k blocks, whose MFMAs carry that
// pair's Philox draw, Box-Muller and drift/drive terms (fenced pieces); after
// the GEMM only dt h is added.  A wave whose rows all lie past the lattice only keeps
// the barriers; k blocks past it are left out, if there are any.  FULL: no such test, for
// lattices whose k blocks fill np, and for np = 512, where 385 to 480 sites step their
// zeros along.  Two of the forms at np = 384 spill with 32 trajectories: FULL one value,
// the other (257 to 352 sites) 13.
template <int TPW, int QG, bool FULL, bool CAPTURE_ONLY>
__global__ void __launch_bounds__(512, 1) mfma_step_kernel(StepArgs g) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NP = 128 * TPW, NKB = NP / 32, LDK = NP + 8;  // LDK: padded row, conflict-free reads
  constexpr int kTB = 16 * QG, kCols = 32 * QG;
  const int n = g.n;
  uint16_t* Xhi = reinterpret_cast<uint16_t*>(smem);
  uint16_t* Xlo = Xhi + kCols * LDK;
  cpx<float>* Prsl = reinterpret_cast<cpx<float>*>(Xlo + kCols * LDK);
  cpx<float>* PU = Prsl + NP;
  cpx<float>* PF = PU + NP;
  double* red = reinterpret_cast<double*>(PF + NP);  // [8 waves][kTB][2]

  // the wave index is uniform: made scalar, the operand addresses become a
  // scalar base plus one per-lane offset instead of a register pair per load
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int col = lane & 15, rg = lane >> 4;
  const float dt = float(g.dt), sig = float(g.dt4);
  const float nl = -1.3862943611198906f * sig * sig;  // -2 ln2 sigma^2 (Box-Muller)
  const bool busy = FULL || wave * TPW * 16 < n;  // the wave has rows
  const int live = (n + 31) / 32;         // k blocks of the lattice
  // site tables pre-scaled by dt for the update's FMA chain:
  //   dt (rsl + i U (|b|^2 - 1)) = (A - dt U.im |b|^2) + i (B + dt U.re |b|^2),
  //   Prsl = (A, B) = (dt (rsl.re + U.im), dt (rsl.im - U.re)), PU = dt U, PF = dt i F
  for (int i = tid; i < NP; i += blockDim.x) {
    const bool in = i < n;
    const cpx<float> r = in ? reinterpret_cast<const cpx<float>*>(g.rsl)[i] : mk(0.f, 0.f);
    const cpx<float> u = in ? reinterpret_cast<const cpx<float>*>(g.U)[i] : mk(0.f, 0.f);
    const cpx<float> f = in ? reinterpret_cast<const cpx<float>*>(g.F)[i] : mk(0.f, 0.f);
    Prsl[i] = mk(dt * (r.re + u.im), dt * (r.im - u.re));
    PU[i] = mk(dt * u.re, dt * u.im);
    PF[i] = mk(-dt * f.im, dt * f.re);
  }
  __syncthreads();

  const uint16_t* Ahi = reinterpret_cast<const uint16_t*>(g.a_hi);
  const uint16_t* Alo = reinterpret_cast<const uint16_t*>(g.a_lo);
  double* part = g.partials + (size_t)blockIdx.x * kQ * n;
  const int nblk = (g.n_traj + kTB - 1) / kTB;

  for (int blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
    int jt[QG];
    bool valid[QG];
    uint64_t traj[QG];
    cpx<float>* gb[QG];
#pragma unroll
    for (int q = 0; q < QG; ++q) {
      jt[q] = blk * kTB + q * 16 + col;
      valid[q] = jt[q] < g.n_traj;
      traj[q] = valid[q] ? g.traj_ids[jt[q]] : 0;
      gb[q] = reinterpret_cast<cpx<float>*>(g.beta) + (size_t)(valid[q] ? jt[q] : 0) * n;
    }
    // first site of this lane's rows, opaque to the compiler (per-site
    // addresses are formed in the block, not held across the steps)
    int ib = wave * TPW * 16 + rg * 4;
    asm volatile("" : "+v"(ib));

    // FP32 state in the result layout: [tile][trajectory group][register]
    float sre[TPW][QG][4], sim[TPW][QG][4];
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int q = 0; q < QG; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = ib + t * 16 + r;
          const cpx<float> v = (valid[q] && i < n) ? gb[q][i] : mk(0.f, 0.f);
          sre[t][q][r] = v.re;
          sim[t][q][r] = v.im;
        }

    if (g.capture) {
      double m2[QG] = {}, m4[QG] = {};
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = ib + t * 16 + r;
          double a = 0.0, b = 0.0, c = 0.0, d = 0.0;
#pragma unroll
          for (int q = 0; q < QG; ++q) {
            const bool use = valid[q] && i < n;
            const double xr = use ? double(sre[t][q][r]) : 0.0, xi = use ? double(sim[t][q][r]) : 0.0;
            const double nn = xr * xr + xi * xi;
            m2[q] += nn;
            m4[q] += nn * nn;
            if (g.dump && use)
              reinterpret_cast<cpx<float>*>(g.traj_out)[((size_t)jt[q] * g.n_frames + g.frame) * n + i] =
                  mk(sre[t][q][r], sim[t][q][r]);
            a += nn;
            b += nn * nn;
            c += xr;
            d += xi;
          }
          // per-site sums over the block's trajectories: the 16 lanes of a
          // row group hold the same site for trajectories q 16 + l % 16
#pragma unroll
          for (int o = 1; o < 16; o <<= 1) {
            a += __shfl_xor(a, o, 64);
            b += __shfl_xor(b, o, 64);
            c += __shfl_xor(c, o, 64);
            d += __shfl_xor(d, o, 64);
          }
          if (col == 0 && i < n) {
            part[i] += a;
            part[n + i] += b;
            part[3 * n + i] += c;
            part[4 * n + i] += d;
          }
        }
      // the four row groups hold the same trajectories
#pragma unroll
      for (int q = 0; q < QG; ++q) {
        m2[q] += __shfl_xor(m2[q], 16, 64);
        m2[q] += __shfl_xor(m2[q], 32, 64);
        m4[q] += __shfl_xor(m4[q], 16, 64);
        m4[q] += __shfl_xor(m4[q], 32, 64);
        if (rg == 0) {
          red[(wave * kTB + q * 16 + col) * 2] = m2[q];
          red[(wave * kTB + q * 16 + col) * 2 + 1] = m4[q];
        }
      }
      __syncthreads();
      if (tid < kTB && blk * kTB + tid < g.n_traj) {
        double a2 = 0.0, a4 = 0.0;
        for (int w = 0; w < 8; ++w) {
          a2 += red[(w * kTB + tid) * 2];
          a4 += red[(w * kTB + tid) * 2 + 1];
        }
        const size_t o = (size_t)(blk * kTB + tid) * g.n_frames + g.frame;
        g.traj_m2[o] = a2 / double(n);
        g.traj_m4[o] = a4 / double(n);
      }
      __syncthreads();
    }
    if (CAPTURE_ONLY) continue;

    int ft_id = 0;
    for (int s = 0; s < g.n_steps; ++s) {
      // stage the state as the BF16 hi/lo B operand: columns q 16 + l % 16 (Re)
      // and 16 QG + q 16 + l % 16 (Im), this lane's four consecutive sites
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int q = 0; q < QG; ++q) {
          const int k0 = (wave * TPW + t) * 16 + rg * 4;
          uint32_t rh[2], rl[2], ih[2], il[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            split_bf16(sre[t][q][2 * e], sre[t][q][2 * e + 1], rh[e], rl[e]);
            split_bf16(sim[t][q][2 * e], sim[t][q][2 * e + 1], ih[e], il[e]);
          }
          const int cr = q * 16 + col, ci = kTB + q * 16 + col;
          *reinterpret_cast<uint2*>(&Xhi[cr * LDK + k0]) = make_uint2(rh[0], rh[1]);
          *reinterpret_cast<uint2*>(&Xlo[cr * LDK + k0]) = make_uint2(rl[0], rl[1]);
          *reinterpret_cast<uint2*>(&Xhi[ci * LDK + k0]) = make_uint2(ih[0], ih[1]);
          *reinterpret_cast<uint2*>(&Xlo[ci * LDK + k0]) = make_uint2(il[0], il[1]);
        }
      if (g.ft_n > 0) {
        // F(t) before this step into the site table (TWMCLiebSolver.cpp:252-256),
        // read during the GEMM after the barrier below; the previous step's
        // readers finished before the barrier that ended its GEMM
        const float fdt = float(drive_interval(g.ft_times, g.ft_n, g.t0 + double(s) * g.dt, ft_id));
        const cpx<float>* fv = reinterpret_cast<const cpx<float>*>(g.ft_vals) + (size_t)ft_id * n;
        const cpx<float>* fs = reinterpret_cast<const cpx<float>*>(g.ft_slopes) + (size_t)ft_id * n;
        for (int i = tid; i < n; i += blockDim.x)
          PF[i] = mk(-dt * fmaf(fdt, fs[i].im, fv[i].im), dt * fmaf(fdt, fs[i].re, fv[i].re));
      }
      __syncthreads();

      constexpr int kPieces = 9, kSpan = 2 / QG, kSlots = 12 * TPW;  // kSpan: k blocks per site pair
      const uint32_t step = uint32_t(g.step0 + (uint64_t)s);
      // opaque to the compiler: the per-pair Philox rounds, the table reads and
      // the operand addresses are formed in the step, not hoisted out of it
      uint32_t pbase = (uint32_t)(wave * TPW * 8 + rg * 2);
      asm volatile("" : "+v"(pbase));
      int zo = 0;
      asm volatile("" : "+s"(zo));
      const uint16_t* Ahw = Ahi + (size_t)(wave * TPW) * NKB * 512 + zo;  // scalar
      const uint16_t* Alw = Alo + (size_t)(wave * TPW) * NKB * 512 + zo;
      auto aload = [&](const uint16_t* A, int t, int kb) {
        return *reinterpret_cast<const bf16x8*>(&(A == Ahi ? Ahw : Alw)[((size_t)t * NKB + kb) * 512 + lane * 8]);
      };
      auto bload = [&](const uint16_t* X, int ct, int kb) {
        const int c = (ct & 1) * kTB + (ct >> 1) * 16 + col;
        return *reinterpret_cast<const bf16x8*>(&X[c * LDK + kb * 32 + rg * 8 + zo]);
      };
      f32x4 acc[TPW][2 * QG];
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int ct = 0; ct < 2 * QG; ++ct) acc[t][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (busy) {
      bf16x8 ah[TPW], al[TPW], bh, bl;
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        ah[t] = aload(Ahi, t, 0);
        al[t] = aload(Alo, t, 0);
      }
      bh = bload(Xhi, 0, 0);
      bl = bload(Xlo, 0, 0);
      u32x4 w;
      float rn[2], cs[2], sn[2];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        // A of the next k block, one block ahead
        bf16x8 ahn[TPW], aln[TPW];
        if (kb + 1 < NKB) {
#pragma unroll
          for (int t = 0; t < TPW; ++t) {
            ahn[t] = aload(Ahi, t, kb + 1);
            aln[t] = aload(Alo, t, kb + 1);
          }
        }
        // site pair kp: row tile tp, trajectory group qp, pair pr of the lane's four sites
        const int kp = kb / kSpan, tp = kp / (2 * QG), qp = (kp >> 1) & (QG - 1), pr = kp & 1;
        auto piece = [&](int pc) __attribute__((always_inline)) {
          if (pc == 0) w = make_counter(traj[qp], TAG_WIENER, step, pbase + (uint32_t)(tp * 8 + pr));
          if (pc < 5) {
            philox_round(w, g.key0, g.key1, 2 * pc);
            philox_round(w, g.key0, g.key1, 2 * pc + 1);
            asm volatile("" : "+v"(w.x), "+v"(w.y), "+v"(w.z), "+v"(w.w));
          } else if (pc < 7) {
            const int h = pc - 5;
            box_muller_f32_scaled(h ? w.z : w.x, h ? w.w : w.y, nl, rn[h], cs[h], sn[h]);
            asm volatile("" : "+v"(rn[h]), "+v"(cs[h]), "+v"(sn[h]));
          } else {
            // increment without dt h: noise + dt iF + drift (TWMCLiebSolver.cpp:259-264)
            const int h = pc - 7, r = 2 * pr + h;
            const int i = (wave * TPW + tp) * 16 + rg * 4 + r;
            const float br = sre[tp][qp][r], bi = sim[tp][qp][r];
            const cpx<float> ab = Prsl[i + zo], u = PU[i + zo], f = PF[i + zo];
            const float mq = fmaf(bi, bi, br * br);
            const float cr = fmaf(-u.im, mq, ab.re), ci = fmaf(u.re, mq, ab.im);
            float dr = fmaf(rn[h], cs[h], f.re);
            dr = fmaf(cr, br, dr);
            dr = fmaf(-ci, bi, dr);
            float di = fmaf(rn[h], sn[h], f.im);
            di = fmaf(cr, bi, di);
            di = fmaf(ci, br, di);
            // added to the state now (the B operand of this step is already
            // staged); dt h follows after the GEMM
            sre[tp][qp][r] = br + dr;
            sim[tp][qp][r] = bi + di;
            asm volatile("" : "+v"(sre[tp][qp][r]), "+v"(sim[tp][qp][r]));
          }
        };
        // the pieces of slot sl of this k block's 6 QG TPW
        auto pieces = [&](int sl) __attribute__((always_inline)) {
          const int at = (kb % kSpan) * 6 * QG * TPW + sl;
#pragma unroll
          for (int pc = (at * kPieces + kSlots - 1) / kSlots; pc < ((at + 1) * kPieces + kSlots - 1) / kSlots; ++pc) piece(pc);
        };
        if (!FULL && kb > 4 * (TPW - 1) && kb >= live) {  // n > 128 (TPW - 1)
#pragma unroll
          for (int sl = 0; sl < 6 * QG * TPW; ++sl) pieces(sl);
          continue;
        }
        // 6 QG TPW MFMAs: column tile ct outer (its B operand loaded one tile
        // ahead), then the products hi.hi, hi.lo, lo.hi, then the row tiles
#pragma unroll
        for (int ct = 0; ct < 2 * QG; ++ct) {
          bf16x8 bhn = bh, bln = bl;
          if (ct + 1 < 2 * QG) {
            bhn = bload(Xhi, ct + 1, kb);
            bln = bload(Xlo, ct + 1, kb);
          } else if (kb + 1 < NKB) {
            bhn = bload(Xhi, 0, kb + 1);
            bln = bload(Xlo, 0, kb + 1);
          }
#pragma unroll
          for (int pm = 0; pm < 3; ++pm)
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
              pieces((ct * 3 + pm) * TPW + t);
              const bf16x8 a = pm < 2 ? ah[t] : al[t];
              const bf16x8 b = pm == 1 ? bl : bh;
              acc[t][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[t][ct], 0, 0, 0);
              __builtin_amdgcn_sched_barrier(0);
            }
          bh = bhn;
          bl = bln;
        }
        if (kb + 1 < NKB) {
#pragma unroll
          for (int t = 0; t < TPW; ++t) {
            ah[t] = ahn[t];
            al[t] = aln[t];
          }
        }
      }
      }
      __syncthreads();  // the next step overwrites the B operand
      // dt h, h = -i Y (h_re = Im Y, h_im = -Re Y), and the update
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int q = 0; q < QG; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = (wave * TPW + t) * 16 + rg * 4 + r + zo;
            if (i < n) {
              sre[t][q][r] = fmaf(dt, acc[t][2 * q + 1][r], sre[t][q][r]);
              sim[t][q][r] = fmaf(-dt, acc[t][2 * q][r], sim[t][q][r]);
            }
          }
    }

    if (!CAPTURE_ONLY) {
#pragma unroll
      for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int q = 0; q < QG; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = ib + t * 16 + r;
            if (valid[q] && i < n) gb[q][i] = mk(sre[t][q][r], sim[t][q][r]);
          }
    }
  }
}

template <int TPW, int QG>
const void* kernel_c(int n, bool capture) {
  if (capture) return (const void*)mfma_step_kernel<TPW, QG, true, true>;
  if constexpr (TPW < 4)
    if (n <= 128 * TPW - 32) return (const void*)mfma_step_kernel<TPW, QG, false, false>;
  return (const void*)mfma_step_kernel<TPW, QG, true, false>;
}

template <int TPW>
const void* kernel_q(int n, int tb, bool capture) {
  if constexpr (TPW < 4)  // four row tiles and four column tiles spill registers
    if (tb == 32) return kernel_c<TPW, 2>(n, capture);
  return kernel_c<TPW, 1>(n, capture);
}

const void* kernel_for(int n, int tb, bool capture) {
  switch (mfma_padded(n) / 128) {
    case 1: return kernel_q<1>(n, tb, capture);
    case 2: return kernel_q<2>(n, tb, capture);
    case 3: return kernel_q<3>(n, tb, capture);
    default: return kernel_q<4>(n, tb, capture);
  }
}

}  // namespace

int mfma_padded(int n) { return (n + 127) / 128 * 128; }

// 16 trajectories per workgroup take about 0.6 of the time of 32 (the A operand
// streams from L2 for either), on twice the workgroups: 16 where that means fewer, or
// no more, rounds of the CUs.  us per step of a round, 32 / 16: np = 256 6.35 / 3.93, 384
// 11.1 / 7.0 (2048 trajectories), 14.5 / 16.9 in two rounds (8192).  At np = 128 several
// workgroups share a CU and 16 is the faster at every batch (8192: 3.03 / 2.96); at 512
// only 16 fits the registers.
int mfma_tb(int np, size_t n_traj, int cus) {
  const size_t r16 = (n_traj + 16 * (size_t)cus - 1) / (16 * (size_t)cus), r32 = (r16 + 1) / 2;
  return np == 128 || np == 512 || 6 * r16 < 10 * r32 ? 16 : 32;
}

// row-major np x np -> fragment order: for 16-row tile T, 32-wide k block b and lane l,
// the 8 consecutive elements A[16 T + l % 16][32 b + 8 (l / 16) + e]
void mfma_swizzle(const double* a, int np, double* out) {
  const int nkb = np / 32;
  for (int T = 0; T < np / 16; ++T)
    for (int b = 0; b < nkb; ++b)
      for (int l = 0; l < 64; ++l)
        for (int e = 0; e < 8; ++e)
          out[(((size_t)T * nkb + b) * 64 + l) * 8 + e] =
              a[(size_t)(T * 16 + l % 16) * np + b * 32 + (l / 16) * 8 + e];
}

size_t mfma_lds_bytes(int np, int tb) {
  return (size_t)2 * 2 * tb * (np + 8) * 2 + (size_t)3 * np * 8 + (size_t)8 * tb * 2 * 8;
}

bool mfma_supported(int n, int hopping, int precision, int param_stride) {
  return hopping == 1 && precision == 32 && param_stride == 0 && n <= 512;
}

hipError_t launch_mfma(const StepArgs& a, int grid, hipStream_t s) {
  const size_t lds = mfma_lds_bytes(a.np, a.tb);
  const void* f = kernel_for(a.n, a.tb, a.n_steps == 0);
  hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  void* args[] = {const_cast<StepArgs*>(&a)};
  return hipLaunchKernel(f, dim3(grid), dim3(512), args, lds, s);
}

hipError_t mfma_occupancy(int n, int tb, int* blocks_per_cu) {
  const size_t lds = mfma_lds_bytes(mfma_padded(n), tb);
  const void* f = kernel_for(n, tb, false);
  hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, f, 512, lds);
}

void mfma_split(const double* a, size_t count, uint16_t* hi, uint16_t* lo) {
  auto rne = [](float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
  };
  auto back = [](uint16_t b) {
    uint32_t u = uint32_t(b) << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
  };
  for (size_t k = 0; k < count; ++k) {
    float f = (float)a[k];
    hi[k] = rne(f);
    lo[k] = rne(f - back(hi[k]));
  }
}

}  // namespace twmc
