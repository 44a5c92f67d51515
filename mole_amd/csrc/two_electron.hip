// Two-electron walker kernels (He singlet with Pade e-e factor; LCAO
// sigma_g^2 with Pade e-e factor).
//
// A walker's positions, the cached psi and the distances it was built from,
// and every accumulator live in VGPRs across all sweeps of the launch; HBM is
// touched once at entry and once at exit (positions as [6][W] and accumulators
// as [column][W], both coalesced).  Each move does what MetropolisBox::move_state does
// (src/metropolis/src/metrop.rs:60-96): three Range draws, one Standard
// draw, psi at the proposal, min(psi'^2/psi^2, 1) > u.  psi at the
// current configuration is the cached value of the same expression, so
// every accept decision equals the reference's two-evaluation form bit
// for bit.  After each sampled sweep the local energy
// -1/2 lap(psi)/psi + V (src/operator/src/operator.rs:177-183) and the
// parameter log-derivatives are formed in closed form and folded into the
// per-walker sums that the energy gradient and the SR matrix need
// (src/optimize/src/util.rs:6-46, src/optimize/src/optimizers.rs:191-233).
#include "../../include/mole_gpu.h"
#include "device_common.hpp"
#include "internal.hpp"
#include "sr_math.hpp"
#include <type_traits>

namespace mole {

// Orbital factor of one electron for the LCAO kind:
// phi = sum_I exp(-zeta r_I), spelled as the value expression requires.
__device__ __forceinline__ double lcao_phi(const Sys2 &sp, double x, double y,
                                           double z) {
  double phi = 0.0;
  for (int I = 0; I < sp.n_nuc; ++I) {
    const double r = norm3(x - sp.nuc[I][0], y - sp.nuc[I][1], z - sp.nuc[I][2]);
    const double e = exp_m(-sp.zeta * r);
    phi = (I == 0) ? e : phi + e;
  }
  return phi;
}

__device__ __forceinline__ double pade(double b, double c, double r) {
  return (b * r) / (1.0 + c * r);
}

// Closed-form local quantities of one configuration: E_L, the laplacian
// ratio sum_i lap_i(psi)/psi, grad ln psi and d ln psi/dp.
struct Local2 {
  double e_local;
  double lap_ratio;
  double g[6];
  double dlog[kNParam2];
};

template <int KIND>
__device__ __forceinline__ Local2 local2(const Sys2 &sp, const double *x) {
  Local2 L;
  const double zeta = sp.zeta, b = sp.b, c = sp.c;
  double V = sp.v_nn;
  double gi[2][3], li[2], dz = 0.0;
  for (int e = 0; e < 2; ++e) {
    const double *xe = x + 3 * e;
    double phi = 0.0, gs[3] = {0.0, 0.0, 0.0}, ls = 0.0, zs = 0.0;
    const int nn = (KIND == MOLE_WF_HELIUM_PADE) ? 1 : sp.n_nuc;
    for (int I = 0; I < sp.n_nuc; ++I) {
      const double d0 = xe[0] - sp.nuc[I][0], d1 = xe[1] - sp.nuc[I][1],
                   d2 = xe[2] - sp.nuc[I][2];
      const double r = norm3(d0, d1, d2);
      const double inv = 1.0 / r;
      V = V - sp.charge[I] * inv;
      if (I < nn) {
        // helium kind: phi = e^{-zeta r}, so the ratios need no exponential
        const double ee = (KIND == MOLE_WF_HELIUM_PADE) ? 1.0 : exp_m(-zeta * r);
        phi += ee;
        const double f = -zeta * ee * inv;
        gs[0] = fma(f, d0, gs[0]);
        gs[1] = fma(f, d1, gs[1]);
        gs[2] = fma(f, d2, gs[2]);
        ls = fma(ee, zeta * zeta - 2.0 * zeta * inv, ls);
        zs = fma(-r, ee, zs);
      }
    }
    const double ip = 1.0 / phi;
    gi[e][0] = gs[0] * ip;
    gi[e][1] = gs[1] * ip;
    gi[e][2] = gs[2] * ip;
    li[e] = ls * ip;
    dz += zs * ip;
  }
  const double d0 = x[0] - x[3], d1 = x[1] - x[4], d2 = x[2] - x[5];
  const double r12 = norm3(d0, d1, d2);
  const double i12 = 1.0 / r12;
  const double den = 1.0 + c * r12;
  const double iden = 1.0 / den;
  const double up = b * iden * iden;
  const double upp = -2.0 * b * c * iden * iden * iden;
  const double J = upp + 2.0 * up * i12 + up * up;
  const double h0 = d0 * i12, h1 = d1 * i12, h2 = d2 * i12;
  const double gd1 = gi[0][0] * h0 + gi[0][1] * h1 + gi[0][2] * h2;
  const double gd2 = gi[1][0] * h0 + gi[1][1] * h1 + gi[1][2] * h2;
  const double k1 = li[0] + J + 2.0 * up * gd1;
  const double k2 = li[1] + J - 2.0 * up * gd2;
  if (sp.hamiltonian == MOLE_H_ELECTRONIC) V = V + i12;
  L.lap_ratio = k1 + k2;
  L.e_local = -0.5 * (k1 + k2) + V;
  L.g[0] = gi[0][0] + up * h0;
  L.g[1] = gi[0][1] + up * h1;
  L.g[2] = gi[0][2] + up * h2;
  L.g[3] = gi[1][0] - up * h0;
  L.g[4] = gi[1][1] - up * h1;
  L.g[5] = gi[1][2] - up * h2;
  L.dlog[0] = dz;
  L.dlog[1] = r12 * iden;
  L.dlog[2] = -b * r12 * r12 * iden * iden;
  return L;
}

template <int KIND>
__device__ __forceinline__ double value2(const Sys2 &sp, const double *x) {
  const double r12 = norm3(x[0] - x[3], x[1] - x[4], x[2] - x[5]);
  if (KIND == MOLE_WF_HELIUM_PADE) {
    const double r1 = norm3(x[0] - sp.nuc[0][0], x[1] - sp.nuc[0][1], x[2] - sp.nuc[0][2]);
    const double r2 = norm3(x[3] - sp.nuc[0][0], x[4] - sp.nuc[0][1], x[5] - sp.nuc[0][2]);
    return exp_m(-sp.zeta * (r1 + r2) + pade(sp.b, sp.c, r12));
  }
  const double phi1 = lcao_phi(sp, x[0], x[1], x[2]);
  const double phi2 = lcao_phi(sp, x[3], x[4], x[5]);
  return (phi1 * phi2) * exp_m(pade(sp.b, sp.c, r12));
}

// Per-walker sample accumulators: energy sums, block means, SR sums, and
// the optional trace / compat-sample writes, in sample order.
struct SampleAcc {
  double acc[kAccColumns2];
  uint32_t fill, sample_idx;

  __device__ __forceinline__ void load(const Sweep2Args &a, int w) {
#pragma unroll
    for (int k = 0; k < kAccColumns2; ++k)
      if (k != kAccAccepted) acc[k] = a.fresh ? 0.0 : a.acc[(size_t)k * a.W + w];
    fill = a.block_fill;
    sample_idx = a.trace_sample0;
  }
  __device__ __forceinline__ void store(const Sweep2Args &a, int w) const {
#pragma unroll
    for (int k = 0; k < kAccColumns2; ++k)
      if (k != kAccAccepted) a.acc[(size_t)k * a.W + w] = acc[k];
  }
  __device__ __forceinline__ void add(const Sweep2Args &a, int w, double E,
                                      const double *dlog, double psi, double inv_block) {
    acc[kAccSumE] += E;
    acc[kAccSumE2] = fma(E, E, acc[kAccSumE2]);
    acc[kAccBlockSum] += E;
    if (++fill == a.block_size) {
      const double bm = acc[kAccBlockSum] * inv_block;
      acc[kAccSumBm] += bm;
      acc[kAccSumBm2] = fma(bm, bm, acc[kAccSumBm2]);
      acc[kAccBlockSum] = 0.0;
      fill = 0;
    }
    double O[kNParam2];
    if (a.o_conv == MOLE_O_REFERENCE) {
      // G = psi ./ (psi * dpsi), dpsi = psi dlog; O = G / psi_s with
      // psi_s = (psi*psi)/psi the "Wavefunction value" sample.  The empty asm
      // keeps these seven divisions behind the branch: without it they are
      // computed for every sample and selected away.
      asm volatile("");
      const double psi_s = (psi * psi) / psi;
#pragma unroll
      for (int k = 0; k < kNParam2; ++k) O[k] = (psi / (psi * (psi * dlog[k]))) / psi_s;
    } else {
#pragma unroll
      for (int k = 0; k < kNParam2; ++k) O[k] = dlog[k];
    }
    int t = 0;
#pragma unroll
    for (int k = 0; k < kNParam2; ++k) {
      acc[kAccSumO + k] += O[k];
      acc[kAccSumOE + k] = fma(O[k], E, acc[kAccSumOE + k]);
#pragma unroll
      for (int l = k; l < kNParam2; ++l, ++t)
        acc[kAccSumOO + t] = fma(O[k], O[l], acc[kAccSumOO + t]);
    }
    if (sample_idx < a.cap_samples) {
      const size_t si = (size_t)w * a.cap_samples + sample_idx;
      const double psi_s = (psi * psi) / psi;
      if (a.trace_e) a.trace_e[si] = E;
      if (a.samp_psi) a.samp_psi[si] = psi_s;
      if (a.samp_g)
#pragma unroll
        for (int k = 0; k < kNParam2; ++k) a.samp_g[si * kNParam2 + k] = O[k] * psi_s;
    }
    ++sample_idx;
  }
};

// One lane per walker, every stage in the same wave: the general path
// (any number of nuclei up to kMaxNuc2).
template <int KIND>
__global__ void __launch_bounds__(256) sweep2_lane_kernel(Sweep2Args a) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= a.W) return;
  Sys2 sp = a.sp;
  if (a.dparams) {  // parameters updated on the device between launches
    sp.zeta = a.dparams[0];
    sp.b = a.dparams[1];
    sp.c = a.dparams[2];
  }
  const int W = a.W;
  double x[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) x[k] = a.pos[(size_t)k * W + w];

  // cached pieces of psi at the current configuration
  double r1 = 0.0, r2 = 0.0, phi1 = 0.0, phi2 = 0.0;
  double r12 = norm3(x[0] - x[3], x[1] - x[4], x[2] - x[5]);
  double psi;
  if (KIND == MOLE_WF_HELIUM_PADE) {
    r1 = norm3(x[0] - sp.nuc[0][0], x[1] - sp.nuc[0][1], x[2] - sp.nuc[0][2]);
    r2 = norm3(x[3] - sp.nuc[0][0], x[4] - sp.nuc[0][1], x[5] - sp.nuc[0][2]);
    psi = exp_m(-sp.zeta * (r1 + r2) + pade(sp.b, sp.c, r12));
  } else {
    phi1 = lcao_phi(sp, x[0], x[1], x[2]);
    phi2 = lcao_phi(sp, x[3], x[4], x[5]);
    psi = (phi1 * phi2) * exp_m(pade(sp.b, sp.c, r12));
  }

  SampleAcc sa;
  sa.load(a, w);
  double accepted = a.fresh ? 0.0 : a.acc[(size_t)kAccAccepted * W + w];
  Stream rng;
  rng.init(a.seed, a.sys, (uint32_t)w, a.epoch);
  uint64_t p = a.draw0;
  const double inv_block = 1.0 / (double)a.block_size;

  for (uint32_t s = 0; s < a.n_sweeps; ++s) {
    uint64_t mask = 0;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const double dx = u64_range(rng.draw(p), a.scale, a.offset);
      const double dy = u64_range(rng.draw(p + 1), a.scale, a.offset);
      const double dz = u64_range(rng.draw(p + 2), a.scale, a.offset);
      const double u = u64_standard(rng.draw(p + 3));
      p += 4;
      const double nx = x[3 * e] + dx, ny = x[3 * e + 1] + dy, nz = x[3 * e + 2] + dz;
      const double n12 = (e == 0) ? norm3(nx - x[3], ny - x[4], nz - x[5])
                                  : norm3(x[0] - nx, x[1] - ny, x[2] - nz);
      double psin, nr = 0.0, nphi = 0.0;
      if (KIND == MOLE_WF_HELIUM_PADE) {
        nr = norm3(nx - sp.nuc[0][0], ny - sp.nuc[0][1], nz - sp.nuc[0][2]);
        const double s12 = (e == 0) ? (nr + r2) : (r1 + nr);
        psin = exp_m(-sp.zeta * s12 + pade(sp.b, sp.c, n12));
      } else {
        nphi = lcao_phi(sp, nx, ny, nz);
        const double jas = exp_m(pade(sp.b, sp.c, n12));
        psin = ((e == 0) ? (nphi * phi2) : (phi1 * nphi)) * jas;
      }
      const double ratio = min_one((psin * psin) / (psi * psi));
      if (ratio > u) {
        x[3 * e] = nx;
        x[3 * e + 1] = ny;
        x[3 * e + 2] = nz;
        r12 = n12;
        psi = psin;
        if (KIND == MOLE_WF_HELIUM_PADE) {
          if (e == 0) r1 = nr; else r2 = nr;
        } else {
          if (e == 0) phi1 = nphi; else phi2 = nphi;
        }
        accepted += 1.0;
        mask |= (uint64_t)1 << e;
      }
    }
    if (a.trace_mask && a.trace_sweep0 + s < a.cap_sweeps)
      a.trace_mask[(size_t)w * a.cap_sweeps + a.trace_sweep0 + s] = mask;
    if (s >= a.sample_start) {
      const Local2 L = local2<KIND>(sp, x);
      sa.add(a, w, L.e_local, L.dlog, psi, inv_block);
    }
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) a.pos[(size_t)k * W + w] = x[k];
  sa.store(a, w);
  a.acc[(size_t)kAccAccepted * W + w] = accepted;
}

// Local energy and d ln psi/dp from a configuration whose distances to the
// nuclei (and, for the LCAO kind, the orbital exponentials) are known.
template <int KIND, int NNUC>
__device__ __forceinline__ void local2_cached(const Sys2 &sp, const double *x,
                                              const double (*r)[NNUC],
                                              const double (*ee)[NNUC], double r12,
                                              double &E, double *dlog) {
  const double zeta = sp.zeta, b = sp.b, c = sp.c;
  double V = sp.v_nn;
  double gi[2][3], li[2], dz = 0.0;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    double phi = 0.0, gs0 = 0.0, gs1 = 0.0, gs2 = 0.0, ls = 0.0, zs = 0.0;
#pragma unroll
    for (int I = 0; I < NNUC; ++I) {
      const double d0 = x[3 * e] - sp.nuc[I][0], d1 = x[3 * e + 1] - sp.nuc[I][1],
                   d2 = x[3 * e + 2] - sp.nuc[I][2];
      const double inv = 1.0 / r[e][I];
      V = V - sp.charge[I] * inv;
      const double eI = (KIND == MOLE_WF_HELIUM_PADE) ? 1.0 : ee[e][I];
      phi += eI;
      const double f = -zeta * eI * inv;
      gs0 = fma(f, d0, gs0);
      gs1 = fma(f, d1, gs1);
      gs2 = fma(f, d2, gs2);
      ls = fma(eI, zeta * zeta - 2.0 * zeta * inv, ls);
      zs = fma(-r[e][I], eI, zs);
    }
    const double ip = 1.0 / phi;
    gi[e][0] = gs0 * ip;
    gi[e][1] = gs1 * ip;
    gi[e][2] = gs2 * ip;
    li[e] = ls * ip;
    dz += zs * ip;
  }
  const double d0 = x[0] - x[3], d1 = x[1] - x[4], d2 = x[2] - x[5];
  const double i12 = 1.0 / r12;
  const double iden = 1.0 / (1.0 + c * r12);
  const double up = b * iden * iden;
  const double upp = -2.0 * b * c * iden * iden * iden;
  const double J = upp + 2.0 * up * i12 + up * up;
  const double h0 = d0 * i12, h1 = d1 * i12, h2 = d2 * i12;
  const double gd1 = gi[0][0] * h0 + gi[0][1] * h1 + gi[0][2] * h2;
  const double gd2 = gi[1][0] * h0 + gi[1][1] * h1 + gi[1][2] * h2;
  const double k1 = li[0] + J + 2.0 * up * gd1;
  const double k2 = li[1] + J - 2.0 * up * gd2;
  if (sp.hamiltonian == MOLE_H_ELECTRONIC) V = V + i12;
  E = -0.5 * (k1 + k2) + V;
  dlog[0] = dz;
  dlog[1] = r12 * iden;
  dlog[2] = -b * r12 * r12 * iden * iden;
}

// Metropolis decision min(a / b, 1) > u (a = psi'^2, b = psi^2) without the
// division where its outcome is beyond rounding: t = a - u b is formed with
// one rounding, and with |t| > 2^-50 b the quotient differs from u by more
// than two units in u's last place (u < 1), so its rounding lies on the same
// side of u.  Close calls, NaN, an infinite b and b < 2^-900 are not `sure`: the
// caller then divides (accept_div), so every decision is the division's (an
// infinite a over a finite b accepts either way).
__device__ __forceinline__ bool accept_fast(double a, double b, double u, bool &sure) {
  const double t = fma(-u, b, a);
  sure = sure && fabs(t) > b * 0x1p-50 && b > 0x1p-900;
  return t > 0.0;
}
__device__ __forceinline__ bool accept_div(double a, double b, double u) { return min_one(a / b) > u; }

constexpr int kQuadXor1 = 0xB1;  // quad_perm [1, 0, 3, 2]
constexpr int kQuadLane0 = 0x00, kQuadLane1 = 0x55, kQuadLane2 = 0xAA;

// v of the lane the quad permutation CTRL names (two 32-bit DPP moves)
template <int CTRL>
__device__ __forceinline__ double quad_mov(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xF, 0xF, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Wave-specialised sweep.  A workgroup of G + 2 waves owns NW = 64 G / L
// walkers:
//   waves 0 .. G-1  the Metropolis chain, L lanes (2 or 4) per walker;
//   wave G          local energy, d ln psi/dp and accumulators of chunk c-1
//                   from snapshots the chain leaves, one lane per walker;
//   wave G + 1      Philox draws of chunk c+1 into LDS (S of every 4 draw
//                   pairs by the sampler wave, to even the two out).
// Chunks are T sweeps, double-buffered, one barrier per chunk.
//
// The chain is a serial sequence of FP64 operations; a wave issues one
// instruction per 4 cycles whatever its kind, so the chain's instruction
// count bounds every walker count that fits the chip at once, and it is
// spread over the lanes.  L = 4: lane q forms the trial position's distance
// and orbital exponential for electron q/2 and nucleus q%2, then one coupled
// part (r12', Jastrow, psi'): lane 0 electron 0's, lane 1 electron 1's if
// electron 0's move is rejected, lanes 2-3 if it is accepted.  L = 2: lane h
// forms electron h's local part for all nuclei, then electron 0's (lane 0) or
// the rejected electron 1's (lane 1) coupled part, and both lanes the accepted
// one.  DPP permutations exchange the results; the decisions and the selects
// of the state update run on all lanes alike.  Every value is the same
// operation on the same operands as in the one-lane kernel, so trajectories
// agree bit for bit.
constexpr int kPairEven = 0xA0;  // quad_perm [0, 0, 2, 2]
constexpr int kPairOdd = 0xF5;   // quad_perm [1, 1, 3, 3]

template <int KIND, int NNUC, int L, int G, int S, int T>
__global__ void __launch_bounds__(64 * (G + 2)) sweep2_ws_kernel(Sweep2Args a) {
  constexpr bool HE = KIND == MOLE_WF_HELIUM_PADE;
  constexpr int NW = 64 * G / L;
  static_assert(NW <= 64, "one sampler lane per walker");
  constexpr int NE = HE ? 0 : 2 * NNUC;        // orbital exponentials kept
  constexpr int SNAP = 6 + 2 * NNUC + NE + 1;  // x, r[e][I], ee[e][I], psi
  struct Lds {
    double rng[2][T][8][NW];
    double snap[2][T][SNAP][NW];
  };
  __shared__ Lds lds;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int w0 = blockIdx.x * NW;
  const int W = a.W;
  Sys2 sp = a.sp;
  if (a.dparams) {  // parameters updated on the device between launches
    sp.zeta = a.dparams[0];
    sp.b = a.dparams[1];
    sp.c = a.dparams[2];
  }
  const uint32_t nchunks = (a.n_sweeps + T - 1) / T;

  if (wave >= G) {
    // draws p .. p+7 of a sweep as (dx, dy, dz, u) per electron, in pairs (one
    // Philox block each when p is even); pairs [b0, b1) of every 4 here
    const uint32_t k0 = (uint32_t)a.seed, k1 = (uint32_t)(a.seed >> 32) ^ a.sys;
    const bool odd = (a.draw0 & 1) != 0;
    auto produce = [&](uint32_t cc, int b0, int nb) {
      const int nt = (int)min((uint32_t)T, a.n_sweeps - cc * T);
      for (int it = lane; it < nt * nb * NW; it += 64) {
        const int wl = it % NW, tb = it / NW;
        const int t = tb / nb, b = b0 + tb % nb;
        const uint64_t blk = ((a.draw0 + 8 * (uint64_t)(cc * T + t)) >> 1) + b;
        const uint32_t wg = (uint32_t)(w0 + wl);
        u32x4 o = philox4x32_10({(uint32_t)blk, (uint32_t)(blk >> 32), wg, a.epoch}, k0, k1);
        if (odd) {  // the pair straddles two blocks
          const u32x4 o2 = philox4x32_10({(uint32_t)(blk + 1), (uint32_t)((blk + 1) >> 32), wg, a.epoch}, k0, k1);
          o = {o.z, o.w, o2.x, o2.y};
        }
        const uint64_t v0 = (uint64_t)o.x | ((uint64_t)o.y << 32), v1 = (uint64_t)o.z | ((uint64_t)o.w << 32);
        double *d = &lds.rng[cc & 1][t][2 * b][wl];
        d[0] = u64_range(v0, a.scale, a.offset);
        d[NW] = (b & 1) ? u64_standard(v1) : u64_range(v1, a.scale, a.offset);
      }
    };
    if (wave > G) {
      if (nchunks > 0) produce(0, S, 4 - S);
      __syncthreads();
      for (uint32_t c = 0; c <= nchunks; ++c) {
        if (c + 1 < nchunks) produce(c + 1, S, 4 - S);
        __syncthreads();
      }
      return;
    }
    const int w = w0 + lane;
    const bool live = lane < NW && w < W;
    const int wl = lane < NW ? lane : 0;
    const double inv_block = 1.0 / (double)a.block_size;
    SampleAcc sa;
    if (live) sa.load(a, w);
    if constexpr (S > 0)
      if (nchunks > 0) produce(0, 0, S);
    __syncthreads();
    for (uint32_t c = 0; c <= nchunks; ++c) {
      if constexpr (S > 0)
        if (c + 1 < nchunks) produce(c + 1, 0, S);
      if (c >= 1) {
        const uint32_t p0 = (c - 1) * T;
        const int nt = (int)min((uint32_t)T, a.n_sweeps - p0);
#pragma unroll 1
        for (int t = a.sample_start > p0 ? (int)min((uint32_t)T, a.sample_start - p0) : 0; t < nt; ++t) {
          const double *sn = &lds.snap[(c - 1) & 1][t][0][wl];
          double xs[6], rs[2][NNUC], es[2][NNUC];
#pragma unroll
          for (int k = 0; k < 6; ++k) xs[k] = sn[k * NW];
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int I = 0; I < NNUC; ++I) {
              rs[e][I] = sn[(6 + e * NNUC + I) * NW];
              es[e][I] = HE ? 1.0 : sn[(6 + 2 * NNUC + e * NNUC + I) * NW];
            }
          const double psis = sn[(SNAP - 1) * NW];
          const double r12 = norm3(xs[0] - xs[3], xs[1] - xs[4], xs[2] - xs[5]);
          double E, dlog[kNParam2];
          local2_cached<KIND, NNUC>(sp, xs, rs, es, r12, E, dlog);
          if (live) sa.add(a, w, E, dlog, psis, inv_block);
        }
      }
      __syncthreads();
    }
    if (live) sa.store(a, w);
    return;
  }

  // ---- chain ----
  const int q = lane & (L - 1);
  const int wl = wave * (64 / L) + lane / L;
  const int w = w0 + wl;
  const bool live = w < W;
  const bool lead = q == 0;
  const bool me = L == 4 ? (q >> 1) != 0 : q != 0;      // this lane's electron is 1
  const bool c0 = q == 0, c1 = q == 1;
  constexpr int NL = L == 4 ? 1 : NNUC;                 // nuclei of this lane's local part
  const int I0 = (L == 4 && NNUC == 2) ? (q & 1) : 0;   // the first of them
  double R[NL][3];
#pragma unroll
  for (int I = 0; I < NL; ++I)
#pragma unroll
    for (int k = 0; k < 3; ++k) R[I][k] = (L == 4 && NNUC == 2 && I0) ? sp.nuc[NNUC - 1][k] : sp.nuc[I][k];
  ExpConst K;
  K.pin();
  const double nzeta = -sp.zeta;
  // the orbital value (LCAO) or nuclear distance (helium) of both electrons
  // from each lane's local parts
  auto exchange = [&](const double *rl, const double *el, double &f0, double &f1) {
    double fe = HE ? rl[0] : el[0];
    if constexpr (!HE && NNUC == 2) fe = fe + (L == 4 ? quad_mov<kQuadXor1>(el[0]) : el[NL - 1]);
    f0 = quad_mov<L == 4 ? kQuadLane0 : kPairEven>(fe);
    f1 = quad_mov<L == 4 ? kQuadLane2 : kPairOdd>(fe);
  };
  double x[6], rl[NL], el[NL], f[2];
#pragma unroll
  for (int k = 0; k < 6; ++k) x[k] = live ? a.pos[(size_t)k * W + w] : 0.0;
#pragma unroll
  for (int I = 0; I < NL; ++I) {
    rl[I] = norm3((me ? x[3] : x[0]) - R[I][0], (me ? x[4] : x[1]) - R[I][1], (me ? x[5] : x[2]) - R[I][2]);
    el[I] = HE ? 1.0 : exp_k(nzeta * rl[I], K);
  }
  exchange(rl, el, f[0], f[1]);
  double psi;
  {
    const double r12 = norm3(x[0] - x[3], x[1] - x[4], x[2] - x[5]);
    psi = HE ? exp_k(nzeta * (f[0] + f[1]) + pade(sp.b, sp.c, r12), K)
             : (f[0] * f[1]) * exp_k(pade(sp.b, sp.c, r12), K);
  }
  double psi2 = psi * psi;
  uint32_t n_acc = 0;
  __syncthreads();

  for (uint32_t c = 0; c <= nchunks; ++c) {
    const uint32_t s0 = c * T;
    const int nt = c < nchunks ? (int)min((uint32_t)T, a.n_sweeps - s0) : 0;
#pragma unroll 1
    for (int t = 0; t < nt; ++t) {
      // the sweep's eight draws together, ahead of the arithmetic
      double d[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) d[k] = lds.rng[c & 1][t][k][wl];
      double n[6];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        n[k] = x[k] + d[k];
        n[3 + k] = x[3 + k] + d[4 + k];
      }
      double nr[NL], ne[NL], nf0, nf1;
      double p0, pr, pa;  // psi' of electron 0's move, and of electron 1's after its rejection / acceptance
      double smin;        // the smallest square root argument
      // FAST leaves out sqrt's range handling; its results stand if every
      // argument is in sqrt_normal's range and every decision is sure (an
      // infinity, zero or NaN under a root makes psi' NaN, which is not)
      auto evaluate = [&](auto fast) {
        constexpr bool FAST = decltype(fast)::value;
        auto root = [&](double v0, double v1, double v2) {
          const double ss = sumsq3(v0, v1, v2);
          if constexpr (FAST) {
            smin = fmin(smin, ss);
            return sqrt_normal(ss);
          } else {
            return sqrt(ss);
          }
        };
        smin = 1.0;
#pragma unroll
        for (int I = 0; I < NL; ++I) {
          nr[I] = root(sel(me, n[3], n[0]) - R[I][0], sel(me, n[4], n[1]) - R[I][1], sel(me, n[5], n[2]) - R[I][2]);
          ne[I] = HE ? 1.0 : exp_k(nzeta * nr[I], K);
        }
        exchange(nr, ne, nf0, nf1);
        auto coupled = [&](const double *A, const double *B, double fa, double fb) {
          const double J = pade(sp.b, sp.c, root(A[0] - B[0], A[1] - B[1], A[2] - B[2]));
          if constexpr (HE) return exp_k(nzeta * (fa + fb) + J, K);
          else return (fa * fb) * exp_k(J, K);
        };
        const bool ko = L == 4 ? c1 : me, kn = L == 4 ? c0 : !me;  // electron 0 / 1 stays put
        double A[3], B[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          A[k] = sel(ko, x[k], n[k]);
          B[k] = sel(kn, x[3 + k], n[3 + k]);
        }
        const double pc = coupled(A, B, sel(ko, f[0], nf0), sel(kn, f[1], nf1));
        if constexpr (L == 4) {
          p0 = quad_mov<kQuadLane0>(pc);
          pr = quad_mov<kQuadLane1>(pc);
          pa = quad_mov<kQuadLane2>(pc);
        } else {
          p0 = quad_mov<kPairEven>(pc);
          pr = quad_mov<kPairOdd>(pc);
          pa = coupled(n, n + 3, nf0, nf1);
        }
      };
      evaluate(std::true_type{});
      double p02 = p0 * p0, pr2 = pr * pr, pa2 = pa * pa;
      bool sure = smin >= 0x1p-767;
      bool acc0 = accept_fast(p02, psi2, d[3], sure);
      bool acc1r = accept_fast(pr2, psi2, d[7], sure);
      bool acc1a = accept_fast(pa2, p02, d[7], sure);
      if (__builtin_expect(__any(!sure), 0)) {
        evaluate(std::false_type{});
        p02 = p0 * p0;
        pr2 = pr * pr;
        pa2 = pa * pa;
        acc0 = accept_div(p02, psi2, d[3]);
        acc1r = accept_div(pr2, psi2, d[7]);
        acc1a = accept_div(pa2, p02, d[7]);
      }
      const bool acc1 = acc0 ? acc1a : acc1r;
      const bool mine = me ? acc1 : acc0;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        x[k] = sel(acc0, n[k], x[k]);
        x[3 + k] = sel(acc1, n[3 + k], x[3 + k]);
      }
      f[0] = sel(acc0, nf0, f[0]);
      f[1] = sel(acc1, nf1, f[1]);
#pragma unroll
      for (int I = 0; I < NL; ++I) {
        rl[I] = sel(mine, nr[I], rl[I]);
        if constexpr (!HE) el[I] = sel(mine, ne[I], el[I]);
      }
      psi = sel(acc1, sel(acc0, pa, pr), sel(acc0, p0, psi));
      psi2 = psi * psi;
      n_acc += (acc0 ? 1u : 0u) + (acc1 ? 1u : 0u);
      if (a.trace_mask) {
        const uint32_t s = s0 + t;
        if (live && lead && a.trace_sweep0 + s < a.cap_sweeps)
          a.trace_mask[(size_t)w * a.cap_sweeps + a.trace_sweep0 + s] = (acc0 ? 1ull : 0ull) | (acc1 ? 2ull : 0ull);
      }
      double *sn = &lds.snap[c & 1][t][0][wl];
      if (lead) {
#pragma unroll
        for (int k = 0; k < 6; ++k) sn[k * NW] = x[k];
        sn[(SNAP - 1) * NW] = psi;
      }
      // (with one nucleus both lanes of a quad's pair write the same value)
      const int ri = (me ? NNUC : 0) + I0;
#pragma unroll
      for (int I = 0; I < NL; ++I) {
        sn[(6 + ri + I) * NW] = rl[I];
        if constexpr (!HE) sn[(6 + 2 * NNUC + ri + I) * NW] = el[I];
      }
    }
    __syncthreads();
  }
  if (live && lead) {
#pragma unroll
    for (int k = 0; k < 6; ++k) a.pos[(size_t)k * W + w] = x[k];
    a.acc[(size_t)kAccAccepted * W + w] = (a.fresh ? 0.0 : a.acc[(size_t)kAccAccepted * W + w]) + (double)n_acc;
  }
}

// One lane per walker, every stage in the same wave, the distances and
// orbital exponentials of the walker kept in registers: for walker counts
// that fill every SIMD with walkers of its own, where the total of issued
// instructions bounds the sweep and the pair's duplicated ones cost more than
// its shorter chain gains.  262,144 walkers of H2: 19.6 -> 6.23 us per sweep
// (the wave-specialised kernel's LDS let one workgroup on a CU).
template <int KIND, int NNUC>
__global__ void __launch_bounds__(256, 2) sweep2_wide_kernel(Sweep2Args a) {
  constexpr bool HE = KIND == MOLE_WF_HELIUM_PADE;
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = w < a.W;
  if (!live) return;
  Sys2 sp = a.sp;
  if (a.dparams) {  // parameters updated on the device between launches
    sp.zeta = a.dparams[0];
    sp.b = a.dparams[1];
    sp.c = a.dparams[2];
  }
  const int W = a.W;
  double x[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) x[k] = a.pos[(size_t)k * W + w];
  double r[2][NNUC], ee[2][NNUC], f[2];
#pragma unroll
  for (int e = 0; e < 2; ++e)
#pragma unroll
    for (int I = 0; I < NNUC; ++I) {
      r[e][I] = norm3(x[3 * e] - sp.nuc[I][0], x[3 * e + 1] - sp.nuc[I][1], x[3 * e + 2] - sp.nuc[I][2]);
      ee[e][I] = HE ? 1.0 : exp_m(-sp.zeta * r[e][I]);
      const double fI = HE ? r[e][I] : ee[e][I];
      f[e] = (I == 0) ? fI : f[e] + fI;
    }
  double r12 = norm3(x[0] - x[3], x[1] - x[4], x[2] - x[5]);
  double psi = HE ? exp_m(-sp.zeta * (f[0] + f[1]) + pade(sp.b, sp.c, r12)) : (f[0] * f[1]) * exp_m(pade(sp.b, sp.c, r12));
  ExpConst K;
  K.pin();
  SampleAcc sa;
  sa.load(a, w);
  uint32_t n_acc = 0;
  Stream rng;
  rng.init(a.seed, a.sys, (uint32_t)w, a.epoch);
  uint64_t p = a.draw0;
  const double inv_block = 1.0 / (double)a.block_size;
  for (uint32_t s = 0; s < a.n_sweeps; ++s) {
    uint64_t mask = 0;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      double n[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) n[k] = x[3 * e + k] + u64_range(rng.draw(p + k), a.scale, a.offset);
      const double u = u64_standard(rng.draw(p + 3));
      p += 4;
      double nr[NNUC], ne[NNUC], nf, n12, psin, smin;
      auto evaluate = [&](auto fast) {  // as in sweep2_ws_kernel
        constexpr bool FAST = decltype(fast)::value;
        smin = 1.0;
        auto root = [&](double v0, double v1, double v2) {
          const double ss = sumsq3(v0, v1, v2);
          if constexpr (FAST) {
            smin = fmin(smin, ss);
            return sqrt_normal(ss);
          } else {
            return sqrt(ss);
          }
        };
#pragma unroll
        for (int I = 0; I < NNUC; ++I) {
          nr[I] = root(n[0] - sp.nuc[I][0], n[1] - sp.nuc[I][1], n[2] - sp.nuc[I][2]);
          ne[I] = HE ? 1.0 : exp_k(-sp.zeta * nr[I], K);
          const double fI = HE ? nr[I] : ne[I];
          nf = (I == 0) ? fI : nf + fI;
        }
        n12 = (e == 0) ? root(n[0] - x[3], n[1] - x[4], n[2] - x[5]) : root(x[0] - n[0], x[1] - n[1], x[2] - n[2]);
        const double fa = e == 0 ? nf : f[0], fb = e == 0 ? f[1] : nf;
        const double J = pade(sp.b, sp.c, n12);
        psin = HE ? exp_k(-sp.zeta * (fa + fb) + J, K) : (fa * fb) * exp_k(J, K);
      };
      evaluate(std::true_type{});
      double pn2 = psin * psin;
      const double ps2 = psi * psi;
      bool sure = smin >= 0x1p-767;
      bool acc = accept_fast(pn2, ps2, u, sure);
      if (__builtin_expect(__any(!sure), 0)) {
        evaluate(std::false_type{});
        pn2 = psin * psin;
        acc = accept_div(pn2, ps2, u);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) x[3 * e + k] = sel(acc, n[k], x[3 * e + k]);
#pragma unroll
      for (int I = 0; I < NNUC; ++I) {
        r[e][I] = sel(acc, nr[I], r[e][I]);
        if constexpr (!HE) ee[e][I] = sel(acc, ne[I], ee[e][I]);
      }
      f[e] = sel(acc, nf, f[e]);
      r12 = sel(acc, n12, r12);
      psi = sel(acc, psin, psi);
      n_acc += acc ? 1u : 0u;
      mask |= acc ? ((uint64_t)1 << e) : 0;
    }
    if (a.trace_mask && a.trace_sweep0 + s < a.cap_sweeps)
      a.trace_mask[(size_t)w * a.cap_sweeps + a.trace_sweep0 + s] = mask;
    if (s >= a.sample_start) {
      double E, dlog[kNParam2];
      local2_cached<KIND, NNUC>(sp, x, r, ee, r12, E, dlog);
      sa.add(a, w, E, dlog, psi, inv_block);
    }
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) a.pos[(size_t)k * W + w] = x[k];
  sa.store(a, w);
  a.acc[(size_t)kAccAccepted * W + w] = (a.fresh ? 0.0 : a.acc[(size_t)kAccAccepted * W + w]) + (double)n_acc;
}

__global__ void init2_kernel(double *pos, int W, uint64_t seed, uint32_t sys,
                             uint32_t epoch) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= W) return;
  Stream rng;
  rng.init(seed, sys, (uint32_t)w, epoch);
  // Range(-1, 1): scale 2, offset -1 - 2
#pragma unroll
  for (int k = 0; k < 6; ++k) pos[(size_t)k * W + w] = u64_range(rng.draw(k), 2.0, -3.0);
}

template <int KIND>
__global__ void eval2_kernel(Eval2Args a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  double x[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) x[k] = a.cfg[i * 6 + k];
  const double psi = value2<KIND>(a.sp, x);
  const Local2 L = local2<KIND>(a.sp, x);
  if (a.value) a.value[i] = psi;
  if (a.grad)
    for (int k = 0; k < 6; ++k) a.grad[i * 6 + k] = psi * L.g[k];
  if (a.lap) a.lap[i] = psi * L.lap_ratio;
  if (a.e_local) a.e_local[i] = L.e_local;
  if (a.pgrad)
    for (int k = 0; k < kNParam2; ++k) a.pgrad[i * kNParam2 + k] = psi * L.dlog[k];
}

// Column sums of a [K][W] array, one workgroup per column, fixed order.
// Column max_col, if in range, is reduced with max instead of +.
__global__ void __launch_bounds__(256) reduce_columns_kernel(const double *acc, int W,
                                                             double *out, int max_first, int max_count) {
  __shared__ double sh[256];
  const int col = blockIdx.x;
  const bool mx = col >= max_first && col < max_first + max_count;
  const double *p = acc + (size_t)col * W;
  double s = 0.0;
  // loads in batches of 16 (all in flight together), added in index order
  int i = threadIdx.x;
  for (; i + 15 * 256 < W; i += 16 * 256) {
    double v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = p[i + q * 256];
#pragma unroll
    for (int q = 0; q < 16; ++q) s = mx ? fmax(s, v[q]) : s + v[q];
  }
  for (; i < W; i += 256) s = mx ? fmax(s, p[i]) : s + p[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off)
      sh[threadIdx.x] = mx ? fmax(sh[threadIdx.x], sh[threadIdx.x + off]) : sh[threadIdx.x] + sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[col] = sh[0];
}

// One workgroup per block: per walker the block's samples summed in order
// times 1/B, then summed over walkers (strided per thread, LDS tree).
__global__ void __launch_bounds__(256) block_records_kernel(const double *trace_e, int W, size_t cap, size_t B,
                                                            size_t first, double *out) {
  __shared__ double s1[256], s2[256];
  const size_t b = first + blockIdx.x;
  const double inv = 1.0 / (double)B;
  double a1 = 0.0, a2 = 0.0;
  for (int w = threadIdx.x; w < W; w += 256) {
    const double *e = trace_e + (size_t)w * cap + b * B;
    double s = 0.0;
    for (size_t k = 0; k < B; ++k) s += e[k];
    const double bm = s * inv;
    a1 += bm;
    a2 = fma(bm, bm, a2);
  }
  s1[threadIdx.x] = a1;
  s2[threadIdx.x] = a2;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      s1[threadIdx.x] += s1[threadIdx.x + off];
      s2[threadIdx.x] += s2[threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = s1[0];
    out[2 * blockIdx.x + 1] = s2[0];
  }
}

// Transposition between columns [D][W] and rows [n][D] of walkers w0 .. w0+n-1
// through a 64 x 32 LDS tile: 512-byte runs of a column, 256-byte runs of a
// row.  The row side is usually pinned host memory, whose link bounds it.
template <bool TO_ROWS>
__global__ void __launch_bounds__(256) transpose_kernel(double *cols, size_t W, int D, size_t w0, size_t n,
                                                        double *rows) {
  __shared__ double tile[32][65];
  const size_t r0 = (size_t)blockIdx.x * 64;
  const int k0 = (int)blockIdx.y * 32;
  auto by_column = [&](auto f) {  // consecutive lanes on consecutive walkers
    const size_t r = r0 + (threadIdx.x & 63);
    for (int k = (int)(threadIdx.x >> 6); k < 32; k += 4)
      if (r < n && k0 + k < D) f(cols[(size_t)(k0 + k) * W + w0 + r], tile[k][threadIdx.x & 63]);
  };
  auto by_row = [&](auto f) {  // consecutive lanes on consecutive columns
    const int k = (int)(threadIdx.x & 31);
    for (int q = (int)(threadIdx.x >> 5); q < 64; q += 8)
      if (r0 + q < n && k0 + k < D) f(rows[(r0 + q) * (size_t)D + k0 + k], tile[k][q]);
  };
  if constexpr (TO_ROWS) {
    by_column([](double &g, double &t) { t = g; });
    __syncthreads();
    by_row([](double &g, double &t) { g = t; });
  } else {
    by_row([](double &g, double &t) { t = g; });
    __syncthreads();
    by_column([](double &g, double &t) { g = t; });
  }
}

__global__ void fill_kernel(double *p, size_t n, double v) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

bool sweep2_wavespec_eligible(const Sys2 &sp) {
  return (sp.kind == MOLE_WF_HELIUM_PADE) ? sp.n_nuc == 1 : sp.n_nuc <= 2;
}

namespace {
template <int KIND, int NNUC, int L, int G, int S, int T>
void launch_ws(const Sweep2Args &a, hipStream_t stream) {
  constexpr int NW = 64 * G / L;
  hipLaunchKernelGGL((sweep2_ws_kernel<KIND, NNUC, L, G, S, T>), dim3((unsigned)((a.W + NW - 1) / NW)),
                     dim3(64 * (G + 2)), 0, stream, a);
}

template <int KIND, int NNUC>
void launch_spec(const Sweep2Args &a, int variant, int bt, int cus, hipStream_t stream) {
  // us per sweep on 256 CUs, helium / H2 (single: the pair kernel's predecessor,
  // one lane per walker in the chain wave):
  //   W         quad, 32/wg   pair, 64/wg   pair, T = 2   wide          single
  //   8,192     0.60 / 0.70   0.69 / 0.85   0.75 / 0.87   1.37 / 1.87   0.80 / 1.24
  //   16,384    0.89 / 1.11   0.71 / 0.86   0.77 / 0.87   1.38 / 1.90   0.83 / 1.26
  //   32,768    1.43 / 2.02   1.08 / 1.71   1.12 / 1.40   1.39 / 1.90   1.59 / 2.45
  //   49,152    2.08 / 2.92   1.62 / 2.61   1.55 / 2.02   1.37 / 1.86   -
  //   262,144   10.1 / 14.5   7.86 / 13.8   6.90 / 9.42   4.40 / 6.23   12.6 / 19.6
  // Up to 32 walkers per CU the quad's shorter chain wins; up to 64 the pair
  // keeps one wave on each SIMD; up to 128 two pair workgroups share a CU if
  // their LDS is small (T = 2); beyond that every SIMD has walkers of its own
  // and the fewest instructions per walker win.
  const int64_t per_cu = ((int64_t)a.W + cus - 1) / cus;
  if (variant == MOLE_VARIANT_LANE || (variant == MOLE_VARIANT_AUTO && per_cu > 128))
    hipLaunchKernelGGL((sweep2_wide_kernel<KIND, NNUC>), dim3((a.W + bt - 1) / bt), dim3(bt), 0, stream, a);
  else if (variant == MOLE_VARIANT_QUAD || (variant == MOLE_VARIANT_AUTO && per_cu <= 32))
    launch_ws<KIND, NNUC, 4, 2, 0, 4>(a, stream);
  else if (variant == MOLE_VARIANT_WAVESPEC || per_cu <= 64)
    launch_ws<KIND, NNUC, 2, 2, 1, 4>(a, stream);
  else
    launch_ws<KIND, NNUC, 2, 2, 1, 2>(a, stream);
}
}  // namespace

hipError_t launch_sweep2(const Sweep2Args &a, int variant, int block_threads, int cus, hipStream_t stream) {
  const bool he = a.sp.kind == MOLE_WF_HELIUM_PADE;
  const int bt = block_threads ? block_threads : 64;
  if (sweep2_wavespec_eligible(a.sp)) {
    if (he)
      launch_spec<MOLE_WF_HELIUM_PADE, 1>(a, variant, bt, cus, stream);
    else if (a.sp.n_nuc == 1)
      launch_spec<MOLE_WF_LCAO2_PADE, 1>(a, variant, bt, cus, stream);
    else
      launch_spec<MOLE_WF_LCAO2_PADE, 2>(a, variant, bt, cus, stream);
    return hipGetLastError();
  }
  const dim3 grid((a.W + bt - 1) / bt);
  if (he)
    hipLaunchKernelGGL((sweep2_lane_kernel<MOLE_WF_HELIUM_PADE>), grid, dim3(bt), 0, stream, a);
  else
    hipLaunchKernelGGL((sweep2_lane_kernel<MOLE_WF_LCAO2_PADE>), grid, dim3(bt), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_init2(double *pos, int W, uint64_t seed, uint32_t sys, uint32_t epoch,
                        hipStream_t stream) {
  hipLaunchKernelGGL(init2_kernel, dim3((W + 255) / 256), dim3(256), 0, stream, pos, W, seed, sys,
                     epoch);
  return hipGetLastError();
}

hipError_t launch_eval2(const Eval2Args &a, hipStream_t stream) {
  const dim3 grid((unsigned)((a.n + 127) / 128));
  if (a.sp.kind == MOLE_WF_HELIUM_PADE)
    hipLaunchKernelGGL((eval2_kernel<MOLE_WF_HELIUM_PADE>), grid, dim3(128), 0, stream, a);
  else
    hipLaunchKernelGGL((eval2_kernel<MOLE_WF_LCAO2_PADE>), grid, dim3(128), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_reduce_columns(const double *acc, int W, int K, double *out, int max_first, int max_count,
                                 hipStream_t stream) {
  hipLaunchKernelGGL(reduce_columns_kernel, dim3(K), dim3(256), 0, stream, acc, W, out, max_first, max_count);
  return hipGetLastError();
}

hipError_t launch_columns_to_rows(const double *cols, size_t W, int D, size_t w0, size_t n, double *rows,
                                  hipStream_t stream) {
  hipLaunchKernelGGL(transpose_kernel<true>, dim3((unsigned)((n + 63) / 64), (unsigned)((D + 31) / 32)), dim3(256), 0,
                     stream, const_cast<double *>(cols), W, D, w0, n, rows);
  return hipGetLastError();
}

hipError_t launch_rows_to_columns(const double *rows, size_t W, int D, size_t w0, size_t n, double *cols,
                                  hipStream_t stream) {
  hipLaunchKernelGGL(transpose_kernel<false>, dim3((unsigned)((n + 63) / 64), (unsigned)((D + 31) / 32)), dim3(256), 0,
                     stream, cols, W, D, w0, n, const_cast<double *>(rows));
  return hipGetLastError();
}

hipError_t launch_fill(double *p, size_t n, double v, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, p, n, v);
  return hipGetLastError();
}

namespace {
__global__ void vmc_step_kernel(const double *red, double n_samples, double *params, mole_optimizer *opt,
                                double *log) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  constexpr int np = kNParam2;
  double so[np], soe[np], soo[np * np], dp[np], pars[np];
  int t = 0;
  for (int k = 0; k < np; ++k) {
    so[k] = red[kAccSumO + k];
    soe[k] = red[kAccSumOE + k];
    pars[k] = params[k];
    for (int l = k; l < np; ++l, ++t) {
      soo[k * np + l] = red[kAccSumOO + t];
      soo[l * np + k] = red[kAccSumOO + t];
    }
  }
  // the parameter count is fixed here (mole_optimize_with checks opt->n_params)
  const int rc = optimizer_update<np>(opt, n_samples, red[kAccSumE], so, soe, soo, pars, dp, nullptr);
  log[0] = red[kAccSumE];
  log[1] = red[kAccSumE2];
  log[2] = red[kAccSumBm];
  log[3] = red[kAccSumBm2];
  log[4] = red[kAccAccepted];
  log[5] = (double)rc;
  log[6] = n_samples;
  log[7] = 0.0;
  if (rc == 0)
    for (int k = 0; k < np; ++k) params[k] = pars[k] + dp[k];
}
}  // namespace

hipError_t launch_block_records(const double *trace_e, int W, size_t cap, size_t B, size_t first, size_t k,
                                double *out, hipStream_t stream) {
  hipLaunchKernelGGL(block_records_kernel, dim3((unsigned)k), dim3(256), 0, stream, trace_e, W, cap, B, first, out);
  return hipGetLastError();
}

hipError_t launch_vmc_step(const double *red, double n_samples, double *params, mole_optimizer *opt, double *log,
                           hipStream_t stream) {
  hipLaunchKernelGGL(vmc_step_kernel, dim3(1), dim3(64), 0, stream, red, n_samples, params, opt, log);
  return hipGetLastError();
}

}  // namespace mole
