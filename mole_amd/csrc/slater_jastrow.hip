// Slater-Jastrow walker kernel: single-electron box moves with
// Sherman-Morrison determinant ratios and updates, periodic Gauss-Jordan
// re-inversion in FP64, and the local energy after sampled sweeps.
//
// A workgroup is one wave.  It owns 64/L walkers of one system (a tile);
// the L lanes of a walker split the parallel stages of a move -- Jastrow terms
// over electrons and nuclei, basis functions, orbitals, Sherman-Morrison
// columns and rows -- and a walker's positions, inverse Slater matrices and
// stage arrays live in LDS for the whole launch, read from and written to HBM
// once.  Every sum is formed in a fixed sequential order, so results do not
// depend on L and equal those of a sequential evaluation bit for bit.
//
// What bounds the kernel is the number of instructions a wave issues: a stage
// costs the same whether one or all of a walker's lanes take part.  So the
// serial parts (sums, decision) run on all lanes alike, which needs no
// broadcast; stages that need no exchange share a phase; and the LDS a walker
// holds is kept small (stage arrays, re-inversion and local-energy scratch
// overlap; counters and determinants in registers; sample sums in HBM), so
// that few lanes per walker still leave two waves per SIMD.
//
// Math (per move of electron i of spin s, column c; B = A_s^-1 with
// A_s[c][k] = phi_k(r_c)):
//   ratio  R_D = sum_k phi_k(r') B[k][c]
//   dJ     = J_i(r') - J_i(r_i),  J_i = sum_{j != i} u_ij + sum_I v_I
//   accept min(R_D^2 exp(2 dJ), 1) > U           (metrop.rs:73-82)
//   update B[k][l] -= B[k][c] f_l (l != c), B[k][c] /= R_D,
//          f_l = (sum_k phi_k(r') B[k][l]) / R_D  (Sherman-Morrison)
#include "../../include/mole_gpu.h"
#include "basis.hpp"
#include "device_common.hpp"
#include "mlp.hpp"
#include "sj_internal.hpp"
#include "sr_math.hpp"

#include <type_traits>

namespace mole {

// LDS layout (bytes); identical on host and device.  Per walker:
//   pos | B | draws of the sweep | scratch
// scratch: the stage arrays of a move, or a Gauss-Jordan re-inversion; the
// local energy's per-electron results take the draws and the scratch together
// (no draw is pending after a sweep).  Per workgroup, ahead of the walkers:
// SJShared.
struct SJLayout {
  uint32_t pos, B, rng, scr, mv, chi, phin, jn, jo, dots, gch, og, jg, le, bytes;
  __host__ __device__ SJLayout(int N, int nu, int nd, int nn, int K, int tsize, int np, int prop) {
    const uint32_t n = nu > nd ? nu : nd, M = N + nn;
    auto up = [](uint32_t x) { return (x + 7u) & ~7u; };
    pos = 0;
    B = pos + 24u * N;
    rng = B + up((uint32_t)tsize * (nu * nu + nd * nd));
    scr = rng + 32u * N;
    // a move's stages
    mv = scr;  // proposed position and drift (Gaussian proposals)
    chi = mv + (prop == kSJPropBox ? 0u : 64u);
    phin = chi + 8u * K;
    jn = phin + up(tsize * n);
    jo = jn + up(tsize * M);
    dots = jo + up(tsize * M);
    gch = dots + up(tsize * n);
    og = gch + (prop == kSJPropDiffuse ? 24u * K : 0u);
    jg = og + (prop == kSJPropDiffuse ? 24u * n : 0u);
    uint32_t end = jg + (prop == kSJPropDiffuse ? 24u * M : 0u);
    // Gauss-Jordan: A, then I (the basis values while A is built)
    const uint32_t second = n * n > (uint32_t)K ? n * n : (uint32_t)K;
    const uint32_t lu = scr + 8u * (n * n + second);
    end = end > lu ? end : lu;
    // per-electron local-energy results, then (1, E, d ln psi/dp)
    le = rng;
    const uint32_t el = le + 8u * ((3u + (uint32_t)np) * N + 8u);
    end = end > el ? end : el;
    // the walkers of a tile sit bytes apart; an odd number of 8-byte words
    // puts the same field of consecutive walkers in different LDS banks
    // (an even count maps many walkers of a wave onto one bank)
    bytes = ((end / 8u) % 2u == 0u) ? end + 8u : end;
  }
};

// (a, b) of sample sum q, packed a | b << 4: the sum gains v[a] v[b] with v =
// (1, E, O_0 .. O_np-1); q = 0, 1 are columns kSJSumE, kSJSumE2, the rest
// follow from kSJSumO on (O, O E, upper triangle of O O^T).
__host__ __device__ constexpr int sj_sample_sums(int np) { return 2 + 2 * np + np * (np + 1) / 2; }
constexpr uint32_t kSJPairBytes = (sj_sample_sums(kSJNParam) + 7) / 8 * 8;

// What the walkers of a workgroup share, at the start of its LDS: the factor
// pairs, the nuclei (x, y, z, -a Z), and -- where they are small -- the basis
// functions (centre x, y, z, exponent, kind) and the orbital coefficients,
// which the lanes of a move read by function and by orbital.  From HBM each of
// these reads is a dependent chain (centre index, then coordinates) of cache
// latencies that two waves per SIMD do not hide (3-4 % of the atoms' sweeps).
// Larger tables cost resident workgroups instead: with up to 128 functions
// staged, a 36-electron molecule of 39 functions went from eight to seven a CU
// and 8,192 walkers of it from 1,066 to 1,487 us per sweep.
constexpr int kSJTabBasis = 8;         // functions
constexpr uint32_t kSJTabCoef = 512;  // bytes
struct SJShared {
  uint32_t nuc, fn, coef, bytes;
  bool has_fn, has_coef;
  __host__ __device__ SJShared(int nn, int K, int n_orb) {
    has_fn = K <= kSJTabBasis;
    has_coef = 8u * (uint32_t)K * (uint32_t)n_orb <= kSJTabCoef;
    nuc = kSJPairBytes;
    fn = nuc + 32u * (uint32_t)nn;
    coef = fn + (has_fn ? 40u * (uint32_t)K : 0u);
    bytes = coef + (has_coef ? 8u * (uint32_t)K * (uint32_t)n_orb : 0u);
  }
};

__host__ size_t sj_lds_per_walker(int N, int nu, int nd, int nn, int K, int tsize, int np, int prop) {
  return SJLayout(N, nu, nd, nn, K, tsize, np, prop).bytes;
}
__host__ size_t sj_lds_per_group(int nn, int K, int n_orb) { return SJShared(nn, K, n_orb).bytes; }

namespace {

// Orders LDS accesses of a one-wave workgroup: the wave's LDS operations
// execute in program order, so only the compiler has to keep it.
__device__ __forceinline__ void sync_wave() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <typename T>
struct SJWalker {
  double *pos, *rng, *scr, *chi, *mv, *le;
  T *Bup, *Bdn, *phin, *jn, *jo, *dots;
};

// Jastrow term num r/(1 + c r) of the points x and q, r = |x - q| (T
// precision): electron pairs with num = b, nuclei with num = -a Z, c = d.
template <typename T>
__device__ __forceinline__ T jastrow_term(T num, T c, const double *x, const double *q);
template <>
__device__ __forceinline__ double jastrow_term<double>(double num, double c, const double *x, const double *q) {
  const double r = norm3(x[0] - q[0], x[1] - q[1], x[2] - q[2]);
  return (num * r) / (1.0 + c * r);
}
template <>
__device__ __forceinline__ float jastrow_term<float>(float num, float c, const double *x, const double *q) {
  const float d0 = (float)(x[0] - q[0]), d1 = (float)(x[1] - q[1]), d2 = (float)(x[2] - q[2]);
  float s = d0 * d0;
  s = s + d1 * d1;
  s = s + d2 * d2;
  const float r = sqrtf(s);
  return (num * r) / (1.0f + c * r);
}

__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return fmaf(a, b, c); }

// e / n for 0 <= e < 4096, 1 <= n <= 64 via a float reciprocal: (e + 1/2)/n
// lies at least 1/(2n) from an integer, far beyond the rounding error.
__device__ __forceinline__ int small_div(int e, float inv_n) { return (int)(((float)e + 0.5f) * inv_n); }

// The workgroup's shared tables (LDS).
struct SJTab {
  const double *nuc, *fn, *coef;
  bool has_fn, has_coef;
};

// A basis function at the point r: displacement, distance, exponent, kind.
struct SJFn {
  double d0, d1, d2, r, z;
  int kind;
};
__device__ __forceinline__ SJFn basis_at(const SJSysDev &S, const SJTab &tab, int m, const double *r) {
  SJFn f;
  double R0, R1, R2;
  if (tab.has_fn) {
    const double *e = tab.fn + 5 * m;
    R0 = e[0];
    R1 = e[1];
    R2 = e[2];
    f.z = e[3];
    f.kind = __double2loint(e[4]);
  } else {
    const double *R = tab.nuc + 4 * S.center[m];
    R0 = R[0];
    R1 = R[1];
    R2 = R[2];
    f.z = S.zeta[m];
    f.kind = S.kind[m];
  }
  f.d0 = r[0] - R0;
  f.d1 = r[1] - R1;
  f.d2 = r[2] - R2;
  f.r = norm3(f.d0, f.d1, f.d2);
  return f;
}

// Basis values chi[m] of the point r into LDS (lanes over basis functions, each
// with its own centre's distance).  gto/pk: Gaussians / p-type STOs may occur
// (otherwise every function is an s-type STO).  No barrier.
__device__ __forceinline__ void basis_to_lds(const SJSysDev &S, const SJTab &tab, const double *r, double *chi, int t,
                                             int L, bool gto, bool pk) {
#pragma unroll 1
  for (int m = t; m < S.n_basis; m += L) {
    const SJFn f = basis_at(S, tab, m, r);
    chi[m] = (gto || pk) ? basis_value<true>(f.kind, f.z, f.d0, f.d1, f.d2, f.r) : exp_m(-f.z * f.r);
  }
}

// The same with the gradients gch[3m + q] (the drift-diffusion proposal, FP64;
// metrop.rs:153-155): the value and the gradient share the exponential.
__device__ __forceinline__ void basis_gradients_to_lds(const SJSysDev &S, const SJTab &tab, const double *r,
                                                       double *chi, double *gch, int t, int L) {
#pragma unroll 1
  for (int m = t; m < S.n_basis; m += L) {
    const SJFn f = basis_at(S, tab, m, r);
    double v, g0, g1, g2, l;
    basis_vgl<true>(f.kind, f.z, f.d0, f.d1, f.d2, f.r, v, g0, g1, g2, l);
    chi[m] = v;
    gch[3 * m] = g0;
    gch[3 * m + 1] = g1;
    gch[3 * m + 2] = g2;
  }
}

// Sequential sums whose loads are issued ahead of the arithmetic, eight bytes
// at a time (x is 8-byte aligned): the same operations in the same order as a
// plain loop.
__device__ __forceinline__ double seq_sum(const double *x, int n) {
  double s = 0.0;
  int j = 0;
  for (; j + 4 <= n; j += 4) {
    const double a = x[j], b = x[j + 1], c = x[j + 2], d = x[j + 3];
    s = (((s + a) + b) + c) + d;
  }
  for (; j < n; ++j) s = s + x[j];
  return s;
}
__device__ __forceinline__ float seq_sum(const float *x, int n) {
  struct alignas(8) F2 {
    float a, b;
  };
  const F2 *v = (const F2 *)x;
  float s = 0.0f;
  int j = 0;
  for (; 2 * j + 8 <= n; j += 4) {
    const F2 p = v[j], q = v[j + 1], r = v[j + 2], t = v[j + 3];
    s = (((s + p.a) + p.b) + q.a) + q.b;
    s = (((s + r.a) + r.b) + t.a) + t.b;
  }
  for (j *= 2; j < n; ++j) s = s + x[j];
  return s;
}

// sum_k a[k] b[k stride] as an fma chain in k order
template <int U, typename T>
__device__ __forceinline__ T seq_dot(const T *a, const T *b, int stride, int n) {
  T s = (T)0;
  int k = 0;
  for (; k + U <= n; k += U) {
    T av[U], bv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      av[u] = a[k + u];
      bv[u] = b[(k + u) * stride];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) s = fma_t(av[u], bv[u], s);
  }
  for (; k < n; ++k) s = fma_t(a[k], b[k * stride], s);
  return s;
}

// phi_k = sum_m c_km chi_m, fma chain in m order; coefficients from the
// [n_basis][n_orb] table (consecutive k on consecutive lanes)
__device__ __forceinline__ double orbital_value(const SJSysDev &S, const SJTab &tab, int k, const double *chi) {
  const int K = S.n_basis, no = S.n_orb;
  double phi = 0.0;
  int m = 0;
  if (tab.has_coef) {
    const double *c = tab.coef + k;
    for (; m + 4 <= K; m += 4) {
      double cv[4], xv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        cv[u] = c[(m + u) * no];
        xv[u] = chi[m + u];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) phi = fma(cv[u], xv[u], phi);
    }
    for (; m < K; ++m) phi = fma(c[m * no], chi[m], phi);
    return phi;
  }
  const double *c = S.coef_t + k;
  for (; m + 8 <= K; m += 8) {
    double cv[8], xv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      cv[u] = c[(size_t)(m + u) * no];
      xv[u] = chi[m + u];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) phi = fma(cv[u], xv[u], phi);
  }
  for (; m < K; ++m) phi = fma(c[(size_t)m * no], chi[m], phi);
  return phi;
}

// The draws of one Gaussian move at stream position q.  Out of line: inlined,
// the constants of log, sin and cos are kept in registers across the sweeps
// and push the moves' own state into scratch memory.
struct SJGauss {
  double z0, z1, z2, u;
};
__device__ __noinline__ SJGauss gauss_draws(uint64_t q, uint32_t k0, uint32_t k1, uint32_t walker, uint32_t epoch) {
  Stream st;
  st.init((uint64_t)k0 | ((uint64_t)k1 << 32), 0, walker, epoch);
  const uint64_t d0 = st.draw(q), d1 = st.draw(q + 1), d2 = st.draw(q + 2), d3 = st.draw(q + 3), d4 = st.draw(q + 4);
  SJGauss g;
  double z3;
  box_muller(d0, d1, &g.z0, &g.z1);
  box_muller(d2, d3, &g.z2, &z3);
  g.u = u64_standard(d4);
  return g;
}

// A walker's counters and determinants, the same on all its lanes.
struct SJBooks {
  double ld[4];     // (mantissa, exponent) of det A_up, det A_dn
  double cond, drift, singular;
};

// What a re-inversion of one spin block found (on every lane).
struct SJRefresh {
  double cond;      // ||A||_1 ||A^-1||_1
  double mant, ex;  // det A = mant 2^ex (mant = 0: singular)
  bool singular;
};

// Gauss-Jordan inverse of the spin-s Slater matrix from the positions, FP64,
// with partial pivoting, into B (as T) when write_B; the determinant from the
// pivots (the row swaps' signs times their product, carried as mant 2^ex).
// A pivot |p| <= n 2^-52 ||A||_1 (or NaN) marks the block singular: its
// division is skipped (the row is zeroed), so the inverse stays finite and
// the determinant reads 0.  All lanes of the workgroup must call it; the
// norms and the pivot search run on every lane alike.
template <typename T>
__device__ __forceinline__ SJRefresh refresh_spin(const SJSysDev &S, const SJTab &tab, SJWalker<T> &wk, int s,
                                                  int t, int L, bool gto, bool pk, bool write_B) {
  SJRefresh res{1.0, 1.0, 0.0, false};
  const int n = s == 0 ? S.n_up : S.n_dn;
  if (n == 0) return res;
  const int first = s == 0 ? 0 : S.n_up;
  T *B = s == 0 ? wk.Bup : wk.Bdn;
  double *M = wk.scr, *I = wk.scr + n * n, *chi = I;
  sync_wave();
  for (int c = 0; c < n; ++c) {
    basis_to_lds(S, tab, wk.pos + 3 * (first + c), chi, t, L, gto, pk);
    sync_wave();
    for (int k = t; k < n; k += L) M[c * n + k] = orbital_value(S, tab, k, chi);
    sync_wave();
  }
  double anorm = 0.0;
  for (int k = 0; k < n; ++k) {
    double cs = 0.0;
    for (int c = 0; c < n; ++c) cs += fabs(M[c * n + k]);
    anorm = cs > anorm ? cs : anorm;
  }
  const double thresh = anorm * ((double)n * 0x1p-52);
  const float inv_n = 1.0f / (float)n;
  for (int e = t; e < n * n; e += L) I[e] = (e == small_div(e, inv_n) * (n + 1)) ? 1.0 : 0.0;
  sync_wave();
  for (int p = 0; p < n; ++p) {
    int piv = p;
    double pv = M[p * n + p];
    for (int r = p + 1; r < n; ++r) {
      const double v = M[r * n + p];
      if (fabs(v) > fabs(pv)) {
        piv = r;
        pv = v;
      }
    }
    const bool bad = !(fabs(pv) > thresh);
    if (bad) {
      res.singular = true;
    } else {
      if (piv != p) res.mant = -res.mant;
      logdet_mul(res.mant, res.ex, pv);
    }
    sync_wave();
    const double ip = bad ? 0.0 : 1.0 / pv;
    // rows p and piv swapped, row p scaled (columns of A before p are done with)
    for (int j = t; j < n; j += L) {
      const double mp = M[p * n + j], mv = M[piv * n + j], ap = I[p * n + j], av = I[piv * n + j];
      if (j >= p) {
        M[piv * n + j] = mp;
        M[p * n + j] = mv * ip;
      }
      I[piv * n + j] = ap;
      I[p * n + j] = av * ip;
    }
    sync_wave();
    // the other rows, one to a lane: row r needs its own element of column p
    // and row p only
    for (int r = t; r < n; r += L) {
      if (r == p) continue;
      const double f = -M[r * n + p];
      auto sweep_row = [&](double *x, const double *y, int j) {
        for (; j + 4 <= n; j += 4) {
          double v[4], w[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            v[u] = x[j + u];
            w[u] = y[j + u];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) x[j + u] = fma(f, w[u], v[u]);
        }
        for (; j < n; ++j) x[j] = fma(f, y[j], x[j]);
      };
      sweep_row(M + r * n, M + p * n, p + 1);
      sweep_row(I + r * n, I + p * n, 0);
    }
    sync_wave();
  }
  if (write_B)
    for (int e = t; e < n * n; e += L) B[e] = (T)I[e];
  double bnorm = 0.0;
  for (int c = 0; c < n; ++c) {
    double cs = 0.0;
    for (int k = 0; k < n; ++k) cs += fabs(I[k * n + c]);
    bnorm = cs > bnorm ? cs : bnorm;
  }
  sync_wave();
  res.cond = anorm * bnorm;
  if (res.singular) {
    res.mant = 0.0;
    res.ex = 0.0;
  }
  return res;
}

// Re-inverts both spin blocks and keeps the books: with count, the condition
// maximum and the singular blocks; the log-determinant state when ld_mode is 1
// (taken from the re-inversion) or 2 (the same, after recording how far the
// value the updates carried drifted from it).
template <typename T>
__device__ __forceinline__ void refresh_walker(const SJSysDev &S, const SJTab &tab, SJWalker<T> &wk, SJBooks &bk,
                                               int t, int L, bool gto, bool pk, bool write_B, bool count,
                                               int ld_mode) {
#pragma unroll 1
  for (int q = 0; q < 2; ++q) {
    const SJRefresh r = refresh_spin<T>(S, tab, wk, q, t, L, gto, pk, write_B);
    if (count) {
      bk.cond = fmax(bk.cond, r.cond);
      if (r.singular) bk.singular += 1.0;
    }
    const double m = q ? bk.ld[2] : bk.ld[0], e = q ? bk.ld[3] : bk.ld[1];
    if (ld_mode == 2 && !r.singular && m != 0.0)
      bk.drift = fmax(bk.drift, fabs(logdet_value(m, e) - logdet_value(r.mant, r.ex)));
    if (ld_mode) {
      bk.ld[0] = q ? bk.ld[0] : r.mant;
      bk.ld[1] = q ? bk.ld[1] : r.ex;
      bk.ld[2] = q ? r.mant : bk.ld[2];
      bk.ld[3] = q ? r.ex : bk.ld[3];
    }
  }
}

// Local energy and d ln psi/dp (five Jastrow parameters) of the walker's
// configuration, whole electrons on lanes: lane t takes electrons t, t+L, ...
// and forms each electron's kinetic term (orbital gradients and laplacians
// as fma chains over the basis, contracted with the inverse column; Jastrow
// gradient and laplacian over partners, electrons then nuclei), potential and
// parameter derivatives in registers; the electrons' results are then added in
// electron order.  Every sum has a fixed order, so the result does not depend
// on L.
// Orbitals per register chunk: 10 take a spin block of up to 10 in one pass
// over the basis and the largest (20) in two (with 8, 9 electrons per spin
// evaluated every basis function twice, and 18 three times).
constexpr int kSJLanesNMax = 10;

// The pieces of the local energy the operator terms need (on every lane).
struct SJParts {
  double kin;  // sum_i lap_i psi / psi
  double vee;  // sum_{i<j} 1/r_ij
  double ven;  // -sum_{I,i} Z_I / |r_i - R_I|
};

// sum_k coef_k term_k of one operator (terms as the C ABI defines them).
__device__ __noinline__ double operator_value(const mole_operator &op, SJParts P, const SJSysDev &S, const double *pos) {
  const int N = S.N;
  double v = 0.0;
  for (uint32_t k = 0; k < op.n_terms; ++k) {
    const mole_term &tm = op.term[k];
    double x = 0.0;
    switch (tm.kind) {
      case MOLE_TERM_KINETIC: x = -0.5 * P.kin; break;
      case MOLE_TERM_IONIC_POTENTIAL: x = P.ven + S.v_nn; break;
      case MOLE_TERM_ELECTRONIC_POTENTIAL: x = P.vee; break;
      case MOLE_TERM_HARMONIC: {
        double s2 = 0.0;
        for (int i = 0; i < N; ++i)
          for (int q = 0; q < 3; ++q) {
            const double dq = pos[3 * i + q] - tm.param[1 + q];
            s2 += dq * dq;
          }
        x = 0.5 * (tm.param[0] * tm.param[0]) * s2;
        break;
      }
      case MOLE_TERM_RADIAL_POWER: {
        const int pw = (int)tm.param[0];
        for (int i = 0; i < N; ++i) {
          const double r = norm3(pos[3 * i] - tm.param[1], pos[3 * i + 1] - tm.param[2], pos[3 * i + 2] - tm.param[3]);
          const double b = pw > 0 ? r : 1.0 / r;
          double y = b;
          for (int e = 1; e < (pw > 0 ? pw : -pw); ++e) y *= b;
          x += y;
        }
        break;
      }
      case MOLE_TERM_DIPOLE:
        for (int i = 0; i < N; ++i)
          x += ((pos[3 * i] - tm.param[0]) * tm.param[3] + (pos[3 * i + 1] - tm.param[1]) * tm.param[4]) +
               (pos[3 * i + 2] - tm.param[2]) * tm.param[5];
        break;
      default: break;
    }
    v += tm.coef * x;
  }
  return v;
}

// Exponent scale s (zeta_m = s zeta0_m): sum_m zeta_m d ln psi / d zeta_m
// of electron i (at xi, column cc of its n x n inverse B), with d chi_m /
// d zeta_m = -r chi_m (s- and p-type STO) or -r^2 chi_m (GTO); fma chains in
// m, then k order.  Out of line: only systems with the scale call it, and the
// sweep kernels keep their code size.
template <typename T, bool EXT>
__device__ __noinline__ double exponent_scale_term(const SJSysDev &S, const T *B, int n, int cc, const double *xi) {
  const int K = S.n_basis, no = S.n_orb;
  double ez = 0.0;
  for (int k0 = 0; k0 < n; k0 += kSJLanesNMax) {
    double oz[kSJLanesNMax];
#pragma unroll
    for (int k = 0; k < kSJLanesNMax; ++k) oz[k] = 0.0;
    for (int m = 0; m < K; ++m) {
      const int I = S.center[m];
      const double d0 = xi[0] - S.nuc[3 * I], d1 = xi[1] - S.nuc[3 * I + 1], d2 = xi[2] - S.nuc[3 * I + 2];
      const double r = norm3(d0, d1, d2);
      const int kd = ((EXT && S.any_gto) || S.any_p) ? S.kind[m] : MOLE_BASIS_STO;
      const double ch = basis_value<EXT>(kd, S.zeta[m], d0, d1, d2, r);
      const double rp = (EXT && kd == MOLE_BASIS_GTO) ? r * r : r;
      const double tz = (-(S.zeta[m] * rp)) * ch;
      const double *cm = S.coef_t + (size_t)m * no + k0;
#pragma unroll
      for (int k = 0; k < kSJLanesNMax; ++k)
        if (k0 + k < n) oz[k] = fma(cm[k], tz, oz[k]);
    }
#pragma unroll
    for (int k = 0; k < kSJLanesNMax; ++k)
      if (k0 + k < n) ez = fma(oz[k], (double)B[(k0 + k) * n + cc], ez);
  }
  return ez;
}

// One compat sample of MonteCarloSampler::data (the extended
// instantiation only): "Wavefunction value" as Sampler::sample stores it,
// psi_s = (psi psi)/psi (src/vmc/src/operators.rs:19-23, samplers.rs:89-90),
// and "Parameter gradient" O_k psi_s with O = d ln psi/dp.  psi = sign
// exp(log|det up| + log|det dn| + J) from the carried determinants ld =
// (mant_up, ex_up, mant_dn, ex_dn) and J = b_anti O_0 + b_para O_1 + a O_3
// (the Pade factor is linear in b_anti, b_para and a).  Out of line: only
// contexts that keep compat samples call it.
__device__ __forceinline__ double sj_psi(const SJSysDev &S, const double *ld, const double *dl) {
  const double J = (S.p[0] * dl[0] + S.p[1] * dl[1]) + S.p[3] * dl[3];
  const double lg = (logdet_value(ld[0], ld[1]) + logdet_value(ld[2], ld[3])) + J;
  const double sg = ((ld[0] < 0.0) != (ld[2] < 0.0)) ? -1.0 : 1.0;
  return sg * exp_m(lg);
}

__device__ __noinline__ void sj_compat_sample(const SJSysDev &S, const double *ld, const double *dl, int np,
                                              size_t at) {
  const double psi = sj_psi(S, ld, dl);
  const double ps = (psi * psi) / psi;
  S.samp_psi[at] = ps;
  for (int k = 0; k < np; ++k) S.samp_g[at * (size_t)np + k] = dl[k] * ps;
}

// g_out (extended kernel, optional): grad_i ln psi of every electron, written
// by the lane that takes the electron as g_out[3 i + q].  Returns the energy
// on every lane and leaves (1, E, d ln psi/dp) at the end of wk.le, whose
// address is *vec.
template <typename T, bool EXT>
__device__ __forceinline__ double local_energy(const SJSysDev &S, SJWalker<T> &wk, int t, int L, double **vec,
                                               SJParts &parts, double *g_out) {
  const int N = S.N, K = S.n_basis, nn = S.n_nuc, no = S.n_orb;
  const double bA = S.p[0], bP = S.p[1], c = S.p[2], a = S.p[3], d = S.p[4];
  // [N][RS]: kinetic term, potential, five Jastrow derivatives, e-e potential
  // (EXT), exponent-scale derivative (with the scale); RS = 3 + np
  double *res = wk.le;
  const int RS = 8 + S.opt_exp;
  const bool kinds = (EXT && S.any_gto) || S.any_p;
  const int nmax = S.n_up > S.n_dn ? S.n_up : S.n_dn;
  sync_wave();
  // FAST leaves out the square root's and the divisions' range handling (a
  // third of a pair's instructions); its results are the same bits while every
  // root's argument is in range, and an electron for which one is not, or a
  // result is NaN, is evaluated again without it.
  const bool tame = fabs(c) < 0x1p100 && fabs(d) < 0x1p100;
  auto electron = [&](int i, auto fast) {
    constexpr bool FAST = decltype(fast)::value;
    RootRange range;
    auto root = [&](double v0, double v1, double v2) {
      const double ss = sumsq3(v0, v1, v2);
      if constexpr (FAST) return range.root(ss);
      else return sqrt(ss);
    };
    auto recip = [](double v) {
      if constexpr (FAST) return recip_normal(v);
      else return 1.0 / v;
    };
    const int s = i < S.n_up ? 0 : 1;
    const int cc = s == 0 ? i : i - S.n_up;
    const int n = s == 0 ? S.n_up : S.n_dn;
    const T *B = s == 0 ? wk.Bup : wk.Bdn;
    const double xi[3] = {wk.pos[3 * i], wk.pos[3 * i + 1], wk.pos[3 * i + 2]};
    // orbitals in register chunks of two halves; the basis values are
    // recomputed per chunk (bit-identical each time), and the chunks add in
    // orbital order, so the width does not change the sums.  Coefficients past
    // the last orbital are read (the table is padded) and their chains not used.
    // The extended instantiations (DMC, operators, Gaussians) carry more live
    // state and take 6, which keeps their spills down.
    constexpr int kHalf = EXT ? 3 : kSJLanesNMax / 2, kCh = 2 * kHalf;
    double Dg0 = 0.0, Dg1 = 0.0, Dg2 = 0.0, Dl = 0.0;
#pragma unroll 1
    for (int k0 = 0; k0 < n; k0 += kCh) {
      double og[kCh][4];
#pragma unroll
      for (int k = 0; k < kCh; ++k) og[k][0] = og[k][1] = og[k][2] = og[k][3] = 0.0;
      // consecutive functions of one centre share its displacement, distance
      // and 1/r, and those of one shell the exponential (a p shell's three)
      int Ip = -1;
      double zp = 0.0, d0 = 0.0, d1 = 0.0, d2 = 0.0, r = 0.0, ir = 0.0, e = 0.0;
      bool have_e = false;
#pragma unroll 1
      for (int m = 0; m < K; ++m) {
        const int I = S.center[m];
        const double z = S.zeta[m];
        const int kd = kinds ? S.kind[m] : MOLE_BASIS_STO;
        if (I != Ip) {
          d0 = xi[0] - S.nuc[3 * I];
          d1 = xi[1] - S.nuc[3 * I + 1];
          d2 = xi[2] - S.nuc[3 * I + 2];
          r = root(d0, d1, d2);
          ir = recip(r);
          Ip = I;
          have_e = false;
        }
        double ch, g0, g1, g2, lc;
        if (EXT && kd == MOLE_BASIS_GTO) {
          basis_vgl<true>(kd, z, d0, d1, d2, r, ch, g0, g1, g2, lc);
        } else {
          if (!have_e || z != zp) {
            e = exp_m(-z * r);
            zp = z;
            have_e = true;
          }
          basis_vgl_sto(kd, z, d0, d1, d2, e, ir, ch, g0, g1, g2, lc);
        }
        const double *cm = S.coef_t + (size_t)m * no + k0;
        auto half = [&](int h) {
#pragma unroll
          for (int k = h; k < h + kHalf; ++k) {
            const double cv = cm[k];
            og[k][0] = fma(cv, g0, og[k][0]);
            og[k][1] = fma(cv, g1, og[k][1]);
            og[k][2] = fma(cv, g2, og[k][2]);
            og[k][3] = fma(cv, lc, og[k][3]);
          }
        };
        half(0);
        if (nmax - k0 > kHalf) half(kHalf);  // the same for all lanes
      }
#pragma unroll
      for (int k = 0; k < kCh; ++k)
        if (k0 + k < n) {
          const double bkc = (double)B[(k0 + k) * n + cc];
          Dg0 = fma(og[k][0], bkc, Dg0);
          Dg1 = fma(og[k][1], bkc, Dg1);
          Dg2 = fma(og[k][2], bkc, Dg2);
          Dl = fma(og[k][3], bkc, Dl);
        }
    }
    // exponent scale s: sum_m zeta_m d ln psi / d zeta_m of electron i's row
    const double ez = S.opt_exp ? exponent_scale_term<T, EXT>(S, B, n, cc, wk.pos + 3 * i) : 0.0;
    double gJ0 = 0.0, gJ1 = 0.0, gJ2 = 0.0, lJ = 0.0;
    double Vi = 0.0, Vee = 0.0, e0 = 0.0, e1 = 0.0, e2 = 0.0, e3 = 0.0, e4 = 0.0;
#pragma unroll 1
    for (int j = 0; j < N; ++j) {
      if (j == i) continue;
      const double *xj = wk.pos + 3 * j;
      const double dv0 = xi[0] - xj[0], dv1 = xi[1] - xj[1], dv2 = xi[2] - xj[2];
      const double r = root(dv0, dv1, dv2);
      const bool same = (j < S.n_up ? 0 : 1) == s;
      const double b = same ? bP : bA;
      // two divisions per pair: 1/r and 1/(1 + c r)
      const double ir = recip(r);
      const double iden = recip(1.0 + c * r);
      const double iden2 = iden * iden;
      const double up = b * iden2;
      const double upp = (-2.0 * b * c) * (iden2 * iden);
      const double ur = up * ir;
      gJ0 += ur * dv0;
      gJ1 += ur * dv1;
      gJ2 += ur * dv2;
      lJ += upp + 2.0 * ur;
      if (j > i) {
        Vi += ir;
        if constexpr (EXT) Vee += ir;
        if (same)
          e1 += r * iden;
        else
          e0 += r * iden;
        e2 += (-b * r * r) * iden2;
      }
    }
#pragma unroll 1
    for (int I = 0; I < nn; ++I) {
      const double d0 = xi[0] - S.nuc[3 * I], d1 = xi[1] - S.nuc[3 * I + 1], d2 = xi[2] - S.nuc[3 * I + 2];
      const double r = root(d0, d1, d2);
      const double Z = S.charge[I];
      const double ir = recip(r);
      const double iden = recip(1.0 + d * r);
      const double iden2 = iden * iden;
      const double aZ = a * Z;
      const double vp = -aZ * iden2;
      const double vpp = (2.0 * aZ * d) * (iden2 * iden);
      const double vr = vp * ir;
      gJ0 += vr * d0;
      gJ1 += vr * d1;
      gJ2 += vr * d2;
      lJ += vpp + 2.0 * vr;
      Vi += -Z * ir;
      e3 += (-Z * r) * iden;
      e4 += (aZ * r * r) * iden2;
    }
    const double dot = Dg0 * gJ0 + Dg1 * gJ1 + Dg2 * gJ2;
    const double gg = gJ0 * gJ0 + gJ1 * gJ1 + gJ2 * gJ2;
    if (EXT && g_out) {
      g_out[3 * i] = Dg0 + gJ0;
      g_out[3 * i + 1] = Dg1 + gJ1;
      g_out[3 * i + 2] = Dg2 + gJ2;
    }
    double *o = res + RS * i;
    o[0] = Dl + 2.0 * dot + lJ + gg;
    o[1] = Vi;
    o[2] = e0;
    o[3] = e1;
    o[4] = e2;
    o[5] = e3;
    o[6] = e4;
    if constexpr (EXT) o[7] = Vee;
    if (S.opt_exp) o[8] = ez;
    if constexpr (FAST) return range.held() && !(o[0] != o[0]) && !(o[1] != o[1]);
    else return true;
  };
#pragma unroll 1
  for (int i = t; i < N; i += L) {
    const bool ok = tame && electron(i, std::true_type{});
    if (__builtin_expect(__any(!ok), 0)) electron(i, std::false_type{});
  }
  sync_wave();
  // sums over electrons, in electron order: lane q forms component q into
  // electron 0's slot (kinetic, potential, derivatives)
  for (int q = t; q < RS; q += L) {
    if (!EXT && q == 7) continue;
    double sum = 0.0;
    int i = 0;
    for (; i + 4 <= N; i += 4) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = res[RS * (i + u) + q];
#pragma unroll
      for (int u = 0; u < 4; ++u) sum += v[u];
    }
    for (; i < N; ++i) sum += res[RS * i + q];
    res[q] = sum;
  }
  sync_wave();
  const double kin = res[0];
  double V = res[1];
  double *v = res + RS * N;  // (1, E, O)
  double *dl = v + 2;
  if (t == 0) {
    v[0] = 1.0;
    for (int q = 0; q < 5; ++q) dl[q] = res[2 + q];
    // d ln psi / d s = (1/s) sum_m zeta_m d ln psi / d zeta_m
    if (S.opt_exp) dl[5] = res[8] / S.p[5];
  }
  if (S.hamiltonian != MOLE_H_ELECTRONIC) {
    V = 0.0;
    for (int i = 0; i < N; ++i)
      for (int I = 0; I < nn; ++I) {
        const double *xi = wk.pos + 3 * i;
        V += -S.charge[I] / norm3(xi[0] - S.nuc[3 * I], xi[1] - S.nuc[3 * I + 1], xi[2] - S.nuc[3 * I + 2]);
      }
  }
  parts.kin = kin;
  double E = -0.5 * kin + V + S.v_nn;
  if (EXT && (S.custom_h || S.n_obs)) {
    double ven = 0.0;
    // IonicPotential::value's order: ions outer, electrons inner
    for (int I = 0; I < nn; ++I)
      for (int i = 0; i < N; ++i) {
        const double *xi = wk.pos + 3 * i;
        ven -= S.charge[I] / norm3(xi[0] - S.nuc[3 * I], xi[1] - S.nuc[3 * I + 1], xi[2] - S.nuc[3 * I + 2]);
      }
    parts.vee = res[7];
    parts.ven = ven;
    if (S.custom_h) E = operator_value(S.ops[0], parts, S, wk.pos);
  }
  if (t == 0) v[1] = E;
  *vec = v;
  sync_wave();
  return E;
}

// Jastrow gradient terms of electron i at r into jg[3j + q] (lanes over
// partners, i's slot zero), FP64.  No barrier.
__device__ __forceinline__ void drift_terms(const SJSysDev &S, const double *nuc, const double *pos, int i,
                                            const double *r, double *jg, int t, int L) {
  const int N = S.N, si = i < S.n_up ? 0 : 1;
#pragma unroll 1
  for (int j = t; j < N + S.n_nuc; j += L) {
    double *o = jg + 3 * j;
    const bool el = j < N;
    const double *xj = el ? pos + 3 * j : nuc + 4 * (j - N);
    const double d0 = r[0] - xj[0], d1 = r[1] - xj[1], d2 = r[2] - xj[2];
    const double rr = norm3(d0, d1, d2);
    // b/(1 + c r)^2 of a pair, -(a Z)/(1 + d r)^2 of a nucleus
    const double num = el ? (((j < S.n_up ? 0 : 1) == si) ? S.p[1] : S.p[0]) : xj[3];
    const double den = 1.0 + (el ? S.p[2] : S.p[4]) * rr;
    const double up = num / (den * den);
    const bool self = j == i;
    o[0] = self ? 0.0 : up * d0 / rr;
    o[1] = self ? 0.0 : up * d1 / rr;
    o[2] = self ? 0.0 : up * d2 / rr;
  }
}

// Orbital gradients og[3k + q] = sum_m c_km gch[3m + q] (lanes over
// orbitals, chains in m order).  No barrier.
__device__ __forceinline__ void orbital_gradients(const SJSysDev &S, const SJTab &tab, int n, const double *gch,
                                                  double *og, int t, int L) {
  const int K = S.n_basis, no = S.n_orb;
  for (int k = t; k < n; k += L) {
    double g0 = 0.0, g1 = 0.0, g2 = 0.0;
    for (int m = 0; m < K; ++m) {
      const double cm = tab.has_coef ? tab.coef[m * no + k] : S.coef_t[(size_t)m * no + k];
      g0 = fma(cm, gch[3 * m], g0);
      g1 = fma(cm, gch[3 * m + 1], g1);
      g2 = fma(cm, gch[3 * m + 2], g2);
    }
    og[3 * k] = g0;
    og[3 * k + 1] = g1;
    og[3 * k + 2] = g2;
  }
}

// g = sum_k og_k B[k][c] (chains in k order) + sum_j jg_j (in j order), each as
// in the CPU restatement, on every lane.
template <typename T>
__device__ __forceinline__ void drift_sum(const double *og, const T *B, int n, int c, const double *jg, int M,
                                          double det_scale, double g[3]) {
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  for (int k = 0; k < n; ++k) {
    const double bkc = (double)B[k * n + c];
    d0 = fma(og[3 * k], bkc, d0);
    d1 = fma(og[3 * k + 1], bkc, d1);
    d2 = fma(og[3 * k + 2], bkc, d2);
  }
  double j0 = 0.0, j1 = 0.0, j2 = 0.0;
  for (int j = 0; j < M; ++j) {
    j0 += jg[3 * j];
    j1 += jg[3 * j + 1];
    j2 += jg[3 * j + 2];
  }
  // det_scale = 1: plain sum; otherwise the determinant part is divided by it
  if (det_scale != 1.0) {
    d0 = d0 / det_scale;
    d1 = d1 / det_scale;
    d2 = d2 / det_scale;
  }
  g[0] = d0 + j0;
  g[1] = d1 + j1;
  g[2] = d2 + j2;
}

}  // namespace

// EXT: the DMC modes, local operators and Gaussian basis functions are
// compiled in (the plain VMC instantiations leave them out, keeping their
// register budget).
// MINW: minimum waves per SIMD the register budget is fitted to (2: up to
// 256 registers; 1: 512, for the learned proposal's larger systems where a
// launch holds no second wave per SIMD anyway).
// One tile's launch: its walkers' state into the workgroup's LDS, the sweeps,
// the state out.
template <typename T, int PROP, bool EXT>
__device__ __forceinline__ void sj_tile(const SJArgs &a, const SJTile tile, unsigned char *lds) {
  constexpr int DPM = sj_draws_per_move(PROP);
  const SJSysDev &S = a.systems[tile.sys];
  const int N = S.N, nu = S.n_up, nd = S.n_dn, L = S.L, W = S.W, nn = S.n_nuc;
  const int lane = threadIdx.x;
  // learned proposal: 16 walkers of 4 lanes, walker s on lanes s, s+16,
  // s+32, s+48 (the sample columns of the MFMA tiles); otherwise L
  // consecutive lanes per walker
  const int slot = PROP == kSJPropLearned ? (lane & 15) : lane / L;
  const int t = PROP == kSJPropLearned ? (lane >> 4) : lane % L;
  const int nslots = 64 / L;
  const int lg_slots = __ffs(nslots) - 1;  // nslots is a power of two
  const bool live = slot < tile.nw;
  const int w = tile.w0 + slot;
  const int np = 5 + S.opt_exp;
  const SJLayout lay(N, nu, nd, nn, S.n_basis, (int)sizeof(T), np, PROP);
  // shared by the workgroup: the sample sums' factor pairs, the nuclei
  uint8_t *pairs = lds;
  const SJShared sh(nn, S.n_basis, S.n_orb);
  double *nuc = (double *)(lds + sh.nuc);
  unsigned char *walkers = lds + sh.bytes;
  const SJTab tab{nuc, (const double *)(lds + sh.fn), (const double *)(lds + sh.coef), sh.has_fn, sh.has_coef};
  unsigned char *base = walkers + (size_t)slot * lay.bytes;
  SJWalker<T> wk;
  wk.pos = (double *)(base + lay.pos);
  wk.Bup = (T *)(base + lay.B);
  wk.Bdn = wk.Bup + nu * nu;
  wk.rng = (double *)(base + lay.rng);
  wk.scr = (double *)(base + lay.scr);
  wk.mv = (double *)(base + lay.mv);
  wk.chi = (double *)(base + lay.chi);
  wk.phin = (T *)(base + lay.phin);
  wk.jn = (T *)(base + lay.jn);
  wk.jo = (T *)(base + lay.jo);
  wk.dots = (T *)(base + lay.dots);
  wk.le = (double *)(base + lay.le);
  const int nB = nu * nu + nd * nd, M = N + nn;
  const bool gto = EXT && S.any_gto;
  const bool pk = S.any_p != 0;
  // DMC steps move walkers the branching gathered: the log-determinant state
  // is not carried there (mole_dmc_diffuse recomputes it at its end)
  const bool dmc_step = EXT && a.dmc == kSJDmcStep;
  const bool track_ld = !dmc_step;

  // ---- state in (a DMC step reads the walkers the branching gathered) ----
  // A partial tile's empty slots start from its first walker: with every
  // electron at the origin their local energy would never be in the fast roots'
  // range, and the wave would evaluate it twice (two electrons in 64 functions,
  // one walker: a sampled sweep at 16 lanes took 39 us instead of 34).  Nothing
  // of theirs is written back.
  const double *pin = dmc_step ? S.dmc_pos_in : S.pos;
  const T *Bg = (const T *)(dmc_step ? S.dmc_B_in : S.B);
  for (int e = lane; e < 3 * N * nslots; e += 64) {
    const int k = e >> lg_slots, sl = e & (nslots - 1);
    double *pp = (double *)(walkers + (size_t)sl * lay.bytes + lay.pos);
    pp[k] = pin[(size_t)k * W + tile.w0 + (sl < tile.nw ? sl : 0)];
  }
  for (int e = lane; e < nB * nslots; e += 64) {
    const int k = e >> lg_slots, sl = e & (nslots - 1);
    T *bb = (T *)(walkers + (size_t)sl * lay.bytes + lay.B);
    bb[k] = Bg[(size_t)k * W + tile.w0 + (sl < tile.nw ? sl : 0)];
  }
  for (int I = lane; I < nn; I += 64) {
    nuc[4 * I] = S.nuc[3 * I];
    nuc[4 * I + 1] = S.nuc[3 * I + 1];
    nuc[4 * I + 2] = S.nuc[3 * I + 2];
    nuc[4 * I + 3] = -(S.p[3] * S.charge[I]);
  }
  const int nsum = sj_sample_sums(np);
  if (lane < nsum) {
    // q = 0, 1: E, E^2; then O_k, O_k E, and the triangle O_k O_l row by row
    int fa = lane == 0 ? 0 : 1, fb = 1;
    if (lane >= 2 + 2 * np) {
      int k = 0, e = lane - 2 - 2 * np;
      while (e >= np - k) e -= np - k++;
      fa = 2 + k;
      fb = 2 + k + e;
    } else if (lane >= 2) {
      fa = lane < 2 + np ? 0 : 1;
      fb = 2 + (lane - 2) % np;
    }
    pairs[lane] = (uint8_t)(fa | fb << 4);
  }
  if (tab.has_fn)
    for (int m = lane; m < S.n_basis; m += 64) {
      double *e = (double *)(lds + sh.fn) + 5 * m;
      const int I = S.center[m];
      e[0] = S.nuc[3 * I];
      e[1] = S.nuc[3 * I + 1];
      e[2] = S.nuc[3 * I + 2];
      e[3] = S.zeta[m];
      e[4] = __longlong_as_double((long long)S.kind[m]);
    }
  if (tab.has_coef)
    for (int e = lane; e < S.n_basis * S.n_orb; e += 64) ((double *)(lds + sh.coef))[e] = S.coef_t[e];
  SJBooks bk{{1.0, 0.0, 1.0, 0.0}, 0.0, 0.0, 0.0};
  double block_sum = 0.0, acc_in = 0.0;
  [[maybe_unused]] double dmc_el = 0.0, dmc_w = 0.0, dmc_eref = 0.0;
  if (live) {
    acc_in = S.acc[(size_t)kSJAccepted * W + w];
    if (dmc_step) {
      dmc_el = S.dmc_el_in[w];
      dmc_w = S.dmc_w_in[w];
      dmc_eref = *S.dmc_eref;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) bk.ld[k] = S.ld[(size_t)k * W + w];
      block_sum = S.acc[(size_t)kSJBlockSum * W + w];
    }
  }
  uint32_t n_acc = 0;
  sync_wave();

  const uint32_t k0 = (uint32_t)a.seed, k1 = (uint32_t)(a.seed >> 32) ^ S.sys_index;
  if (a.init) {
    // Sampler::new: U(-1, 1) from draws 0..3N-1 (samplers.rs:46)
    for (int b = t; 2 * b < 3 * N; b += L) {
      const u32x4 o = philox4x32_10({(uint32_t)b, 0u, (uint32_t)w, a.epoch}, k0, k1);
      const uint64_t v0 = (uint64_t)o.x | ((uint64_t)o.y << 32);
      const uint64_t v1 = (uint64_t)o.z | ((uint64_t)o.w << 32);
      wk.pos[2 * b] = u64_range(v0, 2.0, -3.0);
      if (2 * b + 1 < 3 * N) wk.pos[2 * b + 1] = u64_range(v1, 2.0, -3.0);
    }
    sync_wave();
  }
  const uint32_t lu_period = a.lu_period;
  const SJLaunchState ls = *a.state;
  uint64_t p = S.draw_base + DPM * (uint64_t)N * ls.sweeps_done;
  const uint64_t m0 = S.move_base + (uint64_t)N * ls.sweeps_done;
  // moves until the next re-inversion
  uint32_t lu_left = lu_period ? lu_period - (uint32_t)(m0 % lu_period) : 0;
  uint32_t fill = ls.block_fill;
  uint32_t sidx = ls.trace_samples;
  const double inv_block = 1.0 / (double)a.block_size;
  const T bA = (T)S.p[0], bP = (T)S.p[1], cee = (T)S.p[2], cen = (T)S.p[4];
  // the pass before the first sweep re-inverts where the launch asks for it
  // and takes the local energy of the configurations as they are (DMC's start,
  // mole_eval); one copy of each stage serves it and the sweeps
  const bool entry_refresh = a.init || a.refresh;
  const bool entry_energy = EXT && (a.dmc == kSJDmcInit || a.dmc == kSJEval);

  for (uint32_t pass = entry_refresh || entry_energy ? 0u : 1u; pass <= a.n_sweeps; ++pass) {
    const bool sweep = pass > 0;
    const uint32_t sw = pass - 1;
    if (sweep) {
      if constexpr (PROP == kSJPropBox) {
        // ---- the sweep's draws: [p, p + 4N), lanes over Philox blocks ----
        const uint64_t b0 = p >> 1;
        const int odd = (int)(p & 1), n4 = 4 * N;
        for (int b = t; 2 * b - odd < n4; b += L) {
          const uint64_t bb = b0 + (uint64_t)b;
          const u32x4 o = philox4x32_10({(uint32_t)bb, (uint32_t)(bb >> 32), (uint32_t)w, a.epoch}, k0, k1);
          const uint64_t v0 = (uint64_t)o.x | ((uint64_t)o.y << 32), v1 = (uint64_t)o.z | ((uint64_t)o.w << 32);
          const int r = 2 * b - odd;  // the first of the block's two draws
          // (dx, dy, dz, u) per move: with an even start only second draws are u
          const double d0 = odd && (r & 3) == 3 ? u64_standard(v0) : u64_range(v0, a.scale, a.offset);
          const double d1 = !odd && (r & 3) == 2 ? u64_standard(v1) : u64_range(v1, a.scale, a.offset);
          if (r >= 0) wk.rng[r] = d0;
          if (r + 1 < n4) wk.rng[r + 1] = d1;
        }
      } else {
        // ---- Gaussian proposals: 6 draws per move, lanes over moves; Box-Muller
        // of draws (0,1) and (2,3) -> z0, z1, z2; draw 4 -> the accept uniform
        for (int i = t; i < N; i += L) {
          const SJGauss g = gauss_draws(p + 6 * (uint64_t)i, k0, k1, (uint32_t)w, a.epoch);
          wk.rng[4 * i] = g.z0;
          wk.rng[4 * i + 1] = g.z1;
          wk.rng[4 * i + 2] = g.z2;
          wk.rng[4 * i + 3] = g.u;
        }
      }
      p += DPM * (uint64_t)N;
    }
    sync_wave();
    uint64_t mask = 0;
#pragma unroll 1
    for (int i = sweep ? 0 : N - 1; i < N; ++i) {
      if (sweep) {
        const int s = i < nu ? 0 : 1;
        const int c = s == 0 ? i : i - nu;
        const int n = s == 0 ? nu : nd;
        T *B = s == 0 ? wk.Bup : wk.Bdn;
        const double xi[3] = {wk.pos[3 * i], wk.pos[3 * i + 1], wk.pos[3 * i + 2]};
        const double u = wk.rng[4 * i + 3];
        double xn[3], v[3];
        [[maybe_unused]] double *gch = (double *)(base + lay.gch), *og = (double *)(base + lay.og),
                                *jg = (double *)(base + lay.jg);
        if constexpr (PROP == kSJPropBox) {
          xn[0] = xi[0] + wk.rng[4 * i];
          xn[1] = xi[1] + wk.rng[4 * i + 1];
          xn[2] = xi[2] + wk.rng[4 * i + 2];
        } else if constexpr (PROP == kSJPropLearned) {
          // learned proposal: pass 0, the network at x -> (mu, ln sigma), x' =
          // (x_i + mu) + sigma z; pass 1, the network at x' for the reverse
          // density (all lanes run the MFMA passes).  One loop body keeps a
          // single copy of the features and the network in the kernel's code.
#pragma unroll 1
          for (int ps = 0; ps < 2; ++ps) {
            float fv[4];
            mlp_features(wk.pos, N, S.nuc, nn, i, ps == 0 ? wk.pos + 3 * i : wk.mv, t, fv);
            const f32x4 o = mlp_forward(a.net, features_bf16(fv), nullptr);
            if (t == 0) {
              const double lsg = mlp_log_sigma((double)o[3]);
              const double sg = exp_m(lsg);
              if (ps == 0) {
                double z2 = 0.0;
                for (int q = 0; q < 3; ++q) {
                  const double z = wk.rng[4 * i + q];
                  wk.mv[q] = (xi[q] + (double)o[q]) + sg * z;
                  z2 += z * z;
                }
                wk.mv[3] = -3.0 * lsg - 0.5 * z2;  // log q(x'|x) + const
              } else {
                double e2 = 0.0;
                for (int q = 0; q < 3; ++q) {
                  const double e = (xi[q] - wk.mv[q]) - (double)o[q];
                  e2 += e * e;
                }
                wk.mv[4] = (-3.0 * lsg - e2 / (2.0 * sg * sg)) - wk.mv[3];  // log q(x|x') - log q(x'|x)
              }
            }
            sync_wave();
          }
          xn[0] = wk.mv[0];
          xn[1] = wk.mv[1];
          xn[2] = wk.mv[2];
        } else {
          // drift at x (metrop.rs:150-163): x' = (x_i + tau v) + sqrt(tau) z
          basis_gradients_to_lds(S, tab, xi, wk.chi, gch, t, L);
          drift_terms(S, nuc, wk.pos, i, xi, jg, t, L);
          sync_wave();
          orbital_gradients(S, tab, n, gch, og, t, L);
          sync_wave();
          drift_sum<T>(og, B, n, c, jg, M, 1.0, v);
          for (int q = 0; q < 3; ++q) xn[q] = (xi[q] + v[q] * a.tau) + a.sqrt_tau * wk.rng[4 * i + q];
          sync_wave();
        }
        // Jastrow terms of electron i at r' and at r_i (lanes over electrons,
        // then nuclei; electron i's own slot is 0 and adds nothing)
        for (int j = t; j < M; j += L) {
          const bool el = j < N;
          const double *q = el ? wk.pos + 3 * j : nuc + 4 * (j - N);
          const T num = el ? ((j < nu ? 0 : 1) == s ? bP : bA) : (T)q[3];
          const T cd = el ? cee : cen;
          const T fn = jastrow_term<T>(num, cd, xn, q), fo = jastrow_term<T>(num, cd, xi, q);
          wk.jn[j] = j == i ? (T)0 : fn;
          wk.jo[j] = j == i ? (T)0 : fo;
        }
        if constexpr (PROP == kSJPropDiffuse) {
          basis_gradients_to_lds(S, tab, xn, wk.chi, gch, t, L);
          drift_terms(S, nuc, wk.pos, i, xn, jg, t, L);
        } else {
          basis_to_lds(S, tab, xn, wk.chi, t, L, gto, pk);
        }
        sync_wave();
        for (int k = t; k < n; k += L) wk.phin[k] = (T)orbital_value(S, tab, k, wk.chi);
        if constexpr (PROP == kSJPropDiffuse) orbital_gradients(S, tab, n, gch, og, t, L);
        sync_wave();
        // sum_k phi_k(r') B[k][l] of every column l: the determinant ratio for
        // l = c, the Sherman-Morrison coefficients (times 1/ratio) for the rest
        for (int l = t; l < n; l += L) wk.dots[l] = seq_dot<8>(wk.phin, B + l, n, n);
        sync_wave();
        const T rd = wk.dots[c];
        const T Jn = seq_sum(wk.jn, M);
        const T Jo = seq_sum(wk.jo, M);
        const T dJ = Jn - Jo;
        const double rdd = (double)rd;
        const double R2 = (rdd * rdd) * exp_m(2.0 * (double)dJ);
        bool accept;
        if constexpr (PROP == kSJPropBox) {
          accept = min_one(R2) > u;
        } else if constexpr (PROP == kSJPropLearned) {
          // exact MH ratio of the learned proposal
          accept = min_one(R2 * exp_m(wk.mv[4])) > u;
        } else {
          // metrop.rs:178-197 over electron i's row: reject a sign change,
          // else min(T(x'->x) R^2 / T(x->x'), 1) > u
          double vn[3];
          drift_sum<T>(og, B, n, c, jg, M, rdd, vn);
          double eh[3], el[3];
          for (int q = 0; q < 3; ++q) {
            eh[q] = (xi[q] - xn[q]) - vn[q] * a.tau;
            el[q] = (xn[q] - xi[q]) - v[q] * a.tau;
          }
          const double nh = norm3(eh[0], eh[1], eh[2]);
          const double nl = norm3(el[0], el[1], el[2]);
          const double t_high = exp_m(-(nh * nh) / (2.0 * a.tau));
          const double t_low = exp_m(-(nl * nl) / (2.0 * a.tau));
          accept = !(rdd < 0.0) && min_one((t_high * R2) / t_low) > u;
        }
        sync_wave();
        if (accept) {
          const T inv = (T)1 / rd;
          // det A_s' = R_D det A_s, carried in FP64
          if (track_ld) {
            double m = s ? bk.ld[2] : bk.ld[0], e = s ? bk.ld[3] : bk.ld[1];
            logdet_mul(m, e, rdd);
            bk.ld[0] = s ? bk.ld[0] : m;
            bk.ld[1] = s ? bk.ld[1] : e;
            bk.ld[2] = s ? m : bk.ld[2];
            bk.ld[3] = s ? e : bk.ld[3];
          }
          // row k: B[k][l] -= B[k][c] f_l (l != c), B[k][c] /= R_D -- a row
          // needs no other lane's elements
          for (int k = t; k < n; k += L) {
            T *row = B + k * n;
            const T bkc = row[c];
            int l = 0;
            for (; l + 4 <= n; l += 4) {
              T be[4], f[4];
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                be[q] = row[l + q];
                f[q] = wk.dots[l + q];
              }
#pragma unroll
              for (int q = 0; q < 4; ++q) row[l + q] = fma_t(-bkc, f[q] * inv, be[q]);
            }
            for (; l < n; ++l) row[l] = fma_t(-bkc, wk.dots[l] * inv, row[l]);
            row[c] = bkc * inv;
          }
          if (t == 0) {
            wk.pos[3 * i] = xn[0];
            wk.pos[3 * i + 1] = xn[1];
            wk.pos[3 * i + 2] = xn[2];
          }
          mask |= (uint64_t)1 << i;
          ++n_acc;
        }
        sync_wave();
      }
      bool due = !sweep && entry_refresh;
      if (sweep && lu_period && --lu_left == 0) {
        due = true;
        lu_left = lu_period;
      }
      if (due) {
        // at entry (new configurations) the determinants are taken from the
        // re-inversion, refresh 2 keeping the inverses; after lu_period moves the
        // FP64 log|det| the update chain carried is checked against it
        const bool wb = sweep || a.init || a.refresh == 1;
        refresh_walker<T>(S, tab, wk, bk, t, L, gto, pk, wb, wb, track_ld ? (sweep ? 2 : 1) : 0);
      }
    }
    if (sweep && t == 0 && live && S.trace_mask && ls.trace_sweeps + sw < a.cap_sweeps)
      S.trace_mask[(size_t)w * a.cap_sweeps + ls.trace_sweeps + sw] = mask;
    const bool sample = sweep && sw >= a.sample_start;
    if (!(sample || (!sweep && entry_energy))) continue;

    double *gw = nullptr;
    if (EXT && a.dmc == kSJEval && live && S.ev_grad) gw = S.ev_grad + (size_t)w * 3 * N;
    double *vec;
    SJParts parts;
    const double E = local_energy<T, EXT>(S, wk, t, L, &vec, parts, gw);
    if (EXT && a.dmc == kSJDmcInit) {
      // DmcRunner::new: weight 1; the local energy of the starting configuration
      if (t == 0 && live) {
        S.dmc[w] = 1.0;
        S.dmc[(size_t)W + w] = E;
      }
    } else if (EXT && a.dmc == kSJEval) {
      // mole_eval: psi = sign exp(log|det up| + log|det dn| + J) from the
      // re-inversion's determinants, d psi = psi grad ln psi, lap psi = psi
      // sum_i lap_i psi/psi, E_L and d psi/dp = psi d ln psi/dp
      if (live) {
        const double psi = sj_psi(S, bk.ld, vec + 2);
        if (t == 0) {
          if (S.ev_value) S.ev_value[w] = psi;
          if (S.ev_lap) S.ev_lap[w] = psi * parts.kin;
          if (S.ev_el) S.ev_el[w] = E;
          if (S.ev_pgrad)
            for (int k = 0; k < np; ++k) S.ev_pgrad[(size_t)w * np + k] = psi * vec[2 + k];
        }
        // a lane rescales the gradients it wrote
        if (gw)
          for (int i = t; i < N; i += L)
            for (int q = 0; q < 3; ++q) gw[3 * i + q] = psi * gw[3 * i + q];
      }
    } else if (dmc_step) {
      // DmcRunner::diffuse (src/dmc/src/dmc.rs:88-128): the ensemble terms
      // with the weight before the step, then
      // w *= exp(-tau ((E_old + E_new)/2 - E_ref))
      if (t == 0 && live) {
        S.dmc[2 * (size_t)W + w] = dmc_w * dmc_el;
        S.dmc[3 * (size_t)W + w] = dmc_w;
        S.dmc[w] = dmc_w * exp_m(-a.dmc_tau * ((dmc_el + E) / 2.0 - dmc_eref));
        S.dmc[(size_t)W + w] = E;
      }
    } else {
      if (EXT && t == 0 && live && S.n_obs) {
        // further observables: per-walker sums in HBM (opt-in, sampled sweeps only)
        for (int k = 0; k < S.n_obs; ++k) {
          const double val = operator_value(S.ops[1 + k], parts, S, wk.pos);
          double *o = S.obs_acc + (size_t)(2 * k) * W + w;
          o[0] += val;
          o[(size_t)W] = fma(val, val, o[(size_t)W]);
        }
      }
      // sample sums in HBM, lanes over columns: += v[a] v[b] in one rounding
      if (live) {
        for (int q0 = t; q0 < nsum; q0 += 4 * L) {
          double old[4], va[4], vb[4];
          double *at[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int q = q0 + r * L < nsum ? q0 + r * L : q0;
            const int col = q < 2 ? q : kSJSumO - 2 + q;
            at[r] = S.acc + (size_t)col * W + w;
            old[r] = *at[r];
            const uint8_t f = pairs[q];
            va[r] = vec[f & 15];
            vb[r] = vec[f >> 4];
          }
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (q0 + r * L < nsum) *at[r] = fma(va[r], vb[r], old[r]);
        }
        if (t == 0 && S.trace_e && sidx < a.cap_samples) S.trace_e[(size_t)w * a.cap_samples + sidx] = E;
        if (EXT && t == 0 && S.samp_psi && sidx < a.cap_samples) {
          const double ld[4] = {bk.ld[0], bk.ld[1], bk.ld[2], bk.ld[3]};  // a copy: bk stays in registers
          sj_compat_sample(S, ld, vec + 2, np, (size_t)w * a.cap_samples + sidx);
        }
      }
      block_sum += E;
      if (++fill == a.block_size) {
        if (t == 0 && live) {
          const double bm = block_sum * inv_block;
          double *s1 = S.acc + (size_t)kSJSumBm * W + w, *s2 = S.acc + (size_t)kSJSumBm2 * W + w;
          *s1 += bm;
          *s2 = fma(bm, bm, *s2);
        }
        block_sum = 0.0;
        fill = 0;
      }
      ++sidx;
    }
  }

  // ---- state out ----
  sync_wave();
  for (int e = lane; e < 3 * N * nslots; e += 64) {
    const int k = e >> lg_slots, sl = e & (nslots - 1);
    if (sl < tile.nw)
      S.pos[(size_t)k * W + tile.w0 + sl] = ((double *)(walkers + (size_t)sl * lay.bytes + lay.pos))[k];
  }
  T *Bo = (T *)S.B;
  for (int e = lane; e < nB * nslots; e += 64) {
    const int k = e >> lg_slots, sl = e & (nslots - 1);
    if (sl < tile.nw) Bo[(size_t)k * W + tile.w0 + sl] = ((T *)(walkers + (size_t)sl * lay.bytes + lay.B))[k];
  }
  if (t == 0 && live) {
    auto column = [&](int k) -> double & { return S.acc[(size_t)k * W + w]; };
    column(kSJAccepted) = acc_in + (double)n_acc;
    if (lu_period || entry_refresh) {
      const double c = column(kSJCondMax), g = column(kSJSingular);
      column(kSJCondMax) = fmax(c, bk.cond);
      column(kSJSingular) = g + bk.singular;
    }
    if (!dmc_step) {
      const double d = column(kSJLdDrift);
      column(kSJBlockSum) = block_sum;
      column(kSJLdDrift) = fmax(d, bk.drift);
#pragma unroll
      for (int k = 0; k < 4; ++k) S.ld[(size_t)k * W + w] = bk.ld[k];
    }
  }
}

// One workgroup per tile (the tiles of one LDS footprint class).
template <typename T, int PROP, bool EXT, int MINW>
__global__ void __launch_bounds__(64, MINW) sj_sweep_kernel(SJArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  sj_tile<T, PROP, EXT>(a, a.tiles[blockIdx.x], lds);
}

// Persistent: a grid sized to the resident workgroups takes every tile of the
// context, longest first, each workgroup drawing the next tile index from a
// device ticket until the list is exhausted (every wave reaches the exit).
// The ticket is zero on entry; sj_ticket_reset_kernel zeroes it after.
template <typename T>
__global__ void __launch_bounds__(64, 2) sj_persistent_kernel(SJArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  for (;;) {
    int t = 0;
    if (threadIdx.x == 0) t = (int)atomicAdd(a.ticket, 1u);
    t = __shfl(t, 0);
    if (t >= a.n_tiles) break;
    sj_tile<T, kSJPropBox, false>(a, a.tiles[t], lds);
    __syncthreads();  // the next tile reuses the LDS
  }
}

__global__ void sj_ticket_reset_kernel(uint32_t *ticket) {
  if (threadIdx.x == 0) *ticket = 0u;
}

__global__ void sj_advance_kernel(SJLaunchState *st, uint32_t n_sweeps, uint32_t n_samples,
                                  uint32_t block_size) {
  if (threadIdx.x != 0) return;
  st->sweeps_done += n_sweeps;
  st->block_fill = (uint32_t)(((uint64_t)st->block_fill + n_samples) % block_size);
  st->trace_sweeps += n_sweeps;
  st->trace_samples += n_samples;
}

__global__ void sj_state_set_kernel(SJLaunchState *st, SJLaunchState v) {
  if (threadIdx.x == 0) *st = v;
}

hipError_t launch_sj_state_set(SJLaunchState *state, const SJLaunchState &v, hipStream_t stream) {
  hipLaunchKernelGGL(sj_state_set_kernel, dim3(1), dim3(64), 0, stream, state, v);
  return hipGetLastError();
}

hipError_t launch_sj_advance(SJLaunchState *state, uint32_t n_sweeps, uint32_t n_samples,
                             uint32_t block_size, hipStream_t stream) {
  hipLaunchKernelGGL(sj_advance_kernel, dim3(1), dim3(64), 0, stream, state, n_sweeps, n_samples,
                     block_size);
  return hipGetLastError();
}

template <typename T, int PROP, bool EXT, int MINW>
static hipError_t launch_sj_m(const SJArgs &a, int n_tiles, size_t lds_bytes, hipStream_t stream) {
  if (lds_bytes > 65536) {
    // more than the default 64 KiB of dynamic LDS needs an opt-in per kernel
    const hipError_t e = hipFuncSetAttribute((const void *)sj_sweep_kernel<T, PROP, EXT, MINW>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((sj_sweep_kernel<T, PROP, EXT, MINW>), dim3(n_tiles), dim3(64), lds_bytes, stream, a);
  return hipGetLastError();
}

template <typename T, int PROP, bool EXT>
static hipError_t launch_sj_e(const SJArgs &a, int n_tiles, size_t lds_bytes, hipStream_t stream) {
  if constexpr (PROP == kSJPropLearned)
    if (a.one_wave) return launch_sj_m<T, PROP, EXT, 1>(a, n_tiles, lds_bytes, stream);
  return launch_sj_m<T, PROP, EXT, 2>(a, n_tiles, lds_bytes, stream);
}

template <typename T, int PROP>
static hipError_t launch_sj_t(const SJArgs &a, int n_tiles, size_t lds_bytes, hipStream_t stream) {
  return a.ext ? launch_sj_e<T, PROP, true>(a, n_tiles, lds_bytes, stream)
               : launch_sj_e<T, PROP, false>(a, n_tiles, lds_bytes, stream);
}

template <typename T>
static hipError_t launch_sj_p(const SJArgs &a, int workgroups, size_t lds_bytes, hipStream_t stream) {
  if (lds_bytes > 65536) {
    const hipError_t e = hipFuncSetAttribute((const void *)sj_persistent_kernel<T>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(sj_persistent_kernel<T>, dim3(workgroups), dim3(64), lds_bytes, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(sj_ticket_reset_kernel, dim3(1), dim3(64), 0, stream, a.ticket);
  return hipGetLastError();
}

hipError_t launch_sj_persistent(const SJArgs &a, int workgroups, int fp32, size_t lds_bytes, hipStream_t stream) {
  if (a.n_tiles <= 0 || workgroups <= 0) return hipSuccess;
  return fp32 ? launch_sj_p<float>(a, workgroups, lds_bytes, stream)
              : launch_sj_p<double>(a, workgroups, lds_bytes, stream);
}

int sj_persistent_occupancy(int fp32, size_t lds_bytes) {
  int n = 0;
  const hipError_t e =
      fp32 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, sj_persistent_kernel<float>, 64, lds_bytes)
           : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, sj_persistent_kernel<double>, 64, lds_bytes);
  return e == hipSuccess ? n : 0;
}

namespace {
// One optimiser step of a Slater-Jastrow system on the device (the loop of
// VmcRunner::run_optimization, src/vmc/src/vmc.rs:43-179): the reduced
// sums of the system's NP parameters (columns sj_columns(NP)),
// Optimizer::compute_parameter_update,
// then the parameters the sweep kernel reads (sys->p) and, with the
// exponent scale, the exponents s zeta0_m.
template <int NP>
__global__ void sj_vmc_step_kernel(const double *red, double n_samples, double *params, mole_optimizer *opt,
                                   double *log, SJSysDev *sys, const double *zeta0, double *zeta, int n_basis) {
  __shared__ double scale;
  __shared__ int updated;
  if (threadIdx.x == 0) {
    double so[NP], soe[NP], soo[NP * NP], dp[NP], pars[NP];
    for (int k = 0; k < NP; ++k) {
      so[k] = red[kSJSumO + k];
      soe[k] = red[sj_sum_oe(NP) + k];
      pars[k] = params[k];
      for (int l = k; l < NP; ++l) {
        const int t = k * NP - k * (k - 1) / 2 + (l - k);  // upper-triangle position of (k, l)
        soo[k * NP + l] = red[sj_sum_oo(NP) + t];
        soo[l * NP + k] = red[sj_sum_oo(NP) + t];
      }
    }
    const int rc = optimizer_update<NP>(opt, n_samples, red[kSJSumE], so, soe, soo, pars, dp, nullptr);
    log[0] = red[kSJSumE];
    log[1] = red[kSJSumE2];
    log[2] = red[kSJSumBm];
    log[3] = red[kSJSumBm2];
    log[4] = red[kSJAccepted];
    log[5] = (double)rc;
    log[6] = n_samples;
    log[7] = 0.0;
    updated = rc == 0;
    if (rc == 0)
      for (int k = 0; k < NP; ++k) {
        params[k] = pars[k] + dp[k];
        sys->p[k] = params[k];
      }
    scale = NP == kSJNParam ? params[kSJNParam - 1] : 1.0;
  }
  __syncthreads();
  if (NP == kSJNParam && updated)
    for (int m = threadIdx.x; m < n_basis; m += blockDim.x) zeta[m] = scale * zeta0[m];
}
}  // namespace

hipError_t launch_sj_vmc_step(const double *red, double n_samples, int n_params, double *params, mole_optimizer *opt,
                              double *log, SJSysDev *sys, const double *zeta0, double *zeta, int n_basis,
                              hipStream_t stream) {
  if (n_params == kSJNParam)
    hipLaunchKernelGGL(sj_vmc_step_kernel<kSJNParam>, dim3(1), dim3(64), 0, stream, red, n_samples, params, opt,
                       log, sys, zeta0, zeta, n_basis);
  else
    hipLaunchKernelGGL(sj_vmc_step_kernel<kSJNParam - 1>, dim3(1), dim3(64), 0, stream, red, n_samples, params,
                       opt, log, sys, zeta0, zeta, n_basis);
  return hipGetLastError();
}

hipError_t launch_sj(const SJArgs &a, int n_tiles, int fp32, int proposal, size_t lds_bytes,
                     hipStream_t stream) {
  if (n_tiles <= 0) return hipSuccess;
  if (proposal == kSJPropDiffuse)
    return fp32 ? launch_sj_t<float, kSJPropDiffuse>(a, n_tiles, lds_bytes, stream)
                : launch_sj_t<double, kSJPropDiffuse>(a, n_tiles, lds_bytes, stream);
  if (proposal == kSJPropLearned)
    return fp32 ? launch_sj_t<float, kSJPropLearned>(a, n_tiles, lds_bytes, stream)
                : launch_sj_t<double, kSJPropLearned>(a, n_tiles, lds_bytes, stream);
  return fp32 ? launch_sj_t<float, kSJPropBox>(a, n_tiles, lds_bytes, stream)
              : launch_sj_t<double, kSJPropBox>(a, n_tiles, lds_bytes, stream);
}

}  // namespace mole
