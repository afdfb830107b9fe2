// HIP kernels for CDNA4 (gfx950): rate constants, source term, analytic
// Jacobian and the TR-BDF2 box-model integrator.
//
// Mapping: one cell per 64-lane wavefront (one wavefront per workgroup).
//   * per-species vectors (state, stage values, residuals, Newton updates)
//     live in registers: internal species a on lane a % 64, slot a / 64;
//   * data other lanes read goes through LDS: concentrations, rate
//     constants, rate-of-progress / derivative / segment scratch, and the
//     dense iteration matrix I - c h J with its LU factors;
//   * species are numbered in a fill-reducing elimination order compiled
//     from the mechanism, so the dense LU meets few nonzero multipliers.
// LU with partial pivoting: the pivot row is found with one ballot when the
// diagonal already has the largest magnitude in its column (the common
// case) and with a wavefront arg-max otherwise; rows whose multiplier is
// exactly zero are skipped by the whole wavefront; lanes own the columns of
// the trailing update; the Newton right-hand side is eliminated alongside
// the matrix so only back substitution remains.
// The iteration matrix and its factors are in TA precision (double for the
// all-FP64 form, float for the mixed form); everything else is FP64.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <mutex>

#include "detmath.h"
#include "device_mech.hpp"

namespace tchem_amd {

// Optional per-phase cycle counters for profiling builds (-DTCHEM_PHASE_TIMERS):
// wavefront-summed shader-clock cycles of the source term, Jacobian assembly,
// factorisation, back substitution and whole cells.
#ifdef TCHEM_PHASE_TIMERS
__device__ unsigned long long g_phase_cycles[16];
__shared__ unsigned long long tchem_pt_lds[16][16];  // [wavefront][slot], flushed per cell
#define TCHEM_PT_BEGIN(nm) const unsigned long long tchem_pt_##nm = __builtin_readcyclecounter();
#define TCHEM_PT_END(nm, slot)          \
  if ((threadIdx.x & 63) == 0)          \
    ::tchem_amd::tchem_pt_lds[threadIdx.x >> 6][slot] += __builtin_readcyclecounter() - tchem_pt_##nm;
#define TCHEM_PT_RESET() \
  if ((threadIdx.x & 63) < 16) tchem_pt_lds[threadIdx.x >> 6][threadIdx.x & 63] = 0;
#define TCHEM_PT_FLUSH()                                                                          \
  if ((threadIdx.x & 63) < 16 && tchem_pt_lds[threadIdx.x >> 6][threadIdx.x & 63])                \
    atomicAdd(&g_phase_cycles[threadIdx.x & 63], tchem_pt_lds[threadIdx.x >> 6][threadIdx.x & 63]); \
  if ((threadIdx.x & 63) < 16) tchem_pt_lds[threadIdx.x >> 6][threadIdx.x & 63] = 0;
#else
#define TCHEM_PT_BEGIN(nm)
#define TCHEM_PT_END(nm, slot)
#define TCHEM_PT_RESET()
#define TCHEM_PT_FLUSH()
#endif

}  // namespace tchem_amd

#include "mfma_lu.hpp"

namespace tchem_amd {

namespace {

constexpr int kWave = 64;

// Wavefront-scope barrier for data exchanged through LDS between the lanes
// of one wavefront: the LDS executes a wavefront's operations in order, so
// only compiler reordering has to be prevented (no s_waitcnt, no s_barrier).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double readlane(double v, int l) {
  const long long x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane(int(x & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane(int(x >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ float readlane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

__device__ __forceinline__ unsigned long long ballot(bool p) { return __ballot(p); }

// value of slot `idx` (lane idx % 64, register slot idx / 64) on every lane
template <int QM, typename TA>
__device__ __forceinline__ TA bcast(const TA (&v)[QM], int idx) {
  const int q = idx >> 6, l = idx & 63;
  TA out = TA(0);
#pragma unroll
  for (int s = 0; s < QM; ++s)
    if (s == q) out = readlane(v[s], l);
  return out;
}

// pow(double, int) of the reference for the small integer powers of
// mechanisms: repeated multiplication (x^2 is the correctly rounded square)
__device__ __forceinline__ double pow_small(double x, int n) { return tchem_ipow(x, n); }

// Rate constant of reaction r: src/core/impl/TChem_Impl_KForwardAerosol.hpp:54-131,
// in the reference's expression order, with the portable exp / log / pow of
// detmath.h and no fused operations, so every device and the host give the
// same bits.
__device__ double rate_constant(const DevMech& M, int r, double t, double p, double t_1, double conv,
                                const double* photo) {
#pragma clang fp contract(off)
  const double* P = M.ratePar() + 8 * r;
  const double one = 1.0;
  const int kind = M.rateKind()[r];
  double k;
  if (kind == 0) {  // Arrhenius
    double A = P[0];
    const int slot = M.photoSlot()[r];
    if (photo != nullptr && slot >= 0) A = photo[slot];
    k = A * tchem_exp(P[2] * t_1) * (P[1] == 0.0 ? one : tchem_pow(t / P[3], P[1])) *
        (P[4] == 0.0 ? one : (one + P[4] * p));
  } else if (kind == 1) {  // Troe
    const double k0 = P[0] * (P[2] == 0.0 ? one : tchem_exp(P[2] * t_1)) *
                      (P[1] == 0.0 ? one : tchem_pow(t / 300.0, P[1])) * conv;
    const double k0_kinf = k0 / (P[3] * (P[5] == 0.0 ? one : tchem_exp(P[5] * t_1)) *
                                 (P[4] == 0.0 ? one : tchem_pow(t / 300.0, P[4])));
    const double lg = tchem_log10(k0_kinf) / P[7];
    k = k0 / (1.0 + k0_kinf) * tchem_pow(P[6], 1.0 / (1.0 + lg * lg));
  } else {  // CMAQ_H2O2
    k = P[0] * tchem_exp(P[2] * t_1) * (P[1] == 0.0 ? one : tchem_pow(t / 300.0, P[1])) +
        P[3] * tchem_exp(P[5] * t_1) * (P[4] == 0.0 ? one : tchem_pow(t / 300.0, P[4])) * conv;
  }
  return k * tchem_ipow(conv, M.convExp()[r]);
}

template <typename TA>
struct CellLds {
  TA* A;        // [m][m] iteration matrix / LU factors (row-major, lda = m)
  double* c;    // [nSpec] concentrations: active (internal order) then constant
  double* kf;   // [nReac] rate constants
  double* scr;  // [max(nReac, nPairs)] rate of progress or derivative pairs
  double* seg;  // [nSeg] source-term segment sums
  TA* rdiag;    // [m] reciprocal pivots 1 / u_kk
  int* swp;     // [2m] row interchanges (k, p) of the factorisation
  const double* src;  // nullable: this cell's external sources [m], reference order
};

template <typename TA>
__device__ CellLds<TA> carve(char* base, const DevMech& M, bool withMatrix = true) {
  CellLds<TA> L;
  size_t off = withMatrix ? sizeof(TA) * size_t(M.m) * size_t(M.m) : 0;
  off = (off + 15) & ~size_t(15);
  L.A = reinterpret_cast<TA*>(base);
  L.c = reinterpret_cast<double*>(base + off);
  L.kf = L.c + M.nSpec;
  L.scr = L.kf + M.nReac;
  const int nScr = M.nReac > M.nPairs ? M.nReac : M.nPairs;
  L.seg = L.scr + nScr;
  L.rdiag = reinterpret_cast<TA*>(L.seg + M.nSeg);
  L.swp = reinterpret_cast<int*>(L.seg + M.nSeg + M.m);
  L.src = nullptr;
  return L;
}

// rate of progress of reaction r at the concentrations in LDS
__device__ __forceinline__ double rate_of_progress(const DevMech& M, const double* c, const double* kf, int r) {
  double v = kf[r];
  const int* sp = M.reacSpec() + r * M.maxR;
  const int* pw = M.reacPow() + r * M.maxR;
  for (int j = 0; j < M.maxR; ++j) {
    const int s = sp[j];
    if (s < 0) break;
    v *= pow_small(c[s], pw[j]);
  }
  return v;
}

// omega (internal order) at the concentrations in LDS; result in registers.
// src/core/impl/TChem_Impl_ReactionRatesAerosol.hpp:78-138 as a gather: one
// lane per species adds the emission rate, then nu * rop of every reactant
// and product entry of that species one at a time, in the order of the
// reference's loops (the serial order of its atomic adds), each product
// rounded before the add: the same sum, bit for bit.
template <int QM, typename TA>
__device__ void source_term_from_lds(const DevMech& M, const CellLds<TA>& L, int lane, double (&f)[QM]) {
#pragma clang fp contract(off)
#pragma unroll 2
  for (int r = lane; r < M.nReac; r += kWave) L.scr[r] = rate_of_progress(M, L.c, L.kf, r);
  wave_sync();
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int a = lane + kWave * q;
    double s = 0.0;
    if (a < M.m) {
      s = M.emission()[a];
      if (L.src) s += L.src[M.perm()[a]];
      const int e1 = M.serOmegaPtr()[a + 1];
      for (int e = M.serOmegaPtr()[a]; e < e1; ++e) {
        const double v = M.serOmegaCoef()[e] * L.scr[M.serOmegaReac()[e]];
        s = s + v;
      }
    }
    f[q] = s;
  }
  wave_sync();
}

template <int QM, typename TA>
__device__ void eval_rhs(const DevMech& M, const CellLds<TA>& L, int lane, const double (&u)[QM], double (&f)[QM]) {
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int a = lane + kWave * q;
    if (a < M.m) L.c[a] = u[q];
  }
  wave_sync();
  source_term_from_lds<QM>(M, L, lane, f);
}

// A = diag * I + scale * J at the concentrations in LDS.  J is the analytic
// Jacobian of source_term_from_lds: derivative pairs d rop_r / d c_s, then
// per structural entry the contributions nu * d one at a time in the
// reference loop order (reaction, reactant slot of the derivative, then the
// reactants and products of the reaction), each product rounded before the
// add.  With external_order the entries are placed at the reference's
// species indices.
template <typename TA>
__device__ void assemble_jacobian_from_lds(const DevMech& M, const CellLds<TA>& L, int lane, double diag, double scale,
                                           bool external_order) {
#pragma clang fp contract(off)
  const int m = M.m;
  {
    const size_t bytes = sizeof(TA) * size_t(m) * size_t(m);
    const int n16 = int(bytes / 16);
    uint4* A16 = reinterpret_cast<uint4*>(L.A);
    for (int idx = lane; idx < n16; idx += kWave) A16[idx] = make_uint4(0, 0, 0, 0);
    for (int idx = n16 * int(16 / sizeof(TA)) + lane; idx < m * m; idx += kWave) L.A[idx] = TA(0);
  }
  // derivative pairs: d rop_r / d c_s = k * n_s c_s^(n_s-1) * prod_{j != s} c_j^n_j
  for (int r = lane; r < M.nReac; r += kWave) {
    const int p0 = M.pairPtr()[r], p1 = M.pairPtr()[r + 1];
    if (p0 == p1) continue;
    const int* sp = M.reacSpec() + r * M.maxR;
    const int* pw = M.reacPow() + r * M.maxR;
    for (int p = p0; p < p1; ++p) {
      const int js = M.pairSlot()[p];
      const int ns = pw[js];
      double d = L.kf[r] * double(ns) * pow_small(L.c[sp[js]], ns - 1);
      for (int j = 0; j < M.maxR; ++j) {
        const int s = sp[j];
        if (s < 0) break;
        if (j == js) continue;
        d *= pow_small(L.c[s], pw[j]);
      }
      L.scr[p] = d;
    }
  }
  wave_sync();
  for (int n = lane; n < M.nSerJ; n += kWave) {
    double s = 0.0;
    const int e1 = M.serJPtr()[n + 1];
    for (int e = M.serJPtr()[n]; e < e1; ++e) {
      const double v = M.serJCoef()[e] * L.scr[M.serJPair()[e]];
      s = s + v;
    }
    const int rc = M.serJRowCol()[n];
    int row = rc >> 16, col = rc & 0xffff;
    const double v = (row == col ? diag : 0.0) + scale * s;
    if (external_order) {
      row = M.perm()[row];
      col = M.perm()[col];
    }
    L.A[row * m + col] = TA(v);
  }
  wave_sync();
}

// In-place LU with partial pivoting of the m x m matrix in LDS (row
// interchanges recorded in L.swp, count in nswp), eliminating the right-hand
// side b (row a on lane a % 64, slot a / 64) alongside.  Same arithmetic as
// oracle_lu + the forward half of oracle_lu_solve: pivot = first row of
// largest |a_ik|, l = a_ik * (1 / a_kk), a_ij = fma(-l, a_kj, a_ij),
// b_i = fma(-l, b_k, b_i).  The reciprocal pivots are kept for the back
// substitution.  Returns false for a zero or non-finite pivot.
template <int QM, typename TA>
__device__ bool lu_factor_fused(const CellLds<TA>& L, int m, int lane, TA (&b)[QM], int& nswp) {
#pragma clang fp contract(off)
  TA* A = L.A;
  nswp = 0;
  for (int k = 0; k < m; ++k) {
    TA a[QM], uk[QM];
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      a[q] = (i >= k && i < m) ? A[i * m + k] : TA(0);
      const int j = k + 1 + lane + kWave * q;
      uk[q] = (j < m) ? A[k * m + j] : TA(0);
    }
    const TA akk = bcast<QM>(a, k);
    const TA dabs = fabs(akk);
    unsigned long long gt = 0;
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      gt |= ballot(i > k && i < m && fabs(a[q]) > dabs);
    }
    int p = k;
    TA apiv = akk;
    if (gt != 0 || !(dabs > TA(0))) {
      // arg-max over rows i >= k; ties go to the smallest row index
      TA best = TA(-1);
      int bi = m;
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int i = lane + kWave * q;
        if (i >= k && i < m) {
          const TA v = fabs(a[q]);
          if (v > best) { best = v; bi = i; }
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        const TA ob = __shfl_xor(best, off, kWave);
        const int oi = __shfl_xor(bi, off, kWave);
        if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
      }
      p = __builtin_amdgcn_readfirstlane(bi);
      if (p >= m || !(best > TA(0))) return false;
      apiv = bcast<QM>(a, p);
    }
    if (!isfinite(double(apiv))) return false;
    if (p != k) {
      for (int j = lane; j < m; j += kWave) {
        const TA t = A[k * m + j];
        A[k * m + j] = A[p * m + j];
        A[p * m + j] = t;
      }
      const TA bk = bcast<QM>(b, k), bp = bcast<QM>(b, p);
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int i = lane + kWave * q;
        if (i == k) { a[q] = apiv; b[q] = bp; }
        else if (i == p) { a[q] = akk; b[q] = bk; }
      }
      if (lane == 0) {
        L.swp[2 * nswp] = k;
        L.swp[2 * nswp + 1] = p;
      }
      ++nswp;
      wave_sync();
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int j = k + 1 + lane + kWave * q;
        uk[q] = (j < m) ? A[k * m + j] : TA(0);
      }
    }
    const TA bk = bcast<QM>(b, k);
    const TA inv = TA(1) / apiv;
    if (lane == 0) L.rdiag[k] = inv;
    TA l[QM];
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      l[q] = TA(0);
      if (i > k && i < m && a[q] != TA(0)) {
        l[q] = a[q] * inv;
        A[i * m + k] = l[q];
        b[q] = fma(-l[q], bk, b[q]);
      }
    }
    // trailing update: rows with a nonzero multiplier, two at a time
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      unsigned long long mask = ballot(l[q] != TA(0));
      while (mask) {
        const int b0 = __builtin_ctzll(mask);
        mask &= mask - 1;
        const TA l0 = readlane(l[q], b0);
        const int i0 = kWave * q + b0;
        if (mask) {
          const int b1 = __builtin_ctzll(mask);
          mask &= mask - 1;
          const TA l1 = readlane(l[q], b1);
          const int i1 = kWave * q + b1;
#pragma unroll
          for (int c = 0; c < QM; ++c) {
            const int j = k + 1 + lane + kWave * c;
            if (j < m && uk[c] != TA(0)) {
              const TA x0 = A[i0 * m + j];
              const TA x1 = A[i1 * m + j];
              A[i0 * m + j] = fma(-l0, uk[c], x0);
              A[i1 * m + j] = fma(-l1, uk[c], x1);
            }
          }
        } else {
#pragma unroll
          for (int c = 0; c < QM; ++c) {
            const int j = k + 1 + lane + kWave * c;
            if (j < m && uk[c] != TA(0)) A[i0 * m + j] = fma(-l0, uk[c], A[i0 * m + j]);
          }
        }
      }
    }
    wave_sync();
  }
  return true;
}

// Forward elimination with stored factors: interchanges, then unit-lower L.
template <int QM, typename TA>
__device__ void lu_forward(const CellLds<TA>& L, int m, int lane, TA (&b)[QM], int nswp) {
#pragma clang fp contract(off)
  const TA* A = L.A;
  for (int s = 0; s < nswp; ++s) {
    const int k = L.swp[2 * s], p = L.swp[2 * s + 1];
    const TA bk = bcast<QM>(b, k), bp = bcast<QM>(b, p);
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      if (i == k) b[q] = bp;
      else if (i == p) b[q] = bk;
    }
  }
  TA col[QM];
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    col[q] = (i > 0 && i < m) ? A[i * m] : TA(0);
  }
  for (int k = 0; k < m - 1; ++k) {
    TA nxt[QM];
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      nxt[q] = (i > k + 1 && i < m) ? A[i * m + k + 1] : TA(0);
    }
    const TA yk = bcast<QM>(b, k);
    if (yk != TA(0)) {
#pragma unroll
      for (int q = 0; q < QM; ++q) b[q] = fma(-col[q], yk, b[q]);
    }
#pragma unroll
    for (int q = 0; q < QM; ++q) col[q] = nxt[q];
  }
}

// Back substitution with the upper factor (column order, as oracle_lu_solve);
// the next column is fetched from LDS while the current one is applied.
template <int QM, typename TA>
__device__ void lu_back(const CellLds<TA>& L, int m, int lane, TA (&b)[QM]) {
#pragma clang fp contract(off)
  const TA* A = L.A;
  TA col[QM];
  TA ukk = L.rdiag[m - 1];
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    col[q] = (i < m - 1) ? A[i * m + m - 1] : TA(0);
  }
  for (int k = m - 1; k >= 0; --k) {
    TA nxt[QM];
    TA nkk = TA(1);
#pragma unroll
    for (int q = 0; q < QM; ++q) nxt[q] = TA(0);
    if (k > 0) {
      nkk = L.rdiag[k - 1];
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int i = lane + kWave * q;
        nxt[q] = (i < k - 1) ? A[i * m + k - 1] : TA(0);
      }
    }
    const TA xk = bcast<QM>(b, k) * ukk;  // ukk holds 1 / u_kk
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      if (i == k) b[q] = xk;
    }
    if (xk != TA(0)) {
#pragma unroll
      for (int q = 0; q < QM; ++q) b[q] = fma(-col[q], xk, b[q]);
    }
    ukk = nkk;
#pragma unroll
    for (int q = 0; q < QM; ++q) col[q] = nxt[q];
  }
}

}  // namespace
}  // namespace tchem_amd

#include "sparse_exec.hpp"

namespace tchem_amd {
namespace {

// ---- backends -----------------------------------------------------------------
// Both provide: Lds (per-cell LDS view), Fact (state of the stored factors),
// carve, init, evaluate (f at u; for a Newton iteration also the residual
// and, when refreshing, the iteration matrix), factor_solve (factorise +
// solve; false on a bad pivot) and solve (stored factors).

template <typename TA_, int QM>
struct DenseBackend {
  using TA = TA_;
  static constexpr bool kCollective = false;  // factorisation by the whole workgroup (collective_solve)
  using Lds = CellLds<TA>;
  struct Fact { int nswp = 0; };
  // unknowns, state row length, state column and tolerances of unknown ai
  static __device__ __forceinline__ int unknowns(const IntegratorArgs& a) { return a.M.m; }
  static __device__ __forceinline__ int rowDim(const IntegratorArgs& a) { return a.M.nSpec + 3; }
  static __device__ __forceinline__ int column(const IntegratorArgs& a, int ai) { return 3 + a.M.perm()[ai]; }
  static __device__ __forceinline__ void tolerance(const IntegratorArgs& a, const Lds&, int ai, double& atol,
                                                   double& rtol) {
    const int xs = a.M.perm()[ai];
    atol = a.tol_time[2 * xs];
    rtol = a.tol_time[2 * xs + 1];
  }
  static __device__ __forceinline__ void load_rates(const IntegratorArgs& a, const Lds& L, const double* kf, int lane) {
    for (int r = lane; r < a.M.nReac; r += kWave) L.kf[r] = kf[r];
  }
  // per-cell bindings: this cell's external sources
  static __device__ __forceinline__ void bind(const IntegratorArgs& a, Lds& L, int cell) {
    L.src = a.ext ? a.ext + size_t(cell) * a.M.m : nullptr;
  }
  static __device__ void stage(const IntegratorArgs&, char*) {}
  static __device__ Lds carve(char* base, const IntegratorArgs& a, int) { return tchem_amd::carve<TA>(base, a.M); }
  static __device__ void init(const IntegratorArgs&, const Lds&, int) {}
  // f at u; for a Newton iteration also x = -(u - bc - ch f) and, when
  // refreshing, the iteration matrix I - ch J at the same u
  static __device__ void evaluate(const IntegratorArgs& a, const Lds& L, int lane, const double (&u)[QM],
                                  const double (&bc)[QM], double ch, bool newton, bool refresh, double (&f)[QM],
                                  TA (&x)[QM]) {
#pragma clang fp contract(off)
    eval_rhs<QM>(a.M, L, lane, u, f);
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      x[q] = (newton && i < a.M.m) ? TA(-(u[q] - bc[q] - ch * f[q])) : TA(0);
    }
    if (refresh) assemble_jacobian_from_lds(a.M, L, lane, 1.0, -ch, false);
  }
  static __device__ bool factor_solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM], Fact& fs) {
    if (!lu_factor_fused<QM>(L, a.M.m, lane, x, fs.nswp)) return false;
    lu_back<QM>(L, a.M.m, lane, x);
    return true;
  }
  static __device__ void solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM], const Fact& fs) {
    lu_forward<QM>(L, a.M.m, lane, x, fs.nswp);
    lu_back<QM>(L, a.M.m, lane, x);
  }
};

// time tolerances of unknown ai from the staged table at LDS address tol, or
// (index: its row) from the caller's
template <class Index>
__device__ __forceinline__ void staged_tolerance(const IntegratorArgs& a, unsigned tol, int ai, Index index,
                                                 double& atol, double& rtol) {
  if (a.W.tolStaged) {
    const vec2<double> t = lds_get<vec2<double>>(tol + 16 * ai);
    atol = t.x;
    rtol = t.y;
  } else {
    const int xs = index(ai);
    atol = a.tol_time[2 * xs];
    rtol = a.tol_time[2 * xs + 1];
  }
}

// Sparse form: the encoded programs (lowered.hpp), from device memory or
// staged into the workgroup's LDS.
template <typename TA_, int QM, bool STAGED>
struct SparseBackend {
  using TA = TA_;
  static constexpr bool kCollective = false;  // factorisation by the whole workgroup (collective_solve)
  // QM 4 instances take the programs of cell regions above 64 KiB too
  static constexpr int SH = QM < 4 ? 0 : (sizeof(TA) == 8 ? 3 : 2);
  using Lds = SpLds<TA, STAGED>;
  struct Fact {};
  static __device__ __forceinline__ int unknowns(const IntegratorArgs& a) { return a.M.m; }
  static __device__ __forceinline__ int rowDim(const IntegratorArgs& a) { return a.M.nSpec + 3; }
  static __device__ __forceinline__ int column(const IntegratorArgs& a, int ai) { return 3 + a.M.perm()[ai]; }
  static __device__ __forceinline__ void tolerance(const IntegratorArgs& a, const Lds& L, int ai, double& atol,
                                                   double& rtol) {
    staged_tolerance(a, L.tol, ai, [&](int i) { return a.M.perm()[i]; }, atol, rtol);
  }
  static __device__ __forceinline__ void bind(const IntegratorArgs& a, Lds& L, int cell) {
    L.src = a.ext ? a.ext + size_t(cell) * a.M.m : nullptr;
  }
  static __device__ void stage(const IntegratorArgs& a, char* base) {
    stage_sparse<STAGED>(a.W, reinterpret_cast<const unsigned*>(a.M.ib) + a.W.oWords, a.M.db + a.W.oCoef, base);
    double* tol = reinterpret_cast<double*>(base + sparseStageBytes(a.W, 0, STAGED));
    const int n = a.W.tolStaged ? 2 * a.M.m : 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) tol[i] = a.tol_time[2 * a.M.perm()[i >> 1] + (i & 1)];
    __syncthreads();
  }
  static __device__ Lds carve(char* base, const IntegratorArgs& a, int wave) {
    return carve_sparse<TA, STAGED>(a.W, reinterpret_cast<const unsigned*>(a.M.ib) + a.W.oWords, a.M.m, base,
                                    a.cellBytes, wave);
  }
  static __device__ void init(const IntegratorArgs& a, const Lds& L, int lane) { sp_init(a.W, L, a.M.m, lane); }
  static __device__ __forceinline__ void load_rates(const IntegratorArgs& a, const Lds& L, const double* kf, int lane) {
    sp_load_rates<SH>(a.W, L, kf, lane);
  }
  static __device__ __forceinline__ void put_c(const IntegratorArgs& a, const Lds& L, int lane, const double (&u)[QM]) {
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      if (i < a.M.m) lds_put<double>(L.cell + a.W.oC + 8 * i, u[q]);
    }
    wave_sync();
  }
  static __device__ __forceinline__ void evaluate(const IntegratorArgs& a, const Lds& L, int lane,
                                                  const double (&u)[QM], const double (&bc)[QM], double ch,
                                                  bool newton, bool refresh, double (&f)[QM], TA (&x)[QM]) {
    TCHEM_PT_BEGIN(rates)
    // emission and external sources of this lane's species, on their way while the rates are computed
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      f[q] = 0.0;
      if (i < a.M.m) {
        f[q] = a.M.emission()[i];
        if (L.src) f[q] += L.src[a.M.perm()[i]];
      }
    }
    put_c(a, L, lane, u);
    sp_rates<SH>(a.W, L, lane, refresh);
    wave_sync();
    TCHEM_PT_END(rates, 11)
    TCHEM_PT_BEGIN(rows)
    sp_sums<SH>(L, a.W.oSegHdr, a.W.oSeg, a.W.nSeg, L.coef, L.cell + a.W.oS, lane);
    wave_sync();
    sp_rows<SH, QM>(a.W, L, lane, f);
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      x[q] = (newton && i < a.M.m) ? TA(-(u[q] - bc[q] - ch * f[q])) : TA(0);
      if (newton && i < a.M.m) lds_put<TA>(L.cell + a.W.oR + 2 * sizeof(TA) * i, x[q]);
    }
    wave_sync();
    TCHEM_PT_END(rows, 13)
    TCHEM_PT_BEGIN(sums)
    if (refresh) {
      sp_jacobian<SH>(a.W, L, lane, TA(-ch));
      wave_sync();
    }
    TCHEM_PT_END(sums, 12)
  }
  // after the back substitution the right-hand side holds u_ii x_i
  static __device__ __forceinline__ void get_x(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM]) {
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      x[q] = TA(0);
      if (i < a.M.m) {
        const vec2<TA> v = lds_get<vec2<TA>>(L.cell + a.W.oR + 2 * sizeof(TA) * i);
        x[q] = v.x * v.y;
      }
    }
  }
  static __device__ __forceinline__ bool factor_solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM],
                                                      Fact&) {
    TCHEM_PT_BEGIN(lu)
    sp_lu<SH>(L, L.w, a.W.oLuHdr, a.W.oLu, a.W.oLu1, a.W.nLu, lane);
    const bool ok = sp_pivots<SH, QM>(a.W, L, a.M.m, lane);
    TCHEM_PT_END(lu, 9)
    if (!ok) return false;
    TCHEM_PT_BEGIN(back)
    sp_back<SH>(a.W, L, lane);
    TCHEM_PT_END(back, 10)
    get_x(a, L, lane, x);
    return true;
  }
  static __device__ __forceinline__ void solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM],
                                               const Fact&) {
    sp_lu<SH>(L, L.memory(), a.W.oFwdHdr, a.W.oFwd, a.W.oFwd1, a.W.nFwd, lane);
    sp_back<SH>(a.W, L, lane);
    get_x(a, L, lane, x);
  }
};

struct CellCounters {
  int accepted = 0, rejected = 0, newton_failures = 0, newton_iterations = 0, factorizations = 0, failed = 0;
};

// Whether the rounded quotient a / b is at most 1 (a >= 0; false for NaN, 0 / 0
// and an infinite a), without the division: for finite a and b > 0 the
// quotient rounds above 1 exactly when a > b, since a / b > 1 is at least
// 1 + ulp(b) / b > 1 + 2^-53.  The same for an eighth: 8 a is exact (or
// overflows, and then the quotient is above 1/8 for every b it is compared with).
__device__ __forceinline__ bool ratio_at_most_one(double a, double b) {
  return a < INFINITY && ((a <= b && b > 0.0) || b < 0.0);
}

// One cell of AtmosphericChemistry::runDeviceBatch
// (src/core/TChem_AtmosphericChemistry.cpp:78-163) with the TR-BDF2 step
// control of oracle/oracle.c: integrate_cell, written as a state machine so
// the function evaluation and the linear solve each have a single call site:
//   STEP   start or retry a step: h = min(max(dt, dtmin), tend - t); fail when
//          t + h == t; fetch f(u_n) first if it is not known;
//   FN     f(u_n);
//   NEWTON one Newton iteration of the current stage: residual
//          G(u) = u - bc - ch f(u) and, every jacobian_interval iterations,
//          the iteration matrix I - ch J at the same u; converged when
//          max_i |dx_i| / (atol + rtol |u_i|) <= 1; after max_newton
//          iterations without convergence, or on a zero or non-finite
//          pivot, dt = h/2 and the step is retried (at most 4 attempts);
//   STAGE  f at the converged stage value: after the TR stage set up BDF2;
//          after BDF2 estimate the local error and accept or reject.
// REC: also record the accepted steps for the discrete adjoint (a.rec).
template <class B, int QM, bool REC>
__device__ void integrate_cell(const IntegratorArgs& a, const typename B::Lds& Lw, int cell, int lane) {
  // no implicit fused multiply-adds: the stage, residual and error
  // arithmetic rounds as oracle_run_batch does
#pragma clang fp contract(off)
  using TA = typename B::TA;
  const DevMech& M = a.M;
  const int m = B::unknowns(a), mg = M.m, nSpec = M.nSpec, dim = B::rowDim(a);
  typename B::Lds L = Lw;
  B::bind(a, L, cell);
  const tchem_time_advance_t ta = a.tadv[cell];
  const double tend = ta._tend;
  double* row = a.state + size_t(cell) * dim;
  CellCounters cnt;

  const double t_in = a.t_out[cell];
  if (t_in >= tend || ta._dt < 0.0) {  // skipped (.cpp:83) or already failed
    if (a.stats && lane == 0) a.stats[cell] = tchem_cell_stats_t{0, 0, 0, 0, 0, ta._dt < 0.0 ? 1 : 0, 0, 0};
    if (REC) {
      const int nCkpt0 = a.rec.maxSteps / kAdjointSegment + 1;
      for (int ai = lane; ai < m; ai += kWave) a.rec.ckpt[size_t(cell) * nCkpt0 * m + ai] = row[3 + M.perm()[ai]];
      for (int i = m + lane; i < nSpec; i += kWave) a.rec.consts[size_t(cell) * (nSpec - m) + (i - m)] = row[3 + i];
      if (lane == 0) a.rec.nsteps[cell] = ta._dt < 0.0 ? -1 : 0;
    }
    return;
  }

  const unsigned long long t_start = a.stats ? (unsigned long long)__builtin_amdgcn_s_memrealtime() : 0ull;
  const double gam = 2.0 - 1.41421356237309504880;
  const double c_tr = 0.5 * gam;
  const double a_g = 1.0 / (gam * (2.0 - gam));
  const double a_n = (1.0 - gam) * (1.0 - gam) / (gam * (2.0 - gam));
  const double c_bdf = (1.0 - gam) / (2.0 - gam);
  const double k_err = (-3.0 * gam * gam + 4.0 * gam - 2.0) / (12.0 * (2.0 - gam));

  TCHEM_PT_BEGIN(cell)
  B::load_rates(a, L, a.kf + size_t(cell) * M.nReac, lane);
  for (int i = mg + lane; i < nSpec; i += kWave) L.c[i] = row[3 + i];

  // un (state) and fn (f at un) live across steps; u, bc, est per step
  double un[QM], u[QM], fn[QM], bc[QM], est[QM];
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int ai = lane + kWave * q;
    un[q] = (ai < m) ? row[B::column(a, ai)] : 0.0;
    u[q] = un[q];
    fn[q] = bc[q] = est[q] = 0.0;
  }
  const double atol_n = a.tol_newton[0], rtol_n = a.tol_newton[1];
  const int nCkpt = REC ? a.rec.maxSteps / kAdjointSegment + 1 : 0;
  bool overflow = false;
  if (REC) {
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int ai = lane + kWave * q;
      if (ai < m) a.rec.ckpt[size_t(cell) * nCkpt * m + ai] = un[q];
    }
    for (int i = m + lane; i < nSpec; i += kWave) a.rec.consts[size_t(cell) * (nSpec - m) + (i - m)] = row[3 + i];
  }
  wave_sync();

  const int max_it = ta._num_time_iterations_per_interval;
  const int max_newton = ta._max_num_newton_iterations;
  const int jint = ta._jacobian_interval < 1 ? 1 : ta._jacobian_interval;
  double t = ta._tbeg, dt = ta._dt, h = 0.0, ch = 0.0;
  bool fn_valid = false, failed = false;
  int iter = 0, attempt = 0, stage = 0, nit = 0;
  enum : int { kStep, kFn, kNewton, kStage, kDone };
  int phase = kStep;
  typename B::Fact fs;

  while (phase != kDone) {
    if (phase == kStep) {
      if (iter >= max_it || !(t < tend)) {
        phase = kDone;
        continue;
      }
      h = dt > ta._dtmin ? dt : ta._dtmin;
      if (h > tend - t) h = tend - t;
      if (!(t + h > t)) {  // no representable progress: hard failure
        failed = true;
        phase = kDone;
        continue;
      }
      if (!fn_valid) {
#pragma unroll
        for (int q = 0; q < QM; ++q) u[q] = un[q];
        phase = kFn;
        continue;
      }
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        u[q] = un[q];
        bc[q] = un[q] + c_tr * h * fn[q];
      }
      ch = c_tr * h;
      stage = 0;
      nit = 0;
      phase = kNewton;
      continue;
    }

    if (phase == kNewton && nit >= max_newton) {  // Newton failed: halve the step and retry
      ++cnt.newton_failures;
      dt = 0.5 * h;
      if (++attempt >= 4) {
        failed = true;
        phase = kDone;
      } else {
        phase = kStep;
      }
      continue;
    }
    const bool nw = phase == kNewton;
    const bool refresh = nw && (nit % jint) == 0;
    double f[QM];
    TA x[QM];
    TCHEM_PT_BEGIN(ev)
    B::evaluate(a, L, lane, u, bc, ch, nw, refresh, f, x);
    TCHEM_PT_END(ev, 0)

    if (nw) {
      TCHEM_PT_BEGIN(lin)
      bool ok = true;
      if constexpr (B::kCollective) {  // one call site for the workgroup's factorisation code
        ok = B::collective_solve(a, L, lane, x, refresh);
        if (ok && refresh) ++cnt.factorizations;
      } else if (refresh) {
        ok = B::factor_solve(a, L, lane, x, fs);
        if (ok) ++cnt.factorizations;
      } else {
        B::solve(a, L, lane, x, fs);
      }
      TCHEM_PT_END(lin, refresh ? 2 : 3)
      if (!ok) {  // zero or non-finite pivot
        nit = max_newton;
        continue;
      }
      {
        bool over = false;
#pragma unroll
        for (int q = 0; q < QM; ++q) {
          const int i = lane + kWave * q;
          if (i < m) {
            const double dx = double(x[q]);
            u[q] += dx;
            over |= !ratio_at_most_one(fabs(dx), atol_n + rtol_n * fabs(u[q]));
          }
        }
        ++cnt.newton_iterations;
        ++nit;
        if (ballot(over) == 0) phase = kStage;
      }
      continue;
    }

    if (phase == kFn) {
#pragma unroll
      for (int q = 0; q < QM; ++q) fn[q] = f[q];
      fn_valid = true;
      phase = kStep;
      continue;
    }

    // kStage
    if (stage == 0) {
      // f at the TR-stage value enters the error estimate; the stage value
      // itself only enters the BDF2 constant term
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        est[q] = fn[q] / gam - f[q] / (gam * (1.0 - gam));
        bc[q] = a_g * u[q] - a_n * un[q];
      }
      ch = c_bdf * h;
      stage = 1;
      nit = 0;
      phase = kNewton;
      continue;
    }
    // the largest |lte_i| / (atol_i + rtol_i |u_i|) against 1 (accept) and 1/8 (grow)
    bool above = false, mid = false;
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int ai = lane + kWave * q;
      if (ai < m) {
        double at, rt;
        B::tolerance(a, L, ai, at, rt);
        const double lte = 2.0 * k_err * h * (est[q] + f[q] / (1.0 - gam));
        const double b = at + rt * fabs(u[q]);
        above |= !ratio_at_most_one(fabs(lte), b);
        mid |= !ratio_at_most_one(8.0 * fabs(lte), b);
      }
    }
    const bool reject = ballot(above) != 0, keep = ballot(mid) != 0;
    ++iter;
    attempt = 0;
    phase = kStep;
    if (reject && h > ta._dtmin) {
      ++cnt.rejected;
      dt = 0.25 * h;
      continue;
    }
    t = (h == tend - t) ? tend : t + h;
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      un[q] = u[q];
      fn[q] = f[q];
    }
    dt = keep ? h : 2.0 * h;
    if (dt > ta._dtmax) dt = ta._dtmax;
    if (REC) {
      const int k = cnt.accepted;  // index of this step
      if (k < a.rec.maxSteps) {
        if (lane == 0) a.rec.h[size_t(cell) * a.rec.maxSteps + k] = h;
        if ((k + 1) % kAdjointSegment == 0) {
#pragma unroll
          for (int q = 0; q < QM; ++q) {
            const int ai = lane + kWave * q;
            if (ai < m) a.rec.ckpt[(size_t(cell) * nCkpt + (k + 1) / kAdjointSegment) * m + ai] = un[q];
          }
        }
      } else {
        overflow = true;
      }
    }
    ++cnt.accepted;
  }

  TCHEM_PT_END(cell, 6)
  wave_sync();
  TCHEM_PT_FLUSH()
  double* rowo = a.state_out + size_t(cell) * dim;
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int ai = lane + kWave * q;
    if (ai < m) {
      const int col = B::column(a, ai);
      const double v = failed ? 0.0 : un[q];
      row[col] = v;
      if (rowo != row) rowo[col] = v;
    }
  }
  if (rowo != row)
    for (int i = mg + lane; i < nSpec; i += kWave) rowo[3 + i] = row[3 + i];
  if (lane == 0) {
    rowo[0] = row[0];
    rowo[1] = row[1];
    rowo[2] = row[2];
    a.t_out[cell] = failed ? tend : t;
    a.dt_out[cell] = failed ? -1.0 : dt;
    if (REC) a.rec.nsteps[cell] = (failed || overflow) ? -1 : cnt.accepted;
    if (a.stats) {
      cnt.failed = failed ? 1 : 0;
      a.stats[cell] = tchem_cell_stats_t{cnt.accepted, cnt.rejected, cnt.newton_failures, cnt.newton_iterations,
                                         cnt.factorizations, cnt.failed, t_start,
                                         (unsigned long long)__builtin_amdgcn_s_memrealtime()};
    }
  }
}


// ---- dense LU on the matrix cores (mfma_lu.hpp) ------------------------------
// One cell per workgroup of four wavefronts: wavefront 0 runs integrate_cell
// (FP64 state, residual, error estimate and step control) and hands two
// jobs to the whole workgroup: the FP64 source term (serial per-species
// sums), and at every Newton iteration the assembly of the FP32 iteration
// matrix, which the four wavefronts hold in their registers for the MFMA
// factorisation and solve (mfma::factorAndSolve).  Wavefronts 1-3 wait at
// the workgroup barrier for the next command (source term, factor and
// solve, or finish).

// d rop_r / d c_s of every derivative pair into out (the first part of
// assemble_jacobian_from_lds)
template <typename TO>
__device__ __forceinline__ void derivative_pairs(const DevMech& M, const double* c, const double* kf, TO* out,
                                                 int tid, int nthreads) {
  for (int r = tid; r < M.nReac; r += nthreads) {
    const int p0 = M.pairPtr()[r], p1 = M.pairPtr()[r + 1];
    if (p0 == p1) continue;
    const int* sp = M.reacSpec() + r * M.maxR;
    const int* pw = M.reacPow() + r * M.maxR;
    for (int p = p0; p < p1; ++p) {
      const int js = M.pairSlot()[p];
      const int ns = pw[js];
      double d = kf[r] * double(ns) * pow_small(c[sp[js]], ns - 1);
      for (int j = 0; j < M.maxR; ++j) {
        const int s = sp[j];
        if (s < 0) break;
        if (j == js) continue;
        d *= pow_small(c[s], pw[j]);
      }
      out[p] = TO(d);
    }
  }
}

// LDS bytes of one cell of the MFMA form: the dense cell region without a
// matrix, the FP32 derivative pairs, the source term, then the
// factorisation's region
inline size_t mfmaCellBytes(const DevMech& M, int tiles) {
  auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
  return al(integratorLdsBytes(M, 0)) + al(4 * size_t(M.nPairs + 1)) + al(8 * size_t(M.m)) +
         mfma::luLdsBytes(tiles);
}

// The source term by the whole workgroup (256 threads): rates of progress,
// then the serial per-species gathers of source_term_from_lds into fbuf.
template <class Lds>
__device__ void mfma_rhs_collective(const IntegratorArgs& a, const Lds& L) {
#pragma clang fp contract(off)
  const DevMech& M = a.M;
  const int tid = threadIdx.x;
  for (int r = tid; r < M.nReac; r += 256) L.scr[r] = rate_of_progress(M, L.c, L.kf, r);
  __syncthreads();
  for (int i = tid; i < M.m; i += 256) {
    double s = M.emission()[i];
    if (L.src) s += L.src[M.perm()[i]];
    const int e1 = M.serOmegaPtr()[i + 1];
    for (int e = M.serOmegaPtr()[i]; e < e1; ++e) {
      const double v = M.serOmegaCoef()[e] * L.scr[M.serOmegaReac()[e]];
      s = s + v;
    }
    L.fbuf[i] = s;
  }
  __syncthreads();
}

template <int NB_>
struct MfmaBackend {
  using TA = float;
  static constexpr int NB = NB_, QM = NB / 2;  // 64 unknowns per slot, 32 per tile
  static constexpr bool kCollective = true;  // factorisation by the whole workgroup (collective_solve)
  struct Lds : CellLds<float> {
    float* pairs;   // [nPairs] derivative pairs of the last Jacobian refresh (FP32)
    double* fbuf;   // [m] source term of the workgroup's evaluation
    mfma::Lu lu;
  };
  struct Fact {};
  static __device__ __forceinline__ int unknowns(const IntegratorArgs& a) { return a.M.m; }
  static __device__ __forceinline__ int rowDim(const IntegratorArgs& a) { return a.M.nSpec + 3; }
  static __device__ __forceinline__ int column(const IntegratorArgs& a, int ai) { return 3 + a.M.perm()[ai]; }
  static __device__ __forceinline__ void tolerance(const IntegratorArgs& a, const Lds&, int ai, double& atol,
                                                   double& rtol) {
    const int xs = a.M.perm()[ai];
    atol = a.tol_time[2 * xs];
    rtol = a.tol_time[2 * xs + 1];
  }
  static __device__ __forceinline__ void load_rates(const IntegratorArgs& a, const Lds& L, const double* kf, int lane) {
    for (int r = lane; r < a.M.nReac; r += kWave) L.kf[r] = kf[r];
  }
  static __device__ __forceinline__ void bind(const IntegratorArgs& a, Lds& L, int cell) {
    L.src = a.ext ? a.ext + size_t(cell) * a.M.m : nullptr;
  }
  static __device__ void stage(const IntegratorArgs&, char*) {}
  static __device__ Lds carve(char* base, const IntegratorArgs& a, int) {
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    Lds L;
    static_cast<CellLds<float>&>(L) = tchem_amd::carve<float>(base, a.M, false);
    size_t off = al(integratorLdsBytes(a.M, 0));
    L.pairs = reinterpret_cast<float*>(base + off);
    off += al(4 * size_t(a.M.nPairs + 1));
    L.fbuf = reinterpret_cast<double*>(base + off);
    off += al(8 * size_t(a.M.m));
    L.lu = mfma::carveLu(base + off, NB);
    return L;
  }
  static __device__ void init(const IntegratorArgs&, const Lds&, int) {}
  // f (FP64, serial source term) and the Newton residual; on a refresh c h
  // of the iteration matrix (its derivative pairs and assembly are the
  // workgroup's, in factor_solve)
  static __device__ void evaluate(const IntegratorArgs& a, const Lds& L, int lane, const double (&u)[QM],
                                  const double (&bc)[QM], double ch, bool newton, bool refresh, double (&f)[QM],
                                  TA (&x)[QM]) {
#pragma clang fp contract(off)
    const int m = a.M.m;
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      if (i < m) L.c[i] = u[q];
    }
    if (lane == 0) L.lu.cmd[0] = 2;
    __syncthreads();  // hands the source term to the workgroup
    mfma_rhs_collective(a, L);
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      f[q] = i < m ? L.fbuf[i] : 0.0;
      x[q] = (newton && i < m) ? TA(-(u[q] - bc[q] - ch * f[q])) : TA(0);
    }
    if (refresh) {  // the workgroup computes the derivative pairs in collective_solve
      if (lane == 0) *L.lu.ch = ch;
      wave_sync();
    }
  }
  static __device__ bool factor_solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM], Fact&);
  // factors kept between refreshes: the kept derivative pairs and c h are
  // assembled and factored again (the same matrix, the same factors)
  static __device__ void solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM], const Fact&) {
    collective_solve(a, L, lane, x, false);
  }
  static __device__ bool collective_solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM],
                                          bool refresh);
};

// Assembly of I - c h J (FP32 sums of the serial Jacobian lists) plus the
// identity padding and the right-hand side (stashed in z) as the last column,
// by strips of 64 columns through LDS into the tiles of the four wavefronts,
// then the factorisation and back substitution.
template <int NB>
__device__ __forceinline__ void mfma_collective(const IntegratorArgs& a, const typename MfmaBackend<NB>::Lds& L,
                                                int wave, int lane) {
#pragma clang fp contract(off)
  using namespace mfma;
  const DevMech& M = a.M;
  const int m = M.m;
  const int tid = threadIdx.x;
  TCHEM_PT_BEGIN(dp)
  if (L.lu.cmd[2]) derivative_pairs(M, L.c, L.kf, L.pairs, tid, 256);  // refresh: pairs of the current iterate
  TCHEM_PT_END(dp, 1)
  const float scale = float(-*L.lu.ch);
  f32x16 acc[NB * NB / 4];
  TCHEM_PT_BEGIN(asm)
  constexpr int rows = kTile * NB;
  float4* stage4 = reinterpret_cast<float4*>(L.lu.stage);
#pragma unroll
  for (int q = 0; q < NB / 2; ++q) {  // unrolled: the tiles of strip q are known at compile time
    for (int idx = tid; idx < rows * 65 / 4; idx += 256) stage4[idx] = float4{0.0f, 0.0f, 0.0f, 0.0f};
    __syncthreads();
    {  // this thread's run of terms: coalesced, independent loads
      const int j1 = M.mfjQuarter()[q + 1];
      float sum = 0.0f;
#pragma unroll 4
      for (int j = M.mfjQuarter()[q]; j < j1; ++j) {
        const unsigned w = M.mfjTermW()[size_t(j) * 256 + tid];
        sum = fmaf(M.mfjTermC()[size_t(j) * 256 + tid], L.pairs[w & 0x3fff], sum);
        if (w >> 31) {
          L.lu.stage[(w >> 14) & 0x7fff] = (((w >> 29) & 1u) ? 1.0f : 0.0f) + scale * sum;
          sum = 0.0f;
        }
      }
    }
    for (int p = m + tid; p < rows - 1; p += 256)
      if ((p >> 6) == q) L.lu.stage[p * 65 + (p - 64 * q)] = 1.0f;
    if (q == NB / 2 - 1) {
      for (int i = tid; i < m; i += 256) L.lu.stage[i * 65 + 63] = L.lu.z[i];
      if (tid == 0) L.lu.stage[(rows - 1) * 65 + 63] = 1.0f;
    }
    __syncthreads();
    if constexpr (NB >= 2) if (q == 0) loadStrip<NB, 0>(acc, L.lu.stage, wave, lane);
    if constexpr (NB >= 4) if (q == 1) loadStrip<NB, 1>(acc, L.lu.stage, wave, lane);
    if constexpr (NB >= 6) if (q == 2) loadStrip<NB, 2>(acc, L.lu.stage, wave, lane);
    if constexpr (NB >= 8) if (q == 3) loadStrip<NB, 3>(acc, L.lu.stage, wave, lane);
    __syncthreads();
  }
  TCHEM_PT_END(asm, 4)
  factorAndSolve<NB>(acc, L.lu, wave, lane);
}

template <int NB>
__device__ bool MfmaBackend<NB>::factor_solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM], Fact&) {
  return collective_solve(a, L, lane, x, true);
}

template <int NB>
__device__ bool MfmaBackend<NB>::collective_solve(const IntegratorArgs& a, const Lds& L, int lane, TA (&x)[QM],
                                                  bool refresh) {
  const int m = a.M.m;
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    if (i < m) L.lu.z[i] = x[q];
  }
  if (lane == 0) {
    L.lu.cmd[0] = 1;
    L.lu.cmd[1] = 0;
    L.lu.cmd[2] = refresh ? 1 : 0;
  }
  __syncthreads();  // hands the matrix to the workgroup
  mfma_collective<NB>(a, L, 0, lane);
  // x = -(U^-1 e_last)[0..m)
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    x[q] = (i < m) ? -L.lu.z[i] : TA(0);
  }
  bool ok = L.lu.cmd[1] == 0;
#pragma unroll
  for (int q = 0; q < QM; ++q) ok = ok && isfinite(x[q]);
  return ok;
}

template <int NB>
__global__ __launch_bounds__(256, 1) void trbdf2_mfma_kernel(IntegratorArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  if (a.skip && __builtin_amdgcn_readfirstlane(*a.skip)) return;
  TCHEM_PT_RESET()
  using B = MfmaBackend<NB>;
  constexpr int QM = B::QM;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // uniform: tile choices are scalar branches
  typename B::Lds L = B::carve(lds_raw, a, 0);
  if (wave != 0) {
    // helpers: one collective factorisation per command until told to finish
    for (;;) {
      __syncthreads();
      const int cmd = __builtin_amdgcn_readfirstlane(L.lu.cmd[0]);
      if (cmd == 0) break;
      if (cmd == 2) {
        mfma_rhs_collective(a, L);
      } else {
        mfma_collective<NB>(a, L, wave, lane);
      }
    }
    return;
  }
  // one call site, so integrate_cell (with the collective's register tiles) is inlined
  for (int first = 1;; first = 0) {
    int cell = a.nBatch;
    if (a.persistent) {
      if (lane == 0) cell = atomicAdd(a.queue, 1);
      cell = __builtin_amdgcn_readfirstlane(__shfl(cell, 0, kWave));
    } else if (first) {
      cell = blockIdx.x;
    }
    if (cell >= a.nBatch) break;
    integrate_cell<B, QM, false>(a, L, cell, lane);
    wave_sync();
  }
  if (lane == 0) L.lu.cmd[0] = 0;
  __syncthreads();  // releases the helpers
}

// Batched dense solve A x = b (n <= 255, FP64 in and out, FP32 MFMA
// factorisation without interchanges): the LU of the MFMA form on its own.
// Every wavefront reads its tiles of [A | b | padding] straight into the
// registers of the C layout (a register of a tile is two rows of 32
// consecutive columns), with all loads of a tile row in flight.  Two
// workgroups share a CU at NB = 4 only: at NB = 6 half the registers spill 104
// of them (2048 systems of order 160 464 us, one system 59; with one workgroup
// per CU and no spills 447 and 48).
template <int NB>
__global__ __launch_bounds__(256, NB == 4 ? 2 : 1) void dense_mfma_solve_kernel(int n, int nBatch, const double* A,
                                                                                const double* b, double* x) {
  extern __shared__ __align__(16) char lds_raw[];
  using namespace mfma;
  constexpr int T = NB / 2;
  const int cell = blockIdx.x;
  if (cell >= nBatch) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);  // uniform: tile choices are scalar branches
  const Lu L = carveLu(lds_raw, NB);
  const double* Ac = A + size_t(cell) * n * n;
  const double* bc = b + size_t(cell) * n;
  if (threadIdx.x == 0) L.cmd[1] = 0;
  f32x16 acc[T * T];
#pragma unroll
  for (int o = 0; o < T; ++o) {
#pragma unroll
    for (int p = 0; p < T; ++p) {
      const int i0 = kTile * (2 * o + (wave >> 1)), j = kTile * (2 * p + (wave & 1)) + (lane & 31);
      double v[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = i0 + crow(r, lane);
        const int ic = i < n ? i : n - 1, jc = j < n ? j : n - 1;
        v[r] = Ac[ic * n + jc];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = i0 + crow(r, lane);
        acc[o * T + p][r] = (i < n && j < n) ? float(v[r]) : (i == j ? 1.0f : 0.0f);
      }
      if (p == T - 1 && (wave & 1)) {  // the right-hand side: column 31 of the last block column
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = i0 + crow(r, lane);
          const double rhs = bc[i < n ? i : n - 1];
          if (j == kTile * NB - 1 && i < n) acc[o * T + p][r] = float(rhs);
        }
      }
      if (p & 1) __builtin_amdgcn_sched_barrier(0);  // two tiles' loads in flight, not all (registers)
    }
  }
  factorAndSolve<NB>(acc, L, wave, lane);
  for (int i = threadIdx.x; i < n; i += blockDim.x) x[size_t(cell) * n + i] = L.cmd[1] ? NAN : -double(L.z[i]);
}

// ---- single-particle SIMPOL.1 aerosol integrator ---------------------------
// AerosolChemistry::runDeviceBatch (src/core/TChem_AerosolChemistry.cpp:31-186):
// the gas-phase box model extended by gas-particle partitioning
// (src/core/impl/TChem_Impl_Aerosol_RHS.hpp:64-103,
// TChem_Impl_SIMPOL_phase_transfer.hpp:61-150).  One cell per wavefront,
// FP64 dense LU with partial pivoting over the mt gas + particle unknowns
// (the reference factors a dense Jacobian too); the Jacobian is analytic.

constexpr double kSpRuniv = 8.314472;          // src/core/TChem_Util.hpp:176
constexpr double kSpPi = 3.141592653589793;    // TChem_Util.hpp:212
constexpr double kSpAtmPa = 101325.0;          // TChem_Util.hpp:227-229
constexpr double kSpMinMass = 1.0e-25;         // TChem_Impl_SingleParticleUtils.hpp:25-30
constexpr double kSpMinMw = 0.1;
constexpr double kSpMinDensity = 1800.0;

struct AeroLds : CellLds<double> {
  double* x;    // [mt] unknowns (gas internal order, then particles)
  double* f;    // [mt] source term
  double* sc;   // [nSimpol][4] alpha, mean free path, kg m-3 -> ppm, partitioning constant
  double* ps;   // [nPart][4] effective radius, volume, mass, moles
  double* pd;   // [nPart * nSimpol][6] k_c, k_e, diff, d k_c / dV, (unused) x2
  const double* nc;  // this cell's particle number concentrations
  double T, p;
};

__device__ AeroLds carve_aero(char* base, const DevMech& M, const DevAerosol& X, bool withMatrix = true) {
  AeroLds L;
  const int mt = X.mt;
  size_t off = withMatrix ? sizeof(double) * size_t(mt) * size_t(mt) : 0;
  off = (off + 15) & ~size_t(15);
  L.A = reinterpret_cast<double*>(base);
  L.c = reinterpret_cast<double*>(base + off);
  L.kf = L.c + M.nSpec;
  L.scr = L.kf + M.nReac;
  const int nScr = M.nReac > M.nPairs ? M.nReac : M.nPairs;
  L.seg = L.scr + nScr;
  L.x = L.seg + M.nSeg;
  L.f = L.x + mt;
  L.rdiag = L.f + mt;
  L.sc = L.rdiag + mt;
  L.ps = L.sc + 4 * X.nSimpol;
  L.pd = L.ps + 4 * X.nPart;
  L.swp = reinterpret_cast<int*>(L.pd + 6 * X.nPart * X.nSimpol);
  L.src = nullptr;
  L.nc = nullptr;
  L.T = L.p = 0.0;
  return L;
}

// SIMPOL_constant.hpp:60-128 (same expression order as the reference)
__device__ void simpol_constants(const double* par, double T, double p, double* out) {
  const double B1 = par[0], B2 = par[1], B3 = par[2], B4 = par[3], D = par[4], MW = par[5], Nstar = par[6];
  double alpha = 0.1;
  if (par[7] != 0.0) {
    const double N23 = pow(Nstar, 2.0 / 3.0);
    double dh = -10.0 * (Nstar - 1.0) + 7.53 * (N23 - 1.0) - 1.0;
    double ds = -32.0 * (Nstar - 1.0) + 9.21 * (N23 - 1.0) - 1.3;
    dh = dh * 4184.0;
    ds = ds * 4.184;
    const double dG = dh - T * ds;
    alpha = exp(-dG / (kSpRuniv * T));
    alpha = alpha / (1.0 + alpha);
  }
  const double mfp = 3.0 * D / sqrt(8.0 * kSpRuniv * T / (kSpPi * MW));
  double vp = B1 / T + B2 + B3 * T + B4 * log(T);
  vp = kSpAtmPa * pow(10.0, vp);
  const double conv = kSpRuniv / MW * 1.0e6;
  out[0] = alpha;
  out[1] = mfp;
  out[2] = conv * T / p;
  out[3] = vp / p / MW * 1.0e6;
}

__device__ __forceinline__ double fuchs_sutugin(double Kn, double alpha) {
  return (0.75 * alpha * (1.0 + Kn)) / (Kn * Kn + (1.0 + 0.283 * alpha) * Kn + 0.75 * alpha);
}

// Transfer terms of every (particle, transfer) pair at the unknowns in L.x:
// per-particle sums (lanes over particles), then k_c, k_e, diff and
// d k_c / dV (lanes over pairs).  SingleParticleUtils.hpp:62-160.
template <class LdsT>
__device__ void simpol_terms(const IntegratorArgs& a, const LdsT& L, int lane) {
  const DevAerosol& X = a.X;
  const double* mw = X.db + X.oMw;
  const double* dens = X.db + X.oDens;
  for (int ip = lane; ip < X.nPart; ip += kWave) {
    const double* y = L.x + a.M.m + ip * X.nAero;
    double v = kSpMinMass / kSpMinDensity;
    for (int i = 0; i < X.nAero; ++i) v += y[i] / dens[i];
    double ms = kSpMinMass, mo = kSpMinMass / kSpMinMw;
    for (int i = 0; i < X.nAero; ++i) {
      ms += y[i];
      mo += y[i] / mw[i];
    }
    L.ps[4 * ip + 0] = pow((v * 3.0 / 4.0 / kSpPi), 1.0 / 3.0);
    L.ps[4 * ip + 1] = v;
    L.ps[4 * ip + 2] = ms;
    L.ps[4 * ip + 3] = mo;
  }
  wave_sync();
  const int nPair = X.nPart * X.nSimpol;
  for (int j = lane; j < nPair; j += kWave) {
    const int ip = j / X.nSimpol, s = j - ip * X.nSimpol;
    const double* c4 = L.sc + 4 * s;
    const double alpha = c4[0], D = X.db[X.oPar + 8 * s + 4];
    const double radius = L.ps[4 * ip], volume = L.ps[4 * ip + 1], mass = L.ps[4 * ip + 2];
    const double moles = L.ps[4 * ip + 3];
    const double Kn = c4[1] / radius;
    const double den = Kn * Kn + (1.0 + 0.283 * alpha) * Kn + 0.75 * alpha;
    const double fk = fuchs_sutugin(Kn, alpha);
    const double fp = 0.75 * alpha * (den - (1.0 + Kn) * (2.0 * Kn + 1.0 + 0.283 * alpha)) / (den * den);
    const double kc = 4.0 * kSpPi * radius * D * fk;
    const double ke = kc * 1.0 * (c4[3] * (mass / moles) / mass);
    const int g = X.ib[X.oGas + s], ai = a.M.m + ip * X.nAero + X.ib[X.oAero + s];
    double* o = L.pd + 6 * j;
    o[0] = kc;
    o[1] = ke;
    o[2] = -(ke * L.x[ai]) + kc * L.x[g];
    o[3] = 4.0 * kSpPi * D * (fk - Kn * fp) * (radius / (3.0 * volume));
  }
  wave_sync();
}

// unknown layout and per-cell bindings shared by the aerosol backends
struct AerosolLayout {
  static __device__ __forceinline__ int unknowns(const IntegratorArgs& a) { return a.X.mt; }
  static __device__ __forceinline__ int rowDim(const IntegratorArgs& a) {
    return a.M.nSpec + 3 + a.X.nAero * a.X.nPart;
  }
  static __device__ __forceinline__ int column(const IntegratorArgs& a, int ai) {
    return ai < a.M.m ? 3 + a.M.perm()[ai] : 3 + a.M.nSpec + (ai - a.M.m);
  }
  template <class LdsT>
  static __device__ __forceinline__ void tolerance(const IntegratorArgs& a, const LdsT&, int ai, double& atol,
                                                   double& rtol) {
    const int xs = ai < a.M.m ? a.M.perm()[ai] : ai;
    atol = a.tol_time[2 * xs];
    rtol = a.tol_time[2 * xs + 1];
  }
  template <class LdsT>
  static __device__ __forceinline__ void load_rates(const IntegratorArgs& a, const LdsT& L, const double* kf, int lane) {
    for (int r = lane; r < a.M.nReac; r += kWave) L.kf[r] = kf[r];
  }
  // this cell's number concentrations, temperature and pressure, and the
  // SIMPOL constants (functions of T and p only)
  template <class LdsT>
  static __device__ void bind(const IntegratorArgs& a, LdsT& L, int cell) {
    const double* row = a.state + size_t(cell) * rowDim(a);
    L.nc = a.numberConc + size_t(cell) * a.X.nPart;
    L.T = row[2];
    L.p = row[1];
    const int lane = threadIdx.x & (kWave - 1);
    for (int s = lane; s < a.X.nSimpol; s += kWave) simpol_constants(a.X.db + a.X.oPar + 8 * s, L.T, L.p, L.sc + 4 * s);
    wave_sync();
  }
};

template <int QM>
struct AerosolBackend : AerosolLayout {
  using TA = double;
  static constexpr bool kCollective = false;  // factorisation by the whole workgroup (collective_solve)
  using Lds = AeroLds;
  struct Fact { int nswp = 0; };
  static __device__ void stage(const IntegratorArgs&, char*) {}
  static __device__ Lds carve(char* base, const IntegratorArgs& a, int wave) {
    return carve_aero(base + size_t(wave) * size_t(a.cellBytes), a.M, a.X);
  }
  static __device__ void init(const IntegratorArgs&, const Lds&, int) {}

  // f at u: gas source term, then every transfer in (particle, transfer)
  // order as the reference's serial accumulation; for a Newton iteration
  // also x = -(u - bc - ch f) and, when refreshing, I - ch J
  static __device__ void evaluate(const IntegratorArgs& a, const Lds& L, int lane, const double (&u)[QM],
                                  const double (&bc)[QM], double ch, bool newton, bool refresh, double (&f)[QM],
                                  double (&x)[QM]) {
    const DevMech& M = a.M;
    const DevAerosol& X = a.X;
    const int mt = X.mt;
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int ai = lane + kWave * q;
      if (ai < mt) L.x[ai] = u[q];
      if (ai < M.m) L.c[ai] = u[q];
    }
    wave_sync();
    double fg[QM];
    source_term_from_lds<QM>(M, L, lane, fg);
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int ai = lane + kWave * q;
      if (ai < mt) L.f[ai] = ai < M.m ? fg[q] : 0.0;
    }
    simpol_terms(a, L, lane);  // syncs first
    if (lane == 0) {
      for (int ip = 0; ip < X.nPart; ++ip)
        for (int s = 0; s < X.nSimpol; ++s) {
          const double diff = L.pd[6 * (ip * X.nSimpol + s) + 2];
          const int g = X.ib[X.oGas + s], ai = M.m + ip * X.nAero + X.ib[X.oAero + s];
          L.f[g] += -L.nc[ip] * diff;
          L.f[ai] += diff / L.sc[4 * s + 2];
        }
    }
    wave_sync();
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int ai = lane + kWave * q;
      f[q] = ai < mt ? L.f[ai] : 0.0;
      x[q] = (newton && ai < mt) ? -(u[q] - bc[q] - ch * f[q]) : 0.0;
    }
    if (refresh) assemble(a, L, lane, -ch);
  }

  // A = I + scale * J: gas-phase derivative pairs and Jacobian entries as
  // assemble_jacobian_from_lds (leading dimension mt), then the transfer
  // derivatives of SIMPOL_phase_transfer.hpp differentiated analytically:
  //   d diff / d x_gas = k_c
  //   d diff / d y_i = x_gas d k_c - y_aero d k_e - [i = aero] k_e
  //   d k_c = (d k_c / dV) / rho_i,  d k_e = K_eq d k_c / moles - k_e / (moles MW_i)
  static __device__ void assemble(const IntegratorArgs& a, const Lds& L, int lane, double scale) {
    const DevMech& M = a.M;
    const DevAerosol& X = a.X;
    const int mt = X.mt;
    for (int idx = lane; idx < mt * mt; idx += kWave) L.A[idx] = 0.0;
    wave_sync();
    for (int i = lane; i < mt; i += kWave) L.A[i * mt + i] = 1.0;
    for (int r = lane; r < M.nReac; r += kWave) {
      const int p0 = M.pairPtr()[r], p1 = M.pairPtr()[r + 1];
      if (p0 == p1) continue;
      const int* sp = M.reacSpec() + r * M.maxR;
      const int* pw = M.reacPow() + r * M.maxR;
      for (int pp = p0; pp < p1; ++pp) {
        const int js = M.pairSlot()[pp];
        const int ns = pw[js];
        double d = L.kf[r] * double(ns) * pow_small(L.c[sp[js]], ns - 1);
        for (int j = 0; j < M.maxR; ++j) {
          const int s2 = sp[j];
          if (s2 < 0) break;
          if (j == js) continue;
          d *= pow_small(L.c[s2], pw[j]);
        }
        L.scr[pp] = d;
      }
    }
    wave_sync();
    for (int n = lane; n < M.nnzJ; n += kWave) {
      double sum = 0.0;
      const int e1 = M.jnzPtr()[n + 1];
      for (int e = M.jnzPtr()[n]; e < e1; ++e) sum += M.jcCoef()[e] * L.scr[M.jcPair()[e]];
      const int rc = M.jnzRowCol()[n];
      const int row = rc >> 16, col = rc & 0xffff;
      L.A[row * mt + col] = (row == col ? 1.0 : 0.0) + scale * sum;
    }
    wave_sync();
    if (lane == 0) {
      const double* mw = X.db + X.oMw;
      const double* dens = X.db + X.oDens;
      for (int ip = 0; ip < X.nPart; ++ip) {
        const int base = M.m + ip * X.nAero;
        const double moles = L.ps[4 * ip + 3];
        for (int s = 0; s < X.nSimpol; ++s) {
          const double* o = L.pd + 6 * (ip * X.nSimpol + s);
          const double kc = o[0], ke = o[1], dkdv = o[3];
          const double keq = L.sc[4 * s + 3], kg = L.sc[4 * s + 2], n = L.nc[ip];
          const int g = X.ib[X.oGas + s], ai = base + X.ib[X.oAero + s];
          const double xg = L.x[g], ya = L.x[ai];
          L.A[g * mt + g] += scale * (-n * kc);
          L.A[ai * mt + g] += scale * (kc / kg);
          for (int i = 0; i < X.nAero; ++i) {
            const double dkc = dkdv / dens[i];
            const double dke = keq * dkc / moles - ke / (moles * mw[i]);
            double dd = xg * dkc - ya * dke;
            if (base + i == ai) dd -= ke;
            L.A[g * mt + base + i] += scale * (-n * dd);
            L.A[ai * mt + base + i] += scale * (dd / kg);
          }
        }
      }
    }
    wave_sync();
  }
  static __device__ bool factor_solve(const IntegratorArgs& a, const Lds& L, int lane, double (&x)[QM], Fact& fs) {
    if (!lu_factor_fused<QM>(L, a.X.mt, lane, x, fs.nswp)) return false;
    lu_back<QM>(L, a.X.mt, lane, x);
    return true;
  }
  static __device__ void solve(const IntegratorArgs& a, const Lds& L, int lane, double (&x)[QM], const Fact& fs) {
    lu_forward<QM>(L, a.X.mt, lane, x, fs.nswp);
    lu_back<QM>(L, a.X.mt, lane, x);
  }
};


// Sparse form of the aerosol integrator: the mechanism's compiled programs
// built over the mt unknowns (gas Jacobian pattern + the transfer
// derivatives' pattern, in elimination order: particle species first, then
// the gas species), read from device memory; the transfer terms and their derivatives are added to the
// source term and to the factor entries by one lane, in the dense form's
// order.
struct AeroSpLds : SpLds<double, false> {
  double* A;    // factor slots
  double* x;    // [mt] unknowns, with f, ps and pd in the place of what is dead once the Jacobian is assembled
  double* f;    // [mt] source term
  double* sc;   // [nSimpol][4]
  double* ps;   // [nPart][4]
  double* pd;   // [nPart * nSimpol][6]
  const double* nc;
  double T, p;
};

__device__ AeroSpLds carve_aero_sparse(char* base, const IntegratorArgs& a, int wave) {
  const DevAerosol& X = a.X;
  AeroSpLds L;
  static_cast<SpLds<double, false>&>(L) = carve_sparse<double, false>(
      a.W, reinterpret_cast<const unsigned*>(X.pib) + a.W.oWords, X.mt, base, a.cellBytes, wave);
  char* cell = base + sparseStageBytes(a.W, X.mt, false) + size_t(wave) * size_t(a.cellBytes);
  L.A = reinterpret_cast<double*>(cell);
  L.x = reinterpret_cast<double*>(cell + sparseScratchOffset(a.W));
  L.f = L.x + X.mt;
  L.ps = L.f + X.mt;
  L.pd = L.ps + 4 * X.nPart;
  L.sc = reinterpret_cast<double*>(cell + aerosolScratchEnd(a.W, X));
  L.nc = nullptr;
  L.T = L.p = 0.0;
  return L;
}

template <int QM>
struct AerosolSparseBackend : AerosolLayout {
  using TA = double;
  static constexpr bool kCollective = false;  // factorisation by the whole workgroup (collective_solve)
  static constexpr int SH = QM < 4 ? 0 : 3;
  using Lds = AeroSpLds;
  struct Fact {};
  static __device__ __forceinline__ void tolerance(const IntegratorArgs& a, const Lds& L, int ai, double& atol,
                                                   double& rtol) {
    staged_tolerance(a, L.tol, ai, [&](int i) { return i < a.M.m ? a.M.perm()[i] : i; }, atol, rtol);
  }
  static __device__ void stage(const IntegratorArgs& a, char* base) {
    stage_sparse<false>(a.W, nullptr, a.X.pdb + a.W.oCoef, base);
    double* tol = reinterpret_cast<double*>(base + sparseStageBytes(a.W, 0, false));
    const int n = a.W.tolStaged ? 2 * a.X.mt : 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const int ai = i >> 1, xs = ai < a.M.m ? a.M.perm()[ai] : ai;
      tol[i] = a.tol_time[2 * xs + (i & 1)];
    }
    __syncthreads();
  }
  static __device__ Lds carve(char* base, const IntegratorArgs& a, int wave) { return carve_aero_sparse(base, a, wave); }
  static __device__ void init(const IntegratorArgs& a, const Lds& L, int lane) { sp_init(a.W, L, a.X.mt, lane); }
  static __device__ __forceinline__ void load_rates(const IntegratorArgs& a, const Lds& L, const double* kf, int lane) {
    sp_load_rates<SH>(a.W, L, kf, lane);
  }
  static __device__ void evaluate(const IntegratorArgs& a, const Lds& L, int lane, const double (&u)[QM],
                                  const double (&bc)[QM], double ch, bool newton, bool refresh, double (&f)[QM],
                                  double (&x)[QM]) {
    const DevMech& M = a.M;
    const DevAerosol& X = a.X;
    const int mt = X.mt;
    double fg[QM];
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      fg[q] = i < M.m ? M.emission()[i] : 0.0;
      if (i < M.m) L.c[i] = u[q];
    }
    wave_sync();
    sp_rates<SH>(a.W, L, lane, refresh);
    wave_sync();
    sp_sums<SH>(L, a.W.oSegHdr, a.W.oSeg, a.W.nSeg, L.coef, L.cell + a.W.oS, lane);
    wave_sync();
    sp_rows<SH, QM>(a.W, L, lane, fg);
    wave_sync();
    if (refresh) {
      sp_jacobian<SH>(a.W, L, lane, -ch);
      wave_sync();
    }
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      if (i < mt) L.x[i] = u[q];
      if (i < mt) L.f[i] = i < M.m ? fg[q] : 0.0;
    }
    wave_sync();
    simpol_terms(a, L, lane);
    // Transfer terms and derivatives.  Targets in a particle's own rows or
    // columns are written by that particle's lane, the shared gas-species
    // targets (f_g and the (g, g) entries) by lane 0 afterwards; each target
    // receives its contributions in (particle, transfer) order either way.
    const int nj = 2 + 2 * X.nAero;
    const double scale = -ch;
    for (int ip = lane; ip < X.nPart; ip += kWave) {
      const double* mw = X.db + X.oMw;
      const double* dens = X.db + X.oDens;
      const int base = M.m + ip * X.nAero;
      const double moles = L.ps[4 * ip + 3];
      for (int s = 0; s < X.nSimpol; ++s) {
        const int j = ip * X.nSimpol + s;
        const double* o = L.pd + 6 * j;
        const double kc = o[0], ke = o[1], diff = o[2], dkdv = o[3];
        const double keq = L.sc[4 * s + 3], kg = L.sc[4 * s + 2], n = L.nc[ip];
        const int g = X.ib[X.oGas + s], ai = base + X.ib[X.oAero + s];
        L.f[ai] += diff / kg;
        if (refresh) {
          const int* jp = X.ib + X.oJpos + j * nj;
          const double xg = L.x[g], ya = L.x[ai];
          L.A[jp[1]] += scale * (kc / kg);
          for (int i = 0; i < X.nAero; ++i) {
            const double dkc = dkdv / dens[i];
            const double dke = keq * dkc / moles - ke / (moles * mw[i]);
            double dd = xg * dkc - ya * dke;
            if (base + i == ai) dd -= ke;
            L.A[jp[2 + i]] += scale * (-n * dd);
            L.A[jp[2 + X.nAero + i]] += scale * (dd / kg);
          }
        }
      }
    }
    wave_sync();
    if (lane == 0) {
      for (int ip = 0; ip < X.nPart; ++ip)
        for (int s = 0; s < X.nSimpol; ++s) {
          const int j = ip * X.nSimpol + s;
          const double n = L.nc[ip];
          L.f[X.ib[X.oGas + s]] += -n * L.pd[6 * j + 2];
          if (refresh) L.A[X.ib[X.oJpos + j * nj]] += scale * (-n * L.pd[6 * j]);
        }
    }
    wave_sync();
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      f[q] = i < mt ? L.f[i] : 0.0;
      x[q] = (newton && i < mt) ? -(u[q] - bc[q] - ch * f[q]) : 0.0;
      if (newton && i < mt) lds_put<double>(L.cell + a.W.oR + 16 * pivot(a, i), x[q]);
    }
    if (newton) wave_sync();
  }
  // elimination index of unknown i: particle species first, then the gas
  // species (aerosolPivot)
  static __device__ __forceinline__ int pivot(const IntegratorArgs& a, int i) {
    return i < a.M.m ? i + (a.X.mt - a.M.m) : i - a.M.m;
  }
  static __device__ __forceinline__ void get_x(const IntegratorArgs& a, const Lds& L, int lane, double (&x)[QM]) {
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      x[q] = 0.0;
      if (i < a.X.mt) {
        const vec2<double> v = lds_get<vec2<double>>(L.cell + a.W.oR + 16 * pivot(a, i));
        x[q] = v.x * v.y;
      }
    }
  }
  static __device__ bool factor_solve(const IntegratorArgs& a, const Lds& L, int lane, double (&x)[QM], Fact&) {
    sp_lu<SH>(L, L.w, a.W.oLuHdr, a.W.oLu, a.W.oLu1, a.W.nLu, lane);
    if (!sp_pivots<SH, QM>(a.W, L, a.X.mt, lane)) return false;
    sp_back<SH>(a.W, L, lane);
    get_x(a, L, lane, x);
    return true;
  }
  static __device__ void solve(const IntegratorArgs& a, const Lds& L, int lane, double (&x)[QM], const Fact&) {
    sp_lu<SH>(L, L.memory(), a.W.oFwdHdr, a.W.oFwd, a.W.oFwd1, a.W.nFwd, lane);
    sp_back<SH>(a.W, L, lane);
    get_x(a, L, lane, x);
  }
};

// Batched aerosol source term (gas + transfer) at the state rows: one
// wavefront per cell; omega [nBatch][mt] in the reference's unknown order
// (active gas species, then particle species).
template <int QM>
__global__ __launch_bounds__(64) void aerosol_rhs_kernel(IntegratorArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  const int lane = threadIdx.x, cell = blockIdx.x;
  if (cell >= a.nBatch) return;
  AeroLds L = carve_aero(lds_raw, a.M, a.X, false);  // no iteration matrix
  AerosolBackend<QM>::bind(a, L, cell);
  const double* row = a.state + size_t(cell) * AerosolBackend<QM>::rowDim(a);
  const DevMech& M = a.M;
  const double t_1 = 1.0 / L.T;
  const double conv = M.convPPM * L.p * t_1;
  for (int r = lane; r < M.nReac; r += kWave) L.kf[r] = rate_constant(M, r, L.T, L.p, t_1, conv, nullptr);
  for (int i = M.m + lane; i < M.nSpec; i += kWave) L.c[i] = row[3 + i];
  double u[QM], bc[QM], f[QM], x[QM];
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int ai = lane + kWave * q;
    u[q] = ai < a.X.mt ? row[AerosolBackend<QM>::column(a, ai)] : 0.0;
    bc[q] = 0.0;
  }
  wave_sync();
  AerosolBackend<QM>::evaluate(a, L, lane, u, bc, 0.0, false, false, f, x);
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int ai = lane + kWave * q;
    if (ai < a.X.mt) a.state_out[size_t(cell) * a.X.mt + (ai < M.m ? M.perm()[ai] : ai)] = f[q];
  }
}

// Workgroup = cellsPerGroup wavefronts, one cell per wavefront at a time;
// after staging, wavefronts never synchronise with each other.
//
// What bounds the sparse forms is each wavefront's chain of dependent LDS
// rounds (a wavefront alone on its CU took 66 k cycles per CB05 Newton
// iteration, sixteen took 76 k), not flops or bytes: the encoded programs
// (lowered.hpp, sparse_exec.hpp) replaced an interpreter of the rounds that
// decoded kind, length and indices per round and waited for scalar loads.
// Then slots spread over the LDS banks, and pivots checked (and their
// reciprocals kept for the back substitution) once after the last round; the
// multiplier rounds still invert the pivots they use.  Measured, interpreter -> encoded -> spread: 131040 cells
// mixed, 80 TR-BDF2 iterations 305.2 -> 160.5 -> 145.3 ms; 16411 cells FP64,
// 100 iterations 69.8 -> 36.8 -> 37.4 ms; one cell, 10 iterations 594 -> 309
// -> 300 us; E3SM 40960 cells to 1800 s 63.6 -> 32.3 -> 30.7 ms; CB05 + SOA,
// one particle, 8192 cells, 60 iterations 52.8 -> 33.7 -> 33.6 ms (same bits).
// Reading the stream 4 to 7 rounds ahead instead of 2, or a section's first
// records a section early, gave -4 to +4 %: the rounds wait for their own
// operands and instructions, not for the stream.
template <class B, int QM, int kThreads, bool REC>
__global__ __launch_bounds__(kThreads) void trbdf2_kernel(IntegratorArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  if (a.skip && __builtin_amdgcn_readfirstlane(*a.skip)) return;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  B::stage(a, lds_raw);
  const typename B::Lds L = B::carve(lds_raw, a, wave);
  B::init(a, L, lane);
  TCHEM_PT_RESET()
  if (!a.persistent) {
    const int cell = blockIdx.x * a.cellsPerGroup + wave;
    if (cell < a.nBatch) integrate_cell<B, QM, REC>(a, L, cell, lane);
    return;
  }
  for (;;) {
    int cell = 0;
    if (lane == 0) cell = atomicAdd(a.queue, 1);
    cell = __builtin_amdgcn_readfirstlane(__shfl(cell, 0, kWave));
    if (cell >= a.nBatch) break;
    integrate_cell<B, QM, REC>(a, L, cell, lane);
    wave_sync();
  }
}

// Rate constants of every (cell, reaction), one thread each; read by the
// integrator at the start of a cell.  Keeping the transcendental code out of
// the integrator keeps its register footprint small.
// lscale (nullable): kf_r *= exp(lscale[cell * lstride + r]), the log-scale
// parameters the discrete adjoint differentiates with respect to (lstride 0:
// one set for every cell).
// rowDim: state row length (0: nSpec + 3, the gas-phase box model's rows)
__global__ __launch_bounds__(256) void rates_kernel(DevMech M, int nBatch, const double* state, const double* photo,
                                                   const double* lscale, int lstride, double* kf, const int* skip,
                                                   int rowDim) {
  if (skip && *skip) return;
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long long)nBatch * M.nReac) return;
  const int cell = int(idx / M.nReac), r = int(idx - (long long)cell * M.nReac);
  const double* row = state + size_t(cell) * (rowDim > 0 ? rowDim : M.nSpec + 3);
  const double p = row[1], T = row[2];
  const double t_1 = 1.0 / T;
  const double conv = M.convPPM * p * t_1;
  const double k = rate_constant(M, r, T, p, t_1, conv, photo ? photo + size_t(cell) * M.nPhoto : nullptr);
  kf[idx] = lscale ? k * tchem_exp(lscale[size_t(cell) * lstride + r]) : k;
}

// ---- discrete adjoint --------------------------------------------------------
// Reverse-mode derivative of the recorded TR-BDF2 trajectory (accepted steps
// only, step sizes held fixed) with respect to the initial active species
// and the log-scale parameters theta_r of the rate constants
// (kf_r = k_r exp(theta_r), so d f / d theta_r = nu_r rop_r).  For one step
// u_n -> u_g -> u_{n+1},
//   TR:   u_g - u_n - c_tr h (f(u_g) + f(u_n)) = 0
//   BDF2: u_{n+1} - a_g u_g + a_n u_n - c_bdf h f(u_{n+1}) = 0,
// lambda = dL/du_{n+1} propagates as
//   (I - c_bdf h J(u_{n+1}))^T mu2 = lambda
//   (I - c_tr h J(u_g))^T mu1     = a_g mu2
//   lambda_n = -a_n mu2 + mu1 + c_tr h J(u_n)^T mu1
//   dL/dtheta_r += c_bdf h rop_r(u_{n+1}) (nu_r . mu2)
//                + c_tr h (rop_r(u_g) + rop_r(u_n)) (nu_r . mu1).
// The transposed systems are assembled and factorised directly by the
// transposed programs (I - c h J^T on the transposed factor pattern).
// Checkpoints every kAdjointSegment accepted steps; each segment is replayed
// forward with the forward programs (the same arithmetic as the recording
// integrator, hence the same Newton iterates), its states kept in device
// scratch, then swept in reverse.

template <int QM>
__device__ __forceinline__ void load_vec(const double* src, int m, int lane, double (&u)[QM]) {
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    u[q] = i < m ? src[i] : 0.0;
  }
}
template <int QM>
__device__ __forceinline__ void store_vec(double* dst, int m, int lane, const double (&u)[QM]) {
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    if (i < m) dst[i] = u[q];
  }
}

// One Newton solve of a stage, as the integrator runs it (same refresh
// rule, convergence test and arithmetic).
template <int QM>
__device__ __forceinline__ void replay_newton(const IntegratorArgs& f, const SpLds<double, false>& L, int lane,
                              double (&u)[QM], const double (&bc)[QM], double ch, int max_newton, int jint, double atol, double rtol) {
  using B = SparseBackend<double, QM, false>;
  typename B::Fact fs;
  for (int nit = 0; nit < max_newton; ++nit) {
    const bool refresh = (nit % jint) == 0;
    double fv[QM], x[QM];
    B::evaluate(f, L, lane, u, bc, ch, true, refresh, fv, x);
    if (refresh) {
      if (!B::factor_solve(f, L, lane, x, fs)) return;
    } else {
      B::solve(f, L, lane, x, fs);
    }
    bool over = false;
#pragma unroll
    for (int q = 0; q < QM; ++q) {
      const int i = lane + kWave * q;
      if (i < f.M.m) {
        u[q] += x[q];
        over |= !ratio_at_most_one(fabs(x[q]), atol + rtol * fabs(u[q]));
      }
    }
    if (ballot(over) == 0) return;
  }
}

// Solves (I - ch J^T) mu = rhs at the Jacobian pairs in LDS; mu in registers
// and in L.mu, w = nu . mu.  Returns false on a zero or non-finite pivot.
template <int QM>
__device__ __forceinline__ bool adjoint_solve(const AdjointArgs& a, const SpLds<double, false>& LT, int lane, double ch,
                              const double (&rhs)[QM], double (&mu)[QM]) {
  constexpr int SH = SparseBackend<double, QM, false>::SH;
  const DevLowered& W = a.WT;
  const int m = a.fw.M.m;
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    if (i < m) lds_put<double>(LT.cell + W.oR + 16 * i, rhs[q]);
  }
  sp_jacobian<SH>(W, LT, lane, -ch);
  wave_sync();
  sp_lu<SH>(LT, LT.w, W.oLuHdr, W.oLu, W.oLu1, W.nLu, lane);
  const bool ok = sp_pivots<SH, QM>(W, LT, m, lane);
  sp_back<SH>(W, LT, lane);
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    mu[q] = 0.0;
    if (i < m) {
      const vec2<double> v = lds_get<vec2<double>>(LT.cell + W.oR + 16 * i);
      mu[q] = v.x * v.y;
      lds_put<double>(LT.cell + W.oMu + 8 * i, mu[q]);
    }
  }
  wave_sync();
  sp_sums<SH>(LT, W.oNutHdr, W.oNut, W.nNut, LT.coef, LT.cell + W.oW, lane);
  wave_sync();
  return ok;
}

// grad_r += c rop_r w_r
__device__ __forceinline__ void accumulate_grad(const DevLowered& W, const SpLds<double, false>& L, double* g,
                                                int lane, double c) {
  for (int s = 0; s < W.nRop; ++s) {
    const int r = int(L.w.template rec<unsigned>(W.oKf, s, lane));
    if (r >= 0)
      g[r] += c * lds_get<double>(L.cell + W.oP + 8 * (kWave * s + lane)) *
              lds_get<double>(L.cell + L.w.template rec<unsigned>(W.oWmap, s, lane));
  }
}

template <int QM>
__device__ void adjoint_cell(const AdjointArgs& a, const SpLds<double, false>& L, const SpLds<double, false>& LT,
                             double* g, int cell, int lane) {
  constexpr int SH = SparseBackend<double, QM, false>::SH;
  const IntegratorArgs& f = a.fw;
  const DevMech& M = f.M;
  const int m = M.m, nSpec = M.nSpec, nReac = M.nReac;
  const int maxSteps = f.rec.maxSteps;
  const int nCkpt = maxSteps / kAdjointSegment + 1;
  constexpr int kTraj = 2 * kAdjointSegment + 1;
  double* lam_out = a.lambda_out + size_t(cell) * nSpec;
  double* gout = a.grad + size_t(cell) * nReac;
  // a record of other sizes: only its header (offset 0) is read
  const bool foreign = a.header[0] != f.nBatch || a.header[1] != maxSteps;
  const int n = foreign ? -1 : f.rec.nsteps[cell];
  if (n < 0) {  // failed, overflowed or foreign record
    for (int i = lane; i < nSpec; i += kWave) lam_out[i] = NAN;
    for (int r = lane; r < nReac; r += kWave) gout[r] = NAN;
    return;
  }
  const double gam = 2.0 - 1.41421356237309504880;
  const double c_tr = 0.5 * gam;
  const double a_g = 1.0 / (gam * (2.0 - gam));
  const double a_n = (1.0 - gam) * (1.0 - gam) / (gam * (2.0 - gam));
  const double c_bdf = (1.0 - gam) / (2.0 - gam);
  const double atol = a.tol[0], rtol = a.tol[1];
  const int max_newton = a.newton[2 * cell], jint = a.newton[2 * cell + 1];

  for (int r = lane; r < nReac; r += kWave) g[r] = 0.0;
  for (int i = m + lane; i < nSpec; i += kWave) L.c[i] = f.rec.consts[size_t(cell) * (nSpec - m) + (i - m)];
  double lam[QM];
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int ai = lane + kWave * q;
    lam[q] = ai < m ? a.lambda_in[size_t(cell) * nSpec + M.perm()[ai]] : 0.0;
  }
  wave_sync();
  sp_load_rates<SH>(f.W, L, f.kf + size_t(cell) * nReac, lane);

  using B = SparseBackend<double, QM, false>;
  double* tr = a.traj + size_t(cell) * kTraj * m;
  const double* hrec = f.rec.h + size_t(cell) * maxSteps;
  bool ok = true;
  for (int e = (n + kAdjointSegment - 1) / kAdjointSegment - 1; e >= 0; --e) {
    const int k0 = e * kAdjointSegment;
    const int len = n - k0 < kAdjointSegment ? n - k0 : kAdjointSegment;
    // replay the segment from its checkpoint
    {
      double un[QM], u[QM], fn[QM], bc[QM], x[QM];
      load_vec<QM>(f.rec.ckpt + (size_t(cell) * nCkpt + e) * m, m, lane, un);
      store_vec<QM>(tr, m, lane, un);
#pragma unroll
      for (int q = 0; q < QM; ++q) bc[q] = 0.0;
      B::evaluate(f, L, lane, un, bc, 0.0, false, false, fn, x);
      for (int j = 0; j < len; ++j) {
        const double h = hrec[k0 + j];
#pragma unroll
        for (int q = 0; q < QM; ++q) {
          u[q] = un[q];
          bc[q] = un[q] + c_tr * h * fn[q];
        }
        replay_newton<QM>(f, L, lane, u, bc, c_tr * h, max_newton, jint, atol, rtol);
        store_vec<QM>(tr + size_t(kAdjointSegment + 1 + j) * m, m, lane, u);
#pragma unroll
        for (int q = 0; q < QM; ++q) bc[q] = a_g * u[q] - a_n * un[q];
        replay_newton<QM>(f, L, lane, u, bc, c_bdf * h, max_newton, jint, atol, rtol);
        store_vec<QM>(tr + size_t(j + 1) * m, m, lane, u);
#pragma unroll
        for (int q = 0; q < QM; ++q) un[q] = u[q];
        if (j + 1 < len) B::evaluate(f, L, lane, un, bc, 0.0, false, false, fn, x);
      }
    }
    // reverse sweep; rop and the Jacobian pairs at u_{n+1} are still in LDS
    // from the previous (later) step except for the segment's last step
    for (int j = len - 1; j >= 0; --j) {
      const double h = hrec[k0 + j];
      double u[QM], mu2[QM], mu1[QM], rhs[QM];
      if (j == len - 1) {
        load_vec<QM>(tr + size_t(j + 1) * m, m, lane, u);
        B::put_c(f, L, lane, u);
        sp_rates<SH>(a.WT, LT, lane, true);
        wave_sync();
      }
      ok &= adjoint_solve<QM>(a, LT, lane, c_bdf * h, lam, mu2);
      accumulate_grad(a.WT, LT, g, lane, c_bdf * h);
      load_vec<QM>(tr + size_t(kAdjointSegment + 1 + j) * m, m, lane, u);
      B::put_c(f, L, lane, u);
      sp_rates<SH>(a.WT, LT, lane, true);
      wave_sync();
#pragma unroll
      for (int q = 0; q < QM; ++q) rhs[q] = a_g * mu2[q];
      ok &= adjoint_solve<QM>(a, LT, lane, c_tr * h, rhs, mu1);
      accumulate_grad(a.WT, LT, g, lane, c_tr * h);
      load_vec<QM>(tr + size_t(j) * m, m, lane, u);
      B::put_c(f, L, lane, u);
      sp_rates<SH>(a.WT, LT, lane, true);
      wave_sync();
      accumulate_grad(a.WT, LT, g, lane, c_tr * h);
      sp_sums<SH>(LT, a.WT.oJtvHdr, a.WT.oJtv, a.WT.nJtv, LT.cell, LT.cell + a.WT.oV, lane);
      wave_sync();
#pragma unroll
      for (int q = 0; q < QM; ++q) {
        const int i = lane + kWave * q;
        lam[q] = 0.0;
        if (i < m) {
          const double v = lds_get<double>(LT.cell + LT.w.template rec<unsigned>(a.WT.oVmap, q, lane));
          lam[q] = -a_n * mu2[q] + mu1[q] + c_tr * h * v;
        }
      }
      wave_sync();
    }
  }
  ok = ballot(!ok) == 0;
  for (int i = m + lane; i < nSpec; i += kWave) lam_out[i] = 0.0;
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int ai = lane + kWave * q;
    if (ai < m) lam_out[M.perm()[ai]] = ok ? lam[q] : NAN;
  }
  for (int r = lane; r < nReac; r += kWave) gout[r] = ok ? g[r] : NAN;
}

// One wavefront per cell, cells taken from a device work queue.  Bound by the
// same chain as trbdf2_kernel; gradient of 2000 CB05 cells over 1 ms of model
// time, forward and backward: 583 ms with the rounds interpreted, 248 ms
// encoded.
template <int QM>
__global__ __launch_bounds__(512) __attribute__((flatten)) void adjoint_kernel(AdjointArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const DevMech& M = a.fw.M;
  const unsigned* ib = reinterpret_cast<const unsigned*>(M.ib);
  stage_sparse<false>(a.WT, nullptr, M.db + a.WT.oCoef, lds_raw);
  __syncthreads();
  // one cell region and coefficient table, two instruction streams
  const SpLds<double, false> L = carve_sparse<double, false>(a.fw.W, ib + a.fw.W.oWords, 0, lds_raw, a.cellBytes, wave);
  SpLds<double, false> LT = L;
  LT.w.g = ib + a.WT.oWords;
  LT.w.bytes = 4 * a.WT.words;
  double* g = reinterpret_cast<double*>(lds_raw + sparseStageBytes(a.WT, 0, false) +
                                        size_t(wave) * size_t(a.cellBytes) + adjointRegionBytes(a.fw.W, a.WT));
  sp_init(a.WT, L, M.m, lane);
  if (lane == 0) lds_put<double>(L.cell + a.WT.oMu + 8 * M.m, 0.0);
  wave_sync();
  for (;;) {
    int cell = 0;
    if (lane == 0) cell = atomicAdd(a.fw.queue, 1);
    cell = __builtin_amdgcn_readfirstlane(__shfl(cell, 0, kWave));
    if (cell >= a.fw.nBatch) break;
    adjoint_cell<QM>(a, L, LT, g, cell, lane);
    wave_sync();
  }
}

// Per-cell Newton settings and the record header of an adjoint forward run.
__global__ void adjoint_setup_kernel(int nBatch, int maxSteps, const tchem_time_advance_t* tadv,
                                     const double* tol_newton, int* header, double* tol, int* newton) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    header[0] = nBatch;
    header[1] = maxSteps;
    tol[0] = tol_newton[0];
    tol[1] = tol_newton[1];
  }
  if (i < nBatch) {
    newton[2 * i] = tadv[i]._max_num_newton_iterations;
    newton[2 * i + 1] = tadv[i]._jacobian_interval < 1 ? 1 : tadv[i]._jacobian_interval;
  }
}

// Control words of a captured interval loop: ctl[0] = stopped, ctl[1] =
// intervals run.
__global__ void loop_reset_kernel(int* ctl) {
  if (threadIdx.x == 0) {
    ctl[0] = 0;
    ctl[1] = 0;
  }
}

// The driver's stop test after an interval (src/examples/TChem_AtmosphericChemistry.cpp:340-350):
// stop when mean_i t_out[i] > fraction * tend (tend of cell 0); a fixed
// reduction order, so the decision is reproducible.
__global__ __launch_bounds__(1024) void stop_check_kernel(int n, const double* t_out, const tchem_time_advance_t* tadv,
                                                         double fraction, int* ctl) {
  __shared__ double part[1024];
  if (ctl[0]) return;  // block-uniform
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) s += t_out[i];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0 && part[0] / double(n) > fraction * tadv[0]._tend) ctl[0] = 1;
}

// The autotuner's sample (rows 0, stride, 2 stride, ... of the caller's
// batch) copied by the device: the caller's arrays are never handed to a
// runtime copy (the runtime that owns them may not be the library's, e.g.
// under a profiler that loads its own), and the records get the trial's
// iteration cap, t_out = tbeg and dt_out = 0.  live counts cells with time
// left.
__global__ void autotune_sample_kernel(int n, long long stride, int nb, int np, int iters, const double* state,
                                       const double* photo, const tchem_time_advance_t* tadv, double* st0,
                                       double* ph, tchem_time_advance_t* ta, double* tt0, int* live) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long long src = i * stride;
  for (int j = 0; j < nb; ++j) st0[size_t(i) * nb + j] = state[size_t(src) * nb + j];
  for (int j = 0; j < np; ++j) ph[size_t(i) * np + j] = photo[size_t(src) * np + j];
  tchem_time_advance_t r = tadv[src];
  r._num_time_iterations_per_interval = iters;
  ta[i] = r;
  tt0[i] = r._tbeg;
  tt0[n + i] = 0.0;
  if (r._tend > r._tbeg && r._dt > 0.0) atomicAdd(live, 1);
}

// dst[i] = src[i] for n 4-byte words (device copies of caller arrays)
__global__ void copy_words_kernel(unsigned* dst, const unsigned* src, size_t n) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    dst[i] = src[i];
}

__global__ void reset_counter_kernel(int* counter) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *counter = 0;
}

__global__ void update_tadv_kernel(int n, tchem_time_advance_t* tadv, const double* t_out, const double* dt_out,
                                   int* ctl) {
  if (ctl && ctl[0]) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (ctl && i == 0) ctl[1] += 1;  // intervals run
  if (i < n) {
    tadv[i]._tbeg = t_out[i];
    tadv[i]._dt = dt_out[i];
  }
}

}  // namespace
}  // namespace tchem_amd

#include "batch_kernels.hpp"

namespace tchem_amd {

// ---- launchers (called from the C ABI) --------------------------------------

static int qmOf(int m) { return m <= 64 ? 1 : (m <= 128 ? 2 : (m <= 256 ? 4 : 0)); }
// instance of m unknowns whose encoded programs (sparse forms) hold shifted fields: those with QM 4
static int qmOf(int m, const DevLowered* w) { return w && w->enabled && w->shift ? 4 : qmOf(m); }

template <class B, int QM, int kThreads, bool REC = false>
static const void* integratorFn() {
  return reinterpret_cast<const void*>(&trbdf2_kernel<B, QM, kThreads, REC>);
}

// Largest workgroup of the sparse form: 16 wavefronts (cells) for the mixed
// form, 12 for FP64; 8 for programs with shifted fields, all those of more
// than 128 unknowns among them.  The occupancy of this
// latency-bound kernel sets its throughput, so each workgroup size gets the
// instance with the largest register budget that still lets its wavefronts
// be resident: FP64 up to 8 cells 512 threads (256 VGPRs), 9-12 cells 768
// (168); mixed up to 12 cells 768, 13-16 cells 1024 (128 VGPRs, 4 per SIMD;
// of these the one for 65 to 128 unknowns with staged programs spills 2
// registers, no other sparse instance spills any).
int sparseMaxCellsPerGroup(int precision, const DevLowered& w) {
  if (w.shift) return 8;
  return precision == TCHEM_PRECISION_MIXED ? 16 : 12;
}

// kernel instance for (precision, sparse form: 0 dense, 1 staged programs,
// 2 programs in device memory; species slots per lane; recording for the
// adjoint, FP64 sparse forms only; cells per workgroup); nullptr when there
// is none
static const void* integratorKernel(int precision, int sparse, int qm, bool rec, int cells, int mfmaTiles) {
  if (sparse == 3) {  // dense LU on the matrix cores: mixed precision only
    if (rec || precision != TCHEM_PRECISION_MIXED) return nullptr;
    return mfmaTiles == 4 ? reinterpret_cast<const void*>(&trbdf2_mfma_kernel<4>)
                          : (mfmaTiles == 6 ? reinterpret_cast<const void*>(&trbdf2_mfma_kernel<6>)
                                            : reinterpret_cast<const void*>(&trbdf2_mfma_kernel<8>));
  }
#define TCHEM_PICK_D(TA) \
  return qm == 1 ? integratorFn<DenseBackend<TA, 1>, 1, 64>() \
                 : (qm == 2 ? integratorFn<DenseBackend<TA, 2>, 2, 64>() : integratorFn<DenseBackend<TA, 4>, 4, 64>())
#define TCHEM_PICK_S(TA, T12, ST, REC)                                                        \
  return qm == 1 ? integratorFn<SparseBackend<TA, 1, ST>, 1, T12, REC>()                      \
                 : (qm == 2 ? integratorFn<SparseBackend<TA, 2, ST>, 2, T12, REC>()           \
                            : integratorFn<SparseBackend<TA, 4, ST>, 4, 512, REC>())
  if (rec) {
    if (precision != TCHEM_PRECISION_FP64 || sparse == 0) return nullptr;
    if (cells > 8 && qm <= 2) {
      if (sparse == 1) TCHEM_PICK_S(double, 768, true, true);
      TCHEM_PICK_S(double, 768, false, true);
    }
    if (sparse == 1) TCHEM_PICK_S(double, 512, true, true);
    TCHEM_PICK_S(double, 512, false, true);
  }
  if (precision == TCHEM_PRECISION_FP64) {
    if (cells > 8 && qm <= 2) {
      if (sparse == 1) TCHEM_PICK_S(double, 768, true, false);
      if (sparse == 2) TCHEM_PICK_S(double, 768, false, false);
    }
    if (sparse == 1) TCHEM_PICK_S(double, 512, true, false);
    if (sparse == 2) TCHEM_PICK_S(double, 512, false, false);
    TCHEM_PICK_D(double);
  }
  if (cells > 12 && qm <= 2) {
    if (sparse == 1) TCHEM_PICK_S(float, 1024, true, false);
    if (sparse == 2) TCHEM_PICK_S(float, 1024, false, false);
  }
  if (sparse == 1) TCHEM_PICK_S(float, 768, true, false);
  if (sparse == 2) TCHEM_PICK_S(float, 768, false, false);
  TCHEM_PICK_D(float);
#undef TCHEM_PICK_D
#undef TCHEM_PICK_S
}

hipError_t launchIntegrator(const IntegratorArgs& a, int precision, int grid, size_t lds, hipStream_t stream) {
  const int qm = qmOf(a.M.m, a.sparse == 1 || a.sparse == 2 ? &a.W : nullptr);
  if (qm == 0) return hipErrorInvalidValue;
  const void* fn = integratorKernel(precision, a.sparse, qm, a.rec.h != nullptr, a.cellsPerGroup,
                                    mfma::tilesFor(a.M.m));
  if (!fn) return hipErrorInvalidValue;
  hipFuncAttributes attr;
  const hipError_t ea = hipFuncGetAttributes(&attr, fn);
  if (ea != hipSuccess) return ea;
  const int threads = a.sparse == 3 ? 256 : 64 * a.cellsPerGroup;
  if (threads > attr.maxThreadsPerBlock) return hipErrorInvalidConfiguration;  // instance bound
  IntegratorArgs arg = a;
  void* params[] = {&arg};
  return hipLaunchKernel(fn, dim3(grid), dim3(threads), params, lds, stream);
}

// static LDS of the integrator instance (profiling builds declare some)
size_t integratorStaticLds(int precision, int sparse, int m, const DevLowered& w) {
  const int qm = qmOf(m, &w);
  if (qm == 0) return 0;
  hipFuncAttributes attr;
  if (hipFuncGetAttributes(&attr, integratorKernel(precision, sparse, qm, false, 1, mfma::tilesFor(m))) != hipSuccess) return 0;
  return attr.sharedSizeBytes;
}

hipError_t integratorMaxBlocksPerCU(int precision, int sparse, int m, const DevLowered& w, int threads, size_t lds,
                                    int* blocks, bool rec) {
  const int qm = qmOf(m, sparse == 1 || sparse == 2 ? &w : nullptr);
  if (qm == 0) return hipErrorInvalidValue;
  const void* fn = integratorKernel(precision, sparse, qm, rec, threads / 64, mfma::tilesFor(m));
  if (sparse == 3) threads = 256;
  if (!fn) return hipErrorInvalidValue;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks, fn, threads, lds);
}

hipError_t launchRates(const DevMech& M, int nBatch, const double* state, const double* photo, const double* lscale,
                       int lstride, double* kf, const int* skip, hipStream_t stream, int rowDim) {
  const long long n = (long long)nBatch * M.nReac;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(rates_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, stream, M, nBatch, state, photo,
                     lscale, lstride, kf, skip, rowDim);
  return hipGetLastError();
}

// ---- aerosol integrator launches (FP64 dense, mt <= 128 unknowns) ----
static const void* aerosolKernel(int mt, bool sparse, const DevLowered& w) {
  if (sparse) {
    if (w.shift && mt <= 256) return integratorFn<AerosolSparseBackend<4>, 4, 512>();
    if (mt <= 64) return integratorFn<AerosolSparseBackend<1>, 1, 512>();
    if (mt <= 128) return integratorFn<AerosolSparseBackend<2>, 2, 512>();
    return nullptr;
  }
  if (mt <= 64) return integratorFn<AerosolBackend<1>, 1, 256>();
  if (mt <= 128) return integratorFn<AerosolBackend<2>, 2, 256>();
  return nullptr;
}

// cells (wavefronts) per workgroup of the dense aerosol integrator: up to
// 4, as many as the LDS holds (0 when one cell does not fit or mt > 128)
int aerosolCellsPerGroup(const DevMech& M, const DevAerosol& X, size_t maxLds) {
  if (X.mt > 128) return 0;
  const size_t cb = (aerosolLdsBytes(M, X) + 15) & ~size_t(15);
  int c = int(maxLds / cb);
  return c > 4 ? 4 : c;
}

hipError_t launchAerosol(const IntegratorArgs& a, int grid, size_t lds, hipStream_t stream) {
  const bool sparse = a.sparse != 0;
  const void* fn = aerosolKernel(a.X.mt, sparse, a.W);
  if (!fn || a.cellsPerGroup < 1 || a.cellsPerGroup > (sparse ? 8 : 4)) return hipErrorInvalidValue;
  IntegratorArgs arg = a;
  void* params[] = {&arg};
  return hipLaunchKernel(fn, dim3(grid), dim3(64 * a.cellsPerGroup), params, lds, stream);
}

hipError_t launchAerosolRhs(const IntegratorArgs& a, size_t lds, hipStream_t stream) {
  if (a.nBatch <= 0) return hipSuccess;
  IntegratorArgs arg = a;
  void* params[] = {&arg};
  const void* fn = a.X.mt <= 64 ? reinterpret_cast<const void*>(&aerosol_rhs_kernel<1>)
                  : (a.X.mt <= 128 ? reinterpret_cast<const void*>(&aerosol_rhs_kernel<2>)
                                   : (a.X.mt <= 256 ? reinterpret_cast<const void*>(&aerosol_rhs_kernel<4>) : nullptr));
  if (!fn) return hipErrorInvalidValue;
  return hipLaunchKernel(fn, dim3(a.nBatch), dim3(64), params, lds, stream);
}

static const void* adjointKernel(int qm) {
  return qm == 1 ? reinterpret_cast<const void*>(&adjoint_kernel<1>)
                 : (qm == 2 ? reinterpret_cast<const void*>(&adjoint_kernel<2>)
                            : reinterpret_cast<const void*>(&adjoint_kernel<4>));
}

hipError_t adjointMaxBlocksPerCU(int m, const DevLowered& w, int threads, size_t lds, int* blocks) {
  const int qm = qmOf(m, &w);
  if (qm == 0) return hipErrorInvalidValue;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks, adjointKernel(qm), threads, lds);
}

hipError_t launchAdjoint(const AdjointArgs& a, int grid, size_t lds, hipStream_t stream) {
  const int qm = qmOf(a.fw.M.m, &a.WT);
  if (qm == 0) return hipErrorInvalidValue;
  AdjointArgs arg = a;
  void* params[] = {&arg};
  return hipLaunchKernel(adjointKernel(qm), dim3(grid), dim3(64 * a.cellsPerGroup), params, lds, stream);
}

hipError_t launchAdjointSetup(int nBatch, int maxSteps, const tchem_time_advance_t* tadv, const double* tol_newton,
                              int* header, double* tol, int* newton, hipStream_t stream) {
  const int n = nBatch > 0 ? nBatch : 1;
  hipLaunchKernelGGL(adjoint_setup_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, nBatch, maxSteps, tadv,
                     tol_newton, header, tol, newton);
  return hipGetLastError();
}

// Cells per workgroup of the source term and the E3SM kinetics.  64 keeps a
// wavefront on one reaction and has the highest throughput once its groups
// (one per CU) cover most of the chip; below, 16 and then 4 spread the batch.
// Measured us with 64 / 16 / 4 cells, source term: 131040 cells 188 / 292 /
// 493, 16411: 43 / 47 / 64, 8192: 24 / 21 / 33, 4096: 23 / 18 / 17, 1: 22 /
// 16 / 14; net production rates: 181 / 219 / 335, 41 / 38 / 48, 22 / 17 / 24,
// 22 / 14 / 13, 19 / 14 / 13.  Fewer where the LDS does not hold as many (0:
// not even one).  bytes(C): LDS of a workgroup.
template <class Bytes>
static int cellsPerGroup(int nBatch, int numCUs, size_t maxLds, Bytes bytes) {
  if (nBatch > 40 * (long long)numCUs && bytes(64) <= maxLds) return 64;
  if (nBatch > 12 * (long long)numCUs && bytes(16) <= maxLds) return 16;
  return bytes(4) <= maxLds ? 4 : (bytes(1) <= maxLds ? 1 : 0);
}

size_t e3smGroupBytes(const DevE3sm& E, int C) {
  return sizeof(double) * (size_t(C) * oddStride(E.nSpec + 3) + size_t(E.nReac + 1) * oddStride(C));
}
hipError_t launchE3smKinetics(const DevE3sm& E, int mode, int nBatch, const double* state, const double* photo,
                              int nPhoto, const double* ext, double* out, int ldOut, int numCUs, size_t maxLds,
                              hipStream_t stream) {
  if (nBatch <= 0) return hipSuccess;
  const int C = cellsPerGroup(nBatch, numCUs, maxLds, [&](int c) { return e3smGroupBytes(E, c); });
#define TCHEM_E3SM(c)                                                                                             \
  hipLaunchKernelGGL(e3sm_kinetics_kernel<c>, dim3((nBatch + c - 1) / c), dim3(groupThreads(c)),                  \
                     e3smGroupBytes(E, c), stream, E, mode, nBatch, state, photo, nPhoto, ext, out, ldOut)
  if (C == 64) TCHEM_E3SM(64);
  else if (C == 16) TCHEM_E3SM(16);
  else if (C == 4) TCHEM_E3SM(4);
  else if (C == 1) TCHEM_E3SM(1);
  else return hipErrorInvalidConfiguration;
#undef TCHEM_E3SM
  return hipGetLastError();
}

hipError_t launchAutotuneSample(int n, long long stride, int nb, int np, int iters, const double* state,
                                const double* photo, const tchem_time_advance_t* tadv, double* st0, double* ph,
                                tchem_time_advance_t* ta, double* tt0, int* live, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(autotune_sample_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, n, stride, nb, np, iters,
                     state, photo, tadv, st0, ph, ta, tt0, live);
  return hipGetLastError();
}

hipError_t launchCopyWords(void* dst, const void* src, size_t words, hipStream_t stream) {
  if (words == 0) return hipSuccess;
  const size_t blocks = std::min<size_t>((words + 255) / 256, 4096);
  hipLaunchKernelGGL(copy_words_kernel, dim3(unsigned(blocks)), dim3(256), 0, stream, static_cast<unsigned*>(dst),
                     static_cast<const unsigned*>(src), words);
  return hipGetLastError();
}

hipError_t launchResetCounter(int* counter, hipStream_t stream) {
  hipLaunchKernelGGL(reset_counter_kernel, dim3(1), dim3(64), 0, stream, counter);
  return hipGetLastError();
}

hipError_t launchUpdateTadv(int n, tchem_time_advance_t* tadv, const double* t_out, const double* dt_out, int* ctl,
                            hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(update_tadv_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, n, tadv, t_out, dt_out, ctl);
  return hipGetLastError();
}

hipError_t launchLoopControl(int n, const double* t_out, const tchem_time_advance_t* tadv, double fraction, int* ctl,
                             bool reset, hipStream_t stream) {
  if (reset) hipLaunchKernelGGL(loop_reset_kernel, dim3(1), dim3(64), 0, stream, ctl);
  else hipLaunchKernelGGL(stop_check_kernel, dim3(1), dim3(1024), 0, stream, n, t_out, tadv, fraction, ctl);
  return hipGetLastError();
}

hipError_t launchSourceTerm(const DevMech& M, int nBatch, const double* state, const double* photo, const double* ext,
                            double* omega, int numCUs, size_t maxLds, hipStream_t stream) {
  if (nBatch <= 0) return hipSuccess;
  auto bytes = [&](int c) {
    return sizeof(double) * (size_t(c) * oddStride(M.nSpec + 4) + size_t(M.nReac + 1) * oddStride(c));
  };
  const int C = cellsPerGroup(nBatch, numCUs, maxLds, bytes);
#define TCHEM_SOURCE(c)                                                                                         \
  hipLaunchKernelGGL(sourceterm_kernel<c>, dim3((nBatch + c - 1) / c), dim3(groupThreads(c)), bytes(c), stream, \
                     M, nBatch, state, photo, ext, omega)
  if (C == 64) TCHEM_SOURCE(64);
  else if (C == 16) TCHEM_SOURCE(16);
  else if (C == 4) TCHEM_SOURCE(4);
  else if (C == 1) TCHEM_SOURCE(1);
  else return hipErrorInvalidConfiguration;
#undef TCHEM_SOURCE
  return hipGetLastError();
}

// ---- scratch of the no-allocation entry point ---------------------------------
// Device memory the no-allocation variant of runDeviceBatch uses in place of
// library allocations: the batch's rate constants, then the work-queue
// counter.  Each GPU holds its own copy of the array, at its own address,
// for the life of the process; every call on a GPU shares that GPU's copy,
// so calls that overlap on one GPU race.
constexpr size_t kNoAllocScratchBytes = size_t(16) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

// Device address of the current GPU's scratch, looked up once per device
// (hipGetSymbolAddress with that device current) and kept; host code uses
// this address, never the array's name.
hipError_t noAllocScratch(void** ptr, size_t* bytes) {
  static std::mutex mu;
  static void* cache[256] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 256) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!cache[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    cache[dev] = p;
  }
  *ptr = cache[dev];
  *bytes = kNoAllocScratchBytes;
  return hipSuccess;
}

// LDS of a cell with all 8 x 8 tiles: which mechanisms the form takes
size_t mfmaCellLdsBytes(const DevMech& M) { return mfmaCellBytes(M, 8); }
// LDS of the instance that runs
size_t mfmaLaunchLdsBytes(const DevMech& M) { return mfmaCellBytes(M, mfma::tilesFor(M.m)); }

hipError_t launchDenseMfmaSolve(int n, int nBatch, const double* A, const double* b, double* x, hipStream_t stream) {
  if (nBatch <= 0) return hipSuccess;
  const int tiles = mfma::tilesFor(n);
  auto* fn = tiles == 4 ? dense_mfma_solve_kernel<4> : (tiles == 6 ? dense_mfma_solve_kernel<6> : dense_mfma_solve_kernel<8>);
  hipLaunchKernelGGL(fn, dim3(nBatch), dim3(256), mfma::luLdsBytes(tiles), stream, n, nBatch, A, b, x);
  return hipGetLastError();
}

hipError_t launchJacobian(const DevMech& M, int nBatch, const double* state, const double* photo, double* jac,
                          int numCUs, size_t maxLds, hipStream_t stream) {
  if (nBatch <= 0) return hipSuccess;
  auto bytes = [&](int c) {
    const size_t inner = size_t(c) * oddStride(M.nSpec + 4) + size_t(M.nReac) * oddStride(c);
    const size_t list = size_t(1 + M.nSerJ) * oddStride(c);
    return sizeof(double) * (size_t(M.nPairs + 1) * oddStride(c) + (inner > list ? inner : list));
  };
  // 4 cells (two groups to a CU, one stores while the other computes) or 16,
  // which compute faster and win where one group per CU takes the whole batch:
  // 4096 cells 54 us against 67, but 2000: 48 against 36, 16411: 272 against 242
  int C = nBatch > 10 * (long long)numCUs && nBatch <= 16 * (long long)numCUs ? 16 : 4;
  while (C > 1 && bytes(C) > maxLds) C /= 4;
  if (bytes(C) > maxLds) return hipErrorInvalidConfiguration;
  const size_t map = 4 * ((size_t(M.m) * M.m + 1) / 2);
  const int staged = bytes(C) + map <= maxLds ? 1 : 0;  // else the position table is read from device memory
  const size_t lds = bytes(C) + (staged ? map : 0);
#define TCHEM_JAC(c)                                                                                           \
  hipLaunchKernelGGL(jacobian_kernel<c>, dim3((nBatch + c - 1) / c), dim3(groupThreads(c)), lds, stream, M, nBatch, \
                     state, photo, jac, staged)
  if (C == 16) TCHEM_JAC(16);
  else if (C == 4) TCHEM_JAC(4);
  else TCHEM_JAC(1);
#undef TCHEM_JAC
  return hipGetLastError();
}

}  // namespace tchem_amd

#ifdef TCHEM_PHASE_TIMERS
extern "C" int tchem_debug_phase_cycles(unsigned long long* out, int reset) {
  if (hipMemcpyFromSymbol(out, HIP_SYMBOL(tchem_amd::g_phase_cycles), sizeof(unsigned long long) * 16) != hipSuccess)
    return -1;
  if (reset) {
    const unsigned long long z[16] = {};
    if (hipMemcpyToSymbol(HIP_SYMBOL(tchem_amd::g_phase_cycles), z, sizeof(z)) != hipSuccess) return -1;
  }
  return 0;
}
#endif
