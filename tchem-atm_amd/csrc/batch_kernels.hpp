// Batch functions of a state row: source term, Jacobian, and the E3SM
// kinetics' rate constants, rates of progress and net production rates.
//
// A workgroup takes C cells; thread t works on cell t % C and takes every
// n-th item (reaction, species, Jacobian entry) of its table, n = threads / C.
// With C = 64 a wavefront is 64 cells at one item: no divergence over
// reaction kinds, table reads are scalar, LDS rows are conflict free, and
// every sum runs in the order of the reference's loops without leaving its
// lane.  (One wavefront per cell, items over lanes, spent its time on
// divergent rate kinds, dependent table gathers and, in the E3SM kinetics,
// sums added by one lane.)  Small batches take fewer cells per workgroup so
// that they still spread over the chip: cellsPerGroup.
//
// LDS of a workgroup: state rows [cell][odd stride], then a table
// [item][C | 1] of rate constants, overwritten by rates of progress.
#pragma once

namespace tchem_amd {
namespace {

__host__ __device__ constexpr int oddStride(int n) { return n | 1; }
__host__ __device__ constexpr int groupThreads(int C) { return C == 64 ? 1024 : (C == 16 ? 512 : 256); }

// this thread's cell of the group and first item; the item is a scalar when
// a wavefront holds one
template <int C>
struct GroupThread {
  int cell, sub;
  static constexpr int n = groupThreads(C) / C;
  __device__ __forceinline__ GroupThread() {
    cell = int(threadIdx.x) % C;
    sub = int(threadIdx.x) / C;
    if (C == 64) sub = __builtin_amdgcn_readfirstlane(sub);
  }
};

// C rows of dim values (nc of them in the batch, the others repeat the last
// so that idle lanes compute on real numbers) into LDS rows of stride rs
__device__ __forceinline__ void load_rows(const double* src, int dim, double* dst, int rs, int C, int nc) {
  const int lane = threadIdx.x & (kWave - 1), waves = blockDim.x / kWave;
  for (int c = threadIdx.x / kWave; c < C; c += waves) {
    const double* row = src + size_t(c < nc ? c : nc - 1) * dim;
    for (int i = lane; i < dim; i += kWave) dst[c * rs + i] = row[i];
  }
}
// the first `width` values of nc LDS rows out, rows of ld values, the rest 0
__device__ __forceinline__ void store_rows(const double* rows, int rs, int width, double* dst, int ld, int nc,
                                           const double* add) {
  const int lane = threadIdx.x & (kWave - 1), waves = blockDim.x / kWave;
  for (int c = threadIdx.x / kWave; c < nc; c += waves)
    for (int i = lane; i < ld; i += kWave) {
      const double v = i < width ? rows[c * rs + i] : 0.0;
      dst[size_t(c) * ld + i] = add ? v + add[size_t(c) * ld + i] : v;
    }
}
// item table [item][C | 1] out as rows [nc][n]
template <int C>
__device__ __forceinline__ void store_items(const double* items, int n, double* dst, int nc) {
  const int lane = threadIdx.x & (kWave - 1), waves = blockDim.x / kWave;
  for (int c = threadIdx.x / kWave; c < nc; c += waves)
    for (int i = lane; i < n; i += kWave) dst[size_t(c) * n + i] = items[i * oddStride(C) + c];
}

// Rate constants of the CB05 kinetics, store(r, k) for each of this thread's.
// Reactions come in classes (rateOrder): Arrhenius without temperature
// dependence (photolysis mostly), Arrhenius with an exponential alone, the
// rest; the first two are straight-line code, two reactions at a time.  The
// first keep the factor exp(0 / T) as what it is: 1, or NaN where T is NaN or
// 1 / T is infinite, so that a cell without a temperature has no rates.
template <int C, class Store>
__device__ __forceinline__ void group_rate_constants(const DevMech& M, const GroupThread<C>& g, const double* row,
                                                     const double* photo, Store store) {
#pragma clang fp contract(off)
  const double p = row[1], T = row[2];
  const double t_1 = 1.0 / T;
  const double conv = M.convPPM * p * t_1;
  const double unit = 0.0 * t_1 + 1.0;
  const int* order = M.rateOrder();
  const int n0 = order[M.nReac], n1 = order[M.nReac + 1];  // ends of the first two classes
  int i = g.sub;
#pragma unroll 2
  for (; i < n0; i += g.n) {
    const int r = order[i], slot = M.photoSlot()[r];
    double A = M.ratePar()[8 * r];
    if (photo != nullptr && slot >= 0) A = photo[slot];
    store(r, A * unit * tchem_ipow(conv, M.convExp()[r]));
  }
#pragma unroll 2
  for (; i < n1; i += g.n) {
    const int r = order[i], slot = M.photoSlot()[r];
    double A = M.ratePar()[8 * r];
    if (photo != nullptr && slot >= 0) A = photo[slot];
    store(r, A * tchem_exp(M.ratePar()[8 * r + 2] * t_1) * tchem_ipow(conv, M.convExp()[r]));
  }
  for (; i < M.nReac; i += g.n) {
    const int r = order[i];
    store(r, rate_constant(M, r, T, p, t_1, conv, photo));
  }
}

// Product of the reactants of reaction r in the row, times v: three packed
// fields column | power << 16 (the row ends with a 1 for absent reactants)
__device__ __forceinline__ double times_factor(double v, const double* row, int f) {
#pragma clang fp contract(off)
  const double x = row[f & 0xffff];
  double y = x;
  for (int i = 1; i < (f >> 16); ++i) y = y * x;
  return v * y;
}

// Sum of a padded list (entries of 4, padding of coefficient 0 on the zero
// item), in order, added to s
template <int C, bool FUSED>
__device__ __forceinline__ double list_sum(double s, const int* item, const double* coef, int e, int e1,
                                           const double* items, int cell) {
#pragma clang fp contract(off)
  for (; e < e1; e += 4) {
    double v[4], c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = items[item[e + j] * oddStride(C) + cell];
      c[j] = coef[e + j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) s = FUSED ? fma(c[j], v[j], s) : s + c[j] * v[j];
  }
  return s;
}

// Source term [nBatch][m] in the reference's species order: rate constants,
// rates of progress in place, then per species the serial gather of
// source_term_from_lds (the reference's order of additions), longest lists
// first, dealt to the sub-groups back and forth.
// Bound by latency (scalar table loads, the exponentials' chains, barriers)
// with the 16 wavefronts that 141 KB of LDS leave a CU: 131040 CB05 cells
// 1342 us with one wavefront per cell -> 203 us (193 MB at 5 TB/s: 38 us).
template <int C>
__global__ __launch_bounds__(groupThreads(C)) void sourceterm_kernel(DevMech M, int nBatch, const double* state,
                                                                     const double* photo, const double* ext,
                                                                     double* omega) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) char lds_raw[];
  const int dim = M.nSpec + 3, rs = oddStride(dim + 1), maxR = M.maxR;
  double* rows = reinterpret_cast<double*>(lds_raw);
  double* rop = rows + C * rs;  // [nReac + 1][C | 1], the last item zeros
  const GroupThread<C> g;
  const int cell0 = blockIdx.x * C, nc = nBatch - cell0 < C ? nBatch - cell0 : C;
  load_rows(state + size_t(cell0) * dim, dim, rows, rs, C, nc);
  double* row = rows + g.cell * rs;
  if (g.sub == 0) {
    row[dim] = 1.0;
    rop[M.nReac * oddStride(C) + g.cell] = 0.0;
  }
  __syncthreads();
  const int src = cell0 + (g.cell < nc ? g.cell : nc - 1);
  group_rate_constants<C>(M, g, row, photo ? photo + size_t(src) * M.nPhoto : nullptr, [&](int r, double v) {
    const int* f = M.reacFactor() + r * maxR;
    for (int j = 0; j < maxR; ++j) v = times_factor(v, row, f[j]);
    rop[r * oddStride(C) + g.cell] = v;
  });
  __syncthreads();
  for (int k = 0, b = 0; k < M.m; k += g.n, ++b) {
    const int i = k + ((b & 1) ? g.n - 1 - g.sub : g.sub);
    if (i >= M.m) continue;
    const int a = M.omegaOrder()[i];
    row[M.perm()[a]] = list_sum<C, false>(M.emission()[a], M.padOmegaReac(), M.padOmegaCoef(), M.padOmegaPtr()[a],
                                          M.padOmegaPtr()[a + 1], rop, g.cell);  // the concentrations have been used
  }
  __syncthreads();
  store_rows(rows, rs, M.m, omega + size_t(cell0) * M.m, M.m, nc, ext ? ext + size_t(cell0) * M.m : nullptr);
}

// Jacobian [nBatch][m][m] in the reference's species order: rate constants,
// derivative pairs, then every structural entry summed serially as in
// assemble_jacobian_from_lds into a list of nonzeros, which a wavefront per
// cell spreads over the dense rows through a position table (16-byte stores
// where the rows allow them).  Bound by the stores, 44 KB per CB05 cell, and
// the lists that feed them: 16411 cells 1002 us with the dense matrix of a
// cell in LDS (3 wavefronts per CU) -> 242 us (733 MB at 5 TB/s: 146 us).
template <int C>
__global__ __launch_bounds__(groupThreads(C)) void jacobian_kernel(DevMech M, int nBatch, const double* state,
                                                                   const double* photo, double* jac, int stagedMap) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) char lds_raw[];
  const int dim = M.nSpec + 3, rs = oddStride(dim + 1), m = M.m;
  constexpr int cs = oddStride(C);
  double* dpr = reinterpret_cast<double*>(lds_raw);  // [nPairs + 1][cs], the last item zeros
  double* rows = dpr + (M.nPairs + 1) * cs;          // [C][rs], then kf [nReac][cs]
  double* kf = rows + C * rs;
  double* nz = rows;                                 // [1 + nSerJ][cs] in their place, entry 0 a zero
  const int inner = C * rs + M.nReac * cs, list = (1 + M.nSerJ) * cs;
  unsigned* mapLds = reinterpret_cast<unsigned*>(rows + (inner > list ? inner : list));
  const GroupThread<C> g;
  const int cell0 = blockIdx.x * C, nc = nBatch - cell0 < C ? nBatch - cell0 : C;
  const unsigned* map = M.jacMap();
  const int words = (m * m + 1) / 2;
  if (stagedMap) {
    for (int i = threadIdx.x; i < words; i += blockDim.x) mapLds[i] = map[i];
    map = mapLds;
  }
  load_rows(state + size_t(cell0) * dim, dim, rows, rs, C, nc);
  double* row = rows + g.cell * rs;
  if (g.sub == 0) {
    row[dim] = 1.0;
    dpr[M.nPairs * cs + g.cell] = 0.0;
  }
  __syncthreads();
  const int src = cell0 + (g.cell < nc ? g.cell : nc - 1);
  group_rate_constants<C>(M, g, row, photo ? photo + size_t(src) * M.nPhoto : nullptr,
                          [&](int r, double v) { kf[r * cs + g.cell] = v; });
  __syncthreads();
  // d rop_r / d c_s = k * n_s c_s^(n_s-1) * prod_{j != s} c_j^n_j
  for (int p = g.sub; p < M.nPairs; p += g.n) {
    const int4 w = M.pairRecord()[p];  // reaction | slot of s << 24, column of s | n_s << 16, the other factors
    const int r = w.x & 0xffffff, ns = w.y >> 16;
    double y = ns <= 1 ? 1.0 : row[w.y & 0xffff];
    for (int i = 2; i < ns; ++i) y = y * row[w.y & 0xffff];
    double d = kf[r * cs + g.cell] * double(ns) * y;
    if (M.maxR <= 3) {
      d = times_factor(times_factor(d, row, w.z), row, w.w);
    } else {
      for (int j = 0; j < M.maxR; ++j)
        if (j != (w.x >> 24)) d = times_factor(d, row, M.reacFactor()[r * M.maxR + j]);
    }
    dpr[p * cs + g.cell] = d;
  }
  __syncthreads();
  for (int n = g.sub; n < M.nSerJ; n += g.n)
    nz[(1 + n) * cs + g.cell] =
        list_sum<C, false>(0.0, M.padJPair(), M.padJCoef(), M.padJPtr()[n], M.padJPtr()[n + 1], dpr, g.cell);
  if (g.sub == 0) nz[g.cell] = 0.0;
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1), waves = blockDim.x / kWave;
  const size_t total = size_t(m) * m;
  const bool wide = total % 2 == 0 && reinterpret_cast<size_t>(jac) % 16 == 0;
  for (int c = threadIdx.x / kWave; c < nc; c += waves) {
    double* out = jac + size_t(cell0 + c) * total;
    for (int i = lane; i < words; i += kWave) {
      const unsigned w = map[i];
      const double lo = nz[int(w & 0xffffu) * cs + c], hi = nz[int(w >> 16) * cs + c];
      if (wide) {
        reinterpret_cast<double2*>(out)[i] = make_double2(lo, hi);
      } else {
        out[2 * i] = lo;
        if (size_t(2 * i + 1) < total) out[2 * i + 1] = hi;
      }
    }
  }
}

// ---- E3SM / UCI kinetics batch functions --------------------------------------
// ReactionRates / RateofProgress / NetProductionRates of the reference's
// E3SM kinetics (src/core/impl/TChem_Impl_{KForward,KForwardJPL,AdjustReactions,
// RateofProgress,NetProductionRates}.hpp):
//   mode 0: kf   (ReactionRates)
//   mode 1: rop  (RateofProgress; photolysis rates replace kf of the first nPhoto reactions)
//   mode 2: omega of the active species (NetProductionRates: external sources + nu . rop)
//   mode 3: kf with the photolysis rates applied (the box model's rate constants)
// Species concentrations are the state row's species block (active then constant).

__device__ __forceinline__ double t300_pow(double T, double B) { return B == 0.0 ? 1.0 : pow(T / 300.0, B); }
__device__ __forceinline__ double exp_or_one(double C, double t_1) { return C == 0.0 ? 1.0 : exp(C * t_1); }

//
// 131040 cells of the UCI mechanism, net production rates: 3130 us with one
// wavefront per cell (one lane adding nu . rop) -> 197 us (254 MB at 5 TB/s:
// 50 us); bound like sourceterm_kernel.
template <int C>
__global__ __launch_bounds__(groupThreads(C)) void e3sm_kinetics_kernel(DevE3sm E, int mode, int nBatch,
                                                                        const double* state, const double* photo,
                                                                        int nPhoto, const double* ext, double* out,
                                                                        int ldOut) {
  extern __shared__ __align__(16) char lds_raw[];
  constexpr int cs = oddStride(C);
  const int m = E.nSpec - E.nConst, dim = E.nSpec + 3, rs = oddStride(dim);
  double* rows = reinterpret_cast<double*>(lds_raw);
  double* kf = rows + C * rs;  // [nReac + 1][C | 1], the last item zeros
  const GroupThread<C> g;
  const int cell0 = blockIdx.x * C, nc = nBatch - cell0 < C ? nBatch - cell0 : C;
  load_rows(state + size_t(cell0) * dim, dim, rows, rs, C, nc);
  __syncthreads();
  const int src = cell0 + (g.cell < nc ? g.cell : nc - 1);
  double* row = rows + g.cell * rs;
  double* x = row + 3;
  const double p = row[1], T = row[2];
  const double t_1 = 1.0 / T;
  const double conv = E.convPPM * p * t_1;
  const int* ib = E.ib;
  const double* db = E.db;
  // a rate constant with its adjustments (TChem_Impl_AdjustReactions.hpp:52-96: the reaction's species, in list order)
  auto put = [&](int r, double k) {
    const int e1 = ib[E.oAdjPtr + r + 1];
    for (int e = ib[E.oAdjPtr + r]; e < e1; ++e) k *= x[ib[E.oAdjSpec + e]];
    kf[r * cs + g.cell] = k;
  };
  if (g.sub == 0) kf[E.nReac * cs + g.cell] = 0.0;
  // reactions without a rate form: given photolysis rates, or 0
  for (int i = g.sub; i < E.nGiven; i += g.n) {
    const int r = ib[E.oGiven + i];
    put(r, (mode >= 1 && photo && r < nPhoto) ? photo[size_t(src) * nPhoto + r] : 0.0);
  }
  // KForward (TChem_Impl_KForward.hpp:52-141): Arrhenius and Troe without the
  // conv factor, CMAQ_H2O2 with it
  for (int i = g.sub; i < E.nArr; i += g.n) {
    const double* P = db + E.oArrPar + 5 * i;
    put(ib[E.oArrIdx + i], P[0] * exp(P[2] * t_1) * (P[1] == 0.0 ? 1.0 : pow(T / P[3], P[1])) *
                               (P[4] == 0.0 ? 1.0 : (1.0 + P[4] * p)));
  }
  for (int i = g.sub; i < E.nTroe; i += g.n) {
    const double* P = db + E.oTroePar + 8 * i;
    const double k0 = P[0] * exp_or_one(P[2], t_1) * t300_pow(T, P[1]);
    const double k0_kinf = k0 / (P[3] * exp_or_one(P[5], t_1) * t300_pow(T, P[4]));
    put(ib[E.oTroeIdx + i], k0 / (1.0 + k0_kinf) * pow(P[6], 1.0 / (1.0 + pow(log10(k0_kinf) / P[7], 2.0))));
  }
  for (int i = g.sub; i < E.nCmaq; i += g.n) {
    const double* P = db + E.oCmaqPar + 6 * i;
    const int r = ib[E.oCmaqIdx + i];
    put(r, (P[0] * exp(P[2] * t_1) * t300_pow(T, P[1]) + P[3] * exp(P[5] * t_1) * t300_pow(T, P[4]) * conv) *
               pow(conv, double(ib[E.oConvExp + r])));
  }
  // KForwardJPL (TChem_Impl_KForwardJPL.hpp:44-143), m = [M]
  const double mM = E.M_index >= 0 ? x[E.M_index] : 0.0;
  // from the other end: the sub-groups with one Arrhenius reaction less take these first
  for (int i = g.n - 1 - g.sub; i < E.nJpl + E.nRJpl; i += g.n) {
    const bool rj = i >= E.nJpl;
    const int j = rj ? i - E.nJpl : i;
    const double* P = db + (rj ? E.oRJplPar + 10 * j : E.oJplPar + 7 * j);
    const double k0 = P[0] * exp_or_one(P[2], t_1) * t300_pow(T, P[1]);
    const double kinf = P[3] * exp_or_one(P[5], t_1) * t300_pow(T, P[4]);
    const double xpo = k0 * mM / kinf;
    const double lx = log10(xpo);
    const double factor = P[6] == 1.0 ? 1.0 : pow(P[6], 1.0 / (1.0 + lx * lx));
    double k = k0 / (1.0 + xpo) * factor;
    if (rj) k /= P[7] * exp_or_one(P[9], t_1) * t300_pow(T, P[8]);
    put(ib[(rj ? E.oRJplIdx : E.oJplIdx) + j], k);
  }
  if (E.nProd > 0) {
    __syncthreads();
    if (g.sub == 0)
      for (int i = 0; i < E.nProd; ++i) {
        const int* I = ib + E.oProdI + 7 * i;
        const double* P = db + E.oProdD + 6 * i;
        const double fc = P[0] * exp(P[1] * t_1) * x[I[4]] + P[2] * exp(P[3] * t_1) * x[I[5]] +
                          P[4] * exp(P[5] * t_1) * x[I[6]];
        for (int k = 0; k < 3; ++k) kf[I[k] * cs + g.cell] *= kf[I[3] * cs + g.cell] / fc;
      }
  }
  __syncthreads();
  if (mode == 0 || mode == 3) {
    store_items<C>(kf, E.nReac, out + size_t(cell0) * ldOut, nc);
    return;
  }
  // RateofProgress (TChem_Impl_RateofProgress.hpp:73-87), in place
  for (int r = g.sub; r < E.nReac; r += g.n) {
    double v = kf[r * cs + g.cell];
    const int n = ib[E.oNreac + r];
    for (int j = 0; j < n; ++j)
      v *= pow_small(x[ib[E.oSidx + r * E.maxSpec + j]], abs(int(db[E.oNuki + r * E.maxSpec + j])));
    kf[r * cs + g.cell] = v;
  }
  __syncthreads();
  if (mode == 1) {
    store_items<C>(kf, E.nReac, out + size_t(cell0) * ldOut, nc);
    return;
  }
  // NetProductionRates (TChem_Impl_NetProductionRates.hpp:60-104): external
  // sources, then nu . rop over each active species' reactions in order
  for (int k = 0, b = 0; k < m; k += g.n, ++b) {
    const int i = k + ((b & 1) ? g.n - 1 - g.sub : g.sub);
    if (i >= m) continue;
    const int a = ib[E.oNetOrder + i];
    row[a] = list_sum<C, true>(ext ? ext[size_t(src) * m + a] : 0.0, ib + E.oNetReac, db + E.oNetCoef,
                               ib[E.oNetPtr + a], ib[E.oNetPtr + a + 1], kf, g.cell);  // the state row has been used
  }
  __syncthreads();
  store_rows(rows, rs, m, out + size_t(cell0) * ldOut, ldOut, nc, nullptr);
}

}  // namespace
}  // namespace tchem_amd
