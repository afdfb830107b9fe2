// Execution of the encoded sparse programs (lowered.hpp) by one wavefront.
//
// What bounds this code is the wavefront's own chain: every round is an LDS
// gather, a few dependent multiply-adds and an LDS store that the next round
// reads.  So a round spends no instruction on decoding beyond turning a field
// into an address (one add), its record words are in registers when it
// starts (read two rounds ahead, three register sets in rotation, so nothing
// waits for a load issued in the same round), and no scalar load is in
// flight inside a loop (it would share the LDS wait counter and force full
// waits): what a round does is a bit of a mask held in scalar registers.
// CB05 Newton iteration of one wavefront alone: see trbdf2_kernel.
#pragma once

namespace tchem_amd {
namespace {

using u32x2 = __attribute__((ext_vector_type(2))) unsigned;
using u32x4 = __attribute__((ext_vector_type(4))) unsigned;
template <typename TA>
using vec2 = __attribute__((ext_vector_type(2))) TA;
template <typename TA>
using vec4 = __attribute__((ext_vector_type(4))) TA;

// LDS by 32-bit address; regions of a cell overlap in time, so no
// type-based reordering
template <typename V>
__device__ __forceinline__ V lds_get(unsigned a) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef V __attribute__((may_alias)) VA;
  return *(const __attribute__((address_space(3))) VA*)(a);
#else
  return V();
#endif
}
template <typename V>
__device__ __forceinline__ void lds_put(unsigned a, V v) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef V __attribute__((may_alias)) VA;
  *(__attribute__((address_space(3))) VA*)(a) = v;
#endif
}
__device__ __forceinline__ unsigned lds_address(const char* p) {
#ifdef __HIP_DEVICE_COMPILE__
  return (unsigned)(size_t)(const __attribute__((address_space(3))) char*)p;
#else
  return 0u;
#endif
}

// The instruction stream, in device memory or staged in LDS.  Device memory
// is read through a buffer resource: the lane's offset is one register for
// all records of a size, the record's a scalar, and there is no vector address
// arithmetic.  With plain loads several FP64, aerosol and adjoint instances
// spilled vector registers, and in the 4-slot aerosol one the compiler stored
// a spill (the largest step length) under the wrong lane mask, so its cells
// lost their step control; check_exec_mask.py refuses a build with such a
// store.  Measured, plain -> buffer loads: 131040 CB05 cells mixed 154.1 ->
// 145.5 ms; 363 cells FP64 4177 -> 4058 us; 16411 cells FP64 36.3 -> 37.4 ms.
template <bool STAGED>
struct WordStream {
  const unsigned* g;  // device memory
  unsigned l;         // LDS address
  int bytes;          // stream length in device memory
  // record of this lane in round r of a section at word o
  template <typename V>
  __device__ __forceinline__ V rec(int o, int r, int lane) const {
    constexpr int w = int(sizeof(V) / 4);
    if constexpr (STAGED) return lds_get<V>(l + 4u * unsigned(o + 64 * w * r) + unsigned(4 * w * lane));
#ifdef __HIP_DEVICE_COMPILE__
    const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned*>(g), 0, bytes, 0x00027000);
    // readfirstlane keeps the uniform offset scalar whatever the loop optimiser does
    const int v = 4 * w * lane, s = __builtin_amdgcn_readfirstlane(4 * (o + 64 * w * r));
    if constexpr (w == 1) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(b, v, s, 0));
    else if constexpr (w == 2) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(b, v, s, 0));
    else if constexpr (w == 4) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(b, v, s, 0));
    else {
      static_assert(w == 8 || w <= 4, "record size");
      struct Two { u32x4 a, b; } t;
      t.a = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b, v, s, 0));
      t.b = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b, v + 16, s, 0));
      return __builtin_bit_cast(V, t);
    }
#else
    return V();
#endif
  }
  // a wavefront-uniform 64-bit mask (scalar registers; the stream in device
  // memory is read through the scalar cache)
  __device__ __forceinline__ unsigned long long mask(int word) const {
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (!STAGED) {
      const auto* p = (const __attribute__((address_space(4))) unsigned*)(g + word);
      return (unsigned long long)p[0] | ((unsigned long long)p[1] << 32);
    }
#endif
    const unsigned lo = __builtin_amdgcn_readfirstlane(lds_get<unsigned>(l + 4u * unsigned(word)));
    const unsigned hi = __builtin_amdgcn_readfirstlane(lds_get<unsigned>(l + 4u * unsigned(word + 1)));
    return (unsigned long long)lo | ((unsigned long long)hi << 32);
  }
};

// fields of a word as LDS addresses
template <int SH>
__device__ __forceinline__ unsigned at_lo(unsigned w, unsigned base) {
  return base + ((w & 0xffffu) << SH);
}
template <int SH>
__device__ __forceinline__ unsigned at_hi(unsigned w, unsigned base) {
  return base + ((w >> 16) << SH);
}

// n rounds, records two rounds ahead in three register sets.  The loads past
// the last round read what follows the section (the stream ends with room
// for it).
template <class W, class Load, class Exec>
__device__ __forceinline__ void rotate(int n, Load load, Exec exec) {
  if (n <= 0) return;
  W a, b, c;
  load(a, 0);
  load(b, 1);
  for (int r = 0;;) {
    load(c, r + 2);
    exec(a, r);
    if (++r >= n) return;
    load(a, r + 2);
    exec(b, r);
    if (++r >= n) return;
    load(b, r + 2);
    exec(c, r);
    if (++r >= n) return;
  }
}

// One cell of the sparse forms: LDS addresses, and pointers to what the
// integrator fills itself.
template <typename TA_, bool STAGED_>
struct SpLds {
  using TA = TA_;
  WordStream<STAGED_> w;
  __device__ __forceinline__ WordStream<false> memory() const { return WordStream<false>{w.g, 0u, w.bytes}; }
  unsigned cell;      // cell region
  unsigned coef;      // coefficient table
  unsigned tol;       // (atol, rtol) per unknown
  double* c;          // [nSpec]
  const double* src;  // nullable: this cell's external sources [m], reference order
};

// Slots no program writes: the zeros and the one.
template <typename L>
__device__ __forceinline__ void sp_init(const DevLowered& W, const L& S, int m, int lane) {
  using TA = typename L::TA;
  if (lane == 0) {
    lds_put<TA>(S.cell + W.zeroA, TA(0));
    lds_put<TA>(S.cell + W.oR + 2 * sizeof(TA) * m, TA(0));
    lds_put<TA>(S.cell + W.oR + 2 * sizeof(TA) * m + sizeof(TA), TA(0));
    lds_put<double>(S.cell + W.oneC, 1.0);
    lds_put<double>(S.cell + W.zero8, 0.0);
  }
  wave_sync();
}

// The cell's rate constants into their slots, and the n * kf slots.
template <int SH, typename L>
__device__ __forceinline__ void sp_load_rates(const DevLowered& W, const L& S, const double* kf, int lane) {
  for (int g = 0; g < W.nRop; ++g) {
    const int r = int(S.w.template rec<unsigned>(W.oKf, g, lane));
    lds_put<double>(S.cell + W.oK + 8 * (kWave * g + lane), r >= 0 ? kf[r] : 0.0);
  }
  wave_sync();
  for (int g = 0; g < W.nKfx; ++g) {
    const u32x2 x = S.w.template rec<u32x2>(W.oKfx, g, lane);
    lds_put<double>(at_lo<SH>(x.y, S.cell), lds_get<double>(S.cell + W.oK + 8 * x.x) * double(x.y >> 16));
  }
  wave_sync();
}

// Rates of progress and, with pairs, the derivatives d rop_r / d c_s at the
// concentrations in LDS.
template <int SH, typename L>
__device__ __forceinline__ void sp_rates(const DevLowered& W, const L& S, int lane, bool pairs) {
  using TA = typename L::TA;
  const unsigned cb = S.cell;
  if (W.nPow > 0) {
    for (int g = 0; g < W.nPow; ++g) {
      const u32x2 x = S.w.template rec<u32x2>(W.oPow, g, lane);
      const double v = lds_get<double>(at_lo<SH>(x.x, cb));
      double p = v;
      for (unsigned i = 1; __builtin_amdgcn_ballot_w64(i < x.y) != 0; ++i) p = i < x.y ? p * v : p;
      lds_put<double>(at_hi<SH>(x.x, cb), p);
    }
    wave_sync();
  }
  {
    unsigned k = cb + W.oK + 8 * lane, o = cb + W.oP + 8 * lane;
    rotate<u32x2>(
        W.nRop, [&](u32x2& x, int r) { x = S.w.template rec<u32x2>(W.oRop, r, lane); },
        [&](const u32x2& x, int) {
          const double kf = lds_get<double>(k);
          const double f0 = lds_get<double>(at_lo<SH>(x.x, cb)), f1 = lds_get<double>(at_hi<SH>(x.x, cb));
          const double f2 = lds_get<double>(at_lo<SH>(x.y, cb));
          lds_put<double>(o, kf * f0 * f1 * f2);
          k += 8 * kWave;
          o += 8 * kWave;
        });
  }
  if (!pairs) return;
  unsigned o = cb + W.oD + unsigned(sizeof(TA)) * lane;
  rotate<u32x2>(
      W.nPair, [&](u32x2& x, int r) { x = S.w.template rec<u32x2>(W.oPair, r, lane); },
      [&](const u32x2& x, int) {
        const double kf = lds_get<double>(at_lo<SH>(x.x, cb)), fd = lds_get<double>(at_hi<SH>(x.x, cb));
        const double g0 = lds_get<double>(at_lo<SH>(x.y, cb)), g1 = lds_get<double>(at_hi<SH>(x.y, cb));
        lds_put<TA>(o, TA(kf * fd * g0 * g1));
        o += unsigned(sizeof(TA)) * kWave;
      });
}

// A SUM section: out[64 p + lane] of every group p; the second operands of
// the entries are relative to yBase.
template <int SH, typename L>
__device__ __forceinline__ void sp_sums(const L& S, int oHdr, int oBody, int n, unsigned yBase, unsigned out,
                                        int lane) {
  const unsigned cb = S.cell;
  unsigned o = out + 8 * lane;
  double acc = 0.0;
  for (int r0 = 0; r0 < n; r0 += 64) {
    const unsigned long long first = S.w.mask(oHdr + r0 / 16), last = S.w.mask(oHdr + r0 / 16 + 2);
    rotate<u32x4>(
        n - r0 < 64 ? n - r0 : 64,
        [&](u32x4& x, int r) { x = S.w.template rec<u32x4>(oBody, r0 + r, lane); },
        [&](const u32x4& x, int r) {
          double v[4], y[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[j] = lds_get<double>(at_lo<SH>(x[j], cb));
            y[j] = lds_get<double>(at_hi<SH>(x[j], yBase));
          }
          if ((first >> r) & 1) acc = 0.0;
#pragma unroll
          for (int j = 0; j < 4; ++j) acc = fma(y[j], v[j], acc);
          if ((last >> r) & 1) {
            lds_put<double>(o, acc);
            o += 8 * kWave;
          }
        });
  }
}

// f of the species of this lane: s (emission and external sources) plus
// their segment sums in order
template <int SH, int QM, typename L>
__device__ __forceinline__ void sp_rows(const DevLowered& W, const L& S, int lane, double (&s)[QM]) {
  int o = W.oRow;
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    for (int r = 0; r < W.nRow[q]; ++r) {
      const u32x2 x = S.w.template rec<u32x2>(o, r, lane);
      const double a = lds_get<double>(at_lo<SH>(x.x, S.cell)), b = lds_get<double>(at_hi<SH>(x.x, S.cell));
      const double c = lds_get<double>(at_lo<SH>(x.y, S.cell)), d = lds_get<double>(at_hi<SH>(x.y, S.cell));
      s[q] = s[q] + a;
      s[q] = s[q] + b;
      s[q] = s[q] + c;
      s[q] = s[q] + d;
    }
    o += 128 * W.nRow[q];
  }
}

// A = I + scale * J on the factor pattern (fill positions cleared)
template <int SH, typename L>
__device__ __forceinline__ void sp_jacobian(const DevLowered& W, const L& S, int lane,
                                            typename L::TA scale) {
  using TA = typename L::TA;
  struct Rec {
    u32x4 w;
    vec4<TA> c;
  };
  const unsigned cb = S.cell;
  const auto words = S.memory();
  const int n4 = W.nJ4, n2 = n4 + W.nJ2;
  rotate<Rec>(
      n2 + W.nJ1,
      [&](Rec& x, int r) {
        x.w = words.template rec<u32x4>(W.oJac, r, lane);
        x.c = words.template rec<vec4<TA>>(W.oJacC, r, lane);
      },
      [&](const Rec& x, int r) {
        const TA p0 = lds_get<TA>(at_lo<SH>(x.w.x, cb)), p1 = lds_get<TA>(at_hi<SH>(x.w.x, cb));
        const TA p2 = lds_get<TA>(at_lo<SH>(x.w.y, cb)), p3 = lds_get<TA>(at_hi<SH>(x.w.y, cb));
        if (r < n4) {
          const TA s = fma(x.c.w, p3, fma(x.c.z, p2, fma(x.c.y, p1, x.c.x * p0)));
          const TA v = fma(scale, s, (x.w.w & 1u) ? TA(1) : TA(0));
          lds_put<TA>(at_lo<SH>(x.w.z, cb), (x.w.w & 2u) ? s : v);
        } else if (r < n2) {
          lds_put<TA>(at_lo<SH>(x.w.z, cb), scale * fma(x.c.y, p1, x.c.x * p0));
          lds_put<TA>(at_hi<SH>(x.w.z, cb), scale * fma(x.c.w, p3, x.c.z * p2));
        } else {
          lds_put<TA>(at_lo<SH>(x.w.z, cb), scale * (x.c.x * p0));
          lds_put<TA>(at_hi<SH>(x.w.z, cb), scale * (x.c.y * p1));
          lds_put<TA>(at_lo<SH>(x.w.w, cb), scale * (x.c.z * p2));
          lds_put<TA>(at_hi<SH>(x.w.w, cb), scale * (x.c.w * p3));
        }
      });
  wave_sync();
  for (int g = 0; g < W.nJx; ++g) {
    const u32x2 x = words.template rec<u32x2>(W.oJx, g, lane);
    const int n = int(x.y & 0x7fffffffu);
    const int most = __builtin_amdgcn_readfirstlane(n);  // the first lane's is the largest
    const unsigned zero = cb + W.zeroA;
    unsigned p = at_hi<SH>(x.x, cb);
    TA acc = (x.y >> 31) ? TA(1) : TA(0);
    for (int j = 0; j < most; j += 4) {
      TA v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = lds_get<TA>(j + k < n ? p + unsigned(sizeof(TA)) * k : zero);
#pragma unroll
      for (int k = 0; k < 4; ++k) acc = fma(scale, v[k], acc);
      p += 4 * unsigned(sizeof(TA));
    }
    lds_put<TA>(at_lo<SH>(x.x, cb), acc);
  }
}

// Reciprocal of a pivot: the correctly rounded quotient in FP64; in FP32 the
// hardware reciprocal (within 1 ulp: one instruction instead of the eleven of
// a correctly rounded division, well inside the FP32 factorisation's own
// rounding).  Zero and non-finite pivots give non-finite reciprocals in both.
template <typename TA>
__device__ __forceinline__ TA pivot_recip(TA p) {
  if constexpr (sizeof(TA) == sizeof(float))
    return __builtin_amdgcn_rcpf(p);
  else
    return TA(1) / p;
}

// Rounds of the factorisation (and of the forward substitution with stored
// factors).
template <int SH, typename L, typename Words>
__device__ __forceinline__ void sp_lu(const L& S, const Words& words, int oHdr, int o4, int o1, int n,
                                      int lane) {
  using TA = typename L::TA;
  struct Rec {
    u32x4 w;
    unsigned z;
  };
  const unsigned cb = S.cell;
  for (int r0 = 0; r0 < n; r0 += 64) {
    const unsigned long long mul = words.mask(oHdr + r0 / 16), upd = words.mask(oHdr + r0 / 16 + 2);
    rotate<Rec>(
        n - r0 < 64 ? n - r0 : 64,
        [&](Rec& x, int r) {
          x.w = words.template rec<u32x4>(o4, r0 + r, lane);
          x.z = words.template rec<unsigned>(o1, r0 + r, lane);
        },
        [&](const Rec& x, int r) {
          const unsigned t = at_lo<SH>(x.w.x, cb);
          if ((mul >> r) & 1) {
            const TA p = lds_get<TA>(at_hi<SH>(x.w.x, cb));
            lds_put<TA>(t, lds_get<TA>(t) * pivot_recip(p));
          } else if ((upd >> r) & 1) {
            TA acc = lds_get<TA>(t);
            const TA l0 = lds_get<TA>(at_hi<SH>(x.w.x, cb)), u0 = lds_get<TA>(at_lo<SH>(x.w.y, cb));
            const TA l1 = lds_get<TA>(at_hi<SH>(x.w.y, cb)), u1 = lds_get<TA>(at_lo<SH>(x.w.z, cb));
            const TA l2 = lds_get<TA>(at_hi<SH>(x.w.z, cb)), u2 = lds_get<TA>(at_lo<SH>(x.w.w, cb));
            const TA l3 = lds_get<TA>(at_hi<SH>(x.w.w, cb)), u3 = lds_get<TA>(at_lo<SH>(x.z, cb));
            acc = fma(-l0, u0, acc);
            acc = fma(-l1, u1, acc);
            acc = fma(-l2, u2, acc);
            lds_put<TA>(t, fma(-l3, u3, acc));
          } else {
            const TA p = lds_get<TA>(at_hi<SH>(x.w.y, cb));
            const TA a = lds_get<TA>(at_hi<SH>(x.w.x, cb)), b = lds_get<TA>(at_lo<SH>(x.w.y, cb));
            TA acc = lds_get<TA>(t);
            const TA l0 = lds_get<TA>(at_lo<SH>(x.w.z, cb)), u0 = lds_get<TA>(at_hi<SH>(x.w.z, cb));
            const TA l1 = lds_get<TA>(at_lo<SH>(x.w.w, cb)), u1 = lds_get<TA>(at_hi<SH>(x.w.w, cb));
            const TA inv = pivot_recip(p);
            const TA l = a == TA(0) ? TA(0) : a * inv;
            acc = fma(-l0, u0, acc);
            acc = fma(-l1, u1, acc);
            lds_put<TA>(t, at_hi<SH>(x.w.x, cb) == t ? l : fma(-l, b, acc));
          }
        });
  }
  wave_sync();
}

// Reciprocal pivots of the m rows, kept beside their right-hand sides (the
// multiplier rounds form the same values again).  Returns false when a pivot is zero
// or not finite.
template <int SH, int QM, typename L>
__device__ __forceinline__ bool sp_pivots(const DevLowered& W, const L& S, int m, int lane) {
  using TA = typename L::TA;
  bool bad = false;
#pragma unroll
  for (int q = 0; q < QM; ++q) {
    const int i = lane + kWave * q;
    if (i < m) {
      const TA p = lds_get<TA>(S.cell + S.w.template rec<unsigned>(W.oDiag, q, lane));
      const TA inv = pivot_recip(p);
      lds_put<TA>(S.cell + W.oR + 2 * sizeof(TA) * i + sizeof(TA), inv);
      bad |= !(p != TA(0) && isfinite(p) && isfinite(inv));
    }
  }
  wave_sync();
  return ballot(bad) == 0;
}

// Back substitution: afterwards the right-hand side holds u_ii x_i.
template <int SH, typename L>
__device__ __forceinline__ void sp_back(const DevLowered& W, const L& S, int lane) {
  using TA = typename L::TA;
  const unsigned cb = S.cell;
  rotate<u32x4>(
      W.nBack, [&](u32x4& x, int r) { x = S.w.template rec<u32x4>(W.oBack, r, lane); },
      [&](const u32x4& x, int) {
        const TA u0 = lds_get<TA>(at_hi<SH>(x.x, cb)), u1 = lds_get<TA>(at_hi<SH>(x.z, cb));
        const unsigned t0 = at_lo<SH>(x.x, cb), t1 = at_lo<SH>(x.z, cb);
        const vec2<TA> p0 = lds_get<vec2<TA>>(at_lo<SH>(x.y, cb));
        const TA a0 = lds_get<TA>(t0);
        lds_put<TA>(t0, fma(-u0, p0.x * p0.y, a0));
        const vec2<TA> p1 = lds_get<vec2<TA>>(at_lo<SH>(x.w, cb));
        const TA a1 = lds_get<TA>(t1);
        lds_put<TA>(t1, fma(-u1, p1.x * p1.y, a1));
      });
  wave_sync();
}

// Copies the stream (staged form) and the coefficient table to the start of
// the workgroup's LDS; the unknowns' tolerances and the cell regions follow
// (sparseStageBytes).  The caller synchronises the workgroup.
template <bool STAGED>
__device__ __forceinline__ void stage_sparse(const DevLowered& W, const unsigned* words, const double* coef,
                                             char* base) {
  if constexpr (STAGED) {
    uint4* dst = reinterpret_cast<uint4*>(base);
    const uint4* src = reinterpret_cast<const uint4*>(words);
    for (int i = threadIdx.x; i < W.stagedWords / 4; i += blockDim.x) dst[i] = src[i];
  }
  double* cd = reinterpret_cast<double*>(base + (STAGED ? 4 * size_t(W.stagedWords) : 0));
  for (int i = threadIdx.x; i < W.nCoef; i += blockDim.x) cd[i] = coef[i];
}

// The view of the wave-th cell of the workgroup, m unknowns' tolerances staged.
template <typename TA, bool STAGED>
__device__ __forceinline__ SpLds<TA, STAGED> carve_sparse(const DevLowered& W, const unsigned* words, int m, char* base,
                                                         int cellBytes, int wave) {
  SpLds<TA, STAGED> L;
  const unsigned b = lds_address(base);
  L.w.g = words;
  L.w.l = b;
  L.w.bytes = 4 * W.words;
  L.coef = b + (STAGED ? 4u * unsigned(W.stagedWords) : 0u);
  L.tol = b + unsigned(sparseStageBytes(W, 0, STAGED));
  const size_t at = sparseStageBytes(W, m, STAGED) + size_t(wave) * size_t(cellBytes);
  L.cell = __builtin_amdgcn_readfirstlane(b + unsigned(at));
  L.c = reinterpret_cast<double*>(base + at + W.oC);
  L.src = nullptr;
  return L;
}

}  // namespace
}  // namespace tchem_amd
