// Dense LU on the matrix cores for mechanisms whose factor is dense (no
// counterpart in the reference, which factors a dense m x m matrix with
// Tines per Newton iteration, src/core/problems/TChem_Impl_AtmosphericChemistry.hpp:138-155):
// the FP32 iteration matrix I - c h J of one cell, padded to NB x NB tiles of
// 32 x 32 (NB = 4, 6 or 8: the smallest whose order exceeds m), lives in the
// registers of the four wavefronts of a workgroup (NB^2 / 4 tiles per
// wavefront), and is factored in place without interchanges
// between blocks (the pivots of the fill-reducing order, as in the sparse
// form) by 32 x 32 blocks in Schur-complement form (factorAndSolve):
// the diagonal tile is inverted by one wavefront, and the panel products
// and the trailing update are 32 x 32 x 32 products of 16
// v_mfma_f32_32x32x2f32 instructions each.
// The right-hand side is the last column (rows >= m padded with the
// identity), so the factorisation also does the forward substitution; the
// solution is x = -z[0..m), z = U^-1 e_last, by block back substitution with
// the kept inverses of the diagonal blocks.  Tile (I, J) belongs to wavefront
// 2 (I & 1) + (J & 1), so every trailing update spreads over the four
// wavefronts.
//
// What bounds it: the chain diagonal inverse -> panel -> next diagonal tile of
// the four wavefronts (one per SIMD, the tiles fill the registers), then the
// MFMAs of the trailing update.  So operands lie in LDS as the lanes take them
// (four 16-byte reads per 32 x 32 operand instead of sixteen 4-byte ones), the
// A operand of a block row is read once, the panel goes over all four
// wavefronts, and tiles that would be identity padding do not exist.
// Measured: 2048 systems of order 250 1768 -> 1112 us; the integrator with 160
// species, 603 cells, 30 iterations 21.0 -> 12.7 ms (same bits).
//
// MFMA register layouts (v_mfma_f32_32x32x2f32, D = A B + C):
//   A (32 x 2): lane l holds A[l % 32][l / 32];  B (2 x 32): lane l holds
//   B[l / 32][l % 32];  C/D (32 x 32): register r of lane l holds
//   C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#pragma once

// phase timers of profiling builds (kernels.hip defines them first)
#ifndef TCHEM_PT_BEGIN
#define TCHEM_PT_BEGIN(nm)
#define TCHEM_PT_END(nm, slot)
#endif

namespace mfma {

using f32x16 = __attribute__((ext_vector_type(16))) float;

constexpr int kTile = 32;
constexpr int kLd = kTile + 1;     // LDS row stride of a row-major tile (odd: conflict-free column reads)
constexpr int kTileWords = kTile * kLd;

// tiles per side for m unknowns and the right-hand side
__host__ __device__ constexpr int tilesFor(int m) { return m < 4 * kTile ? 4 : (m < 6 * kTile ? 6 : 8); }

__device__ __forceinline__ int crow(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// Operand tiles of a 32 x 32 x 32 product in LDS: element (o, k), o the outer
// index (row of A, column of B), k the inner one, is where lane
// o + 32 (k & 1) finds its 16 values (inner pairs 0..15) as four 16-byte
// reads.  The four-word groups of an outer index are rotated by o / 4, so 16
// lanes read all 64 banks; the half of odd k starts 16 words on, which keeps
// the stores of a C-layout tile two-way.
constexpr int kOpHalf = kTile * 16 + 16;
constexpr int kOpWords = 2 * kOpHalf;
static_assert(kOpWords <= kTileWords, "an operand tile takes no more room than a row-major one");
__device__ __forceinline__ int opAt(int o, int k) {
  return (k & 1) * kOpHalf + o * 16 + ((((k >> 3) ^ (o >> 2)) & 3) << 2) + ((k >> 1) & 3);
}

// LDS of one cell of the MFMA form (floats unless noted), after the
// integrator's cell region
struct Lu {
  float* stage;    // [32 NB][64 + 1] column strip of the matrix during assembly; reused for the panels
  float* lpanel;   // [NB - 1][kOpWords] A_ik, then -P_ik of the current step (operand A; aliases stage)
  float* upanel;   // [NB - 1][kOpWords] A_kj of the current step (operand B; aliases stage)
  float* invBuf;   // [kTile][kCm] column-major copy of the tile being inverted (aliases stage, past the panels)
  float* diag;     // [kOpWords] D_k^-1 - I of the current step (operand B)
  float* uinv;     // [NB][kTileWords] D_k^-1 of every block (back substitution)
  float* z;        // [32 NB] back substitution unknowns
  float* ypart;    // [4][kTile] partial block sums of the four wavefronts
  int* cmd;        // [2] command word of the driver wavefront, zero-pivot flag
  double* ch;      // [1] c h of the current iteration matrix
};

constexpr int kCm = 36;  // column stride of the column-major copy (16-byte aligned columns)
__host__ __device__ constexpr size_t stageWords(int nb) {
  const size_t panels = size_t(2 * (nb - 1)) * kOpWords + size_t(kTile) * kCm;
  const size_t strip = size_t(kTile) * nb * 65;
  return strip > panels ? strip : panels;
}
__host__ __device__ constexpr size_t luLdsBytes(int nb) {
  return 4 * (stageWords(nb) + size_t(kTileWords) * (1 + nb) + size_t(kTile) * nb + 4 * kTile) + 16 + 16;
}

__device__ inline Lu carveLu(char* base, int nb) {
  Lu L;
  float* f = reinterpret_cast<float*>(base);
  L.stage = f;
  L.lpanel = f;
  L.upanel = f + size_t(nb - 1) * kOpWords;
  L.invBuf = f + size_t(2 * (nb - 1)) * kOpWords;
  L.diag = f + stageWords(nb);
  L.uinv = L.diag + kTileWords;
  L.z = L.uinv + size_t(nb) * kTileWords;
  L.ypart = L.z + kTile * nb;
  char* tail = reinterpret_cast<char*>(L.ypart + 4 * kTile);
  L.cmd = reinterpret_cast<int*>(tail);
  L.ch = reinterpret_cast<double*>(tail + 16);
  return L;
}

// LDS row-major [32][ld] -> C-layout tile
__device__ __forceinline__ f32x16 loadTile(const float* src, int ld, int lane) {
  f32x16 c;
#pragma unroll
  for (int r = 0; r < 16; ++r) c[r] = src[crow(r, lane) * ld + (lane & 31)];
  return c;
}

// C-layout tile -> operand A (outer index: row) and back, operand B (outer
// index: column; a lane's rows 4 j .. 4 j + 3 are two inner pairs)
template <bool NEG>
__device__ __forceinline__ void storeA(const f32x16& c, float* dst, int lane) {
#pragma unroll
  for (int r = 0; r < 16; ++r) dst[opAt(crow(r, lane), lane & 31)] = NEG ? -c[r] : c[r];
}
__device__ __forceinline__ f32x16 loadA(const float* src, int lane) {
  f32x16 c;
#pragma unroll
  for (int r = 0; r < 16; ++r) c[r] = src[opAt(crow(r, lane), lane & 31)];
  return c;
}
__device__ __forceinline__ void storeB(const f32x16& c, float* dst, int lane) {
#pragma unroll
  for (int r = 0; r < 16; r += 4) {
    const int k = crow(r, lane), o = lane & 31;
    *reinterpret_cast<float2*>(dst + opAt(o, k)) = float2{c[r], c[r + 2]};
    *reinterpret_cast<float2*>(dst + opAt(o, k + 1)) = float2{c[r + 1], c[r + 3]};
  }
}

// this lane's values of an operand tile
struct Operand {
  float v[16];
};
__device__ __forceinline__ Operand operand(const float* src, int lane) {
  Operand t;
  const int o = lane & 31, kk = lane >> 5;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float4 f = *reinterpret_cast<const float4*>(src + opAt(o, 8 * g + kk));
    t.v[4 * g] = f.x;
    t.v[4 * g + 1] = f.y;
    t.v[4 * g + 2] = f.z;
    t.v[4 * g + 3] = f.w;
  }
  return t;
}

// acc += A B of 32 x 32 tiles: 16 MFMAs of K = 2
__device__ __forceinline__ f32x16 mma32(f32x16 acc, const Operand& A, const Operand& B) {
#pragma unroll
  for (int s = 0; s < kTile / 2; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(A.v[s], B.v[s], acc, 0, 0, 0);
  return acc;
}

__device__ __forceinline__ void wsync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One wavefront inverts a tile in its own registers (C layout), in place,
// by block Gauss-Jordan with 2 x 2 pivot blocks P = {p, p+1} and no
// interchanges (the pivots of the fill-reducing order, as in the sparse
// form).  With S = M_PP^-1, one step is the rank-2 update
//   M <- M + A B,  A = E_P - M_:P (32 x 2),
//   B = S M_P: with columns P replaced by S + I (2 x 32),
// which leaves S M_PQ in the pivot rows, -M_OP S in the pivot columns, S in
// the pivot block and M_OQ - M_OP S M_PQ elsewhere: after 16 steps the tile
// holds M^-1.  Each step is one v_mfma_f32_32x32x2f32; its operands are
// read from a column-major copy of the tile in LDS (buf, [32][36] floats,
// 16-byte aligned).  A zero or non-finite pivot block sets *bad.
__device__ __forceinline__ void invertTileInPlace(f32x16& acc, float* buf, int lane, bool* bad) {
#pragma clang fp contract(off)
  const int c = lane & 31, h = lane >> 5;
  bool ok = true;
  for (int p = 0; p < kTile; p += 2) {
    // registers 4j..4j+3 hold rows 8j + 4h .. 8j + 4h + 3 of column c
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<float4*>(buf + c * kCm + 8 * j + 4 * h) = float4{acc[4 * j], acc[4 * j + 1], acc[4 * j + 2],
                                                                           acc[4 * j + 3]};
    wsync();
    const float mcol = buf[(p + h) * kCm + c];  // M[c][p + h]
    const float r0 = buf[c * kCm + p], r1 = buf[c * kCm + p + 1];  // M[p][c], M[p + 1][c]
    const float m00 = buf[p * kCm + p], m10 = buf[p * kCm + p + 1];
    const float m01 = buf[(p + 1) * kCm + p], m11 = buf[(p + 1) * kCm + p + 1];
    wsync();  // every read done before the next step's copy
    const float det = m00 * m11 - m01 * m10;
    ok = ok && det != 0.0f && isfinite(det);
    const float rdet = __builtin_amdgcn_rcpf(det);
    const float s0 = h ? -m10 * rdet : m11 * rdet;  // row h of S
    const float s1 = h ? m00 * rdet : -m01 * rdet;
    const float a = (c == p + h ? 1.0f : 0.0f) - mcol;
    float b = s0 * r0 + s1 * r1;
    if (c == p) b = s0 + (h == 0 ? 1.0f : 0.0f);
    if (c == p + 1) b = s1 + (h == 1 ? 1.0f : 0.0f);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
  }
  if (!ok) *bad = true;
}

// After invertTileInPlace: D^-1 into dinvK (kept for the back substitution,
// row-major with stride kLd) and D^-1 - I into L.diag (the panel operand:
// with the identity taken out, P_ik = A_ik D^-1 = A_ik + A_ik (D^-1 - I)).
__device__ __forceinline__ void storeInverse(const f32x16& inv, const Lu& L, float* dinvK, int lane) {
  f32x16 d;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = crow(r, lane), col = lane & 31;
    dinvK[row * kLd + col] = inv[r];
    d[r] = row == col ? inv[r] - 1.0f : inv[r];
  }
  storeB(d, L.diag, lane);
}

// Block LU without interchanges between blocks, Schur-complement form:
//   step k: P_ik = A_ik D_k^-1 (D_k the diagonal tile, inverted by its
//   owner), A_ij -= P_ik A_kj for i, j > k.
// The block row A_kj (j > k) is left as it stands, so the factor is
// A = L U with L_ik = P_ik (unit diagonal blocks) and U_kj = A_kj, U_kk = D_k;
// the right-hand side is the last column, so the elimination also applies L^-1
// to it and the solution needs only the back substitution with U, whose
// diagonal blocks are inverted already.  Look-ahead: in step k's trailing
// update the owner of tile (k+1, k+1) updates it first and inverts it while
// the other wavefronts finish their tiles.  Only two wavefronts own tiles of
// block column k, so the panel products go by block row over all four (a
// product is 16 dependent MFMAs, 1024 cycles): owners put A_ik into LDS, and
// -P_ik replaces it there (the tile itself is not needed any more).
//
// All four wavefronts of the workgroup call this with their own tiles (wave
// = 0..3, acc[a * NB / 2 + b] = tile (2 a + wave / 2, 2 b + wave % 2)); it
// contains the workgroup barriers.  On return z[0..32 NB) holds U^-1 e_last;
// cmd[1] is set when a pivot was zero or not finite.
template <int NB>
__device__ __forceinline__ void factorAndSolve(f32x16 (&acc)[NB * NB / 4], const Lu& L, int wave, int lane) {
  constexpr int T = NB / 2;
  const int wi = wave >> 1, wj = wave & 1;
  bool bad = false;
  TCHEM_PT_BEGIN(d0)
  if (wave == 0) {
    f32x16 d = acc[0];
    invertTileInPlace(d, L.invBuf, lane, &bad);
    storeInverse(d, L, L.uinv, lane);
  }
  TCHEM_PT_END(d0, 5)
#pragma unroll 1
  for (int k = 0; k < NB - 1; ++k) {
    const int odd = k & 1, half = k >> 1, n = k + 1;
    TCHEM_PT_BEGIN(pn)
#pragma unroll
    for (int b = 0; b < T; ++b) {
      if (half != b) continue;
#pragma unroll
      for (int o = 0; o < T; ++o) {
        if (wj == odd && 2 * o + wi > k) storeA<false>(acc[o * T + b], L.lpanel + (2 * o + wi - n) * kOpWords, lane);
        if (wi == odd && 2 * o + wj > k) storeB(acc[b * T + o], L.upanel + (2 * o + wj - n) * kOpWords, lane);
      }
    }
    __syncthreads();
    const Operand dinv = operand(L.diag, lane);
#pragma unroll 1
    for (int i = wave; i < NB - 1 - k; i += 4) {
      float* slot = L.lpanel + i * kOpWords;
      const f32x16 p = mma32(loadA(slot, lane), operand(slot, lane), dinv);
      wsync();
      storeA<true>(p, slot, lane);
    }
    __syncthreads();
    TCHEM_PT_END(pn, 7)
    TCHEM_PT_BEGIN(dg)
    if (wave == 3 * (n & 1)) {  // the owner of tile (n, n)
      const Operand l = operand(L.lpanel, lane), u = operand(L.upanel, lane);
      f32x16 d;
#pragma unroll
      for (int o = 0; o < T; ++o)
        if ((n >> 1) == o) d = mma32(acc[o * T + o], l, u);
      invertTileInPlace(d, L.invBuf, lane, &bad);
      storeInverse(d, L, L.uinv + n * kTileWords, lane);
    }
    TCHEM_PT_END(dg, 5)
    TCHEM_PT_BEGIN(tr)
#pragma unroll
    for (int o = 0; o < T; ++o) {
      if (2 * o + wi <= k) continue;
      const Operand l = operand(L.lpanel + (2 * o + wi - n) * kOpWords, lane);
#pragma unroll
      for (int b = 0; b < T; ++b)
        if (2 * b + wj > k && !(o == b && wi == wj && 2 * o + wi == n))
          acc[o * T + b] = mma32(acc[o * T + b], l, operand(L.upanel + (2 * b + wj - n) * kOpWords, lane));
    }
    __syncthreads();
    TCHEM_PT_END(tr, 8)
  }
  if (bad && lane == 0) L.cmd[1] = 1;
  TCHEM_PT_BEGIN(bs)
  // z = U^-1 e_last: the last block is column 31 of its inverse, then upwards
  if (wave == 0 && lane < kTile) L.z[(NB - 1) * kTile + lane] = L.uinv[size_t(NB - 1) * kTileWords + lane * kLd + 31];
  __syncthreads();
#pragma unroll 1
  for (int I = NB - 2; I >= 0; --I) {
    // the two wavefronts holding block row I: U_IJ z_J of their tiles, row
    // sums by a transposed store (the stage region is free by now)
    if (wi == (I & 1)) {
      float part[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) part[r] = 0.0f;
#pragma unroll
      for (int o = 0; o < T; ++o) {
        if (2 * o + wi != I) continue;
#pragma unroll
        for (int b = 0; b < T; ++b) {
          if (2 * b + wj <= I) continue;
          const float zj = L.z[(2 * b + wj) * kTile + (lane & 31)];
#pragma unroll
          for (int r = 0; r < 16; ++r) part[r] = fmaf(acc[o * T + b][r], zj, part[r]);
        }
      }
      float* yt = L.stage + (wave & 1) * kTileWords;
#pragma unroll
      for (int r = 0; r < 16; ++r) yt[crow(r, lane) * kLd + (lane & 31)] = part[r];
    }
    __syncthreads();
    if (wave == 0) {
      // lane i + 32 h sums row i of half h; y_I = -(both halves)
      const float* yt = L.stage + (lane >> 5) * kTileWords + (lane & 31) * kLd;
      float y = 0.0f;
#pragma unroll
      for (int c = 0; c < kTile; ++c) y += yt[c];
      y += __shfl_xor(y, 32, 64);
      if (lane < kTile) L.ypart[lane] = -y;
      wsync();
      // z_I = D_I^-1 y_I: lane i + 32 h takes columns 16 h .. 16 h + 15 of row i
      const float* ui = L.uinv + size_t(I) * kTileWords + (lane & 31) * kLd + 16 * (lane >> 5);
      const float* yv = L.ypart + 16 * (lane >> 5);
      float zi = 0.0f;
#pragma unroll
      for (int c = 0; c < 16; ++c) zi = fmaf(ui[c], yv[c], zi);
      zi += __shfl_xor(zi, 32, 64);
      if (lane < kTile) L.z[I * kTile + lane] = zi;
    }
    __syncthreads();
  }
  TCHEM_PT_END(bs, 14)
}

// Loads the tiles of wavefront `wave` in column strip Q (columns 64 Q ..
// 64 Q + 63) from the staged strip [32 NB][65].
template <int NB, int Q>
__device__ __forceinline__ void loadStrip(f32x16 (&acc)[NB * NB / 4], const float* stage, int wave, int lane) {
#pragma unroll
  for (int o = 0; o < NB / 2; ++o)
    acc[o * (NB / 2) + Q] = loadTile(stage + ((2 * o + (wave >> 1)) * kTile) * 65 + (wave & 1) * kTile, 65, lane);
}

}  // namespace mfma
