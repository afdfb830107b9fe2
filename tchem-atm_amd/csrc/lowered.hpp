// Device encoding of the sparse programs (schedule.hpp) and of the source
// term and Jacobian around them: the instruction stream one wavefront
// executes per Newton iteration of its cell.
//
// The rounds of schedule.hpp say what is computed and in which order; this
// pass only chooses where operands live and how a round is spelled, so that a
// round costs the device little more than its operand reads:
//   * every operand field is the final LDS address (byte offset in the cell
//     region, >> shift), 16 bits, no indexing or scaling left to do;
//   * a section holds records of one size, read with 8- or 16-byte loads two
//     rounds ahead, and one kind of round wherever the order allows it, so
//     the loop has no per-round dispatch on kind or length;
//   * reactant powers and derivative factors are plain reads: powers c^n
//     (n >= 2) and n * kf are extra slots, an absent reactant reads a slot
//     that holds 1;
//   * right-hand side and reciprocal pivot of a row are neighbours (one read
//     in the back substitution).
//   * reactions, derivative pairs and factor entries are numbered so that the
//     gathers of the rounds fall on distinct LDS banks (spreadOverBanks).
// The value of every slot is the rounds' value bit for bit: the same
// operations on the same operands in the same order per target (a Jacobian
// chain keeps its partial sums of kMaxChain contributions).
//
// Sections (words are 32-bit, a record of w words per lane is stored as
// [lane][w], 64 records per round):
//   POW   w 2: source field | destination field << 16, exponent
//   KF    w 1: reaction whose rate constant is in this slot, -1 for a zero
//         (once per cell)
//   KFX   w 2: slot, destination field | factor << 16   (once per cell)
//   ROP   w 2: f0 | f1 << 16, f2; rop[64 r + lane] = kf[64 r + lane] f0 f1 f2
//   PAIR  w 2: kf | fd << 16, g0 | g1 << 16; dpr[64 r + lane] = kf fd g0 g1
//   SUM   (segments; nu^T mu and J^T mu of the adjoint) w 4: four entries
//         x | y << 16; acc = fma(y, x, acc); sums go to out[64 p + lane] for
//         the p-th group of 64; per 64 rounds a header of two 64-bit masks:
//         rounds that start a group, rounds that end one
//   ROW   w 2: four fields; species sum = emission + them in order
//   JAC   w 4 + four coefficients: dpr fields d0 | d1 << 16, d2 | d3 << 16,
//         targets.  Three kinds in turn: J4 one target, four entries (word 2:
//         target, word 3: bit 0 diagonal, bit 1 the sum alone goes to a
//         partial slot); J2 two targets of two entries (word 2); J1 four
//         targets of one (words 2, 3)
//   JX    w 2: target | first partial << 16, count | diagonal << 31 (largest
//         count first): partials added to the initial value in order
//   LU    w 4 and w 1; per 64 rounds a header of two 64-bit masks: rounds of
//         kind kLMul, rounds of kind kLUpd (others kLMulUpd)
//         kLUpd: target, lo0, hi0, .. lo3, hi3, -
//         kLMulUpd: target, ik, kj, kk, lo0, hi0, lo1, hi1, -, - (a multiplier
//                   lane's target is ik)
//         kLMul: dst, src, -, ..
//   DIAG  w 1: byte offset of the pivot of row 64 r + lane (reciprocal pivots
//         are stored, and pivots checked, once after the last round)
//   FWD   LU rounds of kind kLUpd (factor reuse)
//   BACK  w 4: two single-entry rounds, each target | U << 16, pair
#pragma once

#include <cstdint>
#include <vector>

#include "schedule.hpp"

namespace tchem_amd {

// Plain values shared with the kernels; o* of the cell layout are byte
// offsets in the cell region, o* of sections word offsets in the stream.
struct DevLowered {
  int enabled;
  int shift;      // of every field
  int words;        // stream length, read-ahead included
  int stagedWords;  // of them, those a workgroup that stages the programs copies into LDS: all but JAC, JX, FWD
                    // and the adjoint's sums, which are read from memory (each about as large as the LU section
                    // or rarely run; the LDS they would take holds cells)
  int oWords;     // stream start in the mechanism's int buffer
  int nCoef, oCoef;  // coefficient table (staged into LDS), start in the double buffer
  int tolStaged;     // whether the unknowns' tolerances are staged into LDS too (set by the caller: stageTolerances)
  // cell layout
  int cellBytes;
  int zeroA, trashA;      // slots of the factor array (which starts at 0)
  int oR;                 // (rhs, reciprocal pivot) pairs, rows m (zeros) and m + 1 (trash) after the m unknowns
  int oD, oPS;            // derivative pairs; partial sums (with the segment sums, which are dead then)
  int oC, oneC, trashC;   // concentrations, the slot that holds 1
  int oK, nK, zero8;      // rate constants, with n * kf slots and the slot that holds 0 before them (nK in all)
  int oP, oS;             // rates of progress, segment sums; from the first of oP, oS and oD to the end everything is
                          // dead once the Jacobian is assembled (not in the adjoint)
  // sections
  int oPow, nPow, oKf, oKfx, nKfx, oRop, nRop, oPair, nPair;
  int oSegHdr, oSeg, nSeg;
  int oRow, nRow[4];
  int oJac, oJacC, nJ4, nJ2, nJ1, oJx, nJx;
  int oLuHdr, oLu, oLu1, nLu, oDiag, oBack, nBack, oFwdHdr, oFwd, oFwd1, nFwd;
  // adjoint programs only
  int oNutHdr, oNut, nNut, oJtvHdr, oJtv, nJtv;
  int oMu, oW, oV;  // mu [m + 1] (mu[m] = 0), w sums, v sums (byte offsets in the cell region, the sums in oS's place)
  int oWmap, oVmap;        // byte offset of w_r by slot of reaction r, [64 ceil(m / 64)] of v_i
};

struct LoweredProgram {
  DevLowered d{};
  std::vector<uint32_t> words;
  std::vector<double> coef;  // coefficient table, [0] = 0
  std::vector<int> slot;     // factor slot of the rounds' numbering (SparseSchedule::slotOf) -> slot in the cell
};

// Where reactions, derivative pairs and factor entries live, so that the
// gathers of the rounds fall on distinct LDS banks.  Programs that run on one
// cell region (the adjoint's forward and transposed programs) share the slots
// of reactions and pairs: `shared` are the other program's.
struct LoweredSlots {
  std::vector<int> factor;  // of the rounds' numbering (SparseSchedule::slotOf)
  std::vector<int> pair;    // [64 pairRounds], the first nPairs are the derivative pairs
  std::vector<int> rop;     // [64 ropRounds], the first nReac are the reactions
};
LoweredSlots chooseSlots(const MechTables& t, const SparseSchedule& s, const LoweredSlots* shared = nullptr);

// Lowers the programs of `s` (built from `t`) for matrix entries of
// bytesT bytes (4 or 8).  shift 0 when at most 128 unknowns, and cell region
// and coefficient table are at most 64 KiB each, log2(bytesT) otherwise.
// adjoint: room for mu, w and v, and the transposed
// programs' extra sections; the cell layout depends on sizes only, so the
// forward and transposed programs of one mechanism share it.  Throws
// std::runtime_error when a field does not fit.
LoweredProgram lowerProgram(const MechTables& t, const SparseSchedule& s, int bytesT, bool adjoint,
                            const LoweredSlots& slots);

}  // namespace tchem_amd
