// Prints how many cells of the sparse forms fit a workgroup's LDS: the cell
// regions of the encoded programs (lowered.cpp) beside the coefficient table
// and, where they are staged, the programs.
//
// usage: cells_check <mechanism.yaml> [<aerosol.yaml> <particles>...]
#include <array>
#include <cstdio>
#include <cstdlib>

#include "aerosol_model.hpp"
#include "device_mech.hpp"
#include "kinetic_model.hpp"
#include "lowered.hpp"
#include "mechanism.hpp"
#include "schedule.hpp"
using namespace tchem_amd;

static const size_t kLds = 160 * 1024;
static int cells(size_t stage, size_t cell, int most) {
  const size_t n = stage < kLds ? (kLds - stage) / cell : 0;
  return n < size_t(most) ? int(n) : most;
}

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  const KineticModel km = loadKineticModel(argv[1], nullptr);
  const MechTables t = compileMechanism(km);
  if (argc == 2) {
    const SparseSchedule s = buildSparseSchedule(t);
    const LoweredSlots fs = chooseSlots(t, s);
    for (int bytes : {8, 4}) {
      const DevLowered w = lowerProgram(t, s, bytes, false, fs).d;
      const int most = t.m > 128 ? 8 : (bytes == 8 ? 12 : 16);
      std::printf("fp%d memory %d staged %d\n", 8 * bytes, cells(sparseStageBytes(w, t.m, false), size_t(w.cellBytes), most),
                  cells(sparseStageBytes(w, t.m, true), size_t(w.cellBytes), most));
    }
  }
  for (int i = 3; i < argc; ++i) {
    AerosolModel am = loadAerosolModel(argv[2], km);
    am.nParticles = std::atoi(argv[i]);
    const MechTables ta = aerosolTables(t, am, nullptr);
    const SparseSchedule s = buildSparseSchedule(ta, false);
    const DevLowered w = lowerProgram(ta, s, 8, false, chooseSlots(ta, s)).d;
    DevAerosol X{};
    X.mt = ta.m;
    X.nPart = am.nParticles;
    X.nSimpol = int(am.simpol.size());
    std::printf("particles %d: %d\n", am.nParticles, cells(sparseStageBytes(w, ta.m, false), aerosolSparseCellBytes(w, X), 8));
  }
  return 0;
}
