// Prints how many cells of the sparse forms fit a workgroup's LDS: the cell
// regions of the encoded programs (lowered.cpp) beside the coefficient table
// and, where they are staged, the programs and tolerances.
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

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  const KineticModel km = loadKineticModel(argv[1], nullptr);
  const MechTables t = compileMechanism(km);
  if (argc == 2) {
    const SparseSchedule s = buildSparseSchedule(t, false, false);
    const LoweredSlots fs = chooseSlots(t, s);
    for (int bytes : {8, 4}) {
      DevLowered w = lowerProgram(t, s, bytes, false, fs).d;
      const size_t cell = size_t(w.cellBytes);
      const int most = t.m > 128 ? 8 : (bytes == 8 ? 12 : 16);
      int n[2];
      for (const bool staged : {false, true}) {
        stageTolerances(w, t.m, staged, cell, kLds, most);
        n[staged] = sparseCellsThatFit(w, t.m, staged, cell, kLds, most);
      }
      std::printf("fp%d memory %d staged %d\n", 8 * bytes, n[0], n[1]);
    }
  }
  for (int i = 3; i < argc; ++i) {
    AerosolModel am = loadAerosolModel(argv[2], km);
    am.nParticles = std::atoi(argv[i]);
    const MechTables ta = aerosolTables(t, am, nullptr);
    const SparseSchedule s = buildSparseSchedule(ta, false, false);
    DevLowered w = lowerProgram(ta, s, 8, false, chooseSlots(ta, s)).d;
    DevAerosol X{};
    X.mt = ta.m;
    X.nPart = am.nParticles;
    X.nSimpol = int(am.simpol.size());
    stageTolerances(w, ta.m, false, aerosolSparseCellBytes(w, X), kLds, 8);
    std::printf("particles %d: %d\n", am.nParticles,
                sparseCellsThatFit(w, ta.m, false, aerosolSparseCellBytes(w, X), kLds, 8));
  }
  return 0;
}
