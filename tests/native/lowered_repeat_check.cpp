// The encoded programs over several iterations on one cell region, in the
// kernels' order: regions of a cell share room (lowered.cpp: layout), so what
// an iteration leaves behind must not reach the next one, and what the adjoint
// keeps between its sections must survive them.  Executor and reference are
// those of lowered_check.cpp; the schedules are built as the library builds
// them, their factor positions in order.
//
// usage: lowered_repeat_check <mechanism.yaml> [<aerosol.yaml> <particles>...]
#include <cstdlib>

#define main lowered_check_main
#include "lowered_check.cpp"
#undef main

template <typename T>
struct Cell : Stream<T> {
  using Stream<T>::Stream;
  // an evaluation without derivative pairs (stage values, kept factors)
  void ratesAlone(const std::vector<double>& c) {
    const auto& d = this->d;
    for (size_t i = 0; i < c.size(); ++i) this->template put<double>(d.oC + 8 * int(i), c[i]);
    for (int i = 0; i < 64 * d.nPow; ++i) {
      const uint32_t w = this->word(d.oPow + 2 * i);
      this->template put<double>(this->hi(w), ipow(this->template get<double>(this->lo(w)), int(this->word(d.oPow + 2 * i + 1))));
    }
    for (int i = 0; i < 64 * d.nRop; ++i) {
      const uint32_t w0 = this->word(d.oRop + 2 * i), w1 = this->word(d.oRop + 2 * i + 1);
      this->template put<double>(d.oP + 8 * i, this->template get<double>(d.oK + 8 * i) * this->template get<double>(this->lo(w0)) *
                                                   this->template get<double>(this->hi(w0)) * this->template get<double>(this->lo(w1)));
    }
  }
};

template <typename T>
static void repeat(const MechTables& t, const SS& s, const SS& partner, bool adjoint, const char* what) {
  const LoweredSlots fs = chooseSlots(t, s.transposed ? partner : s);
  const LoweredProgram P = lowerProgram(t, s, int(sizeof(T)), adjoint, s.transposed ? chooseSlots(t, s, &fs) : fs);
  const DevLowered& d = P.d;
  const int m = s.m, before = fails;
  std::mt19937_64 rng(5);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  auto some = [&](int n, double lo, double span) {
    std::vector<double> v(size_t(n), 0.0);
    for (auto& x : v) x = std::pow(10.0, lo + span * U(rng));
    return v;
  };
  Cell<T> S(P, t);
  std::vector<double> w;  // of the last solve
  const std::vector<double> kf = some(t.nReac, -3, 4);
  S.init(kf, m);
  if (adjoint) S.template put<double>(d.oMu + 8 * m, 0.0);
  auto rows = [&](const Rounds<T>& R) {
    for (int a = 0; a + 1 < int(t.rowSegPtr.size()); ++a) {
      double f = t.emission[size_t(a)];
      for (int g = t.rowSegPtr[a]; g < t.rowSegPtr[a + 1]; ++g) f += R.seg[size_t(g)];
      CHECK(same(f, S.row(a, t.emission[size_t(a)])), "%s: source term of species %d", what, a);
    }
  };
  auto progress = [&](const Rounds<T>& R) {
    for (int r = 0; r < t.nReac; ++r)
      CHECK(same(R.rop[size_t(r)], S.template get<double>(d.oP + 8 * S.ropAt[size_t(r)])), "%s: rate of progress %d", what, r);
  };
  auto wKept = [&]() {
    for (size_t r = 0; r < w.size(); ++r)
      CHECK(same(w[r], S.template get<double>(int(S.word(d.oWmap + S.ropAt[r])))), "%s: w %zu", what, r);
  };
  for (int it = 0; it < 4; ++it) {
    const std::vector<double> c = some(t.nSpec, -4, 4);
    const double ch = std::pow(10.0, it - 3);
    Rounds<T> R(t, s);
    R.rates(c, kf);
    if (!s.transposed) {  // a stage evaluation first
      const std::vector<double> c0 = some(t.nSpec, -4, 4);
      Rounds<T> R0(t, s);
      R0.rates(c0, kf);
      R0.eval(1.0, -ch);
      S.ratesAlone(c0);
      progress(R0);
      S.segments();
      rows(R0);
    }
    R.eval(1.0, -ch);
    S.rates(c);
    progress(R);
    wKept();
    if (s.transposed && it > 0) {  // v from the last w and the new pairs
      std::vector<double> v(size_t(m), 0.0);
      for (int r = 0; r < t.nReac; ++r)
        for (int p = t.pairPtr[r]; p < t.pairPtr[r + 1]; ++p) {
          double& x = v[size_t(R.spec(r, t.pairSlot[p]))];
          x = fmaT(double(R.dpr[size_t(p)]), w[size_t(r)], x);
        }
      S.sums(d.oJtvHdr, d.oJtv, d.nJtv, d.oV, [&](uint32_t x) { return S.template get<double>(S.hi(x)); });
      for (int i = 0; i < m; ++i) CHECK(same(v[size_t(i)], S.template get<double>(int(S.word(d.oVmap + i)))), "%s: v %d", what, i);
      progress(R);
    }
    if (!s.transposed) {
      S.segments();
      rows(R);
    }
    S.jacobian(T(-ch));
    for (int p = 0; p < s.nnzF; ++p)
      CHECK(same(R.A[size_t(p)], S.template get<T>(int(sizeof(T)) * P.slot[size_t(p)])), "%s: matrix slot %d, iteration %d", what, p, it);
    for (int i = 0; i < m; ++i) {
      const T b = T(U(rng) - 0.5);
      R.A[size_t(s.nnzF + i)] = b;
      S.template put<T>(d.oR + 2 * int(sizeof(T)) * i, b);
    }
    R.run(0, s.luRounds, 0);
    S.lu(d.oLuHdr, d.oLu, d.oLu1, d.nLu);
    S.pivots(m);
    R.run(s.luRounds, s.backRounds, size_t(s.backBody));
    S.back();
    for (int i = 0; i < m; ++i)
      CHECK(same(R.A[size_t(s.nnzF + i)], S.template get<T>(d.oR + 2 * int(sizeof(T)) * i)), "%s: solution %d, iteration %d", what, i, it);
    if (s.transposed) {
      progress(R);  // the gradient reads them after the solve
      w.assign(size_t(t.nReac), 0.0);
      std::vector<double> mu(size_t(m), 0.0);
      for (int i = 0; i < m; ++i) S.template put<double>(d.oMu + 8 * i, mu[size_t(i)] = U(rng) - 0.5);
      S.sums(d.oNutHdr, d.oNut, d.nNut, d.oW, [&](uint32_t x) { return S.coef(x); });
      for (int a = 0; a < m; ++a)
        for (int e = t.omegaPtr[a]; e < t.omegaPtr[a + 1]; ++e)
          w[size_t(t.omegaReac[e])] = fmaT(t.omegaCoef[e], mu[size_t(a)], w[size_t(t.omegaReac[e])]);
      wKept();
      progress(R);
    }
  }
  std::printf("%s FP%zu: cell %d B%s\n", what, 8 * sizeof(T), d.cellBytes, fails == before ? "" : " FAILED");
}

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  const KineticModel km = loadKineticModel(argv[1], nullptr);
  const MechTables t = compileMechanism(km);
  const SS f = buildSparseSchedule(t, false, false), b = buildSparseSchedule(t, true, false);
  for (const SS* s : {&f, &b})
    for (int q = 0; q < s->nnzF; ++q) CHECK(s->slotOf[size_t(q)] == q, "position %d", q);
  repeat<float>(t, f, f, false, "forward");
  repeat<double>(t, f, f, false, "forward");
  repeat<double>(t, f, b, true, "adjoint forward");
  repeat<double>(t, b, f, true, "adjoint transposed");
  for (int i = 3; i < argc; ++i) {
    AerosolModel am = loadAerosolModel(argv[2], km);
    am.nParticles = std::atoi(argv[i]);
    const MechTables ta = aerosolTables(t, am, nullptr);
    const SS s = buildSparseSchedule(ta, false, false);
    check<double>(ta, s, s, false, "aerosol");
    repeat<double>(ta, s, s, false, "aerosol");
  }
  std::printf("%s (%d failures)\n", fails ? "FAILED" : "OK", fails);
  return fails ? 1 : 0;
}
