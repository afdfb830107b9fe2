// Host-side checker of the device encoding (tchem-atm_amd/csrc/lowered.cpp).
//
// Runs the encoded stream lane by lane the way the kernels do (every lane of
// a round reads before any lane writes, rounds in order) on a cell region
// filled with NaN, and the rounds it was lowered from (schedule.hpp) with
// the same operations on plain arrays.  Every rate of progress, derivative,
// segment sum, matrix entry, factor, pivot and solution must be the same bit
// for bit (zeros may differ in sign), in FP32 and FP64 entries, for the
// forward and the transposed programs; nothing outside the cell region or
// the stream may be touched.
//
// usage: lowered_check <mechanism.yaml> [<aerosol.yaml>]
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "aerosol_model.hpp"
#include "kinetic_model.hpp"
#include "lowered.hpp"
#include "mechanism.hpp"
#include "schedule.hpp"
using namespace tchem_amd;
using SS = SparseSchedule;

static int fails = 0;
#define CHECK(c, ...)               \
  do {                              \
    if (!(c)) {                     \
      if (++fails < 30) {           \
        std::printf("FAIL %s:%d ", __FILE__, __LINE__); \
        std::printf(__VA_ARGS__);   \
        std::printf("\n");          \
      }                             \
    }                               \
  } while (0)

template <typename T>
static T fmaT(T a, T b, T c) { return std::fma(a, b, c); }

template <typename X>
static bool same(X a, X b) { return std::memcmp(&a, &b, sizeof(X)) == 0 || (a == X(0) && b == X(0)); }

static double ipow(double x, int n) {
  double r = n >= 1 ? x : 1.0;
  for (int i = 1; i < n; ++i) r *= x;
  return r;
}

// ---- the rounds, on plain arrays ----------------------------------------------
template <typename T>
struct Rounds {
  const MechTables& t;
  const SS& s;
  std::vector<T> A, rd, dpr;
  std::vector<double> rop, seg;
  bool bad = false;
  Rounds(const MechTables& t_, const SS& s_)
      : t(t_), s(s_), A(size_t(s_.trashSlot) + 1, T(0)), rd(size_t(s_.m) + 2, T(0)), dpr(size_t(s_.pairSlots), T(0)),
        rop(size_t(t_.nReac) + 1, 0.0), seg(size_t(t_.nSeg()) + 1, 0.0) {}
  int spec(int r, int j) const { return j < t.maxReactants ? t.reacSpec[size_t(r) * t.maxReactants + j] : -1; }
  double factor(const std::vector<double>& c, int r, int j) const {
    return spec(r, j) < 0 ? 1.0 : ipow(c[size_t(spec(r, j))], t.reacPow[size_t(r) * t.maxReactants + j]);
  }
  void rates(const std::vector<double>& c, const std::vector<double>& kf) {
    for (int r = 0; r < t.nReac; ++r) rop[size_t(r)] = kf[size_t(r)] * factor(c, r, 0) * factor(c, r, 1) * factor(c, r, 2);
    for (int r = 0; r < t.nReac; ++r)
      for (int p = t.pairPtr[r]; p < t.pairPtr[r + 1]; ++p) {
        const int js = t.pairSlot[p], n = t.reacPow[size_t(r) * t.maxReactants + js];
        double d = kf[size_t(r)] * double(n) * ipow(c[size_t(spec(r, js))], n - 1);
        for (int j = 0; j < 3; ++j)
          if (j != js) d *= factor(c, r, j);
        dpr[size_t(p)] = T(d);
      }
  }
  void eval(double diag, double scale) {  // segment sums and the Jacobian
    size_t off = size_t(s.segBody);
    const int r0 = s.ropRounds + s.pairRounds;
    for (int r = r0; r < r0 + s.segRounds + s.jacRounds; ++r) {
      const int kind = int(s.evalHdr[size_t(r)] >> 16), len = int(s.evalHdr[size_t(r)] & 0xffff);
      for (int l = 0; l < 64; ++l) {
        const unsigned w = s.evalBody[off + size_t(l)];
        auto entry = [&](int j) { return s.evalBody[off + 64 * size_t(1 + j) + size_t(l)]; };
        if (kind == SS::kSeg) {
          const unsigned tg = w & ~SS::kCont;
          double acc = (w & SS::kCont) ? seg[tg] : 0.0;
          for (int j = 0; j < len; ++j) acc = fmaT(s.coefTable[entry(j) >> 16], rop[entry(j) & 0xffff], acc);
          seg[tg] = acc;
        } else {
          const unsigned tg = w & 0x3fffffffu;
          const T init = (w & SS::kCont) ? A[tg] : (((w >> 30) & 1u) ? T(diag) : T(0));
          T sum = T(0);
          for (int j = 0; j < len; ++j) sum = fmaT(T(s.coefTable[entry(j) >> 16]), dpr[entry(j) & 0xffff], sum);
          A[tg] = fmaT(T(scale), sum, init);
        }
      }
      off += 64 * size_t(1 + len);
    }
  }
  void run(int r0, int n, size_t off) {
    const int rhs0 = s.nnzF;
    for (int r = r0; r < r0 + n; ++r) {
      const int kind = int(s.progHdr[size_t(r)] >> 16), len = int(s.progHdr[size_t(r)] & 0xffff);
      std::vector<std::pair<size_t, T>> oA, oR;
      for (int l = 0; l < 64; ++l) {
        auto word = [&](int j) { return s.progBody[off + 64 * size_t(j) + size_t(l)]; };
        if (kind == SS::kMul) {
          const unsigned dst = word(0) & 0xffff, src = word(0) >> 16;
          const T p = A[src], inv = T(1) / p;
          if (dst & 0x8000) {
            oR.push_back({dst & 0x7fff, inv});
            bad |= !(p != T(0) && std::isfinite(p) && std::isfinite(inv));
          } else if (int(dst) != s.trashSlot) {
            oA.push_back({dst, A[dst] * inv});
          }
        } else if (kind == SS::kUpd || kind == SS::kBack) {
          T acc = A[word(0)];
          for (int j = 0; j < len; ++j) {
            const unsigned lo = word(1 + j) & 0xffff, hi = word(1 + j) >> 16;
            const T v = kind == SS::kUpd ? A[hi] : A[size_t(rhs0) + hi] * rd[hi];
            // a chain that has ended reads the zero slot (and, in kBack, the zero column)
            if (kind == SS::kBack && int(lo) >= s.nnzF) continue;
            acc = fmaT(-A[lo], v, acc);
          }
          if (int(word(0)) != s.trashSlot) oA.push_back({word(0), acc});
        } else {
          const unsigned w1 = word(1), w2 = word(2);
          const T p = A[w2 & 0x7fff], inv = T(1) / p, a = A[w1 & 0xffff];
          const T lv = a == T(0) ? T(0) : a * inv;
          T acc = A[word(0)];
          for (int j = 0; j < len - 2; ++j) acc = fmaT(-A[word(3 + j) & 0xffff], A[word(3 + j) >> 16], acc);
          const T val = (w2 & 0x8000u) ? lv : fmaT(-lv, A[w1 >> 16], acc);
          if (int(word(0)) != s.trashSlot) oA.push_back({word(0), val});
          if (int(w2 >> 16) != s.m + 1) {
            oR.push_back({w2 >> 16, inv});
            bad |= !(p != T(0) && std::isfinite(p) && std::isfinite(inv));
          }
        }
      }
      for (auto& x : oA) A[x.first] = x.second;
      for (auto& x : oR) rd[x.first] = x.second;
      off += 64 * size_t(kind == SS::kMul ? 1 : 1 + len);
    }
  }
};

// ---- the encoded stream ----------------------------------------------------------
template <typename T>
struct Stream {
  const LoweredProgram& P;
  const DevLowered& d;
  const MechTables& t;
  std::vector<unsigned char> lds;
  bool bad = false;
  std::vector<int> ropAt;  // slot of each reaction
  Stream(const LoweredProgram& p, const MechTables& t_) : P(p), d(p.d), t(t_), lds(size_t(p.d.cellBytes), 0xff) {}
  uint32_t word(int o) {
    CHECK(o >= 0 && o < d.words && o < int(P.words.size()), "stream word %d of %d", o, d.words);
    return o >= 0 && o < int(P.words.size()) ? P.words[size_t(o)] : 0;
  }
  int lo(uint32_t w) const { return int(w & 0xffff) << d.shift; }
  int hi(uint32_t w) const { return int(w >> 16) << d.shift; }
  template <typename X>
  X get(int a) {
    X v = X(0);
    CHECK(a >= 0 && a + int(sizeof(X)) <= int(lds.size()) && a % int(sizeof(X)) == 0, "read at %d", a);
    if (a >= 0 && a + int(sizeof(X)) <= int(lds.size())) std::memcpy(&v, &lds[size_t(a)], sizeof(X));
    return v;
  }
  template <typename X>
  void put(int a, X v) {
    CHECK(a >= 0 && a + int(sizeof(X)) <= int(lds.size()) && a % int(sizeof(X)) == 0, "write at %d", a);
    if (a >= 0 && a + int(sizeof(X)) <= int(lds.size())) std::memcpy(&lds[size_t(a)], &v, sizeof(X));
  }
  template <typename X>
  using Out = std::vector<std::pair<int, X>>;
  template <typename X>
  void flush(Out<X>& o) {
    for (auto& x : o) put<X>(x.first, x.second);
    o.clear();
  }
  bool bit(int oHdr, int r, int which) {
    const int o = oHdr + 4 * (r / 64) + 2 * which;
    const uint64_t m = uint64_t(word(o)) | (uint64_t(word(o + 1)) << 32);
    return (m >> (r % 64)) & 1;
  }
  double coef(uint32_t w) { return P.coef.at(size_t(hi(w) / 8)); }
  void init(const std::vector<double>& kf, int m) {
    put<T>(d.zeroA, T(0));
    put<T>(d.oR + 2 * int(sizeof(T)) * m, T(0));
    put<T>(d.oR + 2 * int(sizeof(T)) * m + int(sizeof(T)), T(0));
    put<double>(d.oneC, 1.0);
    put<double>(d.zero8, 0.0);
    ropAt.assign(size_t(t.nReac), -1);
    for (int i = 0; i < 64 * d.nRop; ++i) {
      const int r = int(word(d.oKf + i));
      CHECK(r < t.nReac && (r < 0 || ropAt[size_t(r)] < 0), "reaction %d in slot %d", r, i);
      if (r >= 0) ropAt[size_t(r)] = i;
      put<double>(d.oK + 8 * i, r >= 0 ? kf[size_t(r)] : 0.0);
    }
    for (int r = 0; r < t.nReac; ++r) CHECK(ropAt[size_t(r)] >= 0, "reaction %d has no slot", r);
    for (int i = 0; i < 64 * d.nKfx; ++i) {
      const uint32_t w0 = word(d.oKfx + 2 * i), w1 = word(d.oKfx + 2 * i + 1);
      put<double>(lo(w1), get<double>(d.oK + 8 * int(w0)) * double(w1 >> 16));
    }
  }
  void rates(const std::vector<double>& c) {
    for (size_t i = 0; i < c.size(); ++i) put<double>(d.oC + 8 * int(i), c[i]);
    for (int i = 0; i < 64 * d.nPow; ++i) {
      const uint32_t w = word(d.oPow + 2 * i);
      put<double>(hi(w), ipow(get<double>(lo(w)), int(word(d.oPow + 2 * i + 1))));
    }
    for (int i = 0; i < 64 * d.nRop; ++i) {
      const uint32_t w0 = word(d.oRop + 2 * i), w1 = word(d.oRop + 2 * i + 1);
      put<double>(d.oP + 8 * i,
                  get<double>(d.oK + 8 * i) * get<double>(lo(w0)) * get<double>(hi(w0)) * get<double>(lo(w1)));
    }
    for (int i = 0; i < 64 * d.nPair; ++i) {
      const uint32_t w0 = word(d.oPair + 2 * i), w1 = word(d.oPair + 2 * i + 1);
      put<T>(d.oD + int(sizeof(T)) * i,
             T(get<double>(lo(w0)) * get<double>(hi(w0)) * get<double>(lo(w1)) * get<double>(hi(w1))));
    }
  }
  template <class Y>
  void sums(int oHdr, int o, int n, int out, Y y) {
    std::vector<double> acc(64);
    for (int r = 0; r < n; ++r) {
      if (bit(oHdr, r, 0)) std::fill(acc.begin(), acc.end(), 0.0);
      for (int l = 0; l < 64; ++l)
        for (int j = 0; j < 4; ++j) {
          const uint32_t w = word(o + 4 * (64 * r + l) + j);
          acc[size_t(l)] = fmaT(y(w), get<double>(lo(w)), acc[size_t(l)]);
        }
      if (bit(oHdr, r, 1)) {
        for (int l = 0; l < 64; ++l) put<double>(out + 8 * l, acc[size_t(l)]);
        out += 512;
      }
    }
  }
  void segments() { sums(d.oSegHdr, d.oSeg, d.nSeg, d.oS, [&](uint32_t w) { return coef(w); }); }
  double row(int a, double s) {
    const int q = a / 64, l = a % 64;
    int o = d.oRow;
    for (int k = 0; k < q; ++k) o += 128 * d.nRow[k];
    for (int r = 0; r < d.nRow[q]; ++r)
      for (int j = 0; j < 2; ++j) {
        const uint32_t w = word(o + 2 * (64 * r + l) + j);
        s = s + get<double>(lo(w));
        s = s + get<double>(hi(w));
      }
    return s;
  }
  void jacobian(T scale) {
    int r = 0;
    auto cf = [&](int k) {  // coefficient k of the section
      T v;
      uint32_t w[2] = {word(d.oJacC + int(sizeof(T)) / 4 * k), sizeof(T) == 8 ? word(d.oJacC + 2 * k + 1) : 0u};
      std::memcpy(&v, w, sizeof(T));
      return v;
    };
    for (; r < d.nJ4 + d.nJ2 + d.nJ1; ++r) {
      Out<T> out;
      for (int l = 0; l < 64; ++l) {
        const int o = d.oJac + 4 * (64 * r + l);
        const uint32_t x = word(o), y = word(o + 1), z = word(o + 2), w = word(o + 3);
        T c[4], p[4];
        for (int k = 0; k < 4; ++k) c[k] = cf(4 * (64 * r + l) + k);
        p[0] = get<T>(lo(x)), p[1] = get<T>(hi(x)), p[2] = get<T>(lo(y)), p[3] = get<T>(hi(y));
        if (r < d.nJ4) {
          T s = c[0] * p[0];
          for (int k = 1; k < 4; ++k) s = fmaT(c[k], p[k], s);
          out.push_back({lo(z), (w & 2) ? s : fmaT(scale, s, (w & 1) ? T(1) : T(0))});
        } else if (r < d.nJ4 + d.nJ2) {
          out.push_back({lo(z), scale * fmaT(c[1], p[1], c[0] * p[0])});
          out.push_back({hi(z), scale * fmaT(c[3], p[3], c[2] * p[2])});
        } else {
          out.push_back({lo(z), scale * (c[0] * p[0])});
          out.push_back({hi(z), scale * (c[1] * p[1])});
          out.push_back({lo(w), scale * (c[2] * p[2])});
          out.push_back({hi(w), scale * (c[3] * p[3])});
        }
      }
      flush<T>(out);
    }
    for (r = 0; r < d.nJx; ++r) {
      const int most = int(word(d.oJx + 128 * r + 1) & 0x7fffffffu);  // lane 0 has the longest
      Out<T> out;
      for (int l = 0; l < 64; ++l) {
        const uint32_t x = word(d.oJx + 2 * (64 * r + l)), y = word(d.oJx + 2 * (64 * r + l) + 1);
        const int n = int(y & 0x7fffffffu);
        CHECK(n <= most, "join count %d above the round's %d", n, most);
        T acc = (y >> 31) ? T(1) : T(0);
        for (int j = 0; j < n; ++j) acc = fmaT(scale, get<T>(hi(x) + int(sizeof(T)) * j), acc);
        out.push_back({lo(x), acc});
      }
      flush<T>(out);
    }
  }
  void lu(int oHdr, int o4, int o1, int n) {
    for (int r = 0; r < n; ++r) {
      Out<T> out;
      for (int l = 0; l < 64; ++l) {
        uint32_t w[5];
        for (int j = 0; j < 4; ++j) w[j] = word(o4 + 4 * (64 * r + l) + j);
        w[4] = word(o1 + 64 * r + l);
        int f[10];
        for (int j = 0; j < 5; ++j) f[2 * j] = lo(w[j]), f[2 * j + 1] = hi(w[j]);
        if (bit(oHdr, r, 0)) {
          out.push_back({f[0], get<T>(f[0]) * (T(1) / get<T>(f[1]))});
        } else if (bit(oHdr, r, 1)) {
          T acc = get<T>(f[0]);
          for (int j = 0; j < 4; ++j) acc = fmaT(-get<T>(f[1 + 2 * j]), get<T>(f[2 + 2 * j]), acc);
          out.push_back({f[0], acc});
        } else {
          const T p = get<T>(f[3]), a = get<T>(f[1]), b = get<T>(f[2]), inv = T(1) / p;
          const T lv = a == T(0) ? T(0) : a * inv;
          T acc = get<T>(f[0]);
          for (int j = 0; j < 2; ++j) acc = fmaT(-get<T>(f[4 + 2 * j]), get<T>(f[5 + 2 * j]), acc);
          out.push_back({f[0], f[1] == f[0] ? lv : fmaT(-lv, b, acc)});
        }
      }
      flush<T>(out);
    }
  }
  void pivots(int m) {
    for (int i = 0; i < m; ++i) {
      const T p = get<T>(int(word(d.oDiag + i))), inv = T(1) / p;
      put<T>(d.oR + 2 * int(sizeof(T)) * i + int(sizeof(T)), inv);
      bad |= !(p != T(0) && std::isfinite(p) && std::isfinite(inv));
    }
  }
  void back() {
    for (int r = 0; r < d.nBack; ++r)
      for (int k = 0; k < 2; ++k) {
        Out<T> out;
        for (int l = 0; l < 64; ++l) {
          const uint32_t x = word(d.oBack + 4 * (64 * r + l) + 2 * k), y = word(d.oBack + 4 * (64 * r + l) + 2 * k + 1);
          const T b = get<T>(lo(y)), ri = get<T>(lo(y) + int(sizeof(T)));
          out.push_back({lo(x), fmaT(-get<T>(hi(x)), b * ri, get<T>(lo(x)))});
        }
        flush<T>(out);
      }
  }
};

template <typename T>
static void check(const MechTables& t, const SS& s, const SS& partner, bool adjoint, const char* what) {
  // adjoint programs share the slots of the forward one
  const LoweredSlots fs = chooseSlots(t, s.transposed ? partner : s);
  const LoweredProgram P = lowerProgram(t, s, int(sizeof(T)), adjoint, s.transposed ? chooseSlots(t, s, &fs) : fs);
  const DevLowered& d = P.d;
  std::printf("%s FP%zu: cell %d B, stream %d words, shift %d, rounds rop %d pair %d seg %d row %d jac %d+%d+%d join %d lu %d back %d fwd %d\n",
              what, 8 * sizeof(T), d.cellBytes, d.words, d.shift, d.nRop, d.nPair, d.nSeg, d.nRow[0] + d.nRow[1], d.nJ4, d.nJ2,
              d.nJ1, d.nJx, d.nLu, d.nBack, d.nFwd);
  CHECK(d.words == int(P.words.size()) && d.nCoef == int(P.coef.size()) && d.cellBytes % 16 == 0, "sizes");
  if (adjoint) {  // forward and transposed programs run on one cell layout
    const LoweredProgram Q = lowerProgram(t, partner, int(sizeof(T)), true, partner.transposed ? chooseSlots(t, partner, &fs) : fs);
    const DevLowered& e = Q.d;
    for (int i = 0; i < 64 * d.nRop; ++i)
      CHECK(P.words[size_t(d.oKf + i)] == Q.words[size_t(e.oKf + i)], "slot %d holds another reaction", i);
    CHECK(d.zeroA == e.zeroA && d.oR == e.oR && d.oD == e.oD && d.oC == e.oC && d.oneC == e.oneC && d.oK == e.oK && d.nK == e.nK &&
              d.zero8 == e.zero8 && d.oP == e.oP && d.oS == e.oS && d.oMu == e.oMu && d.oW == e.oW && d.oV == e.oV && d.shift == e.shift,
          "cell layouts of the forward and transposed programs differ");
  }
  const int m = s.m;
  std::mt19937_64 rng(11);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  for (int trial = 0; trial < 3; ++trial) {
    std::vector<double> c(size_t(t.nSpec), 0.0), kf(size_t(t.nReac), 0.0);
    for (auto& x : c) x = std::pow(10.0, -4 + 4 * U(rng));
    for (auto& x : kf) x = std::pow(10.0, -3 + 4 * U(rng));
    const double ch = std::pow(10.0, trial - 2);
    Rounds<T> R(t, s);
    Stream<T> S(P, t);
    S.init(kf, m);
    S.rates(c);
    R.rates(c, kf);
    for (int r = 0; r < t.nReac; ++r) CHECK(same(R.rop[size_t(r)], S.template get<double>(d.oP + 8 * S.ropAt[size_t(r)])), "rate of progress %d", r);
    {  // derivative pairs, in some order of slots (the matrix entries below tell which)
      std::vector<T> x(R.dpr.begin(), R.dpr.begin() + t.nPairs()), y;
      for (int p = 0; p < 64 * d.nPair; ++p) y.push_back(S.template get<T>(d.oD + int(sizeof(T)) * p));
      x.resize(y.size(), T(0));
      std::sort(x.begin(), x.end());
      std::sort(y.begin(), y.end());
      CHECK(x == y, "derivative pairs");
    }
    R.eval(1.0, -ch);
    S.segments();
    const int rows = int(t.rowSegPtr.size()) - 1;
    for (int a = 0; a < rows; ++a) {
      double f = t.emission[size_t(a)];
      for (int g = t.rowSegPtr[a]; g < t.rowSegPtr[a + 1]; ++g) f += R.seg[size_t(g)];
      CHECK(same(f, S.row(a, t.emission[size_t(a)])), "source term of species %d", a);
    }
    S.jacobian(T(-ch));
    for (int p = 0; p < s.nnzF; ++p) CHECK(same(R.A[size_t(p)], S.template get<T>(int(sizeof(T)) * P.slot[size_t(p)])), "matrix slot %d", p);
    for (int pass = 0; pass < 2; ++pass) {  // factorise and solve, then solve again with the stored factors
      for (int i = 0; i < m; ++i) {
        const T b = T(U(rng) - 0.5);
        R.A[size_t(s.nnzF + i)] = b;
        S.template put<T>(d.oR + 2 * int(sizeof(T)) * i, b);
      }
      if (pass == 0) {
        R.run(0, s.luRounds, 0);
        S.lu(d.oLuHdr, d.oLu, d.oLu1, d.nLu);
        S.pivots(m);
      } else {
        R.run(s.luRounds + s.backRounds, s.fwdRounds, size_t(s.fwdBody));
        S.lu(d.oFwdHdr, d.oFwd, d.oFwd1, d.nFwd);
      }
      CHECK(R.bad == S.bad && !R.bad, "pivots");
      for (int p = 0; p < s.nnzF; ++p) CHECK(same(R.A[size_t(p)], S.template get<T>(int(sizeof(T)) * P.slot[size_t(p)])), "factor slot %d", p);
      R.run(s.luRounds, s.backRounds, size_t(s.backBody));
      S.back();
      for (int i = 0; i < m; ++i) {
        const int a = d.oR + 2 * int(sizeof(T)) * i;
        CHECK(same(R.A[size_t(s.nnzF + i)], S.template get<T>(a)) && same(R.rd[size_t(i)], S.template get<T>(a + int(sizeof(T)))),
              "solution %d pass %d", i, pass);
      }
    }
    if (adjoint && s.transposed) {
      std::vector<double> mu(size_t(m) + 1, 0.0), w(size_t(t.nReac), 0.0), v(size_t(m), 0.0);
      for (int i = 0; i < m; ++i) mu[size_t(i)] = U(rng) - 0.5;
      for (int i = 0; i <= m; ++i) S.template put<double>(d.oMu + 8 * i, mu[size_t(i)]);
      S.sums(d.oNutHdr, d.oNut, d.nNut, d.oW, [&](uint32_t x) { return S.coef(x); });
      S.sums(d.oJtvHdr, d.oJtv, d.nJtv, d.oV, [&](uint32_t x) { return S.template get<double>(S.hi(x)); });
      for (int a = 0; a < m; ++a)
        for (int e = t.omegaPtr[a]; e < t.omegaPtr[a + 1]; ++e)
          w[size_t(t.omegaReac[e])] = fmaT(t.omegaCoef[e], mu[size_t(a)], w[size_t(t.omegaReac[e])]);
      for (int r = 0; r < t.nReac; ++r)
        for (int p = t.pairPtr[r]; p < t.pairPtr[r + 1]; ++p) {
          double& x = v[size_t(R.spec(r, t.pairSlot[p]))];
          x = fmaT(double(R.dpr[size_t(p)]), w[size_t(r)], x);
        }
      for (int r = 0; r < t.nReac; ++r) CHECK(same(w[size_t(r)], S.template get<double>(int(S.word(d.oWmap + S.ropAt[size_t(r)])))), "w %d", r);
      for (int i = 0; i < m; ++i) CHECK(same(v[size_t(i)], S.template get<double>(int(S.word(d.oVmap + i)))), "v %d", i);
    }
  }
}

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  KineticModel km = loadKineticModel(argv[1], nullptr);
  const MechTables t = compileMechanism(km);
  const SS f = buildSparseSchedule(t), b = buildSparseSchedule(t, true);
  check<float>(t, f, f, false, "forward");
  check<double>(t, f, f, false, "forward");
  check<double>(t, f, b, true, "adjoint forward");
  check<double>(t, b, f, true, "adjoint transposed");
  if (argc > 2) {
    AerosolModel am = loadAerosolModel(argv[2], km);
    for (int particles : {1, 3}) {
      am.nParticles = particles;
      const MechTables ta = aerosolTables(t, am, nullptr);
      const SS s = buildSparseSchedule(ta, false);
      check<double>(ta, s, s, false, "aerosol");
    }
  }
  std::printf("%s (%d failures)\n", fails ? "FAILED" : "OK", fails);
  return fails ? 1 : 0;
}
