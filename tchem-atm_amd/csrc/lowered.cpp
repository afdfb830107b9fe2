// Lowering of the compiled programs to the device encoding (lowered.hpp).
#include "lowered.hpp"

#include <algorithm>
#include <array>
#include <cstring>
#include <map>
#include <numeric>
#include <random>
#include <set>
#include <stdexcept>

namespace tchem_amd {

namespace {

constexpr int kLanes = 64;

int al16(int x) { return (x + 15) & ~15; }
int ceilDiv(int a, int b) { return (a + b - 1) / b; }

// LDS reads of one instruction: the distinct entries 32 lanes (half a
// wavefront) read together.  Entries whose slots are equal modulo 32 conflict
// (32 banks for 4-byte reads, 32 pairs of 64 for 8-byte reads; reads of one
// address do not; stores take the time of two passes anyway).
using Gather = std::vector<int>;

// Slots of n entries such that the gathers take few passes: swaps of two
// entries' slots are kept when they do not add passes.  slot[] holds the
// starting assignment (a permutation); entries >= n of a gather are slots
// that do not move.  Deterministic; at most `tries` swaps.
void spreadOverBanks(std::vector<int>& slot, const std::vector<Gather>& gathers, long tries) {
  constexpr int kBanks = 32;
  const int n = int(slot.size());
  std::vector<std::array<unsigned char, kBanks>> cnt(gathers.size());
  std::vector<std::vector<int>> in(static_cast<size_t>(n));
  for (size_t g = 0; g < gathers.size(); ++g) {
    cnt[g].fill(0);
    for (int e : gathers[g]) {
      ++cnt[g][size_t((e < n ? slot[size_t(e)] : e) % kBanks)];
      if (e < n) in[size_t(e)].push_back(int(g));
    }
  }
  auto passes = [](const std::array<unsigned char, kBanks>& c) { return int(*std::max_element(c.begin(), c.end())); };
  std::mt19937_64 rng(0x5eedULL);
  std::vector<int> mark(gathers.size(), 0);
  int stamp = 0;
  for (long it = 0; it < tries && n > 1; ++it) {
    const size_t a = size_t(rng() % unsigned(n)), b = size_t(rng() % unsigned(n));
    const size_t ra = size_t(slot[a] % kBanks), rb = size_t(slot[b] % kBanks);
    if (ra == rb || (in[a].empty() && in[b].empty())) continue;
    ++stamp;
    for (int g : in[b]) mark[size_t(g)] = stamp;
    int delta = 0;
    auto move = [&](int g, size_t from, size_t to) {
      auto& c = cnt[size_t(g)];
      const int before = passes(c);
      --c[from];
      ++c[to];
      return passes(c) - before;
    };
    std::vector<int> onlyA, onlyB;  // gathers that hold both keep their counts
    for (int g : in[a]) {
      if (mark[size_t(g)] == stamp) mark[size_t(g)] = -stamp;
      else onlyA.push_back(g);
    }
    for (int g : in[b])
      if (mark[size_t(g)] == stamp) onlyB.push_back(g);
    for (int g : onlyA) delta += move(g, ra, rb);
    for (int g : onlyB) delta += move(g, rb, ra);
    if (delta <= 0) {
      std::swap(slot[a], slot[b]);
    } else {
      for (int g : onlyA) move(g, rb, ra);
      for (int g : onlyB) move(g, ra, rb);
    }
  }
}
// the gathers of 64 lanes' entries, half a wavefront each (repeats dropped)
void addGathers(std::vector<Gather>& out, const std::vector<int>& lanes) {
  for (size_t h = 0; h < lanes.size(); h += 32) {
    Gather g(lanes.begin() + long(h), lanes.begin() + long(std::min(lanes.size(), h + 32)));
    std::sort(g.begin(), g.end());
    g.erase(std::unique(g.begin(), g.end()), g.end());
    if (g.size() > 1) out.push_back(std::move(g));
  }
}

// ---- Jacobian chains cut into the records' chunks --------------------------
struct Chunk {
  int target = 0;  // factor position of the rounds' numbering, or -1 - partial slot
  unsigned flags = 0;
  std::vector<std::pair<int, double>> e;  // (pair, coefficient)
};
struct Join {
  int target = 0, first = 0, count = 0;
  bool diag = false;
};
struct Chunks {
  std::vector<Chunk> j4, j2, j1;
  std::vector<Join> joins;
  int nPartial = 0;
};
Chunks jacobianChunks(const MechTables& t, const SparseSchedule& s) {
  Chunks k;
  std::map<std::pair<int, int>, int> at;
  for (int n = 0; n < t.nnzJ(); ++n)
    at[s.transposed ? std::make_pair(t.jnzCol[n], t.jnzRow[n]) : std::make_pair(t.jnzRow[n], t.jnzCol[n])] = n;
  constexpr size_t kC = SparseSchedule::kMaxChain;
  for (int i = 0; i < s.m; ++i)
    for (int q = s.rowPtr[i]; q < s.rowPtr[i + 1]; ++q) {
      const int j = s.colIdx[size_t(q)];
      Chunk c;
      c.target = s.slotOf[size_t(q)];
      const bool diag = i == j;
      const auto it = at.find({i, j});
      if (it != at.end())
        for (int e = t.jnzPtr[it->second]; e < t.jnzPtr[it->second + 1]; ++e) c.e.push_back({t.jcPair[e], t.jcCoef[e]});
      if (!diag && c.e.size() <= 1) {
        k.j1.push_back(c);
      } else if (!diag && c.e.size() == 2) {
        k.j2.push_back(c);
      } else if (c.e.size() <= kC) {
        c.flags = diag ? 1u : 0u;
        k.j4.push_back(c);
      } else {
        Join x;
        x.target = c.target;
        x.first = k.nPartial;
        x.diag = diag;
        for (size_t b = 0; b < c.e.size(); b += kC) {
          Chunk part;
          part.target = -1 - k.nPartial++;
          part.flags = 2u;
          part.e.assign(c.e.begin() + long(b), c.e.begin() + long(std::min(c.e.size(), b + kC)));
          k.j4.push_back(part);
          ++x.count;
        }
        k.joins.push_back(x);
      }
    }
  std::stable_sort(k.joins.begin(), k.joins.end(), [](const Join& a, const Join& b) { return a.count > b.count; });
  return k;
}

// segments by descending length: the order the SUM section takes them in
std::vector<int> segmentOrder(const MechTables& t) {
  std::vector<int> o(size_t(t.nSeg()));
  std::iota(o.begin(), o.end(), 0);
  std::stable_sort(o.begin(), o.end(), [&](int a, int b) { return t.segEnd[a] - t.segBegin[a] > t.segEnd[b] - t.segBegin[b]; });
  return o;
}

// ---- slots: gathers of every round spread over the LDS banks ----------------
std::vector<int> factorSlots(const SparseSchedule& s) {
  using SS = SparseSchedule;
  std::vector<int> slot(size_t(s.nnzF));
  std::iota(slot.begin(), slot.end(), 0);
  std::vector<Gather> gs;
  // right-hand sides sit after the factor, two units apart; the zero slot
  // is nnzF; the trash slot is only read by idle lanes
  const int rhs0 = (s.nnzF + 2 + 3) & ~3;
  auto at = [&](unsigned ix) {
    const int i = int(ix);
    if (i < s.nnzF) return i;
    return i < s.nnzF + s.m ? rhs0 + 2 * (i - s.nnzF) : s.nnzF;
  };
  size_t b = 0;
  for (int r = 0; r < s.luRounds + s.backRounds; ++r) {
    const int kind = int(s.progHdr[size_t(r)] >> 16), len = int(s.progHdr[size_t(r)] & 0xffff);
    const int words = kind == SS::kMul ? 1 : 1 + len;
    auto gather = [&](int j, int shift, unsigned mask) {
      std::vector<int> lanes;
      for (int l = 0; l < kLanes; ++l)
        lanes.push_back(at((s.progBody[b + size_t(kLanes) * size_t(j) + size_t(l)] >> shift) & mask));
      addGathers(gs, lanes);
    };
    if (kind == SS::kMul) {
      gather(0, 16, 0xffffu);
    } else if (kind == SS::kUpd) {
      gather(0, 0, 0xffffu);
      for (int j = 1; j <= len; ++j) gather(j, 0, 0xffffu), gather(j, 16, 0xffffu);
    } else if (kind == SS::kMulUpd) {
      gather(0, 0, 0xffffu);
      gather(1, 0, 0xffffu), gather(1, 16, 0xffffu);
      gather(2, 0, 0x7fffu);
      for (int j = 3; j <= len; ++j) gather(j, 0, 0xffffu), gather(j, 16, 0xffffu);
    } else {
      for (int j = 1; j <= len; ++j) gather(j, 0, 0xffffu);
    }
    b += size_t(kLanes) * size_t(words);
  }
  // CB05: 370 extra passes in order, 122 after 140 tries per entry, 110 after 300, 102 after 600
  spreadOverBanks(slot, gs, std::min<long>(300L * s.nnzF, 400000L));
  return slot;
}
// Live items keep to the first slots, so that the last slots of a section's
// rounds belong to idle lanes and need no room of their own (layout).
std::vector<int> withIdleLanes(std::vector<int> slot, int rounds) {
  for (int i = int(slot.size()); i < kLanes * rounds; ++i) slot.push_back(i);
  return slot;
}
std::vector<int> pairSlots(const SparseSchedule& s, const Chunks& chunks, int nPairs) {
  std::vector<int> pairSlot(static_cast<size_t>(nPairs));
  std::iota(pairSlot.begin(), pairSlot.end(), 0);
  std::vector<Gather> gs;
  auto gather = [&](const std::vector<Chunk>& v, size_t per, size_t k, size_t e) {
    for (size_t r = 0; r * per * kLanes < v.size(); ++r) {
      std::vector<int> lanes;
      for (size_t l = 0; l < size_t(kLanes); ++l) {
        const size_t i = (per * r + k) * kLanes + l;
        lanes.push_back(i < v.size() && e < v[i].e.size() ? v[i].e[e].first : 1 << 20);
      }
      addGathers(gs, lanes);
    }
  };
  for (size_t e = 0; e < 4; ++e) gather(chunks.j4, 1, 0, e);
  for (size_t k = 0; k < 2; ++k)
    for (size_t e = 0; e < 2; ++e) gather(chunks.j2, 2, k, e);
  for (size_t k = 0; k < 4; ++k) gather(chunks.j1, 4, k, 0);
  spreadOverBanks(pairSlot, gs, std::min<long>(120L * long(pairSlot.size()), 60000L));
  return withIdleLanes(std::move(pairSlot), s.pairRounds);
}
// rates of progress and rate constants share their slots
std::vector<int> reactionSlots(const MechTables& t, const SparseSchedule& s, const std::vector<int>& pairSlot) {
  const std::vector<int> segOrder = segmentOrder(t);
  std::vector<int> ropSlot(static_cast<size_t>(t.nReac));
  std::iota(ropSlot.begin(), ropSlot.end(), 0);
  std::vector<Gather> gs;
  for (size_t g = 0; g < segOrder.size(); g += kLanes) {
    const int first = segOrder[g], most = t.segEnd[first] - t.segBegin[first];
    for (int e = 0; e < most; ++e) {
      std::vector<int> lanes;
      for (size_t l = g; l < std::min(segOrder.size(), g + kLanes); ++l) {
        const int at = t.segBegin[segOrder[l]] + e;
        lanes.push_back(at < t.segEnd[segOrder[l]] ? t.omegaReac[at] : 1 << 20);
      }
      addGathers(gs, lanes);
    }
  }
  std::vector<int> reacOf(pairSlot.size(), 1 << 20);
  for (int r = 0; r < t.nReac; ++r)
    for (int p = t.pairPtr[r]; p < t.pairPtr[r + 1]; ++p) reacOf[size_t(pairSlot[size_t(p)])] = r;
  for (size_t i = 0; i < reacOf.size(); i += kLanes)
    addGathers(gs, std::vector<int>(reacOf.begin() + long(i), reacOf.begin() + long(i + kLanes)));
  spreadOverBanks(ropSlot, gs, std::min<long>(200L * long(ropSlot.size()), 60000L));
  return withIdleLanes(std::move(ropSlot), s.ropRounds);
}

struct Lowering {
  const MechTables& t;
  const SparseSchedule& s;
  const int T;
  const bool adjoint;
  const LoweredSlots& slots;
  LoweredProgram out;
  DevLowered& d;
  std::vector<uint32_t>& W;

  Lowering(const MechTables& t_, const SparseSchedule& s_, int bytesT, bool adj, const LoweredSlots& sl)
      : t(t_), s(s_), T(bytesT), adjoint(adj), slots(sl), d(out.d), W(out.words), ropSlot(sl.rop), pairSlot(sl.pair) {}

  int readAhead = 0;  // words a section's loop may read past its end

  unsigned field(int byteOffset) const {
    const int f = byteOffset >> d.shift;
    if (f < 0 || f > 0xffff || (f << d.shift) != byteOffset)
      throw std::runtime_error("lowered programs: address field out of range");
    return unsigned(f);
  }
  static uint32_t pack(unsigned lo, unsigned hi) { return lo | (hi << 16); }
  int begin() {  // sections start 16-byte aligned
    while (W.size() % 4) W.push_back(0);
    return int(W.size());
  }
  // end of a section read by loops that run `ahead` records past it
  void end(int recordWords, int ahead = 2) { readAhead = std::max(readAhead, int(W.size()) + ahead * recordWords); }

  // ---- addresses of the cell region
  int slotA(int p) const { return T * out.slot[size_t(p)]; }  // slot of the rounds' numbering
  int rhs(int i) const { return d.oR + 2 * T * i; }
  // an index of the rounds' matrix array: factor slot, RHS, zero, trash
  unsigned matrix(unsigned ix) const {
    const int i = int(ix);
    if (i < s.nnzF) return field(slotA(i));
    if (i < s.nnzF + s.m) return field(rhs(i - s.nnzF));
    if (i == s.zeroSlot) return field(d.zeroA);
    if (i == s.trashSlot) return field(d.trashA);
    throw std::runtime_error("lowered programs: matrix index out of range");
  }

  const std::vector<int>&ropSlot, &pairSlot;  // of LoweredSlots
  std::vector<std::pair<int, int>> powers;  // (species, exponent >= 2) with a slot of their own
  std::vector<std::pair<int, int>> scaled;  // (reaction, factor >= 2) with a kf slot of their own
  int oPowers = 0, oScaled = 0;             // byte offsets of those slots
  int powerSlot(int sp, int n) {
    if (n <= 0) return d.oneC;
    if (n == 1) return d.oC + 8 * sp;
    const auto it = std::find(powers.begin(), powers.end(), std::make_pair(sp, n));
    return oPowers + 8 * int(it - powers.begin());
  }
  int kfSlot(int r, int n) {
    if (n == 0) return d.zero8;
    if (n == 1) return d.oK + 8 * ropSlot[size_t(r)];
    const auto it = std::find(scaled.begin(), scaled.end(), std::make_pair(r, n));
    return oScaled + 8 * int(it - scaled.begin());
  }
  int spec(int r, int j) const { return j < t.maxReactants ? t.reacSpec[size_t(r) * t.maxReactants + j] : -1; }
  int power(int r, int j) const { return j < t.maxReactants ? t.reacPow[size_t(r) * t.maxReactants + j] : 0; }
  int factorSlot(int r, int j) { return spec(r, j) < 0 ? d.oneC : powerSlot(spec(r, j), power(r, j)); }

  void collect() {
    auto addPower = [&](int sp, int n) {
      if (n >= 2 && std::find(powers.begin(), powers.end(), std::make_pair(sp, n)) == powers.end())
        powers.push_back({sp, n});
    };
    for (int r = 0; r < t.nReac; ++r)
      for (int j = 0; j < t.maxReactants && spec(r, j) >= 0; ++j) addPower(spec(r, j), power(r, j));
    for (int r = 0; r < t.nReac; ++r)
      for (int p = t.pairPtr[r]; p < t.pairPtr[r + 1]; ++p) {
        const int js = t.pairSlot[p], n = power(r, js);
        addPower(spec(r, js), n - 1);
        if (n >= 2) {
          if (std::find(scaled.begin(), scaled.end(), std::make_pair(r, n)) == scaled.end()) scaled.push_back({r, n});
        }
      }
  }

  std::vector<Chunk> j4, j2, j1;
  std::vector<Join> joins;
  int nPartial = 0;

  // Regions share room where one is dead while the other lives: powers and
  // partial sums lie with the segment sums (and, in the adjoint, all of them
  // with w and v).  The slots that the last round of a section writes for its
  // idle lanes fall on the region behind, where that is dead then; the order
  // of a Newton iteration is powers, rates of progress (P), derivative pairs
  // (D), segment sums (S), species rows, Jacobian.  Only the last region pays
  // for its idle lanes, and of the orders S P D, D S P and P D S the smallest
  // is taken, so that as many cells fit a workgroup as there are items for.
  void layout() {
    const int m = s.m;
    const int idleK = 8 * (kLanes * s.ropRounds - t.nReac), idleP = idleK;
    const int idleD = T * (kLanes * s.pairRounds - t.nPairs()), idleS = 8 * (kLanes * ceilDiv(t.nSeg(), kLanes) - t.nSeg());
    const int sizeP = 8 * t.nReac, sizeD = T * t.nPairs(), sizePS = T * nPartial, sizePow = 8 * int(powers.size());
    auto al8 = [](int x) { return (x + 7) & ~7; };
    int o = 0;
    d.zeroA = T * s.nnzF;
    d.trashA = T * (s.nnzF + 1);
    o = al16(T * (s.nnzF + 2));
    d.oR = o;
    o = al16(o + 2 * T * (m + 2));
    d.oC = o;
    d.oneC = o + 8 * t.nSpec;
    d.trashC = d.oneC + 8;
    o = d.trashC + 8;
    if (adjoint) {
      d.oMu = o;
      o += 8 * (m + 1);
    }
    oScaled = o;
    d.zero8 = oScaled + 8 * int(scaled.size());
    d.oK = d.zero8 + 8;
    d.nK = t.nReac + int(scaled.size()) + 1;
    o = d.oK + 8 * t.nReac;  // idle lanes of K: on anything behind, loaded before all of it
    int end = 0;
    if (adjoint) {
      // w v P D: w outlives powers and pairs (gradient), P outlives the
      // Jacobian.  Idle lanes of w fall on v, which has room for its own.
      d.oS = d.oPS = d.oW = o;
      d.oV = oPowers = o + 8 * t.nReac;
      d.oP = std::max({o + 8 * t.nSeg(), o + 8 * t.nSeg() + idleS - sizeP, o + sizePS, oPowers + sizePow,
                       o + 8 * kLanes * ceilDiv(t.nReac, kLanes), d.oV + 8 * kLanes * std::max(1, ceilDiv(m, kLanes))});
      d.oD = d.oP + sizeP;
      end = std::max(d.oD + sizeD + idleD, d.oD + idleP);
    } else {
      // S with powers and partial sums, extra: bytes of the neighbour that
      // partial sums and idle lanes may use too
      auto sizeS = [&](int extra, int atLeast) {
        return al8(std::max({8 * t.nSeg(), sizePow, sizePS - extra, 8 * t.nSeg() + idleS - extra, atLeast}));
      };
      const int spdS = sizeS(sizeP, 0), spd = spdS + sizeP + std::max(sizeD + idleD, idleP);
      const int dspS = sizeS(sizeP, idleD), dsp = al8(sizeD) + dspS + sizeP + idleP;
      const int pdsD = std::max(al8(sizeD), idleP), pdsS = sizeS(0, std::max(idleD, 8 * t.nSeg() + idleS)), pds = sizeP + pdsD + pdsS;
      if (spd <= dsp && spd <= pds) {
        d.oS = o, d.oP = o + spdS, d.oD = d.oP + sizeP, end = o + spd;
      } else if (dsp <= pds) {
        d.oD = o, d.oS = o + al8(sizeD), d.oP = d.oS + dspS, end = o + dsp;
      } else {
        d.oP = o, d.oD = o + sizeP, d.oS = d.oD + pdsD, end = o + pds;
      }
      d.oPS = oPowers = d.oS;
    }
    d.cellBytes = al16(std::max({end, d.oS + 8 * t.nSeg() + idleS, o + idleK}));
    // the fields address the cell region and the coefficient table
    const std::set<double> coefs(t.omegaCoef.begin(), t.omegaCoef.end());
    d.shift = (m > 128 || std::max(size_t(d.cellBytes), 8 * (coefs.size() + 1)) > (1 << 16)) ? (T == 8 ? 3 : 2) : 0;
  }

  void masks(const std::vector<unsigned char>& bits) {  // bit 0 -> first mask, bit 1 -> second
    for (size_t b = 0; b < bits.size(); b += kLanes) {
      uint64_t m0 = 0, m1 = 0;
      for (size_t r = b; r < std::min(bits.size(), b + kLanes); ++r) {
        if (bits[r] & 1) m0 |= uint64_t(1) << (r - b);
        if (bits[r] & 2) m1 |= uint64_t(1) << (r - b);
      }
      for (uint64_t x : {m0, m1}) {
        W.push_back(uint32_t(x));
        W.push_back(uint32_t(x >> 32));
      }
    }
  }

  // SUM section; returns the slot of every chain
  std::vector<int> sums(const std::vector<std::vector<uint32_t>>& chains, uint32_t pad, int* oHdr, int* oBody, int* n) {
    std::vector<int> order(chains.size()), slot(chains.size());
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return chains[a].size() > chains[b].size(); });
    std::vector<unsigned char> bits;
    std::vector<uint32_t> body;
    for (size_t g = 0; g < order.size(); g += kLanes) {
      const int rounds = std::max(1, ceilDiv(int(chains[order[g]].size()), 4));
      for (int r = 0; r < rounds; ++r) {
        bits.push_back((r == 0 ? 1 : 0) | (r + 1 == rounds ? 2 : 0));
        for (int l = 0; l < kLanes; ++l)
          for (int j = 0; j < 4; ++j) {
            uint32_t w = pad;
            if (g + size_t(l) < order.size()) {
              const auto& c = chains[order[g + size_t(l)]];
              if (size_t(4 * r + j) < c.size()) w = c[size_t(4 * r + j)];
            }
            body.push_back(w);
          }
      }
      for (int l = 0; l < kLanes && g + size_t(l) < order.size(); ++l) slot[size_t(order[g + size_t(l)])] = int(g) + l;
    }
    *n = int(bits.size());
    *oHdr = begin();
    masks(bits);
    *oBody = begin();
    W.insert(W.end(), body.begin(), body.end());
    end(4 * kLanes);
    return slot;
  }

  std::map<double, int> coefIx;
  unsigned coef(double c) {
    auto it = coefIx.find(c);
    if (it == coefIx.end()) {
      it = coefIx.emplace(c, int(out.coef.size())).first;
      out.coef.push_back(c);
    }
    return field8(it->second);
  }
  unsigned field8(int ix) const {
    const int f = (8 * ix) >> d.shift;
    if (f > 0xffff) throw std::runtime_error("lowered programs: too many coefficients");
    return unsigned(f);
  }

  void evaluation() {
    coefIx[0.0] = 0;
    out.coef.push_back(0.0);
    // powers and scaled rate constants
    d.oPow = begin();
    d.nPow = ceilDiv(int(powers.size()), kLanes);
    for (int i = 0; i < kLanes * d.nPow; ++i) {
      const bool live = i < int(powers.size());
      W.push_back(live ? pack(field(d.oC + 8 * powers[i].first), field(powerSlot(powers[i].first, powers[i].second)))
                       : pack(field(d.oneC), field(d.trashC)));
      W.push_back(live ? uint32_t(powers[i].second) : 1u);
    }
    std::vector<int> reactionAt(ropSlot.size(), -1);
    for (int r = 0; r < t.nReac; ++r) reactionAt[size_t(ropSlot[size_t(r)])] = r;
    d.oKf = begin();
    for (int r : reactionAt) W.push_back(uint32_t(r));
    d.oKfx = begin();
    d.nKfx = ceilDiv(int(scaled.size()), kLanes);
    for (int i = 0; i < kLanes * d.nKfx; ++i) {
      const bool live = i < int(scaled.size());
      W.push_back(live ? uint32_t(ropSlot[size_t(scaled[i].first)]) : 0u);
      W.push_back(live ? pack(field(kfSlot(scaled[i].first, scaled[i].second)), unsigned(scaled[i].second))
                       : pack(field(d.trashC), 1u));
    }
    // rates of progress
    d.oRop = begin();
    d.nRop = s.ropRounds;
    for (int r : reactionAt) {
      const bool live = r >= 0;
      W.push_back(live ? pack(field(factorSlot(r, 0)), field(factorSlot(r, 1))) : pack(field(d.oneC), field(d.oneC)));
      W.push_back(live ? field(factorSlot(r, 2)) : field(d.oneC));
    }
    end(2 * kLanes);
    // derivative pairs
    d.oPair = begin();
    d.nPair = s.pairRounds;
    {
      std::vector<std::array<uint32_t, 2>> rec(pairSlot.size(), {pack(field(d.zero8), field(d.oneC)),
                                                                 pack(field(d.oneC), field(d.oneC))});
      for (int r = 0; r < t.nReac; ++r)
        for (int p = t.pairPtr[r]; p < t.pairPtr[r + 1]; ++p) {
          const int js = t.pairSlot[p], n = power(r, js);
          std::vector<int> g;
          for (int j = 0; j < 3; ++j)
            if (j != js) g.push_back(factorSlot(r, j));
          rec[size_t(pairSlot[size_t(p)])] = {pack(field(kfSlot(r, n)), field(powerSlot(spec(r, js), n - 1))),
                                              pack(field(g[0]), field(g[1]))};
        }
      for (const auto& x : rec) W.insert(W.end(), x.begin(), x.end());
    }
    end(2 * kLanes);
    // segment sums and species rows
    {
      std::vector<std::vector<uint32_t>> ch;
      for (int g = 0; g < t.nSeg(); ++g) {
        ch.emplace_back();
        for (int e = t.segBegin[g]; e < t.segEnd[g]; ++e)
          ch.back().push_back(pack(field(d.oP + 8 * ropSlot[size_t(t.omegaReac[e])]), coef(t.omegaCoef[e])));
      }
      const std::vector<int> slot = sums(ch, pack(field(d.zero8), 0), &d.oSegHdr, &d.oSeg, &d.nSeg);
      const int rows = int(t.rowSegPtr.size()) - 1;
      d.oRow = begin();
      for (int q = 0; q < 4; ++q) {
        int most = 0;
        for (int a = kLanes * q; a < std::min(rows, kLanes * (q + 1)); ++a)
          most = std::max(most, t.rowSegPtr[a + 1] - t.rowSegPtr[a]);
        d.nRow[q] = ceilDiv(most, 4);
        for (int r = 0; r < d.nRow[q]; ++r)
          for (int l = 0; l < kLanes; ++l) {
            unsigned f[4];
            for (int j = 0; j < 4; ++j) {
              const int a = kLanes * q + l, g = a < rows ? t.rowSegPtr[a] + 4 * r + j : 0;
              f[j] = field(a < rows && g < t.rowSegPtr[a + 1] ? d.oS + 8 * slot[size_t(g)] : d.zero8);
            }
            W.push_back(pack(f[0], f[1]));
            W.push_back(pack(f[2], f[3]));
          }
      }
      end(2 * kLanes);
    }
  }

  void jacobian() {
    auto target = [&](int x) { return field(x < 0 ? d.oPS + T * (-1 - x) : slotA(x)); };
    auto dpr = [&](const Chunk* c, size_t k) { return field(c && k < c->e.size() ? d.oD + T * pairSlot[size_t(c->e[k].first)] : d.zeroA); };
    std::vector<double> cf;
    auto coefs = [&](const Chunk* c, size_t n) {
      for (size_t k = 0; k < n; ++k) cf.push_back(c && k < c->e.size() ? c->e[k].second : 0.0);
    };
    auto get = [](const std::vector<Chunk>& v, size_t i) { return i < v.size() ? &v[i] : nullptr; };
    d.nJ4 = ceilDiv(int(j4.size()), kLanes);
    d.nJ2 = ceilDiv(int(j2.size()), 2 * kLanes);
    d.nJ1 = ceilDiv(int(j1.size()), 4 * kLanes);
    d.oJac = begin();
    for (int r = 0; r < d.nJ4; ++r)
      for (int l = 0; l < kLanes; ++l) {
        const Chunk* c = get(j4, size_t(r * kLanes + l));
        W.push_back(pack(dpr(c, 0), dpr(c, 1)));
        W.push_back(pack(dpr(c, 2), dpr(c, 3)));
        W.push_back(c ? target(c->target) : field(d.trashA));
        W.push_back(c ? c->flags : 0u);
        coefs(c, 4);
      }
    for (int r = 0; r < d.nJ2; ++r)
      for (int l = 0; l < kLanes; ++l) {
        const Chunk* c[2];
        for (int k = 0; k < 2; ++k) c[k] = get(j2, size_t((2 * r + k) * kLanes + l));
        for (int k = 0; k < 2; ++k) {
          W.push_back(pack(dpr(c[k], 0), dpr(c[k], 1)));
          coefs(c[k], 2);
        }
        W.push_back(pack(c[0] ? target(c[0]->target) : field(d.trashA), c[1] ? target(c[1]->target) : field(d.trashA)));
        W.push_back(0u);
      }
    for (int r = 0; r < d.nJ1; ++r)
      for (int l = 0; l < kLanes; ++l) {
        const Chunk* c[4];
        for (int k = 0; k < 4; ++k) c[k] = get(j1, size_t((4 * r + k) * kLanes + l));
        for (int k = 0; k < 4; k += 2) W.push_back(pack(dpr(c[k], 0), dpr(c[k + 1], 0)));
        for (int k = 0; k < 4; k += 2)
          W.push_back(pack(c[k] ? target(c[k]->target) : field(d.trashA),
                           c[k + 1] ? target(c[k + 1]->target) : field(d.trashA)));
        for (int k = 0; k < 4; ++k) coefs(c[k], 1);
      }
    end(4 * kLanes);
    d.oJacC = begin();
    for (double c : cf) {
      if (T == 8) {
        uint64_t b;
        std::memcpy(&b, &c, 8);
        W.push_back(uint32_t(b));
        W.push_back(uint32_t(b >> 32));
      } else {
        const float f = float(c);
        uint32_t b;
        std::memcpy(&b, &f, 4);
        W.push_back(b);
      }
    }
    end(4 * kLanes * (T / 4));
    d.oJx = begin();
    d.nJx = ceilDiv(int(joins.size()), kLanes);
    for (int i = 0; i < kLanes * d.nJx; ++i) {
      const bool live = i < int(joins.size());
      W.push_back(live ? pack(target(joins[i].target), field(d.oPS + T * joins[i].first))
                       : pack(field(d.trashA), field(d.oPS)));
      W.push_back(live ? uint32_t(joins[i].count) | (joins[i].diag ? 0x80000000u : 0u) : 0u);
    }
    end(2 * kLanes);
  }

  // LU-kind rounds [r0, r0 + n) of the rounds' program, body at word b
  void luRounds(int r0, int n, size_t b, int* oHdr, int* o4, int* o1) {
    using SS = SparseSchedule;
    std::vector<unsigned char> bits;
    std::vector<uint32_t> w4, w1;
    const unsigned z = field(d.zeroA), tr = field(d.trashA);
    for (int r = r0; r < r0 + n; ++r) {
      const int kind = int(s.progHdr[size_t(r)] >> 16), len = int(s.progHdr[size_t(r)] & 0xffff);
      auto word = [&](int j, int l) { return s.progBody[b + size_t(kLanes) * size_t(j) + size_t(l)]; };
      bits.push_back(kind == SS::kMul ? 1 : (kind == SS::kUpd ? 2 : 0));
      for (int l = 0; l < kLanes; ++l) {
        unsigned f[10];
        std::fill(f, f + 10, z);
        if (kind == SS::kMul) {
          const unsigned dst = word(0, l) & 0xffff, src = word(0, l) >> 16;
          f[0] = (dst & 0x8000u) ? tr : matrix(dst);
          f[1] = matrix(src);
        } else if (kind == SS::kUpd) {
          f[0] = matrix(word(0, l));
          for (int j = 0; j < len; ++j) {
            f[1 + 2 * j] = matrix(word(1 + j, l) & 0xffff);
            f[2 + 2 * j] = matrix(word(1 + j, l) >> 16);
          }
        } else if (kind == SS::kMulUpd) {
          f[0] = matrix(word(0, l));
          f[1] = matrix(word(1, l) & 0xffff);
          f[2] = matrix(word(1, l) >> 16);
          f[3] = matrix(word(2, l) & 0x7fff);
          for (int j = 0; j < len - 2; ++j) {
            f[4 + 2 * j] = matrix(word(3 + j, l) & 0xffff);
            f[5 + 2 * j] = matrix(word(3 + j, l) >> 16);
          }
          // the device tells a multiplier lane by its target being its own multiplier
          if (((word(2, l) & 0x8000u) != 0) != (f[0] == f[1]))
            throw std::runtime_error("lowered programs: ambiguous multiplier lane");
        } else {
          throw std::runtime_error("lowered programs: unexpected round in the LU program");
        }
        for (int j = 0; j < 8; j += 2) w4.push_back(pack(f[j], f[j + 1]));
        w1.push_back(pack(f[8], f[9]));
      }
      b += size_t(kLanes) * (kind == SS::kMul ? 1 : size_t(1 + len));
    }
    *oHdr = begin();
    masks(bits);
    *o4 = begin();
    W.insert(W.end(), w4.begin(), w4.end());
    end(4 * kLanes);
    *o1 = begin();
    W.insert(W.end(), w1.begin(), w1.end());
    end(kLanes);
  }

  void linearAlgebra() {
    static_assert(SparseSchedule::kMaxChain == 4 && SparseSchedule::kMaxMulUpdChain == 2, "record layout");
    d.nLu = s.luRounds;
    luRounds(0, s.luRounds, 0, &d.oLuHdr, &d.oLu, &d.oLu1);
    d.oDiag = begin();
    for (int i = 0; i < kLanes * ceilDiv(s.m, kLanes); ++i)
      W.push_back(uint32_t(i < s.m ? slotA(s.slotOf[size_t(s.diagIdx[size_t(i)])]) : d.zeroA));
    // back substitution: a round of n-entry chains is n single-entry rounds
    // (no round reads an entry it writes)
    {
      std::vector<std::array<uint32_t, 2 * kLanes>> one;
      size_t b = size_t(s.backBody);
      for (int r = s.luRounds; r < s.luRounds + s.backRounds; ++r) {
        const int len = int(s.progHdr[size_t(r)] & 0xffff);
        for (int j = 0; j < len; ++j) {
          one.emplace_back();
          for (int l = 0; l < kLanes; ++l) {
            const unsigned tgt = s.progBody[b + size_t(l)], e = s.progBody[b + size_t(kLanes) * size_t(1 + j) + size_t(l)];
            // a lane whose chain has ended rests on the trash slot
            const bool live = int(e & 0xffff) < s.nnzF;
            one.back()[size_t(2 * l)] = pack(live ? matrix(tgt) : field(rhs(s.m + 1)), live ? matrix(e & 0xffff) : field(d.zeroA));
            one.back()[size_t(2 * l + 1)] = live ? field(rhs(int(e >> 16))) : field(rhs(s.m));
          }
        }
        b += size_t(kLanes) * size_t(1 + len);
      }
      if (one.size() % 2) {
        one.emplace_back();
        for (int l = 0; l < kLanes; ++l) {
          one.back()[size_t(2 * l)] = pack(field(rhs(s.m + 1)), field(d.zeroA));
          one.back()[size_t(2 * l + 1)] = field(rhs(s.m));
        }
      }
      d.oBack = begin();
      d.nBack = int(one.size() / 2);
      for (size_t r = 0; r < one.size(); r += 2)
        for (int l = 0; l < kLanes; ++l)
          for (size_t k = 0; k < 2; ++k) {
            W.push_back(one[r + k][size_t(2 * l)]);
            W.push_back(one[r + k][size_t(2 * l + 1)]);
          }
      end(4 * kLanes);
    }
  }

  void adjointSums() {
    const int m = s.m;
    std::vector<std::vector<uint32_t>> nu(static_cast<size_t>(t.nReac)), jt(static_cast<size_t>(m));
    for (int a = 0; a < m; ++a)
      for (int e = t.omegaPtr[a]; e < t.omegaPtr[a + 1]; ++e)
        nu[size_t(t.omegaReac[e])].push_back(pack(field(d.oMu + 8 * a), coef(t.omegaCoef[e])));
    const std::vector<int> w = sums(nu, pack(field(d.oMu + 8 * m), 0), &d.oNutHdr, &d.oNut, &d.nNut);
    for (int r = 0; r < t.nReac; ++r)
      for (int p = t.pairPtr[r]; p < t.pairPtr[r + 1]; ++p)
        jt[size_t(spec(r, t.pairSlot[p]))].push_back(pack(field(d.oD + T * pairSlot[size_t(p)]), field(d.oW + 8 * w[size_t(r)])));
    const std::vector<int> v = sums(jt, pack(field(d.zeroA), field(d.zero8)), &d.oJtvHdr, &d.oJtv, &d.nJtv);
    d.oWmap = begin();  // by slot of the reaction
    std::vector<uint32_t> at(ropSlot.size(), uint32_t(d.zero8));
    for (int r = 0; r < t.nReac; ++r) at[size_t(ropSlot[size_t(r)])] = uint32_t(d.oW + 8 * w[size_t(r)]);
    W.insert(W.end(), at.begin(), at.end());
    d.oVmap = begin();
    for (int i = 0; i < kLanes * ceilDiv(m, kLanes); ++i) W.push_back(uint32_t(i < m ? d.oV + 8 * v[size_t(i)] : d.zero8));
  }

  void run() {
    if (T != 4 && T != 8) throw std::runtime_error("lowered programs: entry size");
    if (adjoint && T != 8) throw std::runtime_error("lowered programs: the adjoint is FP64");
    out.slot = slots.factor;
    collect();
    {
      Chunks k = jacobianChunks(t, s);
      j4 = std::move(k.j4), j2 = std::move(k.j2), j1 = std::move(k.j1), joins = std::move(k.joins);
      nPartial = k.nPartial;
    }
    layout();
    evaluation();
    linearAlgebra();
    d.stagedWords = (std::max(int(W.size()), readAhead) + 3) & ~3;
    jacobian();
    d.nFwd = s.fwdRounds;
    luRounds(s.luRounds + s.backRounds, s.fwdRounds, size_t(s.fwdBody), &d.oFwdHdr, &d.oFwd, &d.oFwd1);
    if (adjoint && s.transposed) adjointSums();
    begin();
    while (int(W.size()) < readAhead) W.push_back(0);
    begin();
    d.words = int(W.size());
    d.nCoef = int(out.coef.size());
    d.enabled = 1;
  }
};

}  // namespace

LoweredSlots chooseSlots(const MechTables& t, const SparseSchedule& s, const LoweredSlots* shared) {
  LoweredSlots o;
  o.factor = factorSlots(s);
  if (shared) {
    o.pair = shared->pair;
    o.rop = shared->rop;
  } else {
    o.pair = pairSlots(s, jacobianChunks(t, s), t.nPairs());
    o.rop = reactionSlots(t, s, o.pair);
  }
  return o;
}

LoweredProgram lowerProgram(const MechTables& t, const SparseSchedule& s, int bytesT, bool adjoint,
                            const LoweredSlots& slots) {
  Lowering L(t, s, bytesT, adjoint, slots);
  L.run();
  return std::move(L.out);
}

}  // namespace tchem_amd
