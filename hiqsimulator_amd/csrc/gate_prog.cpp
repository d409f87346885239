// Host side of the gate programs: gates to units, units to passes and stages,
// stages to device records.  See gate_prog.hpp.
#include "gate_prog.hpp"

#include <algorithm>
#include <array>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <stdexcept>

namespace hq {
namespace {

using cplx = std::complex<double>;

inline int popc(uint64_t x) { return __builtin_popcountll(x); }
inline uint64_t low_bit(uint64_t x) { return x & (~x + 1); }

bool is_one(const cplx& z) { return z.real() == 1.0 && z.imag() == 0.0; }
bool finite(const cplx& z) { return std::isfinite(z.real()) && std::isfinite(z.imag()); }

}  // namespace

namespace {
// index bits that some nonzero entry changes
size_t mixed_bits(const cplx* m, size_t targets)
{
     const size_t dim = size_t(1) << targets;
     size_t mixed = 0;
     for (size_t i = 0; i < dim; ++i)
          for (size_t j = 0; j < dim; ++j)
               if (i != j && !(m[i * dim + j] == 0.0)) mixed |= i ^ j;
     return mixed;
}
}  // namespace

bool gate_fits(const cplx* m, size_t targets) { return targets <= 2 || (targets <= 5 && popc(mixed_bits(m, targets)) <= 2); }

bool make_gate_unit(const cplx* m, const std::vector<int64_t>& targets, const std::vector<int64_t>& ctrls, GateUnit& out)
{
     const int t = static_cast<int>(targets.size());
     if (t < 1 || t > 5) return false;
     const size_t dim = size_t(1) << t;
     for (int64_t p: targets)
          if (p < 0 || p >= 62) return false;
     uint64_t cm = 0;
     for (int64_t p: ctrls) {
          if (p < 0 || p >= 62) return false;
          cm |= uint64_t(1) << p;
     }
     const size_t mixed = mixed_bits(m, targets.size());
     const int na = popc(mixed);
     if (na > 2) return false;
     out = GateUnit();
     out.na = na;
     out.d = cm;
     int act[2] = {0, 0}, na_seen = 0;
     int dl[5], nd = 0;
     for (int l = 0; l < t; ++l) {
          const uint64_t bit = uint64_t(1) << targets[l];
          if ((out.a | out.d) & bit) return false;  // repeated position
          if ((mixed >> l) & 1) {
               act[na_seen] = l;
               out.act[na_seen++] = static_cast<uint8_t>(targets[l]);
               out.a |= bit;
          }
          else {
               dl[nd++] = l;
               out.d |= bit;
          }
     }
     const int ad = 1 << na;
     // the block of each setting of the unmixed targets
     auto branch = [&](int s, GateBranch& b) {
          b.cmask = cm;
          b.cval = cm;
          size_t row0 = 0;
          for (int q = 0; q < nd; ++q) {
               const uint64_t bit = uint64_t(1) << targets[dl[q]];
               b.cmask |= bit;
               if ((s >> q) & 1) {
                    b.cval |= bit;
                    row0 |= size_t(1) << dl[q];
               }
          }
          for (int i = 0; i < ad; ++i)
               for (int j = 0; j < ad; ++j) {
                    size_t r = row0, c = row0;
                    for (int l = 0; l < na; ++l) {
                         if ((i >> l) & 1) r |= size_t(1) << act[l];
                         if ((j >> l) & 1) c |= size_t(1) << act[l];
                    }
                    b.u[i * ad + j] = m[r * dim + c];
               }
     };
     out.br.resize(size_t(1) << nd);
     for (int s = 0; s < (1 << nd); ++s) branch(s, out.br[static_cast<size_t>(s)]);
     // the same block in every setting: the unmixed targets do not matter
     bool same = na > 0 && nd > 0;
     for (const auto& b: out.br)
          for (int i = 0; i < ad * ad; ++i) same = same && b.u[i] == out.br[0].u[i];
     if (same) {
          out.br.resize(1);
          out.br[0].cmask = out.br[0].cval = cm;
     }
     if (na == 0 && cm == 0) {
          // the first entry as a factor of everything, the others relative to it
          const cplx f = out.br[0].u[0];
          const double a = std::abs(f);
          if (a > 0.5 && a < 2.0) {
               for (auto& b: out.br) b.u[0] /= f;
               out.br[0].u[0] = f;
               out.br[0].cmask = out.br[0].cval = 0;
          }
     }
     // identity branches do nothing
     auto identity = [&](const GateBranch& b) {
          for (int i = 0; i < ad; ++i)
               for (int j = 0; j < ad; ++j)
                    if (!(i == j ? is_one(b.u[i * ad + j]) : b.u[i * ad + j] == 0.0)) return false;
          return true;
     };
     out.br.erase(std::remove_if(out.br.begin(), out.br.end(), identity), out.br.end());
     // a bit that no branch depends on any more is free (e.g. both settings
     // of a target became identity)
     uint64_t dep = 0;
     for (const auto& b: out.br) dep |= b.cmask;
     out.d &= dep;
     if (out.br.empty()) out.a = 0, out.na = 0;
     return true;
}

// ---------------------------------------------------------------------------
// Which way
// ---------------------------------------------------------------------------
namespace {

bool is_flip(const GateBranch& b) { return b.u[0] == 0.0 && b.u[3] == 0.0 && is_one(b.u[1]) && is_one(b.u[2]); }

constexpr int kGateHostBound = 18;  // up to here the work a gate decides alone

// What an unconditional gate on one qubit is merged with (put_one, layer_phase).
enum Run : uint8_t { kRunNone, kRunPhase, kRunReal, kRunCross, kRunGeneral };

Run run_of(const GateUnit& g)
{
     const auto& u = g.br[0].u;
     if (g.na == 0) return kRunPhase;
     if (u[0].imag() == 0.0 && u[3].imag() == 0.0) {
          if (u[1].imag() == 0.0 && u[2].imag() == 0.0) return kRunReal;
          if (u[1].real() == 0.0 && u[2].real() == 0.0) return kRunCross;
     }
     return kRunGeneral;
}

}  // namespace

// Whether the block is applied without rounded coefficients: entries that are
// zero or the first one's turns by quarters.
bool without_rounded(const GateUnit& g, const GateBranch& b)
{
     const int entries = 1 << (2 * g.na);
     cplx p = 1.0;
     for (int i = 0; g.na && i < entries; ++i)
          if (!(b.u[i] == 0.0)) {
               p = b.u[i];
               break;
          }
     for (int i = 0; i < entries; ++i) {
          const cplx z = b.u[i];
          if (!(z == 0.0 || z == p || z == -p || z == cplx(-p.imag(), p.real()) || z == cplx(p.imag(), -p.real()))) return false;
     }
     return true;
}

// 0 for a unit without rounded coefficients.
uint64_t hash_of(const GateUnit& g)
{
     uint64_t h = 0;
     for (const auto& b: g.br) {
          if (without_rounded(g, b)) continue;
          const int words = 2 << (2 * g.na);
          uint64_t v[32];
          std::memcpy(v, b.u, static_cast<size_t>(words) * 8);
          for (int i = 0; i < words; ++i) {
               h = (h ^ v[i]) * 0x9e3779b97f4a7c15ull;
               h ^= h >> 29;
          }
          h |= 1;
     }
     return h;
}

GateListCost gate_list_cost(const std::vector<GateUnit>& units, int n, Prec prec)
{
     constexpr double kGeneral = 3.7, kTwo = 6.5, kFactor = 0.5, kTested = 2.0;
     constexpr int kWidth = 4;
     GateListCost c;
     const bool need_products = n > kGateHostBound || prec == Prec::C64, need_rounds = prec == Prec::C64;
     // The roundings of gates with the same coefficients come out the same and add
     // up: m of them count as m^2.
     struct Rounding {
          uint64_t same;
          double count;
     };
     std::vector<Rounding> roundings;
     auto round = [&](uint64_t same, double count) {
          if (!need_rounds) return;
          if (same) roundings.push_back({same, count});
          else c.rounds += count;
     };
     Run run[64] = {};    // of each qubit's last gate, while it can still take another
     uint64_t same[64];   // the run's coefficients
     auto end_run = [&](uint64_t bits) {
          for (; bits; bits &= bits - 1) {
               const int p = __builtin_ctzll(bits);
               if (run[p] == kRunNone) continue;
               const bool general = run[p] == kRunGeneral;
               c.work += general ? kGeneral : 1;
               round(same[p], general ? 3 : 1);
               run[p] = kRunNone;
          }
     };
     std::vector<uint64_t> groups;  // qubits of the fused products
     int last[64];                  // a qubit's last one
     std::fill_n(last, 64, -1);
     auto open = [&](int i) {
          for (uint64_t m = groups[i]; m; m &= m - 1)
               if (last[__builtin_ctzll(m)] != i) return false;
          return true;
     };
     double slots = 0;
     uint64_t mixed = 0;  // by the units so far
     for (const GateUnit& g: units) {
          const uint64_t bits = g.a | g.d;
          if (g.br.empty() || !bits) continue;  // (a factor of all amplitudes costs nothing)
          const uint64_t h = need_rounds ? hash_of(g) : 0;
          if (popc(bits) == 1 && (g.na == 0 || (g.br.size() == 1 && !g.br[0].cmask))) {
               const int p = __builtin_ctzll(bits);
               const Run now = run_of(g);
               if (run[p] != kRunNone && run[p] != now) {
                    if (run[p] != kRunPhase && now != kRunPhase && (run[p] == kRunGeneral || now == kRunGeneral)) run[p] = kRunGeneral;
                    else end_run(bits);
               }
               if (run[p] == kRunNone) {
                    run[p] = now;
                    same[p] = h;
               }
               else {
                    same[p] = (same[p] * 0x9e3779b97f4a7c15ull) ^ h;
               }
          }
          else {
               end_run(bits);
               // (a factor on a qubit that nothing has mixed yet goes into a list's product, in FP64)
               const bool listed = g.na == 0 && (bits & ~mixed);
               for (const auto& b: g.br) {
                    if (g.na == 0) c.work += listed ? kFactor : kTested, round(listed ? 0 : h, listed ? 0.25 : 0.75);
                    else if (g.na == 2) c.work += kTwo, round(h, 4);
                    else if (is_flip(b)) c.work += 1;
                    else c.work += kGeneral, round(h, 3);
               }
          }
          mixed |= g.a;
          if (!need_products) continue;
          // the fused product that it would go into
          const int first = last[__builtin_ctzll(bits)];
          bool inside = first >= 0;
          for (uint64_t m = bits; m; m &= m - 1) inside = inside && last[__builtin_ctzll(m)] == first;
          if (inside) continue;
          uint64_t u = bits;
          for (uint64_t m = bits; m; m &= m - 1) {
               const int i = last[__builtin_ctzll(m)];
               if (i < 0 || !(groups[i] & ~u) || !open(i) || popc(u | groups[i]) > kWidth) continue;
               u |= groups[i];
          }
          for (uint64_t m = u; m; m &= m - 1) {
               const int i = last[__builtin_ctzll(m)];
               if (i < 0 || (groups[i] & ~u) || !open(i)) continue;
               slots -= popc(groups[i]);  // grows into the new one
               groups[i] = 0;
          }
          slots += popc(u);
          for (uint64_t m = u; m; m &= m - 1) last[__builtin_ctzll(m)] = static_cast<int>(groups.size());
          groups.push_back(u);
     }
     c.products = slots / 4;
     end_run(~uint64_t(0));
     std::sort(roundings.begin(), roundings.end(), [](const Rounding& a, const Rounding& b) { return a.same < b.same; });
     for (size_t i = 0, j; i < roundings.size(); i = j) {
          double sum = 0;
          for (j = i; j < roundings.size() && roundings[j].same == roundings[i].same; ++j) sum += roundings[j].count;
          c.rounds += sum * static_cast<double>(j - i);
     }
     return c;
}

bool gate_route(const GateListCost& cost, size_t gates, int n, Prec prec, Prec& held)
{
     held = Prec::C128;
     if (n < gate_min_qubits(prec) || n > 40) return false;
     // (two more for the factor of a whole pass)
     if (prec == Prec::C64 && cost.rounds + 2 <= 9.5 * cost.products) {
          held = Prec::C64;
          return true;
     }
     if (n <= 22 && cost.work <= 4.0 * static_cast<double>(gates)) return true;  // bound by the host
     return n > kGateHostBound && cost.work <= (prec == Prec::C128 ? 24.0 : (n <= 24 ? 18.0 : 13.0)) * cost.products;
}

// ---------------------------------------------------------------------------
// Planning
// ---------------------------------------------------------------------------
bool GatePassPlanner::worth_splits(int n, Prec prec)
{
     return std::ldexp(static_cast<double>(amp_bytes(prec)), n) >= 0x1p30;
}

GatePassPlanner::GatePassPlanner(const std::vector<GateUnit>& units, int n, Prec prec, bool splits)
    : units_(units), n_(n), prec_(prec), splits_(splits)
{
     if (n < gate_tile_bits(prec) || n > 62) throw std::runtime_error("gate program: the state is smaller than a tile");
     const uint64_t lim = (uint64_t(1) << n) - 1;
     for (size_t i = 0; i < units.size(); ++i) {
          if ((units[i].a | units[i].d) & ~lim) throw std::runtime_error("gate program: a gate acts beyond the state");
          rem_.push_back(static_cast<int>(i));
     }
}

// k bits of `allowed` (beside `fixed`) such that many units can be taken from
// the front of the list: from the first unit's bits, the bit that lets the
// most units be taken is added until k are there; then bits are exchanged
// while that takes more.  `start`: other bits to begin with.
uint64_t GatePassPlanner::choose(const std::vector<int>& list, uint64_t fixed, uint64_t allowed, int k,
                                 uint64_t start) const
{
     constexpr int kWindow = 96;  // mixing units whose bits are candidates
     uint64_t pool = 0, H = 0;
     int seen = 0;
     for (int i: list) {
          const uint64_t a = units_[i].a;
          if (!a) continue;
          if (!seen) H = (start ? start : a) & ~fixed;
          pool |= a;
          if (++seen >= kWindow) break;
     }
     pool &= allowed & ~fixed;
     // Units that bit set S takes, mixing units counted first; the scan ends
     // when every bit of S is blocked, or where a pass is full.
     const size_t window = std::min(list.size(), kGateMaxPassUnits);
     auto score = [&](uint64_t S) {
          uint64_t ba = 0, bd = 0;
          int s = 0;
          for (size_t at = 0; at < window; ++at) {
               const GateUnit& g = units_[list[at]];
               if (!(g.a & ~S) && !(g.a & (ba | bd)) && !(g.d & ba)) {
                    s += g.a ? 256 : 1;
               }
               else {
                    ba |= g.a;
                    bd |= g.d;
                    if (!(S & ~(ba | bd))) break;
               }
          }
          return s;
     };
     while (popc(H) < k) {
          uint64_t add = 0;
          int best = -1;
          for (uint64_t m = pool & ~H; m; m &= m - 1) {
               const int s = score(fixed | H | low_bit(m));
               if (s > best) {
                    best = s;
                    add = low_bit(m);
               }
          }
          if (!add) break;
          H |= add;
     }
     int best = score(fixed | H);
     for (int round = 0; round < 2; ++round) {
          uint64_t top = H;
          for (uint64_t o = H; o; o &= o - 1)
               for (uint64_t m = pool & ~H; m; m &= m - 1) {
                    const uint64_t H2 = (H & ~low_bit(o)) | low_bit(m);
                    const int s = score(fixed | H2);
                    if (s > best) {
                         best = s;
                         top = H2;
                    }
               }
          if (top == H) break;
          H = top;
     }
     return H;
}

// Moves the units that S takes (at most `cap`) from the list to `out`.
void GatePassPlanner::take(std::vector<int>& list, uint64_t S, size_t cap, std::vector<int>& out) const
{
     uint64_t ba = 0, bd = 0;
     std::vector<int> rest;
     for (int i: list) {
          const GateUnit& g = units_[i];
          if (out.size() < cap && !(g.a & ~S) && !(g.a & (ba | bd)) && !(g.d & ba)) {
               out.push_back(i);
          }
          else {
               ba |= g.a;
               bd |= g.d;
               rest.push_back(i);
          }
     }
     list.swap(rest);
}

// Splits a pass's units into stages, from the back of the list if `back`; with
// `avoid` the first one found keeps off the low bits.  What does not fit stays
// in the list.  Returns the groupings of the pass: one a stage, and one more at
// an end whose registers hold low bits (the compiler's empty stages); 0: none.
size_t GatePassPlanner::make_stages(std::vector<int>& list, GatePassPlan& out, bool back, bool avoid) const
{
     const uint64_t low = (uint64_t(1) << kGateLow) - 1;
     out.regs.clear();
     out.stages.clear();
     if (back) std::reverse(list.begin(), list.end());
     while (!list.empty() && out.stages.size() < kGateMaxStages - 2) {
          uint64_t R;
          if (avoid && out.stages.empty()) {
               uint64_t ba = 0, bd = 0, start = 0;
               for (int i: list) {
                    const GateUnit& g = units_[i];
                    if (g.a && !(g.a & (low | ba | bd)) && !(g.d & ba)) {
                         start = g.a;
                         break;
                    }
                    ba |= g.a;
                    bd |= g.d;
               }
               if (!start) return 0;
               R = choose(list, 0, out.bits & ~low, gate_reg(prec_), start);
          }
          else {
               R = choose(list, 0, out.bits, gate_reg(prec_));
          }
          std::vector<int> stage;
          take(list, R, kGateMaxStageUnits, stage);
          if (stage.empty()) throw std::runtime_error("gate program: no gate could be staged");
          if (back) std::reverse(stage.begin(), stage.end());
          out.regs.push_back(R);
          out.stages.push_back(std::move(stage));
     }
     if (back) {
          std::reverse(list.begin(), list.end());
          std::reverse(out.regs.begin(), out.regs.end());
          std::reverse(out.stages.begin(), out.stages.end());
     }
     return out.stages.size() + ((out.regs.front() & low) != 0) + ((out.regs.back() & low) != 0);
}

bool GatePassPlanner::next(GatePassPlan& out)
{
     if (rem_.empty()) return false;
     const uint64_t low = (uint64_t(1) << kGateLow) - 1;
     const uint64_t all = (uint64_t(1) << n_) - 1;
     out = GatePassPlan();
     out.bits = low | choose(rem_, low, all, gate_high(prec_));
     for (int p = kGateLow; p < n_ && popc(out.bits) < gate_tile_bits(prec_); ++p) out.bits |= uint64_t(1) << p;
     std::vector<int> taken;
     take(rem_, out.bits, kGateMaxPassUnits, taken);
     if (taken.empty()) throw std::runtime_error("gate program: no gate could be planned");
     const std::vector<int> whole = splits_ ? taken : std::vector<int>();
     size_t groupings = make_stages(taken, out, false, false);
     if (splits_ && taken.empty())
          for (int way = 1; way < 4; ++way) {
               GatePassPlan other;
               other.bits = out.bits;
               std::vector<int> list = whole;
               const size_t g = make_stages(list, other, way & 2, way & 1);
               if (g && list.empty() && g < groupings) {
                    groupings = g;
                    out = std::move(other);
               }
          }
     if (!taken.empty()) {  // more stages than a pass holds: the rest stays
          std::vector<int> all_rest(taken.size() + rem_.size());
          std::merge(taken.begin(), taken.end(), rem_.begin(), rem_.end(), all_rest.begin());
          rem_.swap(all_rest);
     }
     return true;
}

// ---------------------------------------------------------------------------
// Compilation
// ---------------------------------------------------------------------------
namespace {

// Where the tile's ranks sit in one stage: thr[j] = rank of thread bit j,
// reg[b] = rank of register bit b.
struct Layout {
     int thr[kGateThr];
     int reg[kGateMaxReg];
};

// The thread order of a stage whose register ranks are given.  The first five
// (complex64: six) lane bits get ranks with independent low slot bits, so that
// 32 lanes of 8 bytes or 64 of 4 hit distinct banks;
// `io`: lanes 0..3 are these ranks (0..3 to load), so that the stage's
// grouping can be loaded or stored in runs of 16 amplitudes; null: any.
Layout make_layout(Prec prec, const std::vector<int>& reg, const int* io)
{
     Layout L{};
     bool in_reg[kGateMaxTile] = {};
     for (size_t b = 0; b < reg.size(); ++b) {
          L.reg[b] = reg[b];
          in_reg[reg[b]] = true;
     }
     const uint32_t low = prec == Prec::C128 ? 31u : 63u;
     const size_t want = prec == Prec::C128 ? 5 : 6;
     std::vector<int> lanes, rest;
     uint32_t basis[6] = {0, 0, 0, 0, 0, 0};  // basis[b]: vector with leading bit b
     std::vector<int> order;
     for (int q = 0; io && q < kGateLow; ++q) {
          if (in_reg[io[q]]) throw std::runtime_error("gate program: internal layout error");
          order.push_back(io[q]);
     }
     for (int r = 0; r < gate_tile_bits(prec); ++r)
          if (!in_reg[r] && std::find(order.begin(), order.end(), r) == order.end()) order.push_back(r);
     const size_t runs = io ? kGateLow : 0;  // lanes that are given, independent or not
     for (size_t q = 0; q < order.size(); ++q) {
          const int r = order[q];
          uint32_t v = gate_slot(prec, r) & low;
          for (int b = 5; b >= 0; --b)
               if ((v >> b) & 1) {
                    if (!basis[b]) break;
                    v ^= basis[b];
               }
          const bool lane = q < runs || (v && lanes.size() < want);
          if (lane && v) basis[31 - __builtin_clz(v)] = v;
          (lane ? lanes : rest).push_back(r);
     }
     lanes.insert(lanes.end(), rest.begin(), rest.end());
     if (lanes.size() != static_cast<size_t>(kGateThr)) throw std::runtime_error("gate program: internal layout error");
     std::copy(lanes.begin(), lanes.end(), L.thr);
     return L;
}

class Compiler {
public:
     Compiler(const std::vector<GateUnit>& units, const GatePassPlan& plan, int n, Prec prec, GatePass& pass,
              std::vector<GateStage>& stages, std::vector<char>& ops, const uint8_t* src_pos)
         : units_(units),
           plan_(plan),
           prec_(prec),
           E_(gate_reg(prec)),
           T_(gate_tile_bits(prec)),
           ob_(gate_op_bytes(prec)),
           pass_(pass),
           stages_(stages),
           ops_(ops)
     {
          int r = 0;
          for (int p = 0; p < 64; ++p) rank_[p] = -1;
          for (int p = 0; p < n; ++p)
               if ((plan.bits >> p) & 1) {
                    if (r >= T_) throw std::runtime_error("gate program: internal tile error");
                    pos_[r] = p;
                    rank_[p] = r++;
               }
          if (r != T_) throw std::runtime_error("gate program: internal tile error");
          for (int q = 0; q < kGateLow; ++q)
               if (pos_[q] != q) throw std::runtime_error("gate program: internal tile error");
          for (int q = 0; q < kGateLow; ++q) {
               in_lanes_[q] = q;
               out_lanes_[q] = src_pos ? rank_[src_pos[q]] : q;
               if (out_lanes_[q] < 0) throw std::runtime_error("gate program: internal tile error");
          }
          for (int p = 0; p < n; ++p) new_pos_[src_pos ? src_pos[p] : p] = static_cast<uint8_t>(p);
          permuted_ = src_pos != nullptr;
          for (int p = 0, j = 0; p < n; ++p) outer_[p] = rank_[p] < 0 ? j++ : -1;
          n_ = n;
          if (ops_.size() >= ob_) ops_.resize(ops_.size() - ob_);  // the spare record moves to the end
     }

     void run()
     {
          pass_ = GatePass{};
          pass_.stage_first = static_cast<uint32_t>(stages_.size());
          for (int j = 0; j < T_ - kGateLow; ++j) pass_.hpos[j] = static_cast<uint8_t>(pos_[kGateLow + j]);
          const size_t ns = plan_.stages.size();
          std::vector<std::vector<int>> regs;
          for (size_t s = 0; s < ns; ++s)
               regs.push_back(reg_ranks(plan_.regs[s], permuted_ && s + 1 == ns ? out_lanes_ : nullptr));
          // a first or last stage whose registers hold ranks of the load's or
          // the store's runs is loaded or stored through an empty stage, and
          // so is a single stage whose runs are not the same ones
          const bool in_empty = holds(regs.front(), in_lanes_);
          if (in_empty) {
               begin_stage(reg_ranks(0, nullptr), in_lanes_);
               set_io(pass_.in_thr, pass_.in_reg);
          }
          bool stored = false;
          for (size_t s = 0; s < ns; ++s) {
               const int* io = nullptr;
               if (s == 0 && !in_empty) io = in_lanes_;
               else if (s + 1 == ns && !holds(regs[s], out_lanes_)) io = out_lanes_;
               begin_stage(regs[s], io);
               if (pass_stages() == 1) set_io(pass_.in_thr, pass_.in_reg);
               emit_stage(plan_.stages[s], s + 1 == ns);
               stored = s + 1 == ns && io && std::equal(io, io + kGateLow, out_lanes_);
          }
          if (!stored) begin_stage(reg_ranks(0, permuted_ ? out_lanes_ : nullptr), out_lanes_);
          set_io(pass_.out_thr, pass_.out_reg);
          if (permuted_) {
               for (int j = 0; j < kGateThr; ++j) pass_.out_thr[j] = new_pos_[pass_.out_thr[j]];
               for (int b = 0; b < E_; ++b) pass_.out_reg[b] = new_pos_[pass_.out_reg[b]];
               int j = 0;
               for (int p = 0; p < n_; ++p)
                    if (!((plan_.bits >> p) & 1)) {
                         if (j >= kGateMaxBase) throw std::runtime_error("gate program: internal tile error");
                         pass_.base_out[j++] = new_pos_[p];
                    }
               pass_.permuted = 1;
          }
          if (pass_stages() > kGateMaxStages) throw std::runtime_error("gate program: too many stages");
          pass_.nstages = static_cast<uint8_t>(pass_stages());
          ops_.resize(ops_.size() + ob_, 0);  // the spare record
     }

private:
     using U2 = std::array<cplx, 4>;
     struct Cond {
          uint32_t rm = 0, rv = 0, tm = 0, tv = 0;
          uint64_t om = 0, ov = 0;
          bool free() const { return !tm && !om; }
     };
     struct Phase {
          Cond c;
          cplx f;
     };
     // The layer that is still open: rotations, then phases, then swaps.
     struct Layer {
          uint32_t kind[kGateMaxReg] = {};
          double p[kGateMaxReg] = {}, q[kGateMaxReg] = {};
          bool has_ph[kGateMaxReg] = {};
          cplx ph[kGateMaxReg];
          std::vector<uint8_t> swaps;
          uint32_t touched = 0;  // bits of the swaps
          uint32_t swapped = 0;  // their targets
          bool used = false;
     };

     size_t pass_stages() const { return stages_.size() - pass_.stage_first; }

     static bool holds(const std::vector<int>& reg, const int* lanes)
     {
          return std::any_of(lanes, lanes + kGateLow,
                             [&](int r) { return std::find(reg.begin(), reg.end(), r) != reg.end(); });
     }

     // Register ranks of a stage, filled up from the top ranks (that are not
     // among `avoid`).
     std::vector<int> reg_ranks(uint64_t bits, const int* avoid) const
     {
          std::vector<int> reg;
          for (uint64_t m = bits; m; m &= m - 1) {
               const int r = rank_[__builtin_ctzll(m)];
               if (r < 0) throw std::runtime_error("gate program: internal stage error");
               reg.push_back(r);
          }
          if (reg.size() > static_cast<size_t>(E_)) throw std::runtime_error("gate program: internal stage error");
          for (int r = T_ - 1; r >= 0 && reg.size() < static_cast<size_t>(E_); --r)
               if (std::find(reg.begin(), reg.end(), r) == reg.end() &&
                   !(avoid && std::find(avoid, avoid + kGateLow, r) != avoid + kGateLow))
                    reg.push_back(r);
          std::sort(reg.begin(), reg.end());
          return reg;
     }

     void begin_stage(const std::vector<int>& reg, const int* io)
     {
          lay_ = make_layout(prec_, reg, io);
          const uint32_t sb = gate_slot_bytes(prec_);
          GateStage st{};
          for (int j = 0; j < kGateThr; ++j) st.thr_lds[j] = static_cast<uint16_t>(gate_slot(prec_, lay_.thr[j]) * sb);
          for (int b = 0; b < E_; ++b) st.reg_lds[b] = static_cast<uint16_t>(gate_slot(prec_, lay_.reg[b]) * sb);
          st.op_first = static_cast<uint32_t>(ops_.size() / ob_);
          stages_.push_back(st);
          for (int p = 0; p < 64; ++p) tbit_[p] = rbit_[p] = -1;
          for (int j = 0; j < kGateThr; ++j) tbit_[pos_[lay_.thr[j]]] = j;
          for (int b = 0; b < E_; ++b) rbit_[pos_[lay_.reg[b]]] = b;
     }

     void set_io(uint8_t* thr, uint8_t* reg) const
     {
          for (int j = 0; j < kGateThr; ++j) thr[j] = static_cast<uint8_t>(pos_[lay_.thr[j]]);
          for (int b = 0; b < E_; ++b) reg[b] = static_cast<uint8_t>(pos_[lay_.reg[b]]);
     }

     Cond split(uint64_t mask, uint64_t val) const
     {
          Cond c;
          for (uint64_t m = mask; m; m &= m - 1) {
               const int p = __builtin_ctzll(m);
               const uint32_t on = static_cast<uint32_t>((val >> p) & 1);
               if (rbit_[p] >= 0) {
                    c.rm |= 1u << rbit_[p];
                    c.rv |= on << rbit_[p];
               }
               else if (tbit_[p] >= 0) {
                    c.tm |= 1u << tbit_[p];
                    c.tv |= on << tbit_[p];
               }
               else {
                    c.om |= uint64_t(1) << p;
                    c.ov |= static_cast<uint64_t>(on) << p;
               }
          }
          return c;
     }

     // ---- records ----
     void put_raw(uint32_t code, uint32_t tcond, uint64_t om, uint64_t ov, const double* c, int nc)
     {
          const size_t at = ops_.size();
          ops_.resize(at + ob_, 0);
          if (prec_ == Prec::C128) put_as<double>(at, code, tcond, om, ov, c, nc);
          else put_as<float>(at, code, tcond, om, ov, c, nc);
          ++nops_;
     }
     template <typename R>
     void put_as(size_t at, uint32_t code, uint32_t tcond, uint64_t om, uint64_t ov, const double* c, int nc)
     {
          GateOp<R> o{};
          o.code = code;
          o.tcond = tcond;
          o.omask = om;
          o.oval = ov;
          for (int i = 0; i < nc; ++i) o.c[i] = static_cast<R>(c[i]);
          std::memcpy(ops_.data() + at, &o, sizeof(o));
     }
     // An op beside the layers; it ends the open layer.
     void put(uint32_t code, const Cond& c, const cplx* u, int nu, uint32_t count = 0, uint32_t aux = 0)
     {
          close_layer();
          item(code | count << 8 | (aux | c.rm | c.rv << 5) << 16, c, u, nu);
     }
     void item(uint32_t code, const Cond& c, const cplx* u, int nu)
     {
          double v[10];
          for (int i = 0; i < nu; ++i) {
               v[2 * i] = u[i].real();
               v[2 * i + 1] = u[i].imag();
          }
          put_raw(code, c.tm | c.tv << 16, c.om, c.ov, v, 2 * nu);
     }

     void close_layer()
     {
          if (!lay.used) return;
          uint32_t aux = 0;
          bool phases = false;
          double c[10] = {}, f[10] = {};
          for (int b = 0; b < E_; ++b) {
               aux |= lay.kind[b] << (2 * b);
               c[2 * b] = lay.p[b];
               c[2 * b + 1] = lay.q[b];
               if (lay.has_ph[b]) {
                    aux |= 1u << (10 + b);
                    phases = true;
                    f[2 * b] = lay.ph[b].real();
                    f[2 * b + 1] = lay.ph[b].imag();
               }
          }
          uint64_t x[2] = {0, 0};
          for (size_t i = 0; i < lay.swaps.size(); ++i) x[i / 8] |= static_cast<uint64_t>(lay.swaps[i]) << (8 * (i % 8));
          put_raw(kGateLayer | (phases ? 1u : 0u) << 8 | aux << 16, static_cast<uint32_t>(lay.swaps.size()), x[0], x[1], c,
                  2 * E_);
          if (phases) put_raw(0, 0, 0, 0, f, 2 * E_);
          lay = Layer();
     }
     // The coefficients as the records hold them.
     double rounded(double a) const { return prec_ == Prec::C128 ? a : static_cast<double>(static_cast<float>(a)); }
     // [[1, p], [q, 1]] times p0 with p and q rounded: the factor that keeps
     // the determinant p0^2 det, so that a rotation stays one (by an angle
     // that differs by the rounding) and norms do not drift.
     double kept_scale(double p0, double det, double rounded_det) const
     {
          const double r = det / rounded_det;
          return r > 0.5 && r < 2.0 ? p0 * std::sqrt(r) : p0;
     }

     void layer_rotation(int b, uint32_t kind, double p, double q)
     {
          if (lay.kind[b] || lay.has_ph[b] || ((lay.touched >> b) & 1)) close_layer();
          lay.kind[b] = kind;
          lay.p[b] = p;
          lay.q[b] = q;
          lay.used = true;
     }
     void layer_phase(int b, const cplx& f)
     {
          if ((lay.swapped >> b) & 1) close_layer();
          lay.ph[b] = lay.has_ph[b] ? lay.ph[b] * f : f;
          lay.has_ph[b] = true;
          lay.used = true;
     }
     void layer_swap(int b, int c)
     {
          if (lay.swaps.size() == 16) close_layer();
          lay.swaps.push_back(static_cast<uint8_t>(b * 8 + c));
          lay.touched |= 1u << b | 1u << c;
          lay.swapped |= 1u << b;
          lay.used = true;
     }

     // The scale that the pass shares, kept within the range of either type.
     void scale(cplx f)
     {
          g_ *= f;
          const double a = std::abs(g_);
          if (!(a > 0x1p-40 && a < 0x1p40)) flush_scale();
     }
     void flush_scale()
     {
          if (!is_one(g_)) put(kGatePAll, Cond(), &g_, 1);
          g_ = 1.0;
     }

     static bool is_real(const U2& u)
     {
          for (const auto& z: u)
               if (z.imag() != 0.0) return false;
          return true;
     }
     // real diagonal, imaginary elsewhere (Rx)
     static bool is_cross(const U2& u)
     {
          return u[0].imag() == 0.0 && u[3].imag() == 0.0 && u[1].real() == 0.0 && u[2].real() == 0.0;
     }

     // An unconditional one-qubit gate on register bit b.
     void put_one(int b, const U2& u)
     {
          const uint32_t ub = static_cast<uint32_t>(b);
          bool fin = true;
          double big = 0;
          for (const auto& z: u) {
               fin = fin && finite(z);
               big = std::max(big, std::max(std::abs(z.real()), std::abs(z.imag())));
          }
          if (fin && u[0] == 0.0 && u[3] == 0.0 && is_one(u[1]) && is_one(u[2])) {
               put(kGateXA + ub, Cond(), nullptr, 0);
               return;
          }
          const double p = u[0].real();
          // a pivot large enough that the other coefficients stay small
          const bool pivot = fin && std::abs(p) >= 0x1p-5 * big && std::abs(p) > 0x1p-20 && std::abs(p) < 0x1p20;
          if (pivot && is_real(u)) {
               const double a = u[1].real() / p, c = u[2].real() / p, w = u[3].real();
               if (w == p || w == -p) {
                    if (w == p) {
                         layer_rotation(b, kGateKindReal, a, c);
                         scale(kept_scale(p, 1 - a * c, 1 - rounded(a) * rounded(c)));
                         return;
                    }
                    if (a == 1.0 && c == 1.0) {
                         layer_rotation(b, kGateKindH, 0, 0);
                    }
                    else {
                         const cplx ac(a, c);
                         put(kGateRM + ub, Cond(), &ac, 1);
                    }
                    scale(p);
                    return;
               }
          }
          if (pivot && is_cross(u) && u[3].real() == p) {
               const double a = u[1].imag() / p, c = u[2].imag() / p;
               layer_rotation(b, kGateKindImag, a, c);
               scale(kept_scale(p, 1 + a * c, 1 + rounded(a) * rounded(c)));
               return;
          }
          if (fin && is_real(u)) {
               const cplx r[2] = {cplx(u[0].real(), u[1].real()), cplx(u[2].real(), u[3].real())};
               put(kGateR4 + ub, Cond(), r, 2);
               return;
          }
          put(kGateG + ub, Cond(), u.data(), 4);
     }

     void flush_one(int b)
     {
          if (!has_one_[b]) return;
          has_one_[b] = false;
          put_one(b, one_[b]);
     }
     void flush_phases(int b)
     {
          put_phases(kGatePA + static_cast<uint32_t>(b), ph_[b]);
     }
     // A list of conditional factors, in as many ops as it takes; the first one
     // begins with tables of the factors that depend on the lane, on the wave or
     // on five bits of the tile number alone, when there are four or more of them.
     void put_phases(uint32_t code, std::vector<Phase>& v)
     {
          const int groups = gate_table_groups(prec_, n_);
          const uint32_t lanes = kGateTableLanes - 1;
          // the table of a condition (-1: none): its first entry, its size, and the bits and value asked there
          struct Place {
               int first = -1, size = 0;
               uint64_t m = 0, on = 0;
          };
          auto place = [&](const Cond& c) {
               Place r;
               if (!c.om && !(c.tm & ~lanes)) r = {0, kGateTableLanes, c.tm, c.tv};
               else if (!c.om && !(c.tm & lanes)) r = {kGateTableLanes, kGateTableWaves, c.tm / kGateTableLanes, c.tv / kGateTableLanes};
               else if (!c.tm) {
                    uint64_t m = 0, on = 0;
                    for (uint64_t q = c.om; q; q &= q - 1) {
                         const int p = __builtin_ctzll(q);
                         m |= uint64_t(1) << outer_[p];
                         on |= ((c.ov >> p) & 1) << outer_[p];
                    }
                    const int g = __builtin_ctzll(m) / kGateTableBits, at = g * kGateTableBits;
                    if (m >> at >> kGateTableBits == 0)
                         r = {kGateTableLanes + kGateTableWaves + (g << kGateTableBits), 1 << kGateTableBits, m >> at, on >> at};
               }
               return r;
          };
          auto tabled = [&](const Phase& p) { return place(p.c).first >= 0; };
          const bool table = std::count_if(v.begin(), v.end(), tabled) >= 4;
          std::vector<cplx> t(table ? gate_table_entries(groups) : 0, cplx(1.0, 0.0));
          if (table) {
               for (const auto& p: v) {
                    const Place r = place(p.c);
                    for (int i = 0; r.first >= 0 && i < r.size; ++i)
                         if ((static_cast<uint64_t>(i) & r.m) == r.on) t[r.first + i] *= p.f;
               }
               v.erase(std::remove_if(v.begin(), v.end(), tabled), v.end());
          }
          const uint32_t block = prec_ == Prec::C128 ? gate_table_records<double>(groups) : gate_table_records<float>(groups);
          for (size_t i = 0; i < v.size() || (table && i == 0);) {
               const bool here = table && i == 0;
               const size_t taken = here ? block : 0;
               const size_t k = std::min<size_t>(v.size() - i, kGateMaxList - taken);
               put(code, Cond(), nullptr, 0, static_cast<uint32_t>(taken + k), here ? 1u + static_cast<uint32_t>(groups) : 0u);
               if (here) {
                    const size_t at = ops_.size();
                    ops_.resize(at + taken * ob_, 0);
                    std::memcpy(ops_.data() + at, t.data(), t.size() * 16);
                    nops_ += taken;
               }
               for (size_t e = 0; e < k; ++e, ++i) {
                    const Cond& c = v[i].c;
                    put_raw(0, c.tm | c.tv << 16, c.om, c.ov, nullptr, 0);
                    const double f[2] = {v[i].f.real(), v[i].f.imag()};  // FP64 in either precision
                    std::memcpy(ops_.data() + ops_.size() - ob_ + offsetof(GateOp<float>, c), f, sizeof(f));
               }
               if (here && k == 0) break;
          }
          v.clear();
     }
     static void add_phase(std::vector<Phase>& v, const Cond& c, const cplx& f)
     {
          for (auto& e: v)
               if (e.c.tm == c.tm && e.c.tv == c.tv && e.c.om == c.om && e.c.ov == c.ov) {
                    e.f *= f;
                    return;
               }
          v.push_back(Phase{c, f});
     }

     void phase(const GateBranch& br)
     {
          if (!br.cmask) {
               scale(br.u[0]);
               return;
          }
          const Cond c = split(br.cmask, br.cval);
          for (int b = 0; b < E_; ++b)
               if ((c.rm >> b) & 1) flush_one(b);
          if (!c.rm) {
               add_phase(pl_, c, br.u[0]);
          }
          else if (popc(c.rm) == 1 && c.rv == c.rm) {
               const int b = __builtin_ctz(c.rm);
               if (c.free()) layer_phase(b, br.u[0]);
               else add_phase(ph_[b], c, br.u[0]);
          }
          else {
               put(kGatePT, c, br.u, 1);
          }
     }

     void one(const GateUnit& g)
     {
          const int b = rbit_[g.act[0]];
          if (b < 0) throw std::runtime_error("gate program: internal stage error");
          if (g.br.size() == 1 && !g.br[0].cmask) {
               const auto& v = g.br[0].u;
               const U2 u = {v[0], v[1], v[2], v[3]};
               flush_phases(b);
               if (has_one_[b]) {
                    const U2& o = one_[b];
                    // one product where it costs no more than the two gates
                    const bool plain = (is_real(o) || is_cross(o)) && (is_real(u) || is_cross(u));
                    if ((is_real(o) && is_real(u)) || (is_cross(o) && is_cross(u)) || !plain) {
                         one_[b] = {u[0] * o[0] + u[1] * o[2], u[0] * o[1] + u[1] * o[3], u[2] * o[0] + u[3] * o[2],
                                    u[2] * o[1] + u[3] * o[3]};
                         return;
                    }
                    flush_one(b);
               }
               one_[b] = u;
               has_one_[b] = true;
               return;
          }
          flush_one(b);
          flush_phases(b);
          for (const auto& br: g.br) {
               const Cond c = split(br.cmask, br.cval);
               for (int q = 0; q < E_; ++q)
                    if ((c.rm >> q) & 1) flush_one(q);
          }
          for (const auto& br: g.br) {
               const Cond c = split(br.cmask, br.cval);
               const uint32_t ub = static_cast<uint32_t>(b);
               if (br.u[0] == 0.0 && br.u[3] == 0.0 && is_one(br.u[1]) && is_one(br.u[2])) {
                    const bool single = popc(c.rm) == 1 && c.rv == c.rm;
                    Cond o = c;
                    o.rm = o.rv = 0;
                    if (single && c.free()) layer_swap(b, __builtin_ctz(c.rm));
                    else if (single) put(kGateXC, o, nullptr, 0, 0, ub * 8 + static_cast<uint32_t>(__builtin_ctz(c.rm)));
                    else if (!c.rm) put(kGateXA + ub, c, nullptr, 0);
                    else put(kGateX + ub, c, nullptr, 0);
               }
               else {
                    put(kGateG + ub, c, br.u, 4);
               }
          }
     }

     void two(const GateUnit& g)
     {
          int b0 = rbit_[g.act[0]], b1 = rbit_[g.act[1]];
          if (b0 < 0 || b1 < 0) throw std::runtime_error("gate program: internal stage error");
          const bool swapped = b0 > b1;
          for (int b: {b0, b1}) {
               flush_one(b);
               flush_phases(b);
          }
          if (swapped) std::swap(b0, b1);
          for (const auto& br: g.br) {
               const Cond c = split(br.cmask, br.cval);
               for (int q = 0; q < E_; ++q)
                    if ((c.rm >> q) & 1) flush_one(q);
               put(kGateG2 + gate_pair(b0, b1), c, nullptr, 0, 4);
               auto at = [&](int i) { return swapped ? ((i & 1) << 1) | (i >> 1) : i; };
               for (int r = 0; r < 4; ++r) {
                    cplx row[4];
                    for (int k = 0; k < 4; ++k) row[k] = br.u[at(r) * 4 + at(k)];
                    item(0, Cond(), row, 4);
               }
          }
     }

     void emit_stage(const std::vector<int>& list, bool last)
     {
          nops_ = 0;
          for (int i: list) {
               const GateUnit& g = units_[i];
               if (g.na == 0)
                    for (const auto& br: g.br) phase(br);
               else if (g.na == 1) one(g);
               else two(g);
          }
          for (int b = 0; b < E_; ++b) flush_one(b);
          for (int b = 0; b < E_; ++b) flush_phases(b);
          put_phases(kGatePL, pl_);
          if (last) flush_scale();
          close_layer();
          if (nops_ > 0xffffu) throw std::runtime_error("gate program: too many gates in one stage");
          stages_.back().nops = static_cast<uint16_t>(nops_);
     }

     const std::vector<GateUnit>& units_;
     const GatePassPlan& plan_;
     const Prec prec_;
     const int E_, T_;
     const size_t ob_;
     GatePass& pass_;
     std::vector<GateStage>& stages_;
     std::vector<char>& ops_;
     int rank_[64], pos_[kGateMaxTile];
     int in_lanes_[kGateLow], out_lanes_[kGateLow];  // ranks of the load's and the store's runs
     uint8_t new_pos_[64] = {};                      // of an index bit, after the permutation
     int outer_[64];  // an index bit's place in the tile number
     bool permuted_ = false;
     int n_ = 0;
     int tbit_[64], rbit_[64];
     Layout lay_{};
     size_t nops_ = 0;
     cplx g_ = 1.0;  // factor of every amplitude still to be applied
     U2 one_[kGateMaxReg];  // one-qubit gates still to be emitted
     bool has_one_[kGateMaxReg] = {};
     std::vector<Phase> ph_[kGateMaxReg], pl_;  // conditional factors still to be emitted
     Layer lay;
};

}  // namespace

void compile_gate_pass(const std::vector<GateUnit>& units, const GatePassPlan& plan, int n, Prec prec, GatePass& pass,
                       std::vector<GateStage>& stages, std::vector<char>& ops, const uint8_t* src_pos)
{
     Compiler(units, plan, n, prec, pass, stages, ops, src_pos).run();
}

bool split_gate_pass(GatePassPlan& plan, GatePassPlan& second)
{
     second = GatePassPlan();
     second.bits = plan.bits;
     if (plan.stages.size() > 1) {
          const size_t half = plan.stages.size() / 2;
          second.regs.assign(plan.regs.begin() + static_cast<long>(half), plan.regs.end());
          second.stages.assign(plan.stages.begin() + static_cast<long>(half), plan.stages.end());
          plan.regs.resize(half);
          plan.stages.resize(half);
          return true;
     }
     std::vector<int>& only = plan.stages.at(0);
     if (only.size() < 2) return false;
     const auto half = only.begin() + static_cast<long>(only.size() / 2);
     second.regs = plan.regs;
     second.stages.emplace_back(half, only.end());
     only.erase(half, only.end());
     return true;
}

bool widen_for_permutation(const std::vector<GateUnit>& units, GatePassPlan& plan, int n, Prec prec,
                           const uint8_t* src_pos)
{
     uint64_t bits = (uint64_t(1) << kGateLow) - 1;
     for (const auto& st: plan.stages)
          for (int i: st) bits |= units[i].a;
     for (int q = 0; q < kGateLow; ++q) bits |= uint64_t(1) << src_pos[q];
     const int T = gate_tile_bits(prec);
     if (popc(bits) > T) return false;
     for (uint64_t m = plan.bits & ~bits; m && popc(bits) < T; m &= m - 1) bits |= low_bit(m);
     for (int p = 0; p < n && popc(bits) < T; ++p) bits |= uint64_t(1) << p;
     plan.bits = bits;
     return true;
}

void check_gate_pass(const GatePass& pass, const std::vector<GateStage>& stages, const std::vector<char>& ops,
                     Prec prec, int n)
{
     auto fail = [] { throw std::runtime_error("gate program: internal bounds check failed"); };
     const int E = gate_reg(prec), T = gate_tile_bits(prec);
     const uint32_t sb = gate_slot_bytes(prec);
     const size_t ob = gate_op_bytes(prec), nrec = ops.size() / ob;
     if (n < T || n > 40 || pass.nstages < 1 || pass.stage_first + size_t(pass.nstages) > stages.size()) fail();
     uint64_t bits = (uint64_t(1) << kGateLow) - 1;
     for (int j = 0; j < T - kGateLow; ++j) {
          if (pass.hpos[j] < kGateLow || pass.hpos[j] >= n || (j && pass.hpos[j] <= pass.hpos[j - 1])) fail();
          bits |= uint64_t(1) << pass.hpos[j];
     }
     for (int io = 0; io < 2; ++io) {
          const uint8_t* thr = io ? pass.out_thr : pass.in_thr;
          const uint8_t* reg = io ? pass.out_reg : pass.in_reg;
          uint64_t got = 0;
          for (int j = 0; j < kGateThr; ++j) got |= uint64_t(1) << thr[j];
          for (int b = 0; b < E; ++b) got |= uint64_t(1) << reg[b];
          uint64_t want = bits;
          if (io && pass.permuted) {  // every bit of the new index once
               if (n - T > kGateMaxBase) fail();
               for (int j = 0; j < n - T; ++j) got |= uint64_t(1) << pass.base_out[j];
               want = (uint64_t(1) << n) - 1;
          }
          if (got != want) fail();
     }
     for (int s = 0; s < pass.nstages; ++s) {
          const GateStage& st = stages[pass.stage_first + s];
          // the offsets are a basis of the 2^T slots: rank over GF(2)
          uint32_t basis[kGateMaxTile] = {};
          int rank = 0;
          for (int i = 0; i < T; ++i) {
               const uint32_t byte = i < kGateThr ? st.thr_lds[i] : st.reg_lds[i - kGateThr];
               if (byte % sb) fail();
               uint32_t v = byte / sb;
               if (v >> T) fail();
               for (int b = T - 1; b >= 0 && v; --b)
                    if ((v >> b) & 1) {
                         if (!basis[b]) {
                              basis[b] = v;
                              ++rank;
                              break;
                         }
                         v ^= basis[b];
                    }
          }
          if (rank != T) fail();
          if (st.op_first + size_t(st.nops) + 1 > nrec) fail();  // and the record read ahead
          // lists end inside their stage
          for (size_t p = 0; p < st.nops;) {
               uint32_t w, tc;
               std::memcpy(&w, ops.data() + (st.op_first + p) * ob, 4);
               std::memcpy(&tc, ops.data() + (st.op_first + p) * ob + 4, 4);
               if ((w & 0xff) >= kGateCodes || ((w & 0xff) == kGateLayer && tc > 16)) fail();
               const uint32_t code = w & 0xff, count = (w >> 8) & 0xff;
               if (code >= kGatePA && code < kGateG2 && (w >> 16)) {
                    const int g = static_cast<int>(w >> 16) - 1;
                    if (g != gate_table_groups(prec, n)) fail();
                    if (count < (prec == Prec::C128 ? gate_table_records<double>(g) : gate_table_records<float>(g))) fail();
               }
               p += 1 + count;
               if (p > st.nops) fail();
          }
     }
}

}  // namespace hq
