// Host-only run of the gate programs, built with AddressSanitizer and
// UndefinedBehaviorSanitizer: random gate lists are split into units, planned
// and compiled, the records are checked, and a plain interpreter of the
// records (tile by tile, thread by thread, with the regrouping through a
// slot array) must leave the state that applying the gates one by one does.
// The lists hold every form that the compiler tells apart: real and imaginary
// rotations, Hadamards, general and non-unitary matrices, zero pivots,
// phases, diagonals on several qubits, controls on register, thread and outer
// bits, controlled and plain swaps, two-qubit gates in either bit order,
// block-diagonal matrices, identities and long runs on few qubits.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "../../hiqsimulator_amd/csrc/gate_prog.hpp"

#define CHECK(c)                                                                   \
     do {                                                                          \
          if (!(c)) {                                                              \
               std::fprintf(stderr, "check failed line %d: %s\n", __LINE__, #c);   \
               std::exit(1);                                                       \
          }                                                                        \
     } while (0)

namespace {

using namespace hq;
using cplx = std::complex<double>;
using State = std::vector<cplx>;

struct Gate {
     std::vector<cplx> m;
     std::vector<int64_t> t, c;
};

void apply(State& psi, const Gate& g)
{
     const int k = static_cast<int>(g.t.size());
     const size_t D = size_t(1) << k;
     uint64_t cm = 0, tm = 0;
     for (auto p: g.c) cm |= uint64_t(1) << p;
     for (auto p: g.t) tm |= uint64_t(1) << p;
     std::vector<cplx> v(D);
     for (uint64_t i = 0; i < psi.size(); ++i) {
          if ((i & tm) || (i & cm) != cm) continue;
          auto at = [&](size_t j) {
               uint64_t o = i;
               for (int l = 0; l < k; ++l)
                    if ((j >> l) & 1) o |= uint64_t(1) << g.t[l];
               return o;
          };
          for (size_t j = 0; j < D; ++j) v[j] = psi[at(j)];
          for (size_t r = 0; r < D; ++r) {
               cplx s = 0;
               for (size_t j = 0; j < D; ++j) s += g.m[r * D + j] * v[j];
               psi[at(r)] = s;
          }
     }
}

template <typename R>
cplx factor(const GateOp<R>* o, uint32_t count, uint64_t base, uint64_t tix, uint32_t tid, uint32_t tables)
{
     cplx f = 1;
     if (tables) {  // products by lane, by wave and by five bits of the tile number, in the place of records
          const uint32_t skip = gate_table_records<R>(static_cast<int>(tables) - 1);
          CHECK(count >= skip);
          std::vector<double> t(2 * gate_table_entries(static_cast<int>(tables) - 1));
          std::memcpy(t.data(), o, t.size() * sizeof(double));
          auto at = [&](size_t i) { return cplx(t[2 * i], t[2 * i + 1]); };
          f *= at(tid % kGateTableLanes) * at(kGateTableLanes + tid / kGateTableLanes);
          for (uint32_t g = 1; g < tables; ++g)
               f *= at(kGateTableLanes + kGateTableWaves + ((g - 1) << kGateTableBits) +
                       ((tix >> ((g - 1) * kGateTableBits)) & ((1u << kGateTableBits) - 1)));
          o += skip;
          count -= skip;
     }
     for (uint32_t e = 0; e < count; ++e)
          if ((base & o[e].omask) == o[e].oval && (tid & (o[e].tcond & 0xffff)) == (o[e].tcond >> 16)) {
               double u[2];
               std::memcpy(u, o[e].c, sizeof(u));
               f *= cplx(u[0], u[1]);
          }
     return f;
}

// One pass as the kernel runs it, in double.
template <typename R>
void interpret(State& psi, int n, const GatePass& P, const std::vector<GateStage>& stages, const std::vector<char>& ob)
{
     constexpr Prec prec = sizeof(R) == 8 ? Prec::C128 : Prec::C64;
     constexpr int E = gate_reg(prec), T = gate_tile_bits(prec);
     constexpr uint32_t A = 1u << E;
     std::vector<GateOp<R>> ops(ob.size() / sizeof(GateOp<R>));
     std::memcpy(ops.data(), ob.data(), ob.size());
     auto bits = [](uint32_t v, const uint8_t* pos, int cnt) {
          uint64_t i = 0;
          for (int j = 0; j < cnt; ++j) i |= static_cast<uint64_t>((v >> j) & 1) << pos[j];
          return i;
     };
     auto slot = [](uint32_t v, const uint16_t* m, int cnt) {
          uint32_t s = 0;
          for (int j = 0; j < cnt; ++j)
               if ((v >> j) & 1) s ^= m[j];
          return s / gate_slot_bytes(prec);
     };
     std::vector<cplx> x(size_t(kGateThreads) * A), lds(size_t(1) << T);
     State other(P.permuted ? psi.size() : 0, cplx(NAN, NAN));  // where a permuted pass stores
     for (uint64_t tix = 0; tix < (uint64_t(1) << (n - T)); ++tix) {
          uint64_t base = tix << kGateLow;
          for (int j = 0; j < T - kGateLow; ++j) {
               const uint64_t lo = base & ((uint64_t(1) << P.hpos[j]) - 1);
               base = ((base ^ lo) << 1) | lo;
          }
          for (uint32_t t = 0; t < kGateThreads; ++t)
               for (uint32_t k = 0; k < A; ++k) x[t * A + k] = psi.at(base + bits(t, P.in_thr, kGateThr) + bits(k, P.in_reg, E));
          for (int s = 0; s < P.nstages; ++s) {
               const GateStage& st = stages.at(P.stage_first + s);
               if (s) {
                    const GateStage& pv = stages.at(P.stage_first + s - 1);
                    for (uint32_t t = 0; t < kGateThreads; ++t)
                         for (uint32_t k = 0; k < A; ++k) lds.at(slot(t, pv.thr_lds, kGateThr) ^ slot(k, pv.reg_lds, E)) = x[t * A + k];
                    for (uint32_t t = 0; t < kGateThreads; ++t)
                         for (uint32_t k = 0; k < A; ++k) x[t * A + k] = lds.at(slot(t, st.thr_lds, kGateThr) ^ slot(k, st.reg_lds, E));
               }
               for (uint32_t t = 0; t < kGateThreads; ++t) {
                    cplx* v = &x[t * A];
                    auto pairs = [&](int b, auto&& f) {
                         for (uint32_t k = 0; k < A; ++k)
                              if (!((k >> b) & 1)) f(v[k], v[k | (1u << b)], k);
                    };
                    auto swap_if = [&](int b, uint32_t rm, uint32_t rv) {
                         pairs(b, [&](cplx& a, cplx& z, uint32_t k) {
                              if ((k & rm) == rv) std::swap(a, z);
                         });
                    };
                    for (size_t p = 0; p < st.nops;) {
                         const GateOp<R>& o = ops.at(st.op_first + p);
                         const uint32_t code = o.code & 0xff, count = (o.code >> 8) & 0xff, aux = o.code >> 16;
                         const uint32_t rm = aux & 31, rv = (aux >> 5) & 31;
                         const GateOp<R>* list = &ops.at(st.op_first + p + 1);
                         p += 1 + count;
                         if (code == kGateLayer) {
                              for (int b = 0; b < E; ++b) {
                                   const uint32_t kind = (aux >> (2 * b)) & 3;
                                   const double c0 = o.c[2 * b], c1 = o.c[2 * b + 1];
                                   pairs(b, [&](cplx& a, cplx& z, uint32_t) {
                                        const cplx a0 = a, z0 = z;
                                        if (kind == kGateKindReal) a = a0 + c0 * z0, z = z0 + c1 * a0;
                                        if (kind == kGateKindH) a = a0 + z0, z = a0 - z0;
                                        if (kind == kGateKindImag) a = a0 + cplx(0, c0) * z0, z = z0 + cplx(0, c1) * a0;
                                   });
                              }
                              for (int b = 0; b < E; ++b)
                                   if ((aux >> (10 + b)) & 1)
                                        for (uint32_t k = 0; k < A; ++k)
                                             if ((k >> b) & 1) v[k] *= cplx(list->c[2 * b], list->c[2 * b + 1]);
                              for (uint32_t i = 0; i < o.tcond; ++i) {
                                   const uint32_t by = ((i < 8 ? o.omask : o.oval) >> (8 * (i % 8))) & 0xff;
                                   CHECK(by / 8 != by % 8 && by / 8 < uint32_t(E) && by % 8 < uint32_t(E));
                                   swap_if(by / 8, 1u << (by % 8), 1u << (by % 8));
                              }
                              continue;
                         }
                         if ((base & o.omask) != o.oval || (t & (o.tcond & 0xffff)) != (o.tcond >> 16)) continue;
                         const cplx c0(o.c[0], o.c[1]), c1(o.c[2], o.c[3]), c2(o.c[4], o.c[5]), c3(o.c[6], o.c[7]);
                         if (code < kGateR4) {
                              pairs(code - kGateRM, [&](cplx& a, cplx& z, uint32_t) {
                                   const cplx a0 = a, z0 = z;
                                   a = a0 + c0.real() * z0, z = -z0 + c0.imag() * a0;
                              });
                         }
                         else if (code < kGateG) {
                              pairs(code - kGateR4, [&](cplx& a, cplx& z, uint32_t) {
                                   const cplx a0 = a, z0 = z;
                                   a = c0.real() * a0 + c0.imag() * z0, z = c1.real() * a0 + c1.imag() * z0;
                              });
                         }
                         else if (code < kGateXA) {
                              pairs(code - kGateG, [&](cplx& a, cplx& z, uint32_t k) {
                                   const cplx a0 = a, z0 = z;
                                   if ((k & rm) == rv) a = c0 * a0 + c1 * z0, z = c2 * a0 + c3 * z0;
                              });
                         }
                         else if (code < kGateX) {
                              swap_if(code - kGateXA, 0, 0);
                         }
                         else if (code < kGateXC) {
                              swap_if(code - kGateX, rm, rv);
                         }
                         else if (code == kGateXC) {
                              CHECK(aux / 8 != aux % 8 && aux / 8 < uint32_t(E) && aux % 8 < uint32_t(E));
                              swap_if(aux / 8, 1u << (aux % 8), 1u << (aux % 8));
                         }
                         else if (code < kGateG2) {
                              cplx f = c0;
                              if (code >= kGatePA) f = factor(list, count, base, tix, t, aux);
                              for (uint32_t k = 0; k < A; ++k) {
                                   bool on = true;
                                   if (code == kGatePT) on = (k & rm) == rv;
                                   else if (code >= kGatePA && code < kGatePL) on = (k >> (code - kGatePA)) & 1;
                                   if (on) v[k] *= f;
                              }
                         }
                         else {
                              CHECK(count == 4 && code < kGateCodes);
                              for (int b1 = 1; b1 < E; ++b1)
                                   for (int b0 = 0; b0 < b1; ++b0) {
                                        if (gate_pair(b0, b1) != code - kGateG2) continue;
                                        for (uint32_t k = 0; k < A; ++k) {
                                             if (((k >> b0) & 1) || ((k >> b1) & 1) || (k & rm) != rv) continue;
                                             const uint32_t at[4] = {k, k | 1u << b0, k | 1u << b1, k | 1u << b0 | 1u << b1};
                                             cplx w[4];
                                             for (int q = 0; q < 4; ++q) w[q] = v[at[q]];
                                             for (int r = 0; r < 4; ++r) {
                                                  cplx sum = 0;
                                                  for (int q = 0; q < 4; ++q) sum += cplx(list[r].c[2 * q], list[r].c[2 * q + 1]) * w[q];
                                                  v[at[r]] = sum;
                                             }
                                        }
                                   }
                         }
                    }
               }
          }
          const uint64_t to = P.permuted ? bits(static_cast<uint32_t>(tix), P.base_out, n - T) : base;
          for (uint32_t t = 0; t < kGateThreads; ++t)
               for (uint32_t k = 0; k < A; ++k)
                    (P.permuted ? other : psi).at(to + bits(t, P.out_thr, kGateThr) + bits(k, P.out_reg, E)) = x[t * A + k];
          // runs of 16 amplitudes are loaded and stored by 16 lanes
          for (int j = 0; j < kGateLow; ++j) CHECK(P.in_thr[j] == j && P.out_thr[j] == j);
     }
     if (P.permuted) psi.swap(other);
}

struct Maker {
     std::mt19937 rng;
     int n;
     double u(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
     std::vector<int64_t> qubits(int k, int span)
     {
          std::vector<int64_t> q(span);
          for (int i = 0; i < span; ++i) q[i] = (i + first) % n;
          std::shuffle(q.begin(), q.end(), rng);
          q.resize(k);
          return q;
     }
     int first = 0;
     std::vector<cplx> random(int d)
     {
          std::vector<cplx> m(d * d);
          for (auto& z: m) z = cplx(u(-1, 1), u(-1, 1)) / std::sqrt(double(d));
          return m;
     }
     Gate gate(int span)
     {
          Gate g;
          const double th = u(0, 6.3), c = std::cos(th), s = std::sin(th);
          const int kind = static_cast<int>(rng() % 20);
          const int nc = rng() % 3 ? 0 : 1 + static_cast<int>(rng() % 2);
          int k = 1;
          switch (kind) {
               case 0: g.m = {M_SQRT1_2, M_SQRT1_2, M_SQRT1_2, -M_SQRT1_2}; break;
               case 1: g.m = {c, cplx(0, -s), cplx(0, -s), c}; break;
               case 2: g.m = {c, -s, s, c}; break;
               case 3: g.m = {std::polar(1.0, -th), 0, 0, std::polar(1.0, th)}; break;
               case 4: g.m = {1, 0, 0, std::polar(1.0, th)}; break;
               case 5: g.m = {0, 1, 1, 0}; break;
               case 6: g.m = {0, cplx(0, -1), cplx(0, 1), 0}; break;
               case 7: g.m = random(2); break;
               case 8: g.m = {1, 0, 0, 0}; break;                       // projector
               case 9: g.m = {1e-9, 1, -1, 1e-9}; break;                // tiny pivot
               case 10: g.m = {2, 1, 1, -3}; break;                     // real, no rotation
               case 11: g.m = {1, 0, 0, 1}; break;                      // identity
               case 12: g.m = {1, 0, 0, 0, 0, 0, 0, 1, 0, 0, 1, 0, 0, 1, 0, 0}, k = 2; break;  // cyclic permutation
               case 13: g.m = {1, 0, 0, 0, 0, 0, 1, 0, 0, 1, 0, 0, 0, 0, 0, 1}, k = 2; break;  // swap
               case 14: g.m = random(4), k = 2; break;
               case 15: {  // controlled U as a plain matrix, either bit first
                    const auto v = random(2);
                    g.m.assign(16, 0);
                    k = 2;
                    const bool hi = rng() & 1;
                    for (int i = 0; i < 2; ++i) g.m[hi ? i * 4 + i : 2 * i * 4 + 2 * i] = 1;
                    for (int i = 0; i < 2; ++i)
                         for (int j = 0; j < 2; ++j) g.m[hi ? (2 + i) * 4 + 2 + j : (2 * i + 1) * 4 + 2 * j + 1] = v[i * 2 + j];
                    break;
               }
               case 16: {  // diagonal on three qubits, one entry one
                    k = 3;
                    g.m.assign(64, 0);
                    for (int i = 0; i < 8; ++i) g.m[i * 9] = i == 5 ? cplx(1) : std::polar(rng() % 4 ? 1.0 : 0.3, u(0, 6));
                    break;
               }
               case 17: {  // multiplexed: both blocks act
                    const auto a = random(2), b = random(2);
                    k = 2;
                    g.m = {a[0], a[1], 0, 0, a[2], a[3], 0, 0, 0, 0, b[0], b[1], 0, 0, b[2], b[3]};
                    break;
               }
               case 18: {  // the same block twice
                    const auto a = random(2);
                    k = 2;
                    g.m = {a[0], a[1], 0, 0, a[2], a[3], 0, 0, 0, 0, a[0], a[1], 0, 0, a[2], a[3]};
                    break;
               }
               default: {  // block diagonal in one of three qubits
                    k = 3;
                    const auto a = random(4);
                    g.m.assign(64, 0);
                    for (int i = 0; i < 4; ++i)
                         for (int j = 0; j < 4; ++j) g.m[(2 * i) * 8 + 2 * j] = a[i * 4 + j];
                    for (int i = 0; i < 4; ++i) g.m[(2 * i + 1) * 8 + 2 * i + 1] = 1;
               }
          }
          const auto q = qubits(std::min(span, k + nc), span);
          g.t.assign(q.begin(), q.begin() + k);
          g.c.assign(q.begin() + k, q.end());
          return g;
     }
};

// permute: the last pass also takes the bits of the index to other places, if
// it can; returns whether it did.
// Controlled phases between all pairs of a register whose qubits come in
// rotated order, with Hadamards: lists of many factors.
struct Qft {
     int n, turn;
     std::vector<Gate> gates() const
     {
          std::vector<Gate> out;
          const double r = std::sqrt(0.5);
          for (int j = n - 1; j >= 0; --j) {
               const int q = (j + turn) % n;
               out.push_back({{r, r, r, -r}, {q}, {}});
               for (int m = j - 1; m >= 0; --m)
                    out.push_back({{1, 0, 0, std::polar(1.0, 2 * 3.14159265358979323846 / double(uint64_t(1) << (j - m + 1)))}, {q}, {(m + turn) % n}});
          }
          return out;
     }
};

bool run_case(int n, int ngates, int span, int first, Prec prec, unsigned seed, size_t min_passes = 1,
              bool permute = false, int qft_turn = -1, bool splits = false)
{
     Maker mk{std::mt19937(seed), n};
     mk.first = first;
     std::vector<Gate> gates = qft_turn >= 0 ? Qft{n, qft_turn}.gates() : std::vector<Gate>();
     if (qft_turn >= 0) ngates = static_cast<int>(gates.size());
     else
          for (int i = 0; i < ngates; ++i) gates.push_back(mk.gate(span));
     std::vector<GateUnit> units;
     for (const Gate& g: gates) {
          GateUnit u;
          CHECK(make_gate_unit(g.m.data(), g.t, g.c, u));
          units.push_back(u);
     }
     State psi(size_t(1) << n), ref;
     for (auto& z: psi) z = cplx(mk.u(-1, 1), mk.u(-1, 1));
     ref = psi;
     for (const auto& g: gates) apply(ref, g);
     GatePassPlanner planner(units, n, prec, splits);
     GatePassPlan plan;
     std::vector<GateStage> stages;
     std::vector<char> ops;
     std::vector<GatePass> passes;
     std::vector<int> seen(units.size(), 0);
     std::vector<uint8_t> src_pos;
     bool permuted = false;
     if (permute) {
          for (int q: mk.qubits(n, n)) src_pos.push_back(static_cast<uint8_t>(q));
          CHECK(src_pos.size() == static_cast<size_t>(n));
     }
     while (planner.next(plan)) {
          const uint64_t tile = plan.bits;
          permuted = permute && planner.remaining().empty() && widen_for_permutation(units, plan, n, prec, src_pos.data());
          if (!permuted) CHECK(plan.bits == tile);
          for (size_t s = 0; s < plan.stages.size(); ++s) {
               CHECK(!(plan.regs[s] & ~plan.bits));
               for (int i: plan.stages[s]) ++seen[i];
          }
          GatePass p;
          compile_gate_pass(units, plan, n, prec, p, stages, ops, permuted ? src_pos.data() : nullptr);
          passes.push_back(p);
     }
     if (permuted) {
          State moved(ref.size());
          for (uint64_t i = 0; i < ref.size(); ++i) {
               uint64_t from = 0;
               for (int p = 0; p < n; ++p) from |= ((i >> p) & 1) << src_pos[p];
               moved[i] = ref[from];
          }
          ref.swap(moved);
     }
     for (int c: seen) CHECK(c == 1);
     CHECK(passes.size() >= min_passes);
     for (const auto& p: passes) {
          check_gate_pass(p, stages, ops, prec, n);
          if (prec == Prec::C128) interpret<double>(psi, n, p, stages, ops);
          else interpret<float>(psi, n, p, stages, ops);
     }
     double err = 0, norm = 0;
     for (size_t i = 0; i < psi.size(); ++i) {
          err = std::max(err, std::abs(psi[i] - ref[i]));
          norm = std::max(norm, std::abs(ref[i]));
     }
     // a gate rounds each amplitude a few times, relative to the largest of
     // its pair: 8 eps a gate, of the coefficients' type
     const double eps = prec == Prec::C128 ? 0x1p-52 : 0x1p-23;
     if (!(err <= 8 * eps * ngates * norm + 1e-300)) {
          std::fprintf(stderr, "n=%d gates=%d span=%d prec=%d seed=%u: err %.3e norm %.3e\n", n, ngates, span,
                       static_cast<int>(prec), seed, err, norm);
          std::exit(1);
     }
     return permuted;
}

}  // namespace

int main()
{
     unsigned seed = 1;
     for (Prec prec: {Prec::C128, Prec::C64}) {
          for (int n: {gate_tile_bits(prec), gate_tile_bits(prec) + 1, 16}) {
               run_case(n, 1, n, 0, prec, seed++);
               run_case(n, 7, n, 0, prec, seed++);
               for (int r = 0; r < 6; ++r) run_case(n, 40 + 7 * r, n, 0, prec, seed++);
               for (int f: {0, 4, n - 5}) run_case(n, 60, 5, f, prec, seed++);  // few qubits: long stages
          }
          run_case(18, 80, 18, 0, prec, seed++, 2);
     }
     // long lists: tables and records
     for (Prec prec: {Prec::C128, Prec::C64})
          for (int n: {gate_tile_bits(prec), 16, 18})
               for (int turn: {0, 5, n - 3}) {
                    run_case(n, 0, n, 0, prec, seed++, 1, false, turn);
               }
     // the best of four ways to split a pass into stages
     for (Prec prec: {Prec::C128, Prec::C64})
          for (int n: {gate_tile_bits(prec), 16}) {
               for (int r = 0; r < 4; ++r) run_case(n, 1 + 24 * r, n, 0, prec, seed++, 1, r == 2, -1, true);
               run_case(n, 60, 5, 0, prec, seed++, 1, false, -1, true);
               run_case(n, 0, n, 0, prec, seed++, 1, false, 3, true);
          }
     // the last pass permutes
     seed = 1000;
     for (Prec prec: {Prec::C128, Prec::C64}) {
          const int T = gate_tile_bits(prec);
          for (int r = 0; r < 8; ++r) CHECK(run_case(T, 1 + 9 * r, T, 0, prec, seed++, 1, true));  // one tile: always
          int did = 0;
          for (int n: {T + 1, 17, 18})
               for (int r = 0; r < 8; ++r) did += run_case(n, 1 + 12 * r, n, 0, prec, seed++, 1, true);
          for (int f: {0, 4, 12}) did += run_case(17, 60, 5, f, prec, seed++, 1, true);
          CHECK(did >= 8 && did < 27);  // both outcomes
     }
     // more gates than one stage or one pass holds
     {
          std::vector<GateUnit> units;
          std::vector<Gate> gates;
          for (int i = 0; i < 2000; ++i) {
               Gate g;
               const double th = 0.01 * i;
               g.m = {std::cos(th), -std::sin(th), std::sin(th), std::cos(th)};
               g.t = {i % 13};
               g.c = {(i + 12) % 13};  // controlled by the last target: a serial chain
               GateUnit u;
               CHECK(make_gate_unit(g.m.data(), g.t, g.c, u));
               units.push_back(u);
               gates.push_back(g);
          }
          GatePassPlanner planner(units, 13, Prec::C128);
          GatePassPlan plan;
          State psi(size_t(1) << 13, cplx(0.01, -0.02)), ref = psi;
          psi[5] = ref[5] = 1;
          for (const auto& g: gates) apply(ref, g);
          int np = 0;
          while (planner.next(plan)) {
               GatePass p;
               std::vector<GateStage> stages;
               std::vector<char> ops;
               CHECK(plan.stages.size() <= kGateMaxStages - 2);
               compile_gate_pass(units, plan, 13, Prec::C128, p, stages, ops);
               check_gate_pass(p, stages, ops, Prec::C128, 13);
               interpret<double>(psi, 13, p, stages, ops);
               ++np;
          }
          CHECK(np > 1);
          for (size_t i = 0; i < psi.size(); ++i) CHECK(std::abs(psi[i] - ref[i]) < 1e-10);
     }
     // what is not taken: three mixed bits, repeated or negative positions
     {
          GateUnit u;
          std::vector<cplx> m(64);
          for (int i = 0; i < 8; ++i) m[i * 8 + (7 - i)] = 1;
          CHECK(!make_gate_unit(m.data(), {0, 1, 2}, {}, u));
          std::vector<cplx> x = {0, 1, 1, 0};
          CHECK(!make_gate_unit(x.data(), {3}, {3}, u));
          CHECK(!make_gate_unit(x.data(), {-1}, {}, u));
          std::vector<GateUnit> far(1);
          far[0].a = 1ull << 20;
          bool threw = false;
          try {
               GatePassPlanner p(far, 14, Prec::C64);
          } catch (const std::runtime_error&) {
               threw = true;
          }
          CHECK(threw);
     }
     std::printf("gate programs ok\n");
     return 0;
}
