// Host run of the engine's gate lists over a stand-in for the HIP runtime, with
// an allocation or a launch that fails: whatever was applied has left the
// queue, and what was not is still there, so that a caller who goes on gets
// every gate once.  Lists through apply_tiled allocate before their first pass.
#define main gate_prog_main
#include "gate_prog_test.cpp"
#undef main

#include "../../hiqsimulator_amd/csrc/engine.hpp"
#include "fake_hip.hpp"

namespace hq {

long passes_run = 0, fail_launch = -1;  // passes until one fails
long allocations_at_first_pass = 0;

hipError_t launch_gate_pass(void* psi, Prec prec, Prec held, int n, const GatePass& pass, const GateStage* stages, const void* ops,
                            hipStream_t, void* dst)
{
     CHECK(prec == Prec::C128 && held == Prec::C128);
     if (fail_launch >= 0 && fail_launch-- == 0) return hipErrorLaunchFailure;
     if (passes_run++ == 0) allocations_at_first_pass = fake::allocations;
     auto* const p = static_cast<cplx*>(psi);
     State s(p, p + (size_t(1) << n));
     std::vector<GateStage> st(stages, stages + pass.stage_first + pass.nstages);
     size_t nrec = 0;
     for (const auto& x: st) nrec = std::max<size_t>(nrec, x.op_first + size_t(x.nops) + 1);
     const char* const o = static_cast<const char*>(ops);
     interpret<double>(s, n, pass, st, std::vector<char>(o, o + nrec * gate_op_bytes(prec)));
     std::copy(s.begin(), s.end(), static_cast<cplx*>(dst));
     return hipSuccess;
}
hipError_t init_reduce_scratch(double*, hipStream_t) { return hipSuccess; }
hipError_t launch_fill(void* psi, Prec, uint64_t n, double re, double im, hipStream_t)
{
     std::fill_n(static_cast<cplx*>(psi), n, cplx(re, im));
     return hipSuccess;
}
hipError_t launch_copy(void* dst, const void* src, Prec, uint64_t n, hipStream_t)
{
     std::copy_n(static_cast<const cplx*>(src), n, static_cast<cplx*>(dst));
     return hipSuccess;
}
hipError_t launch_permute(void* dst, const void* src, Prec, int n, const uint8_t* src_pos, hipStream_t)
{
     for (uint64_t j = 0; j < uint64_t(1) << n; ++j) {
          uint64_t i = 0;
          for (int p = 0; p < n; ++p) i |= ((j >> p) & 1) << src_pos[p];
          static_cast<cplx*>(dst)[j] = static_cast<const cplx*>(src)[i];
     }
     return hipSuccess;
}
Readback::~Readback() {}
void Readback::read(const void* psi, Prec, uint64_t n, std::complex<double>* out, hipStream_t)
{
     std::copy_n(static_cast<const cplx*>(psi), n, out);
}

}  // namespace hq

namespace {

std::vector<int64_t> iota(int n)
{
     std::vector<int64_t> v(n);
     for (int i = 0; i < n; ++i) v[i] = i;
     return v;
}
Mat mat_of(const Gate& g)
{
     Mat m;
     m.dim = size_t(1) << g.t.size();
     m.a = g.m;
     return m;
}
// Gates of a state that keep its norm near one.
std::vector<Gate> list(int n, int count, unsigned seed)
{
     Maker mk{std::mt19937(seed), n};
     std::vector<Gate> out;
     while (static_cast<int>(out.size()) < count) {
          Gate g = mk.gate(n);
          bool unitary = true;
          const size_t D = size_t(1) << g.t.size();
          for (size_t i = 0; i < D; ++i)
               for (size_t j = 0; j < D; ++j) {
                    cplx s = 0;
                    for (size_t k = 0; k < D; ++k) s += g.m[i * D + k] * std::conj(g.m[j * D + k]);
                    unitary = unitary && std::abs(s - (i == j ? 1.0 : 0.0)) < 1e-9;
               }
          if (unitary) out.push_back(g);
     }
     return out;
}
State applied(int n, const std::vector<Gate>& gates)
{
     State s(size_t(1) << n);
     s[0] = 1;
     for (const auto& g: gates) apply(s, g);
     return s;
}
State permuted(const State& s, const std::vector<int64_t>& ids)
{
     State out(s.size());
     for (uint64_t j = 0; j < s.size(); ++j) {
          uint64_t i = 0;
          for (size_t p = 0; p < ids.size(); ++p) i |= ((j >> p) & 1) << ids[p];
          out[j] = s[i];
     }
     return out;
}
double distance(const State& a, const State& b)
{
     double e = 0;
     for (size_t i = 0; i < a.size(); ++i) e = std::max(e, std::abs(a[i] - b[i]));
     return e;
}
State state_of(Engine& e, int n)
{
     State s(size_t(1) << n);
     e.get_state_c128(s.data());
     return s;
}
void queue_gates(Engine& e, const std::vector<Gate>& gates)
{
     for (const auto& g: gates) {
          e.apply_gate(mat_of(g), g.t, g.c);
          e.run();
     }
}

enum What { kWait, kList, kReorder };

// One call with the given failure; returns whether it failed.
bool attempt(int n, const std::vector<Gate>& gates, What what, long alloc, long launch)
{
     Engine e(1, n, 5, Prec::C128, 0);
     e.allocate_qureg(iota(n), 0);
     std::vector<int64_t> order = iota(n);
     std::mt19937 rng(5);
     std::shuffle(order.begin(), order.end(), rng);
     std::vector<Engine::Gate> tiled;
     if (what == kList)
          for (const auto& g: gates) {
               Engine::Gate x;
               x.m = mat_of(g);
               x.targets = g.t;
               x.ctrls = g.c;
               tiled.push_back(x);
          }
     else queue_gates(e, gates);
     passes_run = 0;
     fake::fail_alloc = alloc;
     fail_launch = launch;
     bool threw = false;
     try {
          if (what == kList) e.apply_tiled(tiled, 4);
          else if (what == kReorder) e.permute_qubits(order);
          else e.synchronize();
     } catch (const std::runtime_error&) {
          threw = true;
     }
     fake::fail_alloc = fail_launch = -1;
     const double tol = 1e-12;
     if (what == kList) {
          if (!threw) CHECK(distance(state_of(e, n), applied(n, gates)) < tol);
          // nothing was applied by a call that ran out of memory
          else if (launch < 0) CHECK(distance(state_of(e, n), applied(n, {})) < tol);
          CHECK(fake::allocations >= allocations_at_first_pass);
     }
     else {
          // a second call goes on where the first one stopped
          if (what == kReorder && threw) e.permute_qubits(order);
          State ref = applied(n, gates);
          if (what == kReorder) ref = permuted(ref, order);
          CHECK(distance(state_of(e, n), ref) < tol);
          CHECK(e.queued_gates() == 0);
     }
     return threw;
}

}  // namespace

int main()
{
     const int n = 15;
     const auto gates = list(n, 130, 3);
     for (What what: {kWait, kList, kReorder}) {
          int failed = 0;
          long k = 0;
          while (attempt(n, gates, what, k, -1)) ++k, ++failed;  // until every allocation succeeds
          CHECK(failed >= 1);
          for (k = 0; attempt(n, gates, what, -1, k); ++k) ++failed;
          CHECK(k >= 2);  // more than one pass
     }
     // a pass whose records exceed a staging slot: no allocation after the first pass
     {
          const int m = 13;
          const auto many = list(m, 4000, 9);
          Engine e(1, m, 5, Prec::C128, 0);
          e.allocate_qureg(iota(m), 0);
          std::vector<Engine::Gate> tiled;
          for (const auto& g: many) {
               Engine::Gate x;
               x.m = mat_of(g);
               x.targets = g.t;
               x.ctrls = g.c;
               tiled.push_back(x);
          }
          passes_run = 0;
          CHECK(e.apply_tiled(tiled, 4) > 1);
          CHECK(fake::allocations == allocations_at_first_pass);
          CHECK(distance(state_of(e, m), applied(m, many)) < 1e-11);
     }
     std::printf("gate failures ok\n");
     return 0;
}
