// Planning time of long gate lists on few qubits and of Pauli sums with many
// strings, on the host: eight times the length may take at most sixteen times as
// long (a plan that looks at everything left at every step takes sixty-four).
#include <chrono>
#include <cmath>
#include <cstdio>
#include <random>

#include "../../hiqsimulator_amd/csrc/gate_prog.hpp"
#include "../../hiqsimulator_amd/csrc/pauli_prog.hpp"

using namespace hq;
using cplx = std::complex<double>;

namespace {

template <typename F>
double best_of_three(F&& f)
{
     double best = 1e30;
     for (int r = 0; r < 3; ++r) {
          const auto t0 = std::chrono::steady_clock::now();
          f();
          best = std::min(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
     }
     return best;
}

// CNOTs and rotations on all qubits but one.
double plan_gates(int n, int count)
{
     std::mt19937 rng(1);
     std::vector<GateUnit> units(count);
     for (auto& u: units) {
          const int a = static_cast<int>(rng() % (n - 1)), b = (a + 1 + static_cast<int>(rng() % (n - 2))) % (n - 1);
          const std::vector<cplx> rot = {0.6, 0.8, 0.8, -0.6}, x = {0, 1, 1, 0};
          const bool cnot = rng() & 1;
          if (!make_gate_unit((cnot ? x : rot).data(), {a}, cnot ? std::vector<int64_t>{b} : std::vector<int64_t>{}, u)) return -1;
     }
     return best_of_three([&] {
          GatePassPlanner planner(units, n, Prec::C128);
          GatePassPlan plan;
          size_t seen = 0;
          while (planner.next(plan))
               for (const auto& s: plan.stages) seen += s.size();
          if (seen != units.size()) std::printf("gates lost\n");
     });
}

double plan_strings(int n, int count)
{
     std::mt19937 rng(2);
     std::vector<PauliTermIn> in;
     for (int i = 0; i < count; ++i) {
          uint64_t x = 0, z = 0;
          for (int k = 0; k < 8; ++k) {
               const int q = static_cast<int>(rng() % n), s = static_cast<int>(rng() % 3);
               if (s < 2) x |= uint64_t(1) << q;
               if (s > 0) z |= uint64_t(1) << q;
          }
          in.push_back({x, z, cplx(0.1, 0)});
     }
     return best_of_three([&] { (void)plan_pauli(in, n, true); });
}

bool scales(const char* what, double small, double large)
{
     std::printf("%s: %.1f and %.1f ms\n", what, 1e3 * small, 1e3 * large);
     return small > 0 && large < 16 * small;
}

}  // namespace

int main()
{
     bool ok = scales("gates", plan_gates(14, 12500), plan_gates(14, 100000));
     ok = scales("strings", plan_strings(20, 5000), plan_strings(20, 40000)) && ok;
     if (ok) std::printf("planning scales\n");
     return ok ? 0 : 1;
}
