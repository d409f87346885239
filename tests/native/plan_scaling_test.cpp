// Planning time of long gate lists on few qubits, on the host: eight times the length may take at most sixteen times as
// long (a plan that looks at everything left at every step takes sixty-four).
#include <chrono>
#include <cmath>
#include <cstdio>
#include <random>

#include "../../hiqsimulator_amd/csrc/gate_prog.hpp"

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

bool scales(const char* what, double small, double large)
{
     std::printf("%s: %.1f and %.1f ms\n", what, 1e3 * small, 1e3 * large);
     return small > 0 && large < 16 * small;
}

}  // namespace

int main()
{
     const bool ok = scales("gates", plan_gates(14, 12500), plan_gates(14, 100000));
     if (ok) std::printf("planning scales\n");
     return ok ? 0 : 1;
}
