// Host-only run of the Pauli sum planner, built with AddressSanitizer and
// UndefinedBehaviorSanitizer: a plain interpreter of the planned records
// (tile by tile, as the kernels evaluate them) plus the terms left over must
// give what applying the terms one by one gives, for expectation values and
// for applying the sum: chains, random strings, strings wider than a tile,
// repeated terms, complex and zero coefficients, identities.
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../hiqsimulator_amd/csrc/pauli_prog.hpp"

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

double parity(uint64_t m) { return __builtin_popcountll(m) & 1 ? -1.0 : 1.0; }

// (sums over the state are long double, so that their own rounding does not
// enter the comparison)
using lcplx = std::complex<long double>;

lcplx expect_one(const State& psi, const PauliTermIn& t)
{
     lcplx s = 0;
     for (uint64_t i = 0; i < psi.size(); ++i) s += lcplx(std::conj(psi[i ^ t.x]) * psi[i] * parity(i & t.z));
     return lcplx(t.c) * s;
}

void apply_one(State& dst, const State& src, const PauliTermIn& t)
{
     for (uint64_t i = 0; i < src.size(); ++i) dst[i ^ t.x] += t.c * parity(i & t.z) * src[i];
}

void run_case(int n, int nterms, int max_weight, bool complex_c, unsigned seed)
{
     std::mt19937 rng(seed);
     auto u = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); };
     std::vector<PauliTermIn> list;
     for (int i = 0; i < nterms; ++i) {
          PauliTermIn t{0, 0, complex_c ? cplx(u(-1, 1), u(-1, 1)) : cplx(u(-1, 1), 0)};
          const int w = static_cast<int>(rng() % (max_weight + 1));
          for (int k = 0; k < w; ++k) {
               const uint64_t b = uint64_t(1) << (rng() % n);
               const int p = static_cast<int>(rng() % 3);
               if (p < 2) t.x |= b;
               if (p > 0) t.z |= b;
          }
          if (i % 7 == 3 && i) t = list[rng() % i];
          if (i % 11 == 5) t.c = 0;
          list.push_back(t);
     }
     State psi(size_t(1) << n);
     for (auto& z: psi) z = cplx(u(-1, 1), u(-1, 1));
     const int T = pauli_tile_bits(n);
     for (bool apply: {false, true}) {
          const PauliPlan plan = plan_pauli(list, n, apply);
          CHECK(!plan.terms.empty());
          lcplx ref = 0, got = 0;
          State rdst(psi.size()), dst(psi.size());
          for (const auto& t: list) {
               ref += expect_one(psi, t);
               apply_one(rdst, psi, t);
          }
          for (const auto& t: plan.others) {
               CHECK(__builtin_popcountll(t.x >> kPauliLow) > T - kPauliLow);
               got += expect_one(psi, t);
               apply_one(dst, psi, t);
          }
          for (const auto& P: plan.passes) {
               int pos[kPauliMaxTile];
               uint64_t bits = 0;
               for (int r = 0; r < T; ++r) {
                    pos[r] = r < kPauliLow ? r : P.hpos[r - kPauliLow];
                    CHECK(pos[r] < n && (r == 0 || pos[r] > pos[r - 1]));
                    bits |= uint64_t(1) << pos[r];
               }
               auto index = [&](uint64_t base, uint32_t rank) {
                    for (int r = 0; r < T; ++r) base |= static_cast<uint64_t>((rank >> r) & 1) << pos[r];
                    return base;
               };
               CHECK(P.first + P.count < plan.terms.size());  // and the record read ahead
               for (uint64_t base = 0; base < psi.size(); ++base) {
                    if (base & bits) continue;
                    std::vector<double> w(size_t(1) << T, 0.0);
                    uint32_t group = P.first;
                    for (uint32_t i = P.first; i < P.first + P.count; ++i) {
                         const PauliTerm& t = plan.terms[i];
                         const uint32_t zt = t.z_tile & 0xffffu;
                         CHECK(!(t.x >> T) && !(zt >> T) && t.x == plan.terms[group].x);
                         for (uint32_t r = 0; r < (1u << T); ++r) w[r] += t.c * parity(base & t.z_out) * parity(r & zt);
                         if (i > group && !(plan.terms[i - 1].z_tile & kPauliClassEnd))
                              CHECK((plan.terms[i - 1].z_tile & 0xffffu) >> kPauliThr == zt >> kPauliThr);
                         if (!(t.z_tile & kPauliGroupEnd)) continue;
                         CHECK(t.z_tile & kPauliClassEnd);
                         group = i + 1;
                         for (uint32_t r = 0; r < (1u << T); ++r) {
                              const cplx x = psi[index(base, r)], y = psi[index(base, r ^ t.x)];
                              const bool im = t.z_tile & kPauliImag;
                              if (apply) {
                                   dst[index(base, r)] += (im ? cplx(0, w[r]) : cplx(w[r], 0)) * y;
                              }
                              else {
                                   // the half that the kernel takes
                                   if ((t.x >> kPauliLane) && ((r >> (31 - __builtin_clz(t.x))) & 1)) continue;
                                   const cplx q = std::conj(y) * x;
                                   const double v = w[r] * (im ? q.imag() : q.real());
                                   got += t.z_tile & kPauliOut1 ? lcplx(0, v) : lcplx(v, 0);
                              }
                         }
                         w.assign(size_t(1) << T, 0.0);
                    }
                    CHECK(group == P.first + P.count);
               }
          }
          double scale = 0;
          for (const auto& t: list) scale += std::abs(t.c);
          const double tol = 1e-15 * (scale + 1) * static_cast<double>(psi.size());
          if (apply) {
               for (size_t i = 0; i < psi.size(); ++i) CHECK(std::abs(dst[i] - rdst[i]) <= 1e-14 * (scale + 1) * (nterms + 1));
          }
          else {
               CHECK(std::abs(got - ref) <= tol);
          }
     }
}

}  // namespace

int main()
{
     unsigned seed = 1;
     for (int n: {9, 10, 11, 12, 13, 15}) {
          run_case(n, 0, 2, false, seed++);
          run_case(n, 1, 1, false, seed++);
          run_case(n, 30, 2, false, seed++);
          run_case(n, 24, 4, true, seed++);
          run_case(n, 12, n + 4, true, seed++);
     }
     // a chain: neighbours share passes
     std::vector<PauliTermIn> chain;
     for (int i = 0; i + 1 < 26; ++i) {
          const uint64_t m = uint64_t(3) << i;
          chain.push_back({m, 0, 1.0});
          chain.push_back({m, m, -1.0});
          chain.push_back({0, m, 1.0});
     }
     const PauliPlan plan = plan_pauli(chain, 26, false);
     CHECK(plan.passes.size() <= 4 && plan.others.empty());
     std::printf("pauli plans ok, %zu passes\n", plan.passes.size());
     return 0;
}
