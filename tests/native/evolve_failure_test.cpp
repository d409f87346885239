// Host run of the engine's time evolution over a stand-in for the HIP runtime:
// results of one and of several segments of the series, with and without
// controls, and with an allocation or a launch that fails, after which the
// state is what it was.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <random>
#include <stdexcept>
#include <vector>

#include "../../hiqsimulator_amd/csrc/engine.hpp"
#include "fake_hip.hpp"

#define CHECK(c)                                                                   \
     do {                                                                          \
          if (!(c)) {                                                              \
               std::fprintf(stderr, "check failed line %d: %s\n", __LINE__, #c);   \
               std::exit(1);                                                       \
          }                                                                        \
     } while (0)

namespace hq {

using State = std::vector<cplx>;
long applies = 0, fail_apply = -1;  // products until one fails

cplx* amps(void* p) { return static_cast<cplx*>(p); }
const cplx* amps(const void* p) { return static_cast<const cplx*>(p); }

hipError_t launch_pauli_apply(const PauliApply& a, Prec prec, int n, const PauliPass& pass, const PauliTerm* terms, hipStream_t)
{
     CHECK(prec == Prec::C128 && a.src != a.dst);
     if (fail_apply >= 0 && fail_apply-- == 0) return hipErrorLaunchFailure;
     ++applies;
     const int T = pauli_tile_bits(n);
     auto index_bits = [&](uint32_t ranks) {
          uint64_t m = ranks & ((1u << kPauliLow) - 1);
          for (int r = kPauliLow; r < T; ++r) m |= static_cast<uint64_t>((ranks >> r) & 1) << pass.hpos[r - kPauliLow];
          return m;
     };
     const State src(amps(a.src), amps(a.src) + (size_t(1) << n));
     const State add = a.add ? State(amps(a.add), amps(a.add) + src.size()) : State(src.size());
     for (uint64_t j = 0; j < src.size(); ++j) {
          cplx o = 0;
          for (uint32_t t = pass.first; t < pass.first + pass.count; ++t) {
               const uint64_t z = terms[t].z_out | index_bits(terms[t].z_tile & 0xffff), x = index_bits(terms[t].x);
               cplx w = __builtin_popcountll(j & z) & 1 ? -terms[t].c : terms[t].c;
               if (terms[t].z_tile & kPauliImag) w *= cplx(0, 1);
               o += w * src[j ^ x];
          }
          const cplx b = cplx(a.fr, a.fi) * o + a.g * add[j];
          amps(a.dst)[j] = b;
          if (a.o_dst) amps(a.o_dst)[j] = (a.o_src ? a.h * amps(a.o_src)[j] : cplx(0)) + cplx(a.er, a.ei) * src[j] + cplx(a.cr, a.ci) * b;
     }
     return hipSuccess;
}
hipError_t launch_pauli_accumulate(void* dst, const void* src, Prec, uint64_t n, uint64_t x, uint64_t z, double cr, double ci, hipStream_t)
{
     CHECK(x == 0 && z == 0);
     for (uint64_t i = 0; i < n; ++i) amps(dst)[i] += cplx(cr, ci) * amps(src)[i];
     return hipSuccess;
}
hipError_t launch_normalize(void* psi, Prec, uint64_t n, uint64_t msk, uint64_t val, double f, const double* norm, hipStream_t)
{
     CHECK(!norm);
     for (uint64_t i = 0; i < n; ++i) amps(psi)[i] = (i & msk) == val ? amps(psi)[i] * f : cplx(0);
     return hipSuccess;
}
hipError_t launch_scale(void* psi, Prec, uint64_t n, double re, double im, hipStream_t)
{
     for (uint64_t i = 0; i < n; ++i) amps(psi)[i] *= cplx(re, im);
     return hipSuccess;
}
hipError_t launch_copy(void* dst, const void* src, Prec, uint64_t n, hipStream_t)
{
     std::copy_n(amps(src), n, amps(dst));
     return hipSuccess;
}
hipError_t launch_fill(void* psi, Prec, uint64_t n, double re, double im, hipStream_t)
{
     std::fill_n(amps(psi), n, cplx(re, im));
     return hipSuccess;
}
hipError_t init_reduce_scratch(double*, hipStream_t) { return hipSuccess; }
Readback::~Readback() {}
void Readback::read(const void* psi, Prec, uint64_t n, std::complex<double>* out, hipStream_t) { std::copy_n(amps(psi), n, out); }

}  // namespace hq

namespace {

using namespace hq;

struct Sum {
     std::vector<uint64_t> x, z;
     std::vector<cplx> c;
};

// H psi on the qubits of the masks (Y = i X Z), where all controls are set.
State applied(const Sum& h, const State& psi, uint64_t cmask)
{
     State out(psi.size());
     for (size_t t = 0; t < h.x.size(); ++t) {
          cplx f = h.c[t];
          for (int k = __builtin_popcountll(h.x[t] & h.z[t]) & 3; k; --k) f *= cplx(0, 1);
          for (uint64_t i = 0; i < psi.size(); ++i)
               if ((i & cmask) == cmask) out[i ^ h.x[t]] += (__builtin_popcountll(i & h.z[t]) & 1 ? -f : f) * psi[i];
     }
     return out;
}
// exp(-i t H) psi in many short Taylor steps.
State evolved(const Sum& h, State psi, double t, uint64_t cmask)
{
     double l1 = 0;
     for (const auto& c: h.c) l1 += std::abs(c);
     const int steps = 1 + static_cast<int>(2 * std::abs(t) * l1);
     for (int s = 0; s < steps; ++s) {
          State a = psi;
          for (int k = 1; k < 24; ++k) {
               a = applied(h, a, cmask);
               for (size_t i = 0; i < a.size(); ++i) psi[i] += a[i] *= cplx(0, -t / steps / k);
          }
     }
     return psi;
}

double distance(const State& a, const State& b)
{
     double e = 0;
     for (size_t i = 0; i < a.size(); ++i) e = std::max(e, std::abs(a[i] - b[i]));
     return e;
}

std::vector<int64_t> iota(int n)
{
     std::vector<int64_t> v(n);
     for (int i = 0; i < n; ++i) v[i] = i;
     return v;
}

// Evolves a random state; returns whether the call failed.
bool run(int n, int qubits, const std::vector<int64_t>& ctrls, double t, long alloc, long apply, bool identity)
{
     std::mt19937 rng(9);
     std::normal_distribution<double> g;
     Engine e(1, n, 4, Prec::C128, 0);
     e.allocate_qureg(iota(n), 0);
     State psi(size_t(1) << n);
     for (auto& z: psi) z = cplx(g(rng), g(rng)) / std::sqrt(double(2 << n));
     e.set_state_c128(psi.data(), psi.size());
     Sum h;
     auto term = [&](uint64_t x, uint64_t z, double c) {
          h.x.push_back(x);
          h.z.push_back(z);
          h.c.push_back(c);
     };
     for (int i = 0; i + 1 < qubits; ++i) term(0, 3u << i, 0.5 + 0.05 * i);
     for (int i = 0; i < qubits; i += 2) term(1u << i, 0, 0.3);
     term(3, 2, 0.2);  // Y X
     if (identity) term(0, 0, 0.7);
     uint64_t cmask = 0;
     for (auto c: ctrls) cmask |= uint64_t(1) << c;
     fake::fail_alloc = alloc;
     fail_apply = apply;
     bool threw = false;
     try {
          e.time_evolution(h.x, h.z, h.c, t, iota(qubits), ctrls);
     } catch (const std::runtime_error&) {
          threw = true;
     }
     fake::fail_alloc = fail_apply = -1;
     State got(psi.size());
     e.get_state_c128(got.data());
     if (threw) CHECK(distance(got, psi) == 0);
     else CHECK(distance(got, evolved(h, psi, t, cmask)) < 1e-10);
     return threw;
}

}  // namespace

int main()
{
     // reaches around one and two segments, forwards and backwards
     for (double t: {0.01, 0.7, -3.0, 37.0, -60.0, 120.0}) CHECK(!run(9, 9, {}, t, -1, -1, t > 1));
     for (double t: {0.5, -60.0, 90.0}) CHECK(!run(11, 9, {10, 9}, t, -1, -1, true));
     for (double t: {0.5, 60.0})
          for (bool ctrl: {false, true}) {
               const int n = ctrl ? 10 : 9;
               const std::vector<int64_t> c = ctrl ? std::vector<int64_t>{9} : std::vector<int64_t>{};
               long k = 0;
               while (run(n, 9, c, t, k, -1, false)) ++k;
               CHECK(k >= 3);
               applies = 0;
               CHECK(!run(n, 9, c, t, -1, -1, false));
               const long all = applies;
               for (long q: {0L, 1L, 2L, 3L, all / 2, all - 2, all - 1}) CHECK(run(n, 9, c, t, -1, q, false));
          }
     std::printf("evolution failures ok\n");
     return 0;
}
