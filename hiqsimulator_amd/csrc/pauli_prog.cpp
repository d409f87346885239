// Planning of Pauli sums.  See pauli_prog.hpp.
#include "pauli_prog.hpp"

#include <algorithm>
#include <cmath>
#include <map>
#include <utility>

namespace hq {

namespace {
inline int popc(uint64_t x) { return __builtin_popcountll(x); }
}  // namespace

PauliPlan plan_pauli(const std::vector<PauliTermIn>& in, int n, bool apply)
{
     PauliPlan plan;
     const int T = pauli_tile_bits(n), H = T - kPauliLow;
     const uint64_t low = (uint64_t(1) << kPauliLow) - 1;
     // real coefficients by (x, kind); terms of one x stay in list order
     struct Z {
          uint64_t z;
          double c;
     };
     std::vector<uint64_t> xs;  // in order of first use
     std::map<std::pair<uint64_t, uint32_t>, std::vector<Z>> by;
     std::map<uint64_t, bool> known;
     for (const auto& t: in) {
          if (popc(t.x & ~low) > H) {
               plan.others.push_back(t);
               continue;
          }
          // Expectation: the pair i, i ^ x of a term adds twice the real part
          // of conj(psi[i ^ x]) psi[i] when |x & z| is even, twice i times
          // its imaginary part when it is odd.  Apply: the sign at the source
          // i = j ^ x is the one at j times (-1)^{|x & z|}.
          const bool odd = popc(t.x & t.z) & 1;
          std::complex<double> c = t.c;
          uint32_t kind = 0;
          if (apply) {
               if (odd) c = -c;
          }
          else if (odd) {
               kind = 1;
               c = std::complex<double>(-c.imag(), c.real());
          }
          if (known.emplace(t.x, true).second) xs.push_back(t.x);
          // real part of the coefficient, then its imaginary part
          if (!(c.real() == 0.0)) by[{t.x, kind}].push_back(Z{t.z, c.real()});
          if (!(c.imag() == 0.0)) by[{t.x, apply ? 1u : kind | 2u}].push_back(Z{t.z, c.imag()});
     }
     std::vector<uint64_t> left;
     bool diagonal = false;
     for (uint64_t x: xs) {
          if (x) left.push_back(x);
          else diagonal = true;
     }
     while (!left.empty() || diagonal) {
          // the first x left, then always the one that needs the fewest new bits
          uint64_t bits = low;
          std::vector<uint64_t> here;
          if (diagonal) here.push_back(0);
          diagonal = false;
          for (;;) {
               // (a sweep takes all that need none: at most H + 1 sweeps a pass)
               int best = -1, need = H + 1;
               size_t kept = 0;
               for (uint64_t x: left) {
                    const int k = popc(x & ~bits);
                    if (k == 0) {
                         here.push_back(x);
                         continue;
                    }
                    if (popc(bits) + k <= T && k < need) {
                         need = k;
                         best = static_cast<int>(kept);
                    }
                    left[kept++] = x;
               }
               left.resize(kept);
               if (best < 0) break;
               bits |= left[best];
          }
          for (int p = 0; p < n && popc(bits) < T; ++p) bits |= uint64_t(1) << p;
          int rank[64], r = 0;
          PauliPass pass{};
          for (int p = 0; p < 64; ++p) {
               rank[p] = -1;
               if (!((bits >> p) & 1)) continue;
               if (r >= kPauliLow) pass.hpos[r - kPauliLow] = static_cast<uint8_t>(p);
               rank[p] = r++;
          }
          auto to_tile = [&](uint64_t m) {
               uint32_t t = 0;
               for (uint64_t b = m & bits; b; b &= b - 1) t |= 1u << rank[__builtin_ctzll(b)];
               return t;
          };
          pass.first = static_cast<uint32_t>(plan.terms.size());
          for (uint64_t x: here)
               for (uint32_t kind = 0; kind < 4; ++kind) {
                    const auto it = by.find({x, kind});
                    if (it == by.end()) continue;
                    auto& zs = it->second;
                    auto cls = [&](const Z& z) { return to_tile(z.z) >> kPauliThr; };
                    std::stable_sort(zs.begin(), zs.end(), [&](const Z& a, const Z& b) { return cls(a) < cls(b); });
                    const uint32_t xt = to_tile(x);
                    // Expectation: i and i ^ x contribute the same; where the
                    // highest bit of x tells waves or amplitudes of a thread
                    // apart, the kernel takes the one half, twice.
                    const double f = !apply && (xt >> kPauliLane) ? 2.0 : 1.0;
                    for (size_t i = 0; i < zs.size(); ++i) {
                         PauliTerm t{};
                         t.z_out = zs[i].z & ~bits;
                         t.c = f * zs[i].c;
                         t.z_tile = to_tile(zs[i].z) | ((kind & 1u) ? kPauliImag : 0u) | ((kind & 2u) ? kPauliOut1 : 0u);
                         t.x = xt;
                         const bool last = i + 1 == zs.size();
                         if (last) t.z_tile |= kPauliGroupEnd;
                         if (last || cls(zs[i]) != cls(zs[i + 1])) t.z_tile |= kPauliClassEnd;
                         plan.terms.push_back(t);
                    }
               }
          pass.count = static_cast<uint32_t>(plan.terms.size()) - pass.first;
          plan.passes.push_back(pass);
     }
     plan.terms.push_back(PauliTerm{});
     return plan;
}

std::vector<double> bessel_series(double z)
{
     if (!(z > 1e-300)) return {1.0};
     // far enough above the turning point k = z that J_k is below 1e-60 there
     const int top = static_cast<int>(z + 24.0 * std::cbrt(z) + 60.0) | 1;
     std::vector<long double> j(static_cast<size_t>(top) + 2, 0.0L);
     j[static_cast<size_t>(top)] = 1e-300L;
     long double even = 0.0L;
     for (int k = top; k >= 1; --k) {
          j[k - 1] = 2.0L * k / z * j[k] - j[k + 1];
          if (std::fabs(j[k - 1]) > 1e250L)
               for (int q = k - 1; q <= top; ++q) j[q] *= 1e-250L;
     }
     for (int k = 2; k <= top; k += 2) even += j[k];
     const long double norm = 1.0L / (j[0] + 2.0L * even);
     std::vector<double> out;
     for (int k = 0; k <= top; ++k) out.push_back(static_cast<double>(j[k] * norm));
     while (out.size() > 1 && std::fabs(out.back()) < 1e-17) out.pop_back();
     return out;
}

}  // namespace hq
