// The running sums of block probabilities as the sampler's workgroup forms them
// (running_sums.hpp), thread by thread with the same tree: sums never fall, are
// equal over empty blocks, and the first one that exceeds (or reaches) any u
// below the total belongs to a block that holds something.  Probabilities with
// many roundings, runs of empty blocks of every length and whole empty runs.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <random>
#include <vector>

#include "../../hiqsimulator_amd/csrc/running_sums.hpp"

using namespace hq;

#define CHECK(c)                                                                 \
     do {                                                                        \
          if (!(c)) {                                                            \
               std::fprintf(stderr, "check failed line %d: %s\n", __LINE__, #c); \
               std::exit(1);                                                     \
          }                                                                      \
     } while (0)

namespace {

constexpr int kThreads = 1024;

std::vector<double> running(const std::vector<double>& p)
{
     const int nb = static_cast<int>(p.size()), per = nb > kThreads ? nb / kThreads : 1;
     std::vector<BlockRun> run(kThreads);
     std::vector<double> part(kThreads), end(kThreads), out(nb);
     for (int t = 0; t < kThreads; ++t) {
          for (int i = 0; i < per && t * per + i < nb; ++i) run[t].add(p[t * per + i], i);
          part[t] = run[t].sum;
     }
     // inside the waves, then over them
     auto scan = [](std::vector<double>& v, int first, int count) {
          for (int o = 1; o < count; o <<= 1)
               for (int i = count - 1; i >= o; --i) v[first + i] += v[first + i - o];
     };
     std::vector<double> waves(kThreads / 64);
     for (int w = 0; w < kThreads / 64; ++w) {
          scan(part, 64 * w, 64);
          waves[w] = part[64 * w + 63];
     }
     scan(waves, 0, kThreads / 64);
     for (int t = 64; t < kThreads; ++t) part[t] += waves[t / 64 - 1];
     for (int t = 0; t < kThreads; ++t) {
          end[t] = run[t].end(part[t]);
          if (t) end[t] = larger(end[t - 1], end[t]);
     }
     for (int t = 0; t < kThreads; ++t) {
          double s = t ? end[t - 1] : 0.0;
          for (int i = 0; i < per && t * per + i < nb; ++i) {
               s += p[t * per + i];
               out[t * per + i] = running_sum(s, i, run[t].last, end[t]);
          }
     }
     return out;
}

void check_sums(const std::vector<double>& p, std::mt19937& rng)
{
     const auto c = running(p);
     double exact = 0, before = 0;
     for (double x: p) exact += x;
     for (size_t i = 0; i < p.size(); ++i) {
          CHECK(c[i] >= before);
          if (p[i] == 0.0) CHECK(c[i] == before);
          before = c[i];
     }
     CHECK(std::abs(before - exact) <= 1e-12 * exact);
     // the points around every value that is there, and some between
     std::vector<double> us = {0x1p-1074};
     for (int k = 0; k < 200; ++k) {
          const double v = c[rng() % c.size()];
          us.push_back(v);
          us.push_back(std::nextafter(v, 0.0));
          us.push_back(std::nextafter(v, 2.0));
          us.push_back(before * std::uniform_real_distribution<double>(0, 1)(rng));
     }
     for (double u: us) {
          const auto above = std::upper_bound(c.begin(), c.end(), u) - c.begin();
          if (u < before) CHECK(p[above] > 0.0);
          const auto reach = std::lower_bound(c.begin(), c.end(), u) - c.begin();
          if (u > 0.0 && u <= before) CHECK(p[reach] > 0.0);
     }
}

}  // namespace

int main()
{
     std::mt19937 rng(5);
     std::uniform_real_distribution<double> u(0, 1);
     for (int nb: {1, 2, 32, 512, 1024, 2048, 4096, 8192, 32768})
          for (int kind = 0; kind < 6; ++kind)
               for (int r = 0; r < 4; ++r) {
                    std::vector<double> p(nb);
                    for (auto& x: p) x = u(rng) / nb;
                    if (kind >= 1)
                         for (auto& x: p)
                              if (u(rng) < (kind == 1 ? 0.3 : 0.95)) x = 0;
                    if (kind >= 3)  // long empty stretches
                         for (int i = 0; i < nb; ++i)
                              if ((i * 7 / std::max(1, nb / 16)) % 3) p[i] = 0;
                    if (kind == 4)
                         for (auto& x: p) x *= std::pow(10.0, -30 * u(rng));
                    if (kind == 5) std::fill(p.begin(), p.end(), 0.0);
                    p[rng() % nb] = 0.1 + u(rng);
                    check_sums(p, rng);
               }
     // NaN reaches the total
     for (int nb: {32, 1024, 32768}) {
          std::vector<double> p(nb, 1.0 / nb);
          p[rng() % nb] = std::numeric_limits<double>::quiet_NaN();
          CHECK(std::isnan(running(p).back()));
     }
     std::printf("running sums ok\n");
     return 0;
}
