// Which way gate lists go, on the host: gate programs or tile programs, and for
// complex64 states the precision that the amplitudes are held in.
#define main gate_prog_main
#include "gate_prog_test.cpp"
#undef main

namespace {

struct Lists {
     int n;
     std::mt19937 rng{7};
     double u() { return std::uniform_real_distribution<double>(0, 6.28)(rng); }
     std::vector<cplx> rx(double t) { return {std::cos(t), cplx(0, -std::sin(t)), cplx(0, -std::sin(t)), std::cos(t)}; }
     std::vector<cplx> ry(double t) { return {std::cos(t), -std::sin(t), std::sin(t), std::cos(t)}; }
     std::vector<cplx> rz(double t) { return {std::polar(1.0, -t), 0, 0, std::polar(1.0, t)}; }
     const std::vector<cplx> x{0, 1, 1, 0};
     std::vector<cplx> dense(int d)
     {
          std::vector<cplx> m(d * d);
          for (auto& z: m) z = cplx(u(), u());
          return m;
     }
     // one of `one` for every qubit, then CNOTs, layer by layer
     template <typename F>
     std::vector<Gate> layers(int count, const std::vector<int64_t>& qs, F&& one)
     {
          std::vector<Gate> out;
          for (int l = 0; l < count; ++l) {
               for (int64_t q: qs) one(out, q);
               for (size_t i = l % 2; i + 1 < qs.size(); i += 2) out.push_back({x, {qs[i + 1]}, {qs[i]}});
          }
          return out;
     }
     std::vector<int64_t> all() const
     {
          std::vector<int64_t> q(n);
          for (int i = 0; i < n; ++i) q[i] = i;
          return q;
     }
     std::vector<Gate> random_layers(int count)
     {
          return layers(count, all(), [&](std::vector<Gate>& out, int64_t q) {
               const int k = static_cast<int>(rng() % 3);
               out.push_back({k == 0 ? rx(u()) : (k == 1 ? ry(u()) : rz(u())), {q}, {}});
          });
     }
     std::vector<Gate> equal_layers(int count)
     {
          return layers(count, all(), [&](std::vector<Gate>& out, int64_t q) { out.push_back({rx(0.4), {q}, {}}); });
     }
     std::vector<Gate> zxzxz(int count, const std::vector<int64_t>& qs)
     {
          return layers(count, qs, [&](std::vector<Gate>& out, int64_t q) {
               for (int i = 0; i < 5; ++i) out.push_back({i % 2 ? rx(u()) : rz(u()), {q}, {}});
          });
     }
     std::vector<Gate> ising(int steps)
     {
          std::vector<Gate> out;
          const cplx a = std::polar(1.0, 0.3), b = std::polar(1.0, -0.3);
          for (int s = 0; s < steps; ++s) {
               for (int i = 0; i + 1 < n; ++i) out.push_back({{a, 0, 0, 0, 0, b, 0, 0, 0, 0, b, 0, 0, 0, 0, a}, {i, i + 1}, {}});
               for (int i = 0; i < n; ++i) out.push_back({rx(0.4), {i}, {}});
          }
          return out;
     }
     std::vector<Gate> ladder()
     {
          std::vector<Gate> out;
          for (int r = 0; r < 8; ++r)
               for (int i = 0; i + 1 < n; ++i) out.push_back({x, {i + 1}, {i}});
          return out;
     }
     std::vector<Gate> bricks(const std::vector<int64_t>& qs, int count)
     {
          std::vector<Gate> out;
          for (int l = 0; l < count; ++l)
               for (size_t i = l % 2; i + 1 < qs.size(); i += 2) out.push_back({dense(4), {qs[i], qs[i + 1]}, {}});
          return out;
     }
     std::vector<Gate> pair(int count)
     {
          std::vector<Gate> out;
          for (int i = 0; i < count; ++i) out.push_back({dense(4), {1, n - 2}, {}});
          return out;
     }
};

enum Way { kTiles, kFp64, kFp32 };

Way way(const std::vector<Gate>& gates, int n, Prec prec)
{
     std::vector<GateUnit> units(gates.size());
     for (size_t i = 0; i < gates.size(); ++i) CHECK(make_gate_unit(gates[i].m.data(), gates[i].t, gates[i].c, units[i]));
     const GateListCost c = gate_list_cost(units, n, prec);
     CHECK(c.work >= 0 && c.products >= 0 && c.rounds >= 0);
     Prec held;
     if (!gate_route(c, gates.size(), n, prec, held)) return kTiles;
     return held == Prec::C128 ? kFp64 : kFp32;
}

}  // namespace

int main()
{
     for (int n: {21, 24, 28, 34}) {
          Lists l{n};
          const std::vector<int64_t> few = {1, 5, n - 2, n / 2};
          const bool large = n > 22;
          // repeated angles, many rotations a qubit and long lists on few qubits are
          // never held in FP32; layers of different angles are
          for (int count: {2, 4, 20, 60}) {
               CHECK(way(l.random_layers(count), n, Prec::C64) == kFp32);
               CHECK(way(l.equal_layers(count), n, Prec::C64) == kFp64);
          }
          // and a few rotations among many CNOTs
          for (bool equal: {false, true}) {
               std::vector<Gate> g;
               for (int i = 0; i < 1000; ++i) {
                    const int q = 5 * i % (n - 4);
                    for (int k = 0; k < 4; ++k) g.push_back({l.x, {q + k + 1}, {q + k}});
                    g.push_back({l.rx(equal ? 0.4 : 0.4 + 0.001 * i), {q}, {}});
               }
               CHECK(way(g, n, Prec::C64) == (equal ? kFp64 : kFp32));
          }
          CHECK(way(l.ising(1), n, Prec::C64) == kFp64);
          for (int steps: {5, 40}) CHECK(way(l.ising(steps), n, Prec::C64) == (large ? kTiles : kFp64));
          for (int count: {1, 10, 200}) CHECK(way(l.zxzxz(count, few), n, Prec::C64) != kFp32);
          CHECK(way(Qft{n, 0}.gates(), n, Prec::C64) == kFp32);
          CHECK(way(Qft{n, 5}.gates(), n, Prec::C64) == kFp32);
          CHECK(way(l.ladder(), n, Prec::C64) == kFp32);
          // lists that fuse into few products run as those
          for (Prec prec: {Prec::C128, Prec::C64}) {
               CHECK((way(l.zxzxz(200, few), n, prec) == kTiles) == large);
               CHECK((way(l.zxzxz(6, l.all()), n, prec) == kTiles) == large);
               CHECK(way(l.pair(40), n, prec) == kTiles);
          }
          // and those that do not as gate programs
          CHECK(way(l.random_layers(20), n, Prec::C128) == kFp64);
          CHECK(way(l.ising(5), n, Prec::C128) == kFp64);
          CHECK(way(l.ladder(), n, Prec::C128) == kFp64);
          CHECK(way(Qft{n, 3}.gates(), n, Prec::C128) == kFp64);
          CHECK(way(l.bricks(l.all(), 6), n, Prec::C128) == kFp64);
     }
     // small states
     for (int n: {13, 16, 18}) {
          Lists l{n};
          CHECK(way(l.random_layers(20), n, Prec::C128) == kFp64);
          CHECK(way(l.zxzxz(200, {1, 5, n - 2, n / 2}), n, Prec::C128) == kFp64);
          CHECK(way(l.bricks(l.all(), 6), n, Prec::C128) == kTiles);
          CHECK(way(l.random_layers(20), n, Prec::C64) == kTiles);
     }
     CHECK(way(Lists{12}.random_layers(3), 12, Prec::C128) == kTiles);
     // what is asked before the units are made agrees with them
     {
          Maker mk{std::mt19937(3), 9};
          int fit = 0, total = 0;
          auto ask = [&](const std::vector<cplx>& m, size_t k) {
               GateUnit u;
               const std::vector<int64_t> t = {2, 0, 5, 7, 1};
               const bool made = make_gate_unit(m.data(), {t.begin(), t.begin() + static_cast<long>(k)}, {}, u);
               CHECK(gate_fits(m.data(), k) == made);
               fit += made;
               ++total;
          };
          for (int i = 0; i < 200; ++i) {
               const Gate g = mk.gate(9);
               ask(g.m, g.t.size());
          }
          for (size_t k: {3u, 4u, 5u}) {
               const size_t d = size_t(1) << k;
               std::vector<cplx> m(d * d);
               for (size_t i = 0; i < d; ++i) m[i * d + i] = 1;
               ask(m, k);
               m[1] = 0.5, ask(m, k);      // one qubit
               m[d + 3] = 0.5, ask(m, k);  // two
               m[3 * d + 7] = 0.5, ask(m, k);
               ask(mk.random(static_cast<int>(d)), k);
          }
          CHECK(fit > 100 && fit < total);
     }
     // empty lists, identities and factors of everything
     {
          Lists l{24};
          Prec held;
          CHECK(gate_route(gate_list_cost({}, 24, Prec::C128), 0, 24, Prec::C128, held));
          std::vector<Gate> id(10, Gate{{1, 0, 0, 1}, {3}, {}});
          CHECK(way(id, 24, Prec::C64) == kFp64);
          id.push_back(Gate{{cplx(0, 1), 0, 0, cplx(0, 1)}, {2}, {}});
          CHECK(way(id, 24, Prec::C128) == kFp64);
     }
     std::printf("gate routes ok\n");
     return 0;
}
