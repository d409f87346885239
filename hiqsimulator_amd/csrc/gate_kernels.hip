// gfx950 kernels of the gate programs (gate_prog.hpp).
//
// Bound: HBM (one read and one write of the state a pass) up to about forty
// gates a pass: 30 random qubits in complex128 take 7.8 ms a pass then, of
// which a bare copy in this shape takes 6.8 ms.  Vector issue (the gates and the
// regrouping between stages) comes on top with more, 11.2 ms for 74 gates.
// The 1780 gates of a 30-qubit circuit take 24 passes and 269 ms; as fused
// dense ops on LDS tiles they took 50 passes and 426 ms.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.hpp"
#include "gate_prog.hpp"

namespace hq {
namespace {

template <typename R>
struct Shape;
template <>
struct Shape<double> {
     static constexpr int E = gate_reg(Prec::C128), T = gate_tile_bits(Prec::C128);
};
template <>
struct Shape<float> {
     static constexpr int E = gate_reg(Prec::C64), T = gate_tile_bits(Prec::C64);
};

// A record read as 32-bit words at a wave-uniform address (scalar loads).
template <typename T>
__device__ __forceinline__ T load_record(const T* __restrict__ p)
{
     constexpr int N = sizeof(T) / 4;
     const uint32_t* const q = reinterpret_cast<const uint32_t*>(p);
     uint32_t w[N];
#pragma unroll
     for (int i = 0; i < N; ++i) w[i] = q[i];
     T r;
     __builtin_memcpy(&r, w, sizeof(T));
     return r;
}

// Every pair of amplitudes that differ in register bit B: f(a, z, index of a).
template <int B, int A, typename V, typename F>
__device__ __forceinline__ void for_pairs(V (&x)[A], F&& f)
{
#pragma unroll
     for (int j = 0; j < A / 2; ++j) {
          const int i = ((j >> B) << (B + 1)) | (j & ((1 << B) - 1));
          f(x[i], x[i | (1 << B)], i);
          __builtin_amdgcn_sched_barrier(0);  // a pair's temporaries die with it
     }
}

// A copy the compiler cannot see through.  Every op below updates the
// amplitudes in place, each new value written when the old one is dead; where
// an old value is needed again, it is copied first.  Without that the new
// values of an op live in other registers until the end of its case of the
// opcode switch, which takes the tile's registers twice and spills.
__device__ __forceinline__ double copy_of(double a)
{
     double r;
     asm("v_mov_b64 %0, %1" : "=v"(r) : "v"(a));
     return r;
}
__device__ __forceinline__ float copy_of(float a)
{
     float r;
     asm("v_mov_b32 %0, %1" : "=v"(r) : "v"(a));
     return r;
}
template <typename V>
__device__ __forceinline__ V copy_amp(const V& a)
{
     V r;
     r.x = copy_of(a.x);
     r.y = copy_of(a.y);
     return r;
}

template <typename V, typename R>
__device__ __forceinline__ void cmul(V& a, R fr, R fi)
{
     const R u = a.y * fi, t = a.x * fi;
     a.x = fma(a.x, fr, -u);
     a.y = fma(a.y, fr, t);
}

template <int B, int A, typename V, typename R>
__device__ __forceinline__ void op_real(V (&x)[A], R p, R q)
{
     for_pairs<B>(x, [&](V& a, V& z, int) {
          const V t = copy_amp(a);
          a.x = fma(p, z.x, a.x);
          a.y = fma(p, z.y, a.y);
          z.x = fma(q, t.x, z.x);
          z.y = fma(q, t.y, z.y);
     });
}

template <int B, int A, typename V, typename R>
__device__ __forceinline__ void op_real_minus(V (&x)[A], R p, R q)
{
     for_pairs<B>(x, [&](V& a, V& z, int) {
          const V t = copy_amp(a);
          a.x = fma(p, z.x, a.x);
          a.y = fma(p, z.y, a.y);
          z.x = fma(q, t.x, -z.x);
          z.y = fma(q, t.y, -z.y);
     });
}

template <int B, int A, typename V, typename R>
__device__ __forceinline__ void op_imag(V (&x)[A], R p, R q)
{
     for_pairs<B>(x, [&](V& a, V& z, int) {
          const V t = copy_amp(a);
          a.x = fma(-p, z.y, a.x);
          a.y = fma(p, z.x, a.y);
          z.x = fma(-q, t.y, z.x);
          z.y = fma(q, t.x, z.y);
     });
}

template <int B, int A, typename V, typename R>
__device__ __forceinline__ void op_real4(V (&x)[A], const R (&c)[10])
{
     for_pairs<B>(x, [&](V& a, V& z, int) {
          const R tx = c[2] * a.x, ty = c[2] * a.y;
          a.x *= c[0];
          a.y *= c[0];
          a.x = fma(c[1], z.x, a.x);
          a.y = fma(c[1], z.y, a.y);
          z.x = fma(c[3], z.x, tx);
          z.y = fma(c[3], z.y, ty);
     });
}

template <int B, int A, typename V, typename R>
__device__ __forceinline__ void op_general(V (&x)[A], const R (&c)[10], uint32_t rm, uint32_t rv)
{
     for_pairs<B>(x, [&](V& a, V& z, int i) {
          if ((static_cast<uint32_t>(i) & rm) != rv) return;  // uniform
          const V t = copy_amp(a);
          a.x = fma(-c[3], z.y, fma(c[2], z.x, fma(-c[1], t.y, c[0] * t.x)));
          a.y = fma(c[3], z.x, fma(c[2], z.y, fma(c[1], t.x, c[0] * t.y)));
          const R zx = copy_of(z.x);
          z.x = fma(-c[7], z.y, fma(c[6], z.x, fma(-c[5], t.y, c[4] * t.x)));
          z.y = fma(c[7], zx, fma(c[6], z.y, fma(c[5], t.x, c[4] * t.y)));
     });
}

// Exchanges two registers in place (an ordinary swap of array elements makes
// the compiler keep both orders of the whole array apart at the joins of the
// opcode switch, which spills).
__device__ __forceinline__ void swap_regs(uint32_t& a, uint32_t& b) { asm("v_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
__device__ __forceinline__ void swap_amps(float2& a, float2& z)
{
     uint32_t ax = __float_as_uint(a.x), ay = __float_as_uint(a.y);
     uint32_t zx = __float_as_uint(z.x), zy = __float_as_uint(z.y);
     swap_regs(ax, zx);
     swap_regs(ay, zy);
     a = make_float2(__uint_as_float(ax), __uint_as_float(ay));
     z = make_float2(__uint_as_float(zx), __uint_as_float(zy));
}
__device__ __forceinline__ void swap_half(double& a, double& z)
{
     uint32_t al = __double2loint(a), ah = __double2hiint(a), zl = __double2loint(z), zh = __double2hiint(z);
     swap_regs(al, zl);
     swap_regs(ah, zh);
     a = __hiloint2double(ah, al);
     z = __hiloint2double(zh, zl);
}
__device__ __forceinline__ void swap_amps(double2& a, double2& z)
{
     swap_half(a.x, z.x);
     swap_half(a.y, z.y);
}

template <int B, int A, typename V>
__device__ __forceinline__ void op_swap(V (&x)[A], uint32_t rm, uint32_t rv)
{
     for_pairs<B>(x, [&](V& a, V& z, int i) {
          if ((static_cast<uint32_t>(i) & rm) != rv) return;  // uniform
          swap_amps(a, z);
     });
}

template <int B, int A, typename V>
__device__ __forceinline__ void op_swap_all(V (&x)[A])
{
     for_pairs<B>(x, [&](V& a, V& z, int) { swap_amps(a, z); });
}

// H without its factor, in place.
template <int B, int A, typename V>
__device__ __forceinline__ void op_sum_difference(V (&x)[A])
{
     for_pairs<B>(x, [&](V& a, V& z, int) {
          a.x += z.x;
          a.y += z.y;
          z.x = fma(static_cast<decltype(a.x)>(-2), z.x, a.x);
          z.y = fma(static_cast<decltype(a.y)>(-2), z.y, a.y);
     });
}

// Swap of register bit B where register bit C is set.
template <int B, int C, int A, typename V>
__device__ __forceinline__ void op_cswap(V (&x)[A])
{
     if constexpr (B != C)
          for_pairs<B>(x, [&](V& a, V& z, int i) {
               if (!((i >> C) & 1)) return;  // compile time
               swap_amps(a, z);
          });
}

template <int B, int A, typename V, typename R>
__device__ __forceinline__ void op_phase(V (&x)[A], R fr, R fi)
{
#pragma unroll
     for (int i = 0; i < A; ++i)
          if (B < 0 || ((i >> (B < 0 ? 0 : B)) & 1)) {
               cmul(x[i], fr, fi);
               __builtin_amdgcn_sched_barrier(0);
          }
}

template <int A, typename V, typename R>
__device__ __forceinline__ void op_phase_tested(V (&x)[A], R fr, R fi, uint32_t rm, uint32_t rv)
{
#pragma unroll
     for (int i = 0; i < A; ++i)
          if ((static_cast<uint32_t>(i) & rm) == rv) {
               cmul(x[i], fr, fi);
               __builtin_amdgcn_sched_barrier(0);
          }
}

// 4 x 4 matrix on register bits B0 < B1; row r in the coefficients of m[r].
template <int B0, int B1, int A, typename V, typename R>
__device__ __forceinline__ void op_two(V (&x)[A], const GateOp<R>* __restrict__ m, uint32_t rm, uint32_t rv)
{
#pragma unroll
     for (int j = 0; j < A / 4; ++j) {
          int i = ((j >> B0) << (B0 + 1)) | (j & ((1 << B0) - 1));
          i = ((i >> B1) << (B1 + 1)) | (i & ((1 << B1) - 1));
          if ((static_cast<uint32_t>(i) & rm) != rv) continue;  // uniform
          const int at[4] = {i, i | (1 << B0), i | (1 << B1), i | (1 << B0) | (1 << B1)};
          V v[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) v[k] = copy_amp(x[at[k]]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
               R re = 0, im = 0;
#pragma unroll
               for (int k = 0; k < 4; ++k) {
                    const R mr = m[r].c[2 * k], mi = m[r].c[2 * k + 1];
                    re = fma(-mi, v[k].y, fma(mr, v[k].x, re));
                    im = fma(mi, v[k].x, fma(mr, v[k].y, im));
               }
               x[at[r]].x = re;
               x[at[r]].y = im;
          }
          __builtin_amdgcn_sched_barrier(0);
     }
}

// An opcode whose value the compiler takes as unknown at each use.
__device__ __forceinline__ uint32_t opaque_code(uint32_t c)
{
     asm volatile("" : "+s"(c));
     return c;
}

// What a list needs of a record: its conditions and the two doubles at the
// start of its coefficients.  The scalar unit moves every word of a record
// that is loaded ahead, and has as much to do here as the vector unit.
struct ListRecord {
     uint32_t tcond;
     uint64_t omask, oval;
     double fx, fy;
};
template <typename R>
__device__ __forceinline__ ListRecord load_list_record(const GateOp<R>* __restrict__ p)
{
     const uint32_t* const q = reinterpret_cast<const uint32_t*>(p);
     uint32_t w[9];
#pragma unroll
     for (int i = 0; i < 9; ++i) w[i] = q[i + 1];
     ListRecord r;
     r.tcond = w[0];
     __builtin_memcpy(&r.omask, w + 1, 8);
     __builtin_memcpy(&r.oval, w + 3, 8);
     __builtin_memcpy(&r.fx, w + 5, 8);
     __builtin_memcpy(&r.fy, w + 7, 8);
     return r;
}

// The product of the factors of ops[0..count) whose conditions hold for this
// thread's tile and index; with tables > 0, the list begins with those.  In
// FP64 for either type: a list multiplies one amplitude by many factors, and
// their rounded moduli would add up.
template <typename V, typename R>
__device__ __forceinline__ V factor_product(const GateOp<R>* __restrict__ ops, uint32_t count, uint64_t base,
                                            uint64_t tix, uint32_t tid, uint32_t tables)
{
     double2 f = make_double2(1, 0);
     if (tables) {
          const double* t = reinterpret_cast<const double*>(ops);
          const uint32_t lane = tid & (kGateTableLanes - 1u);
          const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(tid / kGateTableLanes)));
          f.x = t[2 * lane];
          f.y = t[2 * lane + 1];
          t += 2 * kGateTableLanes;
          cmul(f, t[2 * wave], t[2 * wave + 1]);
          t += 2 * kGateTableWaves;
          uint32_t left = static_cast<uint32_t>(tix);  // (n <= 40: 27 bits at most)
          for (uint32_t g = 1; g < tables; ++g) {
               const uint32_t i = left & ((1u << kGateTableBits) - 1u);
               cmul(f, t[2 * i], t[2 * i + 1]);
               t += 2 << kGateTableBits;
               left >>= kGateTableBits;
          }
          const uint32_t skip = static_cast<uint32_t>((gate_table_entries(static_cast<int>(tables) - 1) * 16 + sizeof(GateOp<R>) - 1) / sizeof(GateOp<R>));
          ops += skip;
          count -= skip;
     }
     ListRecord cur = load_list_record(ops);  // (a list is never the last record)
#pragma unroll 2
     for (uint32_t e = 0; e < count; ++e) {
          asm volatile("" : "+s"(cur.tcond));
          __builtin_amdgcn_sched_barrier(0);
          const ListRecord nxt = load_list_record(ops + e + 1);
          if ((base & cur.omask) == cur.oval) {  // uniform
               if (cur.tcond == 0) cmul(f, cur.fx, cur.fy);
               if (opaque_code(cur.tcond) != 0) {
                    const bool on = (tid & (cur.tcond & 0xffffu)) == (cur.tcond >> 16);
                    cmul(f, on ? cur.fx : 1.0, on ? cur.fy : 0.0);
               }
          }
          cur = nxt;
     }
     V r;
     r.x = static_cast<R>(f.x);
     r.y = static_cast<R>(f.y);
     return r;
}

// Ties every amplitude to one register for all paths that join here.
template <int A, typename V>
__device__ __forceinline__ void pin(V (&x)[A])
{
#pragma unroll
     for (int k = 0; k < A; ++k) asm volatile("" : "+v"(x[k].x), "+v"(x[k].y));
}

#define HQ_IN(LO, HI) if (opaque_code(code) - static_cast<uint32_t>(LO) < static_cast<uint32_t>((HI) - (LO)))
#define HQ_AT(K) if (opaque_code(code) == static_cast<uint32_t>(K))
// CALL with B = code - K, for the E register bits.
#define HQ_BITS(K, CALL)                                                       \
     HQ_IN(K, K + E)                                                           \
     {                                                                         \
          HQ_AT(K + 0) { constexpr int B = 0; CALL; }                          \
          HQ_AT(K + 1) { constexpr int B = 1; CALL; }                          \
          HQ_AT(K + 2) { constexpr int B = 2; CALL; }                          \
          HQ_AT(K + 3) { constexpr int B = 3; CALL; }                          \
          if constexpr (E > 4) HQ_AT(K + 4) { constexpr int B = E - 1; CALL; } \
     }

// Swap of bit `code` / 8 under bit `code` % 8.
template <int E, typename V, int A>
__device__ __forceinline__ void coded_swap(V (&x)[A], const uint32_t pair)
{
     const uint32_t c = pair & 7u;
     const uint32_t code = pair >> 3;
#define HQ_CTRL(C) if (opaque_code(c) == C) op_cswap<B, C>(x);
     HQ_BITS(0, HQ_CTRL(0) HQ_CTRL(1) HQ_CTRL(2) HQ_CTRL(3) if constexpr (E > 4) { HQ_CTRL(E - 1) })
#undef HQ_CTRL
}

// A layer: rotations, phases, swaps.
template <typename R, int E, typename V, int A>
__device__ __forceinline__ void run_layer(V (&x)[A], const GateOp<R>& o, const GateOp<R>* __restrict__ next)
{
     const uint32_t aux = o.code >> 16;
#define HQ_ROT(B)                                                                          \
     {                                                                                     \
          const uint32_t code = (aux >> (2 * (B))) & 3u;                                   \
          HQ_AT(kGateKindReal) { op_real<B>(x, o.c[2 * (B)], o.c[2 * (B) + 1]); }          \
          HQ_AT(kGateKindH) { op_sum_difference<B>(x); }                                   \
          HQ_AT(kGateKindImag) { op_imag<B>(x, o.c[2 * (B)], o.c[2 * (B) + 1]); }          \
     }
     if (opaque_code(aux) & ((1u << 2 * E) - 1u)) {
          HQ_ROT(0)
          HQ_ROT(1)
          HQ_ROT(2)
          HQ_ROT(3)
          if constexpr (E > 4) HQ_ROT(E - 1)
     }
#undef HQ_ROT
     if (opaque_code(aux) >> 10) {
          const GateOp<R> f = load_record(next);
#define HQ_PH(B) \
     if (opaque_code(aux) & (1u << (10 + (B)))) op_phase<B>(x, f.c[2 * (B)], f.c[2 * (B) + 1]);
          HQ_PH(0)
          HQ_PH(1)
          HQ_PH(2)
          HQ_PH(3)
          if constexpr (E > 4) { HQ_PH(E - 1) }
#undef HQ_PH
     }
     uint64_t lo = o.omask, hi = o.oval;
     for (uint32_t i = 0; i < o.tcond; ++i) {
          coded_swap<E>(x, static_cast<uint32_t>(lo) & 0xffu);
          lo = (lo >> 8) | (hi << 56);
          hi >>= 8;
          pin(x);
     }
}

// Stage ops on the registers, in order.
//
// The dispatch is made of nested one-sided ifs, each on a code the compiler
// cannot relate to the others: a switch (or an else) is rebuilt into a form
// that keeps the amplitudes before and after each branch alive together,
// which takes their registers twice and spills.
template <typename R, typename V, int A>
__device__ __forceinline__ void run_ops(V (&x)[A], const GateOp<R>* __restrict__ ops, const uint32_t nops,
                                        const uint64_t base, const uint64_t tix, const uint32_t tid)
{
     constexpr int E = Shape<R>::E;
     if (nops == 0) return;
     GateOp<R> cur = load_record(ops);
     uint32_t p = 0;
     do {
          // cur is here before the next record's loads are issued, so that
          // nothing waits for those until the op is done.
          asm volatile("" : "+s"(cur.code));
          __builtin_amdgcn_sched_barrier(0);
          const uint32_t count = (cur.code >> 8) & 0xffu;
          const GateOp<R>* const list = ops + p + 1;
          p += 1 + count;
          const GateOp<R> nxt = load_record(ops + p);  // (one spare record at the end)
          const uint32_t code = cur.code & 0xffu;
          HQ_AT(kGateLayer) { run_layer<R, E>(x, cur, list); }
          if (opaque_code(code) != kGateLayer && (base & cur.omask) == cur.oval &&
              (tid & (cur.tcond & 0xffffu)) == (cur.tcond >> 16)) {
               const uint32_t rm = (cur.code >> 16) & 31u, rv = (cur.code >> 21) & 31u;
               HQ_IN(kGateRM, kGateXC)
               {
                    HQ_IN(kGateRM, kGateXA)
                    {
                         HQ_BITS(kGateRM, op_real_minus<B>(x, cur.c[0], cur.c[1]))
                         HQ_BITS(kGateR4, op_real4<B>(x, cur.c))
                         HQ_BITS(kGateG, op_general<B>(x, cur.c, rm, rv))
                    }
                    HQ_BITS(kGateXA, op_swap_all<B>(x))
                    HQ_BITS(kGateX, op_swap<B>(x, rm, rv))
               }
               HQ_IN(kGateXC, kGateG2)
               {
                    HQ_AT(kGateXC) { coded_swap<E>(x, cur.code >> 16); }
                    HQ_AT(kGatePAll) { op_phase<-1>(x, cur.c[0], cur.c[1]); }
                    HQ_AT(kGatePT) { op_phase_tested(x, cur.c[0], cur.c[1], rm, rv); }
                    HQ_IN(kGatePA, kGateG2)
                    {
                         const V f = factor_product<V, R>(list, count, base, tix, tid, rm);
                         HQ_BITS(kGatePA, op_phase<B>(x, f.x, f.y))
                         HQ_AT(kGatePL) { op_phase<-1>(x, f.x, f.y); }
                    }
               }
               HQ_IN(kGateG2, kGateCodes)
               {
                    HQ_AT(kGateG2 + gate_pair(0, 1)) { op_two<0, 1>(x, list, rm, rv); }
                    HQ_AT(kGateG2 + gate_pair(0, 2)) { op_two<0, 2>(x, list, rm, rv); }
                    HQ_AT(kGateG2 + gate_pair(1, 2)) { op_two<1, 2>(x, list, rm, rv); }
                    HQ_AT(kGateG2 + gate_pair(0, 3)) { op_two<0, 3>(x, list, rm, rv); }
                    HQ_AT(kGateG2 + gate_pair(1, 3)) { op_two<1, 3>(x, list, rm, rv); }
                    HQ_AT(kGateG2 + gate_pair(2, 3)) { op_two<2, 3>(x, list, rm, rv); }
                    if constexpr (E > 4) {
                         HQ_AT(kGateG2 + gate_pair(0, 4)) { op_two<0, E - 1>(x, list, rm, rv); }
                         HQ_AT(kGateG2 + gate_pair(1, 4)) { op_two<1, E - 1>(x, list, rm, rv); }
                         HQ_AT(kGateG2 + gate_pair(2, 4)) { op_two<2, E - 1>(x, list, rm, rv); }
                         HQ_AT(kGateG2 + gate_pair(3, 4)) { op_two<3, E - 1>(x, list, rm, rv); }
                    }
               }
          }
          pin(x);
          cur = nxt;
     } while (p < nops);
}
#undef HQ_BITS
#undef HQ_AT
#undef HQ_IN

// A value the compiler takes as new: what is computed from it is computed
// again at each use instead of being held in registers beside the tile.
__device__ __forceinline__ uint32_t fresh(uint32_t v)
{
     asm volatile("" : "+v"(v));
     return v;
}

// Byte offset of a thread's bits: the XOR of the offsets of its set bits.
__device__ __forceinline__ uint32_t thread_slot(uint32_t tid, const uint16_t (&m)[kGateThr])
{
     uint32_t s = 0;
#pragma unroll
     for (int j = 0; j < kGateThr; ++j) s ^= static_cast<uint32_t>(-static_cast<int32_t>((tid >> j) & 1u)) & m[j];
     return s;
}

__device__ __forceinline__ uint32_t reg_slot(int k, const uint16_t (&m)[kGateMaxReg])
{
     uint32_t s = 0;
#pragma unroll
     for (int b = 0; b < kGateMaxReg; ++b)
          if ((k >> b) & 1) s ^= m[b];
     return s;
}

// The tile from one stage's grouping to the next one's, through 64 KiB of
// LDS: the real parts, then the imaginary parts, so that two workgroups share
// a CU.  w, r: the thread's slots in the two groupings; a, b: their register
// bits' offsets.
template <typename R, typename V, int A>
__device__ __forceinline__ void regroup(V (&x)[A], char* lds, uint32_t w, uint32_t r,
                                        const uint16_t (&a)[kGateMaxReg], const uint16_t (&b)[kGateMaxReg])
{
     // The fences keep the addresses of a few accesses at a time in
     // registers, not those of all.
     __syncthreads();  // the previous regrouping has been read
#pragma unroll
     for (int k = 0; k < A; ++k) {
          *reinterpret_cast<R*>(lds + (w ^ reg_slot(k, a))) = x[k].x;
          if ((k & 3) == 3) __builtin_amdgcn_sched_barrier(0);
     }
     __syncthreads();
#pragma unroll
     for (int k = 0; k < A; ++k) x[k].x = *reinterpret_cast<const R*>(lds + (r ^ reg_slot(k, b)));
     __syncthreads();
     w = fresh(w);
     r = fresh(r);
#pragma unroll
     for (int k = 0; k < A; ++k) {
          *reinterpret_cast<R*>(lds + (w ^ reg_slot(k, a))) = x[k].y;
          if ((k & 3) == 3) __builtin_amdgcn_sched_barrier(0);
     }
     __syncthreads();
#pragma unroll
     for (int k = 0; k < A; ++k) x[k].y = *reinterpret_cast<const R*>(lds + (r ^ reg_slot(k, b)));
}

__device__ __forceinline__ uint64_t thread_index(uint32_t tid, const uint8_t (&pos)[kGateThr])
{
     uint64_t i = 0;
#pragma unroll
     for (int j = 0; j < kGateThr; ++j) i |= static_cast<uint64_t>((tid >> j) & 1u) << pos[j];
     return i;
}

__device__ __forceinline__ uint64_t reg_index(int k, const uint8_t (&pos)[kGateMaxReg])
{
     uint64_t i = 0;
#pragma unroll
     for (int b = 0; b < kGateMaxReg; ++b) i |= static_cast<uint64_t>((k >> b) & 1) << pos[b];
     return i;
}

template <typename R, typename V>
__device__ __forceinline__ VT<R> converted(const V& a)
{
     VT<R> r;
     r.x = static_cast<R>(a.x);
     r.y = static_cast<R>(a.y);
     return r;
}

// S: the state's type; R: the type that the amplitudes have while the pass
// holds them.
// Copies that the register allocator cannot merge away.  The loads and stores
// work on whole amplitudes in consecutive registers while the regrouping
// moves real and imaginary parts separately; tied to the loads' registers the
// whole array ends up twice in the register file, and spills.
template <typename S, typename R>
__device__ __forceinline__ void gate_program(VT<S>* psi, const GatePass& P,
                                             const GateStage* __restrict__ stages,
                                             const GateOp<R>* __restrict__ ops, const uint64_t tix, char* lds,
                                             VT<S>* dst)
{
     using V = VT<R>;
     constexpr int E = Shape<R>::E, A = 1 << E, H = Shape<R>::T - kGateLow;
     const uint32_t tid = threadIdx.x;
     uint64_t base = tix << kGateLow;
#pragma unroll
     for (int j = 0; j < H; ++j) {
          const uint64_t lo = base & ((1ull << P.hpos[j]) - 1ull);
          base = ((base ^ lo) << 1) | lo;
     }
     V x[A];
     {
          const VT<S>* const p = psi + base + thread_index(tid, P.in_thr);
          if constexpr (sizeof(S) == sizeof(R)) {
#pragma unroll
               for (int k = 0; k < A; ++k) {
                    x[k] = ld_nt(p + reg_index(k, P.in_reg));
                    if ((k & 3) == 3) __builtin_amdgcn_sched_barrier(0);
               }
#pragma unroll
               for (int k = 0; k < A; ++k) x[k] = copy_amp(x[k]);
          }
          else {
               VT<S> in[A];
#pragma unroll
               for (int k = 0; k < A; ++k) {
                    in[k] = ld_nt(p + reg_index(k, P.in_reg));
                    if ((k & 3) == 3) __builtin_amdgcn_sched_barrier(0);
               }
#pragma unroll
               for (int k = 0; k < A; ++k) x[k] = converted<R>(in[k]);
          }
     }
     uint32_t s = 0, slot = 0;
     do {
          const GateStage st = load_record(stages + s);
          const uint32_t to = thread_slot(tid, st.thr_lds);
          if (s > 0) regroup<R>(x, lds, slot, to, load_record(stages + s - 1).reg_lds, st.reg_lds);
          slot = to;
          run_ops<R>(x, ops + st.op_first, st.nops, base, tix, tid);
     } while (++s < P.nstages);
     uint64_t to = base;
     if (P.permuted) {
          to = 0;
#pragma unroll
          for (int j = 0; j < kGateMaxBase; ++j) to |= ((tix >> j) & 1) << P.base_out[j];
     }
     VT<S>* const p = dst + to + thread_index(fresh(tid), P.out_thr);
#pragma unroll
     for (int k = 0; k < A; ++k) {
          st_nt(p + reg_index(k, P.out_reg), converted<S>(copy_amp(x[k])));
          if ((k & 3) == 3) __builtin_amdgcn_sched_barrier(0);
     }
}

template <typename S, typename R>
__global__ void __launch_bounds__(kGateThreads) __attribute__((amdgpu_waves_per_eu(4)))
    k_gate_pass(VT<S>* psi, const GatePass P, const GateStage* __restrict__ stages,
                const GateOp<R>* __restrict__ ops, const int swz, const uint64_t nblocks, VT<S>* dst)
{
     __shared__ __align__(16) char lds[sizeof(R) << Shape<R>::T];
     const uint64_t b = block_linear();
     if (b >= nblocks) return;  // padding of the 2-D grid (whole block)
     gate_program<S, R>(psi, P, stages + P.stage_first, ops, swizzle_block(b, swz), lds, dst);
}

}  // namespace

hipError_t launch_gate_pass(void* psi, Prec prec, Prec held, int n_qubits, const GatePass& pass, const GateStage* stages,
                            const void* ops, hipStream_t s, void* dst)
{
     if (pass.permuted ? (!dst || dst == psi) : (dst && dst != psi)) return hipErrorInvalidValue;
     if (!dst) dst = psi;
     const int T = gate_tile_bits(held);
     if (n_qubits < T || n_qubits > 40 || pass.nstages < 1) return hipErrorInvalidValue;
     for (int j = 0; j < T - kGateLow; ++j)
          if (pass.hpos[j] < kGateLow || pass.hpos[j] >= n_qubits || (j && pass.hpos[j] <= pass.hpos[j - 1]))
               return hipErrorInvalidValue;
     const uint64_t blocks = 1ull << (n_qubits - T);
     const int bits = get_block_swizzle();
     const int swz = (bits > 0 && bits <= 16 && blocks % (1ull << bits) == 0) ? bits : 0;
     if (prec == Prec::C128 && held == Prec::C128)
          hipLaunchKernelGGL((k_gate_pass<double, double>), grid_2d(blocks), dim3(kGateThreads), 0, s,
                             static_cast<double2*>(psi), pass, stages, static_cast<const GateOp<double>*>(ops), swz,
                             blocks, static_cast<double2*>(dst));
     else if (prec == Prec::C64 && held == Prec::C128)
          hipLaunchKernelGGL((k_gate_pass<float, double>), grid_2d(blocks), dim3(kGateThreads), 0, s,
                             static_cast<float2*>(psi), pass, stages, static_cast<const GateOp<double>*>(ops), swz,
                             blocks, static_cast<float2*>(dst));
     else if (prec == Prec::C64)
          hipLaunchKernelGGL((k_gate_pass<float, float>), grid_2d(blocks), dim3(kGateThreads), 0, s,
                             static_cast<float2*>(psi), pass, stages, static_cast<const GateOp<float>*>(ops), swz,
                             blocks, static_cast<float2*>(dst));
     else return hipErrorInvalidValue;
     return hipGetLastError();
}

}  // namespace hq
