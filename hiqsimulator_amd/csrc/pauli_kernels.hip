// gfx950 kernels of the planned Pauli sums (pauli_prog.hpp).
//
// Bound: HBM for a few groups a pass (one read of the state; apply: a read
// and one or two writes more), vector issue and LDS beyond about twenty terms.
// Before, every term was a pass of its own.  Expectation of 101 terms (26
// qubits, complex128): 101 passes of 0.2 ms, 3 of 0.36 ms now, 0.17 ms of each
// for the read; evolution under 39 terms (20 qubits): 2883 passes, 57 of 13.9
// us now.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.hpp"
#include "pauli_prog.hpp"

namespace hq {
namespace {

template <typename T>
__device__ __forceinline__ T load_words(const T* __restrict__ p)
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

// Where a tile lies and where a thread's amplitudes lie in it: amplitude k of
// thread t is tile rank index k * 2^THR + t.
template <int A, int THR>
struct TileAt {
     static constexpr int KB = A == 8 ? 3 : (A == 4 ? 2 : (A == 2 ? 1 : 0));
     static constexpr int H = THR + KB - kPauliLow;
     uint64_t lane;   // index bits of the thread
     uint64_t reg[A]; // index bits of the amplitude number (uniform)

     __device__ __forceinline__ TileAt(const PauliPass& P, uint32_t tid)
     {
          lane = tid & ((1u << kPauliLow) - 1u);
#pragma unroll
          for (int j = 0; j < THR - kPauliLow; ++j)
               lane |= static_cast<uint64_t>((tid >> (kPauliLow + j)) & 1u) << P.hpos[j];
#pragma unroll
          for (int k = 0; k < A; ++k) {
               uint64_t o = 0;
#pragma unroll
               for (int j = 0; j < KB; ++j) o |= static_cast<uint64_t>((k >> j) & 1) << P.hpos[THR - kPauliLow + j];
               reg[k] = o;
          }
     }
     __device__ __forceinline__ uint64_t base(const PauliPass& P, uint64_t tix) const
     {
          uint64_t b = tix << kPauliLow;
#pragma unroll
          for (int j = 0; j < H; ++j) {
               const uint64_t lo = b & ((1ull << P.hpos[j]) - 1ull);
               b = ((b ^ lo) << 1) | lo;
          }
          return b;
     }
};

// The parity of k & zk as a factor +-1 (uniform).
__device__ __forceinline__ double amp_sign(int k, uint32_t zk)
{
     return __hiloint2double(0x3ff00000 | static_cast<int>(__popc(static_cast<uint32_t>(k) & zk) << 31), 0);
}

// Runs the records of a pass on one tile: done(t, w) for every group, t its
// last record and w[k] = sum over its terms of c (-1)^{|i & z|} for amplitude
// k.  The sign splits into the tile's (uniform), the thread's and the
// amplitude number's (uniform).  Classes (terms that share the amplitude
// number's part) are those of kPauliThr thread bits, which is right for more
// of them, too.
template <int A, int THR, typename Done>
__device__ __forceinline__ void run_terms(const PauliTerm* __restrict__ terms, const uint32_t count, const uint64_t base,
                                          const uint32_t tid, Done&& done)
{
     double w[A], v = 0;
#pragma unroll
     for (int k = 0; k < A; ++k) w[k] = 0;
     PauliTerm cur = load_words(terms);
     for (uint32_t t = 0; t < count; ++t) {
          asm volatile("" : "+s"(cur.z_tile));
          __builtin_amdgcn_sched_barrier(0);
          const PauliTerm nxt = load_words(terms + t + 1);  // (one spare record at the end)
          const uint32_t uni = static_cast<uint32_t>(__popcll(base & cur.z_out));
          const uint32_t sgn = (__popc(tid & cur.z_tile & ((1u << THR) - 1u)) + uni) << 31;
          v += __hiloint2double(__double2hiint(cur.c) ^ static_cast<int>(sgn), __double2loint(cur.c));
          if (cur.z_tile & kPauliClassEnd) {
               const uint32_t zk = (cur.z_tile & 0xffffu) >> THR;
#pragma unroll
               for (int k = 0; k < A; ++k) w[k] = fma(v, amp_sign(k, zk), w[k]);
               v = 0;
               if (cur.z_tile & kPauliGroupEnd) {
                    done(cur, w);
#pragma unroll
                    for (int k = 0; k < A; ++k) w[k] = 0;
               }
          }
          cur = nxt;
     }
}

// sum_k w[k] Re (IM: Im) of conj(y_k) x_k, y the amplitude at i ^ x; KB >= 0:
// only the amplitudes whose number has bit KB clear.
template <int KB, bool IM, typename V, int A>
__device__ __forceinline__ double group_part(const V (&x)[A], const double (&w)[A], const V* tile, uint32_t tid, uint32_t xm)
{
     double s = 0;
#pragma unroll
     for (int k = 0; k < A; ++k) {
          if (KB >= 0 && ((k >> (KB < 0 ? 0 : KB)) & 1)) continue;
          const V y = tile[(k * kPauliThreads + tid) ^ xm];
          const double yr = y.x, yi = y.y, xr = x[k].x, xi = x[k].y;
          s = fma(w[k], IM ? fma(yr, xi, -(yi * xr)) : fma(yr, xr, yi * xi), s);
     }
     return s;
}
template <int KB, typename V, int A>
__device__ __forceinline__ double group_sum(const V (&x)[A], const double (&w)[A], const V* tile, uint32_t tid, uint32_t xm,
                                            bool im)
{
     return im ? group_part<KB, true>(x, w, tile, tid, xm) : group_part<KB, false>(x, w, tile, tid, xm);
}

template <typename R, int A>
__global__ void __launch_bounds__(kPauliThreads)
    k_pauli_sum(const VT<R>* __restrict__ psi, const PauliPass P, const PauliTerm* __restrict__ terms,
                const uint64_t ntiles, double* __restrict__ partials)
{
     using V = VT<R>;
     __shared__ V tile[kPauliThreads * A];
     const uint32_t tid = threadIdx.x;
     const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(tid)));
     const TileAt<A, kPauliThr> at(P, tid);
     double acc[2] = {0.0, 0.0};
     for (uint64_t tix = blockIdx.x; tix < ntiles; tix += gridDim.x) {
          const uint64_t base = at.base(P, tix);
          V x[A];
#pragma unroll
          for (int k = 0; k < A; ++k) x[k] = ld_nt(psi + base + at.lane + at.reg[k]);
          __syncthreads();  // the previous tile has been read
#pragma unroll
          for (int k = 0; k < A; ++k) tile[k * kPauliThreads + tid] = x[k];
          __syncthreads();
          run_terms<A, kPauliThr>(terms + P.first, P.count, base, tid, [&](const PauliTerm& t, const double (&w)[A]) {
               const bool im = t.z_tile & kPauliImag;
               double s = 0;
               // the half that the highest bit of x selects (pauli_prog.cpp)
               const uint32_t kx = t.x >> kPauliThr;
               const uint32_t wx = t.x & ((1u << kPauliThr) - (1u << kPauliLane));
               if (kx >= 4u) {
                    if constexpr (A >= 8) s = group_sum<2>(x, w, tile, tid, t.x, im);
               }
               else if (kx >= 2u) {
                    if constexpr (A >= 4) s = group_sum<1>(x, w, tile, tid, t.x, im);
               }
               else if (kx) {
                    if constexpr (A >= 2) s = group_sum<0>(x, w, tile, tid, t.x, im);
               }
               else if (wx) {
                    if (!((wave >> (31 - __clz(static_cast<int>(wx)))) & 1u)) s = group_sum<-1>(x, w, tile, tid, t.x, im);
               }
               else {
                    s = group_sum<-1>(x, w, tile, tid, t.x, im);
               }
               if (t.z_tile & kPauliOut1) acc[1] += s;
               else acc[0] += s;
          });
     }
     // wave sums, then one partial a block
     __shared__ double red[2][kPauliThreads / 64];
#pragma unroll
     for (int o = 0; o < 2; ++o) {
          double v = acc[o];
          for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
          if ((tid & 63) == 0) red[o][tid >> 6] = v;
     }
     __syncthreads();
     if (tid < 2) {
          double v = 0;
          for (int i = 0; i < kPauliThreads / 64; ++i) v += red[tid][i];
          partials[tid * gridDim.x + blockIdx.x] = v;
     }
}

// Sum of the partials of NOUT outputs; with skip (below) the old value stays.
__global__ void __launch_bounds__(kBlock)
    k_sum_partials(const double* __restrict__ partials, const int nblocks, double* __restrict__ out,
                   const double* __restrict__ skip, const double skip_below)
{
     const int o = blockIdx.x;
     if (skip && skip[0] < skip_below) {
          if (threadIdx.x == 0) out[o] = skip[0];
          return;
     }
     double v = 0;
     for (int i = threadIdx.x; i < nblocks; i += kBlock) v += partials[o * nblocks + i];
     for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
     __shared__ double red[kBlock / 64];
     if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
     __syncthreads();
     if (threadIdx.x == 0) {
          double s = 0;
          for (int i = 0; i < kBlock / 64; ++i) s += red[i];
          out[o] = s;
     }
}

template <typename R>
struct ApplyArgs {
     const VT<R>* src;
     VT<R>* dst;
     const VT<R>* add;
     const VT<R>* o_src;
     VT<R>* o_dst;
     const double* skip;
     double skip_below;
     R fr, fi, g, h, cr, ci, er, ei;
};

template <typename R, int A, int THR>
__global__ void __launch_bounds__(1 << THR)
    k_pauli_apply(const ApplyArgs<R> a, const PauliPass P, const PauliTerm* __restrict__ terms,
                  const uint64_t ntiles, double* __restrict__ partials)
{
     using V = VT<R>;
     constexpr int kThreads = 1 << THR;
     if (a.skip && a.skip[0] < a.skip_below) return;  // the whole grid
     __shared__ V tile[kThreads * A];
     const uint32_t tid = threadIdx.x;
     const TileAt<A, THR> at(P, tid);
     double norm = 0;
     for (uint64_t tix = blockIdx.x; tix < ntiles; tix += gridDim.x) {
          const uint64_t base = at.base(P, tix);
          V o[A];
#pragma unroll
          for (int k = 0; k < A; ++k) o[k] = a.src[base + at.lane + at.reg[k]];
          __syncthreads();  // the previous tile has been read
#pragma unroll
          for (int k = 0; k < A; ++k) {
               tile[k * kThreads + tid] = o[k];
               o[k].x = o[k].y = 0;
          }
          V d[A];  // what the result is added to, on its way meanwhile
#pragma unroll
          for (int k = 0; k < A; ++k) d[k].x = d[k].y = 0;
          if (a.add) {
#pragma unroll
               for (int k = 0; k < A; ++k) d[k] = a.add[base + at.lane + at.reg[k]];
          }
          __syncthreads();
          run_terms<A, THR>(terms + P.first, P.count, base, tid, [&](const PauliTerm& t, const double (&w)[A]) {
               // two one-sided ifs on a flag the compiler cannot relate: an
               // if-else would keep the sums before and after both alive
               uint32_t real = ~t.z_tile & kPauliImag;
               asm volatile("" : "+s"(real));
               if (real) {
#pragma unroll
                    for (int k = 0; k < A; ++k) {
                         const V y = tile[(k * kThreads + tid) ^ t.x];
                         const R v = static_cast<R>(w[k]);
                         o[k].x = fma(v, y.x, o[k].x);
                         o[k].y = fma(v, y.y, o[k].y);
                    }
               }
               if (t.z_tile & kPauliImag) {
#pragma unroll
                    for (int k = 0; k < A; ++k) {
                         const V y = tile[(k * kThreads + tid) ^ t.x];
                         const R v = static_cast<R>(w[k]);
                         o[k].x = fma(-v, y.y, o[k].x);
                         o[k].y = fma(v, y.x, o[k].y);
                    }
               }
          });
#pragma unroll
          for (int k = 0; k < A; ++k) {
               const uint64_t i = base + at.lane + at.reg[k];
               V b;
               b.x = fma(-a.fi, o[k].y, a.fr * o[k].x);
               b.y = fma(a.fi, o[k].x, a.fr * o[k].y);
               b.x = fma(a.g, d[k].x, b.x);
               b.y = fma(a.g, d[k].y, b.y);
               a.dst[i] = b;
               if (a.o_dst) {
                    const V e = tile[k * kThreads + tid];
                    V s;
                    s.x = fma(-a.ei, e.y, a.er * e.x);
                    s.y = fma(a.ei, e.x, a.er * e.y);
                    if (a.o_src) {
                         const V t = a.o_src[i];
                         s.x = fma(a.h, t.x, s.x);
                         s.y = fma(a.h, t.y, s.y);
                    }
                    s.x = fma(-a.ci, b.y, fma(a.cr, b.x, s.x));
                    s.y = fma(a.ci, b.x, fma(a.cr, b.y, s.y));
                    a.o_dst[i] = s;
                    const double br = b.x, bi = b.y;
                    norm = fma(br, br, fma(bi, bi, norm));
               }
          }
     }
     if (!partials) return;
     for (int d = 32; d > 0; d >>= 1) norm += __shfl_xor(norm, d, 64);
     __shared__ double red[kThreads / 64];
     if ((tid & 63) == 0) red[tid >> 6] = norm;
     __syncthreads();
     if (tid == 0) {
          double v = 0;
          for (int i = 0; i < kThreads / 64; ++i) v += red[i];
          partials[blockIdx.x] = v;
     }
}

bool pass_fits(const PauliPass& p, int n)
{
     if (n < kPauliMinQubits || n > 40) return false;
     const int H = pauli_tile_bits(n) - kPauliLow;
     for (int j = 0; j < H; ++j)
          if (p.hpos[j] < kPauliLow || p.hpos[j] >= n || (j && p.hpos[j] <= p.hpos[j - 1])) return false;
     return true;
}

template <typename R, int A>
void sum_launch(const void* psi, const PauliPass& p, const PauliTerm* t, uint64_t ntiles, int grid,
                double* scratch, hipStream_t s)
{
     hipLaunchKernelGGL((k_pauli_sum<R, A>), dim3(grid), dim3(kPauliThreads), 0, s, static_cast<const VT<R>*>(psi), p, t,
                        ntiles, scratch);
}
template <typename R, int A>
void apply_launch(const PauliApply& a, const PauliPass& p, const PauliTerm* t, uint64_t ntiles,
                  int grid, hipStream_t s)
{
     ApplyArgs<R> k{};
     k.src = static_cast<const VT<R>*>(a.src);
     k.dst = static_cast<VT<R>*>(a.dst);
     k.o_src = static_cast<const VT<R>*>(a.o_src);
     k.o_dst = static_cast<VT<R>*>(a.o_dst);
     k.skip = a.skip;
     k.skip_below = a.skip_below;
     k.add = static_cast<const VT<R>*>(a.add);
     k.fr = static_cast<R>(a.fr);
     k.fi = static_cast<R>(a.fi);
     k.g = static_cast<R>(a.g);
     k.h = static_cast<R>(a.h);
     k.cr = static_cast<R>(a.cr);
     k.ci = static_cast<R>(a.ci);
     k.er = static_cast<R>(a.er);
     k.ei = static_cast<R>(a.ei);
     // One workgroup a CU at most: twice the threads, half the amplitudes each,
     // hide more of each other's latency (20 qubits, complex128: 14.8 us a pass
     // with 512 threads, 13.9 us with 1024).  With more tiles two workgroups of
     // 512 share a CU and overlap.
     if constexpr (A > 1)
          if (ntiles <= 256) {
               hipLaunchKernelGGL((k_pauli_apply<R, A / 2, kPauliThr + 1>), dim3(grid), dim3(2 * kPauliThreads), 0, s, k, p,
                                  t, ntiles, a.norm ? a.scratch : nullptr);
               return;
          }
     hipLaunchKernelGGL((k_pauli_apply<R, A, kPauliThr>), dim3(grid), dim3(kPauliThreads), 0, s, k, p, t, ntiles,
                        a.norm ? a.scratch : nullptr);
}

// f<A>() for the amplitudes a thread of an n-qubit state's tile holds.
#define HQ_PAULI(RR, CALL)                                  \
     switch (pauli_tile_bits(n) - kPauliThr) {              \
          case 0: { using R = RR; constexpr int A = 1; CALL; } break; \
          case 1: { using R = RR; constexpr int A = 2; CALL; } break; \
          case 2: { using R = RR; constexpr int A = 4; CALL; } break; \
          default: { using R = RR; constexpr int A = 8; CALL; } break; \
     }

}  // namespace

hipError_t launch_pauli_sum(const void* psi, Prec prec, int n, const PauliPass& pass, const PauliTerm* terms,
                            double* scratch, double* out, hipStream_t s)
{
     if (!pass_fits(pass, n)) return hipErrorInvalidValue;
     const uint64_t ntiles = 1ull << (n - pauli_tile_bits(n));
     const int grid = static_cast<int>(ntiles < kReduceBlocks ? ntiles : kReduceBlocks);
     if (prec == Prec::C128) HQ_PAULI(double, (sum_launch<R, A>(psi, pass, terms, ntiles, grid, scratch, s)))
     else HQ_PAULI(float, (sum_launch<R, A>(psi, pass, terms, ntiles, grid, scratch, s)))
     const hipError_t e = hipGetLastError();
     if (e != hipSuccess) return e;
     hipLaunchKernelGGL(k_sum_partials, dim3(2), dim3(kBlock), 0, s, scratch, grid, out, nullptr, 0.0);
     return hipGetLastError();
}

hipError_t launch_pauli_apply(const PauliApply& a, Prec prec, int n, const PauliPass& pass, const PauliTerm* terms,
                              hipStream_t s)
{
     if (!pass_fits(pass, n) || a.src == a.dst || (a.norm && (!a.o_dst || !a.scratch)))
          return hipErrorInvalidValue;
     const uint64_t ntiles = 1ull << (n - pauli_tile_bits(n));
     const int grid = static_cast<int>(ntiles < kReduceBlocks ? ntiles : kReduceBlocks);
     if (prec == Prec::C128) HQ_PAULI(double, (apply_launch<R, A>(a, pass, terms, ntiles, grid, s)))
     else HQ_PAULI(float, (apply_launch<R, A>(a, pass, terms, ntiles, grid, s)))
     const hipError_t e = hipGetLastError();
     if (e != hipSuccess || !a.norm) return e;
     hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(kBlock), 0, s, a.scratch, grid, a.norm, a.skip, a.skip_below);
     return hipGetLastError();
}

#undef HQ_PAULI

}  // namespace hq
