// Device-to-host copies of states, widened to complex128.
#include "readback.hpp"
#include "device_common.hpp"
#include <chrono>
#include <cstring>
#include <stdexcept>
#include <string>

namespace hq {
namespace {

constexpr int kThreads = 1024;

template <typename V>
__global__ void __launch_bounds__(kThreads)
    k_read_out(double2* __restrict__ dst, const V* __restrict__ src, const uint64_t n)
{
     const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
     if (i >= n) return;
     const V a = src[i];
     dst[i] = make_double2(a.x, a.y);
}

template <typename V>
__global__ void __launch_bounds__(kThreads)
    k_read_out_one(double2* __restrict__ dst, const V* __restrict__ src, const int n, uint64_t* __restrict__ flag,
                   const uint64_t seq)
{
     for (int i = threadIdx.x; i < n; i += kThreads) dst[i] = make_double2(src[i].x, src[i].y);
     // (host memory is not cached on the device: once a wave's stores are out,
     // they are ahead of the flag)
     asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
     __syncthreads();
     if (threadIdx.x == 0) __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

void ok(hipError_t e, const char* what)
{
     if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

}  // namespace

Readback::~Readback()
{
     for (auto e: ev_)
          if (e) (void)hipEventDestroy(e);
     if (h_one_) (void)hipHostFree(h_one_);
     if (h_) (void)hipHostFree(h_);
}

// What the first small or large read needs.
void Readback::ensure(bool one)
{
     if (one && !h_one_) {
          ok(hipHostMalloc(reinterpret_cast<void**>(&h_one_), kOneGroup * 16 + 64, hipHostMallocDefault),
             "hipHostMalloc(readback)");
          std::memset(h_one_ + kOneGroup * 16, 0, 64);
     }
     if (one || h_) return;
     for (auto& e: ev_)
          if (!e) ok(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
     ok(hipHostMalloc(reinterpret_cast<void**>(&h_), 2 * kChunk * 16, hipHostMallocDefault), "hipHostMalloc(readback)");
}

void Readback::read(const void* psi, Prec prec, uint64_t n, std::complex<double>* out, hipStream_t s)
{
     ensure(n <= kOneGroup);
     if (n <= kOneGroup) {
          auto* const flag = reinterpret_cast<uint64_t*>(h_one_ + kOneGroup * 16);
          auto* const d = reinterpret_cast<double2*>(h_one_);
          ++seq_;
          if (prec == Prec::C128)
               hipLaunchKernelGGL((k_read_out_one<double2>), dim3(1), dim3(kThreads), 0, s, d,
                                  static_cast<const double2*>(psi), static_cast<int>(n), flag, seq_);
          else
               hipLaunchKernelGGL((k_read_out_one<float2>), dim3(1), dim3(kThreads), 0, s, d,
                                  static_cast<const float2*>(psi), static_cast<int>(n), flag, seq_);
          ok(hipGetLastError(), "read_out");
          const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
          while (__atomic_load_n(flag, __ATOMIC_ACQUIRE) != seq_)
               if (std::chrono::steady_clock::now() > until) {
                    ok(hipStreamSynchronize(s), "hipStreamSynchronize");
                    break;
               }
          std::memcpy(out, h_one_, n * 16);
          return;
     }
     const uint64_t chunks = (n + kChunk - 1) / kChunk;
     auto launch = [&](uint64_t c) {
          const uint64_t first = c * kChunk, count = n - first < kChunk ? n - first : kChunk;
          auto* const d = reinterpret_cast<double2*>(h_ + (c & 1) * kChunk * 16);
          const dim3 grid(static_cast<unsigned>((count + kThreads - 1) / kThreads));
          if (prec == Prec::C128)
               hipLaunchKernelGGL((k_read_out<double2>), grid, dim3(kThreads), 0, s, d,
                                  static_cast<const double2*>(psi) + first, count);
          else
               hipLaunchKernelGGL((k_read_out<float2>), grid, dim3(kThreads), 0, s, d,
                                  static_cast<const float2*>(psi) + first, count);
          ok(hipGetLastError(), "read_out");
          ok(hipEventRecord(ev_[c & 1], s), "hipEventRecord");
     };
     launch(0);
     for (uint64_t c = 0; c < chunks; ++c) {
          // (the other buffer was copied out in the step before)
          if (c + 1 < chunks) launch(c + 1);
          ok(hipEventSynchronize(ev_[c & 1]), "hipEventSynchronize");
          const uint64_t first = c * kChunk, count = n - first < kChunk ? n - first : kChunk;
          std::memcpy(out + first, h_ + (c & 1) * kChunk * 16, count * 16);
     }
}

}  // namespace hq
