// States to host memory as complex128.
#pragma once
#include "kernels.hpp"
#include <hip/hip_runtime.h>
#include <complex>
#include <cstdint>

namespace hq {

// Chunks of a state are widened to complex128 by a kernel that writes into one
// of two pinned buffers, while the host copies the other one to its
// destination: no pageable copy, no second host array for complex64 states and
// no conversion on the host.  Bound by the host's copy and its page faults.
// Times of get_state before (copy into pageable memory) and now: 2^4
// amplitudes 20 / 7 us, complex128 2^15 226 / 31 us, 2^20 0.94 / 0.70 ms, 2^27
// 206 / 162 ms; complex64 2^12 130 / 14 us, 2^18 0.41 / 0.18 ms, 2^27 389 / 162
// ms.  The buffers (16 KiB for states of one workgroup, 2 MiB for others) are
// allocated by the first read that needs them and freed with the object.
class Readback {
public:
     Readback() = default;
     ~Readback();
     Readback(const Readback&) = delete;
     Readback& operator=(const Readback&) = delete;
     // Throws std::runtime_error.  Work that writes psi is on `s` or done.
     void read(const void* psi, Prec prec, uint64_t n, std::complex<double>* out, hipStream_t s);

     static constexpr uint64_t kChunk = uint64_t(1) << 16;  // amplitudes
     // Up to here one workgroup copies, and a flag tells the host (8 us for 2^10
     // amplitudes; one workgroup for 2^12 took 16 us, several and an event 14).
     static constexpr uint64_t kOneGroup = 1024;

private:
     void ensure(bool one);
     char* h_one_ = nullptr;  // kOneGroup amplitudes, then the flag
     char* h_ = nullptr;      // two chunks
     hipEvent_t ev_[2] = {nullptr, nullptr};
     uint64_t seq_ = 0;
};

}  // namespace hq
