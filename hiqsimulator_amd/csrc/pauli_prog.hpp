// Pauli sums, many terms in one pass over the state.
//
// A term P = i^{|x & z|} X^x Z^z takes amplitude i to i ^ x with the sign
// (-1)^{|i & z|}.  Terms with the same x share the amplitudes they read, and
// terms whose x lies inside a tile's index bits find them in the tile: a
// workgroup loads 2^12 amplitudes (index bits 0..3 and eight chosen bits)
// into LDS once and evaluates every group of such terms there, each thread
// for its eight amplitudes.  z is unrestricted: bits outside the tile give a
// sign that the whole tile shares.  A nearest-neighbour Hamiltonian on 26
// qubits (101 terms) takes three passes over the state instead of 101.
#pragma once

#include <hip/hip_runtime.h>

#include <complex>
#include <cstdint>
#include <vector>

#include "kernels.hpp"

namespace hq {

constexpr int kPauliLow = 4;         // index bits 0..3 are always tile bits
constexpr int kPauliThr = 9;         // tile ranks of the thread index
constexpr int kPauliLane = 6;        // of these, ranks 0..5 are the lane's
constexpr int kPauliThreads = 1 << kPauliThr;
constexpr int kPauliMaxTile = 12;
constexpr int kPauliMaxHigh = kPauliMaxTile - kPauliLow;
constexpr int kPauliMinQubits = 9;   // a tile gives every thread an amplitude
inline int pauli_tile_bits(int n) { return n < kPauliMaxTile ? n : kPauliMaxTile; }

// ---- device records ---------------------------------------------------------
// The terms of a pass are one stream of records (one scalar load each, read
// one ahead).  Terms of one x and kind form a group; inside a group, terms
// whose z agrees on the amplitude-number bits (the tile ranks above the
// thread's) form a class, whose signed coefficients are summed once for the
// thread and then added to its amplitudes' weights.
struct PauliTerm {
     uint64_t z_out;   // index bits outside the tile
     double c;
     uint32_t z_tile;  // tile ranks; kPauli* flags above
     uint32_t x;       // tile ranks
};
static_assert(sizeof(PauliTerm) == 24, "record size");
constexpr uint32_t kPauliClassEnd = 1u << 16;  // last record of its class
constexpr uint32_t kPauliGroupEnd = 1u << 17;  // last record of its group
constexpr uint32_t kPauliImag = 1u << 18;      // imaginary part (expectation) / factor i (apply)
constexpr uint32_t kPauliOut1 = 1u << 19;      // expectation: imaginary output
struct PauliPass {
     uint8_t hpos[kPauliMaxHigh];  // the chosen bits, ascending
     uint32_t first, count;        // records
};

// ---- host -------------------------------------------------------------------
struct PauliTermIn {
     uint64_t x, z;
     std::complex<double> c;  // coefficient with i^{|x & z|} folded in
};
struct PauliPlan {
     std::vector<PauliPass> passes;
     std::vector<PauliTerm> terms;     // ends in one spare record (the kernels read one ahead)
     std::vector<PauliTermIn> others;  // terms whose x does not fit a tile
};
// Plan of a sum on a state of n >= kPauliMinQubits qubits: for its expectation
// value (`apply` false) or for applying it.
PauliPlan plan_pauli(const std::vector<PauliTermIn>& terms, int n, bool apply);
// Bessel functions J_0(z), J_1(z), ... up to the last one above 1e-17, by
// Miller's backward recurrence J_{k-1} = (2k / z) J_k - J_{k+1}, normalised
// with J_0 + 2 (J_2 + J_4 + ...) = 1.  z >= 0, at most 1e6.
std::vector<double> bessel_series(double z);

// ---- launches (pauli_kernels.hip) -------------------------------------------
// out[0], out[1] = real and imaginary part of the pass's share of
// sum_t c_t <psi| X^x Z^z |psi>.  scratch: kReduceScratchDoubles.
hipError_t launch_pauli_sum(const void* psi, Prec prec, int n, const PauliPass& pass, const PauliTerm* terms,
                            double* scratch, double* out, hipStream_t s);

// dst = f * (the pass's share of the sum applied to src) + g * add (add may be
// dst; dst != src).  With o_dst: o_dst = h * o_src + e * src + c * dst
// afterwards (o_src may be o_dst, or null for zero), and with norm: norm[0] = |dst|^2 (through scratch).  With
// skip: nothing is done when skip[0] < skip_below, and norm[0] = skip[0].
struct PauliApply {
     const void* src = nullptr;
     void* dst = nullptr;
     double fr = 1, fi = 0;
     const void* add = nullptr;
     double g = 1;
     const void* o_src = nullptr;
     void* o_dst = nullptr;
     double h = 1, cr = 1, ci = 0, er = 0, ei = 0;
     const double* skip = nullptr;
     double skip_below = 0;
     double* scratch = nullptr;
     double* norm = nullptr;
};
hipError_t launch_pauli_apply(const PauliApply& a, Prec prec, int n, const PauliPass& pass, const PauliTerm* terms,
                              hipStream_t s);

}  // namespace hq
