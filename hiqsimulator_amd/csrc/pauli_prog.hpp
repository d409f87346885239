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
constexpr int kPauliThreads = 1 << kPauliThr;
constexpr int kPauliMaxTile = 12;
constexpr int kPauliMaxHigh = kPauliMaxTile - kPauliLow;
constexpr int kPauliMinQubits = 9;   // a tile gives every thread an amplitude
inline int pauli_tile_bits(int n) { return n < kPauliMaxTile ? n : kPauliMaxTile; }

// ---- device records ---------------------------------------------------------
// Terms [first, first + count) with one x (a mask over tile ranks).
struct PauliGroup {
     uint32_t x;
     uint32_t kind;  // bit 0: imaginary part (expectation) / factor i (apply); bit 1: imaginary output
     uint32_t first, count;
};
struct PauliTerm {
     uint64_t z_out;   // index bits outside the tile
     uint32_t z_tile;  // tile ranks
     uint32_t pad;
     double c;
};
static_assert(sizeof(PauliGroup) == 16 && sizeof(PauliTerm) == 24, "record sizes");
struct PauliPass {
     uint8_t hpos[kPauliMaxHigh];  // the chosen bits, ascending
     uint32_t group_first, ngroups;
};

// ---- host -------------------------------------------------------------------
struct PauliTermIn {
     uint64_t x, z;
     std::complex<double> c;  // coefficient with i^{|x & z|} folded in
};
struct PauliPlan {
     std::vector<PauliPass> passes;
     std::vector<PauliGroup> groups;
     std::vector<PauliTerm> terms;     // ends in one spare record (the kernels read one ahead)
     std::vector<PauliTermIn> others;  // terms whose x does not fit a tile
};
// Plan of a sum on a state of n >= kPauliMinQubits qubits: for its expectation
// value (`apply` false) or for applying it.
PauliPlan plan_pauli(const std::vector<PauliTermIn>& terms, int n, bool apply);

// ---- launches (pauli_kernels.hip) -------------------------------------------
// out[0], out[1] = real and imaginary part of the pass's share of
// sum_t c_t <psi| X^x Z^z |psi>.  scratch: kReduceScratchDoubles.
hipError_t launch_pauli_sum(const void* psi, Prec prec, int n, const PauliPass& pass, const PauliGroup* groups,
                            const PauliTerm* terms, double* scratch, double* out, hipStream_t s);

// dst (+)= f * (the pass's share of the sum applied to src); dst != src.
// With o_dst: o_dst = o_src + dst afterwards, and norm[0] = |dst|^2 (through
// scratch).  With skip: nothing is done when skip[0] < skip_below, and
// norm[0] = skip[0].
struct PauliApply {
     const void* src = nullptr;
     void* dst = nullptr;
     bool accumulate = false;
     double fr = 1, fi = 0;
     const void* o_src = nullptr;
     void* o_dst = nullptr;
     const double* skip = nullptr;
     double skip_below = 0;
     double* scratch = nullptr;
     double* norm = nullptr;
};
hipError_t launch_pauli_apply(const PauliApply& a, Prec prec, int n, const PauliPass& pass, const PauliGroup* groups,
                              const PauliTerm* terms, hipStream_t s);

}  // namespace hq
