// Gate programs: a gate list applied to a state tile by tile, gate by gate.
//
// A tile program (batch.hpp) multiplies fused 2^k x 2^k matrices into LDS
// tiles; its cost is that of the dense products, whatever the gates were.
// Most gates are one-qubit gates, controlled gates and phases, and applied by
// themselves they take a fraction of the fused product's operations: with one
// coefficient factored out into a scale that a whole pass shares, H, Rx and
// Ry cost two fused multiply-adds an amplitude, a phase two, a CNOT none
// (against 48 for a 4-qubit product that holds about eight such gates).
// Also, only the qubits that a gate mixes have to lie in the tile: control
// and diagonal qubits are conditions on the index, which a tile can evaluate
// wherever they are, so a pass takes gates that a dense plan cannot.
//
// Below, a precision is the one that the amplitudes have in a pass.  A
// complex64 state is held in complex128 for lists whose roundings in FP32, gate
// after gate, could be more than those of the fused products (gate_route).
//
// A pass covers tiles of 2^13 amplitudes in complex128 and 2^14 in complex64:
// index bits 0..3 (runs of 16 amplitudes: 256 and 128 bytes) and nine or ten
// chosen bits.  A workgroup of 512 threads holds its tile in registers, 16 or
// 32 amplitudes (four or five tile bits, 64 registers either way) a thread.
// The pass is a list of stages; each keeps four or five tile bits in the
// thread and applies every gate that mixes only those, in program order, and
// between stages the tile is regrouped through LDS.
//
// This header: the device records, the host planner (which gates go into
// which pass and stage) and the compiler from gates to records.
#pragma once

#include <hip/hip_runtime.h>

#include <complex>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "kernels.hpp"

namespace hq {

constexpr int kGateLow = 4;                     // index bits 0..3 are always tile bits
constexpr int kGateThr = 9;                     // tile bits of the thread index
constexpr int kGateThreads = 1 << kGateThr;
// Tile bits in a thread's registers, and all tile bits.
constexpr int gate_reg(Prec p) { return p == Prec::C128 ? 4 : 5; }
constexpr int gate_tile_bits(Prec p) { return kGateThr + gate_reg(p); }
constexpr int gate_high(Prec p) { return gate_tile_bits(p) - kGateLow; }  // chosen bits
// Smallest states that run as gate programs.  Complex128: from one tile on.
// The kernels alone cross over at 21 qubits (20 random layers: 224 against
// 166 us at 16 qubits, 315 against 280 at 20, 368 against 436 at 21, 8.2
// against 11.5 ms at 26), where the tiles fill the chip; below that a call is
// bound by its host work, which is less (703 against 877 us a call at 16
// qubits, 1189 against 1265 at 20).  Complex64 keeps the tile programs there:
// their kernels are ahead by more (20 qubits: 221 against 314 us; 22: 459
// against 403, held in FP32).
constexpr int gate_min_qubits(Prec p) { return p == Prec::C128 ? 13 : 21; }
constexpr int kGateMaxReg = 5, kGateMaxTile = kGateThr + kGateMaxReg, kGateMaxHigh = kGateMaxTile - kGateLow;
constexpr size_t kGateMaxStages = 255;      // a pass's stage count is a byte
constexpr size_t kGateMaxStageUnits = 512;  // and a stage's record count 16 bits
// Units of a pass: far beyond what its reads and writes are worth, and a bound
// for the planner's scans (100000 gates on 13 qubits were planned in 1.2 s, each
// pass over all that were left; 0.13 s now).
constexpr size_t kGateMaxPassUnits = 4096;

// ---- device records ---------------------------------------------------------
// Opcodes.  b is the register bit (0..4) an op acts on.
enum GateCode : uint32_t {
     // A layer: rotations on any of the register bits, then phases on them,
     // then controlled swaps between them, in one record.  aux: rotation kind
     // of bit b at 2 b (kGateKind*), phase flag of bit b at 10 + b.  c: two
     // coefficients a bit.  With phases, `count` is 1 and the next record's c
     // holds a factor a bit.  omask and oval are no condition but up to 16
     // bytes (target * 8 + control), tcond their number.
     kGateLayer = 0,
     kGateRM = 1,     // +b: a' = a + c0 z, z' = -z + c1 a (real c)
     kGateR4 = 6,     // +b: real 2 x 2 matrix c0..c3
     kGateG = 11,     // +b: complex 2 x 2 matrix c0..c7, where the register condition holds
     kGateXA = 16,    // +b: a and z change places
     kGateX = 21,     // +b: the same where the register condition holds
     kGateXC = 26,    // the same for target aux / 8 under control aux % 8, register bits
     kGatePAll = 27,  // every amplitude times c0 + i c1
     kGatePT = 28,    // the same where the register condition holds
     kGatePA = 29,    // +b: amplitudes with bit b times the product of the next `count`
                      // records' factors (two doubles at c) whose conditions hold
     kGatePL = 34,    // the same for every amplitude
     kGateG2 = 35,    // + pair: complex 4 x 4 matrix in the coefficients of the next four
                      // records, on the register pair, where the register condition holds
     kGateCodes = 45
};
// Rotation kinds of a layer.
enum GateKind : uint32_t {
     kGateKindNone = 0,
     kGateKindReal = 1,  // a' = a + c0 z, z' = z + c1 a
     kGateKindH = 2,     // a' = a + z, z' = a - z
     kGateKindImag = 3   // a' = a + i c0 z, z' = z + i c1 a
};
// Register pairs of kGateG2: (0,1) (0,2) (1,2) (0,3) (1,3) (2,3) (0,4) (1,4) (2,4) (3,4).
constexpr uint32_t gate_pair(int b0, int b1) { return static_cast<uint32_t>(b1 * (b1 - 1) / 2 + b0); }
constexpr uint32_t kGateMaxList = 255;  // `count` is a byte
// A list (kGatePA, kGatePL) whose aux is 1 + g begins with tables in the place
// of records: the products of its factors whose conditions are on lane bits
// only, for each of the 64 lanes; on wave bits only, for each of the 8 waves;
// and on bits 5 i .. 5 i + 4 of the tile number only, for each of their 32
// values, i < g (g covers the whole number).  Pairs of doubles.  A factor from
// a record takes some sixteen vector and thirty scalar instructions; a table
// takes one load and one product.  Worth it from four such factors on: the QFT
// of 29 qubits in complex64 took 12.7 ms with records, 10.7 ms with tables.
constexpr int kGateTableLanes = 64, kGateTableWaves = kGateThreads / 64;
constexpr int kGateTableBits = 5;
constexpr int gate_table_groups(Prec p, int n) { return (n - gate_tile_bits(p) + kGateTableBits - 1) / kGateTableBits; }
constexpr size_t gate_table_entries(int groups)
{
     return kGateTableLanes + kGateTableWaves + (static_cast<size_t>(groups) << kGateTableBits);
}

// One op.  But for layers it applies where (tile base index & omask) == oval,
// (thread & tmask) == tval and, for the ops that say so, (amplitude &
// regmask) == regval.
template <typename R>
struct GateOp {
     uint32_t code;   // opcode | count << 8 | aux << 16; aux = regmask | regval << 5 where that is asked
     uint32_t tcond;  // tmask | tval << 16
     uint64_t omask, oval;
     R c[10];
};
static_assert(sizeof(GateOp<double>) == 104 && sizeof(GateOp<float>) == 64 &&
                  offsetof(GateOp<double>, c) == offsetof(GateOp<float>, c),
              "record sizes");
// Records that the tables take the place of.
template <typename R>
constexpr uint32_t gate_table_records(int groups)
{
     return static_cast<uint32_t>((gate_table_entries(groups) * 16 + sizeof(GateOp<R>) - 1) / sizeof(GateOp<R>));
}
inline size_t gate_op_bytes(Prec p) { return p == Prec::C128 ? sizeof(GateOp<double>) : sizeof(GateOp<float>); }

// One stage: LDS byte offsets of the thread bits and the register bits (the
// slot of an amplitude is the XOR of its bits' offsets) and its ops.
struct GateStage {
     uint16_t thr_lds[kGateThr];
     uint16_t reg_lds[kGateMaxReg];
     uint16_t nops, pad;
     uint32_t op_first;
};
static_assert(sizeof(GateStage) == 36, "record size");

// One pass over a state: the chosen bits, the index bits of the first
// stage's (load) and the last stage's (store) thread and register bits, and
// the stages.  A permuted pass stores into another buffer, with the index bits
// permuted: its out_* are bits of the new index, and base_out[j] is the new
// place of the j-th lowest bit outside the tile.
constexpr int kGateMaxBase = 40 - 13;
struct GatePass {
     uint8_t hpos[kGateMaxHigh];
     uint8_t in_thr[kGateThr], in_reg[kGateMaxReg];
     uint8_t out_thr[kGateThr], out_reg[kGateMaxReg];
     uint8_t base_out[kGateMaxBase];
     uint8_t nstages, permuted, pad[3];
     uint32_t stage_first;
};
static_assert(sizeof(GatePass) == 76, "record size");

// Slot of tile rank r in LDS, as an XOR mask over the slots: the low bits
// hold the low rank bits XOR-ed with a linear map of the others.  64 banks of
// 4 bytes serve 32 lanes without a conflict when their low five (8-byte
// slots, complex128) or six (4-byte slots, complex64) slot bits are distinct.
// The columns below form binary linear codes of minimum distance 5: whichever
// ranks are in registers, five of the others have independent columns, and
// those are given to the first five lane bits.
inline uint32_t gate_slot(Prec p, int rank)
{
     constexpr uint8_t c5[13] = {1, 2, 4, 8, 16, 31, 7, 25, 11, 10, 5, 23, 20};
     constexpr uint8_t c6[14] = {1, 2, 4, 8, 16, 32, 47, 25, 51, 29, 30, 59, 60, 53};
     if (p == Prec::C128) return (rank >= 5 ? 1u << rank : 0u) | c5[rank];
     return (rank >= 6 ? 1u << rank : 0u) | c6[rank];
}
constexpr uint32_t gate_slot_bytes(Prec p) { return p == Prec::C128 ? 8 : 4; }

// ---- host: gates ------------------------------------------------------------
// A gate split by what it does to each of its index bits: `a` are the bits it
// mixes (at most two), `d` the bits it only depends on (controls, and
// targets in which its matrix is block diagonal).  Branch: what happens to
// the mixed bits where (index & cmask) == cval; u is the factor (no mixed
// bit), the 2 x 2 or the 4 x 4 matrix (bit l <-> act[l]), row-major.
// Identity branches are left out.
struct GateBranch {
     uint64_t cmask = 0, cval = 0;
     std::complex<double> u[16];
};
struct GateUnit {
     uint64_t a = 0, d = 0;
     int na = 0;
     uint8_t act[2] = {0, 0};
     std::vector<GateBranch> br;
};
// The unit of a gate (2^t x 2^t matrix m, row-major, bit l <-> targets[l];
// positions below 62); false when it mixes more than two bits.
bool make_gate_unit(const std::complex<double>* m, const std::vector<int64_t>& targets,
                    const std::vector<int64_t>& ctrls, GateUnit& out);

// Whether the matrix mixes at most two of its targets.  Asked before the units
// of a list are made: a list with one gate that mixes three spent 0.1 ms on 470
// units (0.92 ms as tile programs on 16 qubits).
bool gate_fits(const std::complex<double>* m, size_t targets);

// ---- host: which way a list goes --------------------------------------------
// What a list takes either way, counted in one sweep over its units.
//   work      of a gate program: a rotation, a phase or a CNOT is 1, a general
//             2 x 2 block 3.7, a 4 x 4 block 6.5, a conditional factor 0.5, or 2
//             when its qubits are all mixed by gates before it (they are then
//             often in registers together, where the factor is applied by
//             itself); runs that become one matrix count once.
//   products  fused products on four qubits that a tile program needs about:
//             a quarter of the qubits of greedily grown groups of up to four.
//   rounds    roundings of an amplitude that a gate program makes in the
//             precision it is held in, as their squares add up: one for a
//             rotation or a phase, three for a general block, four for a 4 x 4
//             block, 0.25 (or 0.75, where its work is 2) for a conditional
//             factor; m gates of the same rounded coefficients make m^2, for
//             theirs are the same each time.  (For complex64 states.)
struct GateListCost {
     double work = 0, products = 0, rounds = 0;
};
// (products are left 0 where gate_route does not ask for them)
GateListCost gate_list_cost(const std::vector<GateUnit>& units, int n, Prec prec);
// The precision that a gate program of the list would hold the amplitudes of
// an n-qubit state in; false: the list runs as tile programs.
//
// Time.  Tile programs over gate programs, with work per product in brackets.
// Complex128, 28 qubits: QFT (2) 7.5, CNOT ladder (3) 2.2, layers of rotations
// and CNOTs (12) 1.6, Trotter steps of an Ising chain (20) 1.4, 2-qubit Haar
// bricks (23) 1.2, three rotations a qubit and layer (27) 0.92, one-qubit Haar
// and CNOT (31) 0.82, five rotations (40) 0.72, 200 layers on 4 qubits (1046)
// 0.12: up to 24.  Complex64 held in FP64 against products in FP32, 28 qubits:
// CNOT ladder 1.6, layers (12) 1.0, H and CZ (14) 0.82, Ising steps 0.75, 2-qubit
// bricks 0.71, three rotations 0.58: up to 13, and up to 18 for 24 qubits or
// less, where the host takes a good part of it (Heisenberg steps (17) 1.5 at 23
// qubits, 1.2 at 24).  Up to 22 qubits the host and a workgroup's latency bound
// both ways (0.5 us a unit of work against 1.25 us a gate for the fusion): of
// these lists only those of dense 2-qubit blocks are faster as products (0.66 at
// 13 qubits, 0.9 at 16, 1.1 at 20).
//
// Roundings.  Error of gate programs held in FP32 over that of tile programs (l2,
// complex64, 25 qubits, random states), with roundings per product in brackets:
// QFT (1) 0.54, factors on three qubits (3) 0.5, H on every qubit (4) 0.52, layers
// with random angles and CNOTs (8) 0.75, of Ry alone 0.64, 40 layers on 8 qubits
// (10) 0.79; one-qubit Haar (12) 0.86 and, from |0..0>, 1.4; H and CZ (10) 0.68
// and 2.7; one-qubit Haar and CNOT (22) 1.1, three rotations (24) 1.1, five (37)
// 1.4, 200 layers on 4 qubits (700) 6.4; the same angles again and again: QAOA
// (240) 1.3, four Heisenberg steps (290) 2.4, 40 Ising steps (9400) 2.9.  So FP32
// up to 9.5; layers with random angles from |0..0> are within a tenth of tile
// programs there (0.9 to 1.1).  Held in FP64 the error is 0.05 to 0.2 of that of
// tile programs, and a list takes 1.25 times (23 qubits) to 1.65 times (28) as long
// as in FP32.
bool gate_route(const GateListCost& cost, size_t gates, int n, Prec prec, Prec& held);

// ---- host: planning ---------------------------------------------------------
struct GatePassPlan {
     uint64_t bits = 0;                     // the tile's index bits
     std::vector<uint64_t> regs;            // per stage: the bits its gates mix
     std::vector<std::vector<int>> stages;  // per stage: unit indices, program order
};

// One pass at a time from the front of the list.  A unit is taken if the bits
// it mixes lie in the tile and it commutes with every unit skipped before it:
// neither mixes a bit that the other touches.
class GatePassPlanner {
public:
     // splits: every pass is split into stages in four ways, and the one with the
     // fewest groupings kept (worth_splits).
     GatePassPlanner(const std::vector<GateUnit>& units, int n, Prec prec, bool splits = false);
     // Where a pass takes longer than its planning: a grouping less saves 0.4 to
     // 0.9 ms of a pass on 30 qubits in complex128, and 0.04 ms of planning find
     // 0.4 of one on average (of 4.1; complex64, 23 qubits: 0.6 of 5.6).
     static bool worth_splits(int n, Prec prec);
     bool next(GatePassPlan& out);
     // Indices of the units not planned yet, in program order.
     const std::vector<int>& remaining() const { return rem_; }

private:
     uint64_t choose(const std::vector<int>& list, uint64_t fixed, uint64_t allowed, int k, uint64_t start = 0) const;
     size_t make_stages(std::vector<int>& list, GatePassPlan& out, bool back, bool avoid) const;
     void take(std::vector<int>& list, uint64_t S, size_t cap, std::vector<int>& out) const;
     const std::vector<GateUnit>& units_;
     int n_;
     Prec prec_;
     bool splits_;
     std::vector<int> rem_;
};

// ---- host: compilation ------------------------------------------------------
// Appends the records of one pass: its stages to `stages`, its ops (of the
// state's precision) to `ops`.  pass.stage_first and the stages' op_first
// count from the beginning of the arrays.  `ops` always ends in one spare
// record (the kernel reads one ahead).
// src_pos: if given, the pass also permutes the index bits: bit p of the new
// index is bit src_pos[p] of the old one; bits src_pos[0..kGateLow) have to
// lie in the tile (widen_for_permutation).
void compile_gate_pass(const std::vector<GateUnit>& units, const GatePassPlan& plan, int n, Prec prec,
                       GatePass& pass, std::vector<GateStage>& stages, std::vector<char>& ops,
                       const uint8_t* src_pos = nullptr);
// Leaves the plan the first half of its stages (or of the units of its only
// one) and puts the other half into `second`, to run right behind it; false for
// a single unit.
bool split_gate_pass(GatePassPlan& plan, GatePassPlan& second);
// Puts bits src_pos[0..kGateLow) into the plan's tile, in the place of bits that
// its units do not mix, so that the permuted state is stored in runs of 2^kGateLow
// amplitudes; false, and nothing changed, when they do not fit.  At 30 qubits
// in complex128 a permutation takes 6.3 ms by itself and about 2 ms in a pass;
// of five random layers of gates between permutations two thirds end in a pass
// with room for it.
bool widen_for_permutation(const std::vector<GateUnit>& units, GatePassPlan& plan, int n, Prec prec,
                           const uint8_t* src_pos);
// Throws unless every record of the pass stays inside the tile, the arrays
// and a state of 2^n amplitudes.
void check_gate_pass(const GatePass& pass, const std::vector<GateStage>& stages, const std::vector<char>& ops,
                     Prec prec, int n);

// ---- launches (gate_kernels.hip) --------------------------------------------
// One pass over a state of 2^n amplitudes (gate_tile_bits(held) <= n <= 40) of
// precision prec, planned and compiled for precision held, which the
// amplitudes have while the pass holds them; stages and ops are device arrays,
// ops with one spare record at the end.  dst: where a permuted
// pass stores (another buffer than psi).
hipError_t launch_gate_pass(void* psi, Prec prec, Prec held, int n_qubits, const GatePass& pass, const GateStage* stages,
                            const void* ops, hipStream_t s, void* dst = nullptr);
}  // namespace hq
