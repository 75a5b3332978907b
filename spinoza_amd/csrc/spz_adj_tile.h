// spz_adj_tile.h -- reverse tile sweeps of the adjoint gradient: one pass over
// psi and lambda that undoes a run of gates on both and sums their gradient
// terms (see spz_adj_tile.hip).
#pragma once

#include "spz_internal.h"
#include "spz_tile.h"

namespace spz {

constexpr int kAdjK = 12;       // tile qubits: 16 amplitudes of each state per thread
constexpr int kAdjSlots = 64;   // gradients of one sweep (LDS rows of their partial sums)

// One reverse sweep over psi (read from src) and lam.  A gate of the program
// whose `pad` is k + 1 writes the compensated sum (S, C) of its gradient terms
// over each tile to part[2 (k tiles + tile)].
int launch_adj_tile(const spz_state_s *src, spz_state_s *psi, spz_state_s *lam, const TileDesc &d,
                    const TileOp *d_ops, int slots, double *part);
// grad[idx[k]] = the sum of slot k's partials, for every slot.
int launch_adj_sum(const double *part, uint64_t tiles, const uint32_t *d_idx, int slots,
                   double *grad);

// Bytes of partial sums that adjoint_undo needs for a state of N amplitudes
// (more than one tile; a smaller one needs 2 kChipRows doubles per op).
inline size_t adj_part_bytes(uint64_t N) { return (N >> kAdjK) * kAdjSlots * 2 * sizeof(double); }

// The sweeps that undo ops[lo, hi) (validated; host only).
struct ChipPlan;
int adjoint_plan(int n, const spz_op *ops, uint64_t lo, uint64_t hi, ChipPlan &out);

// Undo ops[lo, hi) (validated, hi > lo, FP64 states) on psi, whose
// amplitudes are taken from src (another state or psi itself), and on lam, and
// write dE/dtheta of each parametric one to the device array grad[0, hi).
int adjoint_undo(const spz_state_s *src, spz_state_s *psi, spz_state_s *lam, const spz_op *ops,
                 uint64_t lo, uint64_t hi, double *part, double *grad);

// The same for FP32 storage (spz_adj_group.hip), in place, and its scratch.
int adjoint_undo_groups(spz_state_s *psi, spz_state_s *lam, const spz_op *ops, uint64_t lo,
                        uint64_t hi, double *part, double *grad);
size_t adj_group_part_bytes(uint64_t N);

// The inverse of one op.
spz_op inverse_op(const spz_op &o);

}  // namespace spz
