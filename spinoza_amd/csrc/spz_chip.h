// spz_chip.h -- tile sweeps of many circuits per launch, and of circuits that
// fit in one tile (see spz_chip.hip).
#pragma once

#include <vector>

#include "spz_internal.h"
#include "spz_tile.h"

namespace spz {

constexpr int kChipK = 12;          // tile qubits (states of fewer are padded to a tile)
constexpr int kChipRows = 16;       // gradient pairs a tile writes per slot (one per 16 lanes)

enum ChipFlags : uint32_t {
    CHIP_INIT = 1u,   // start from |0...0> instead of loading psi
    CHIP_STORE = 2u,  // write psi (and lambda) back
};

// One sweep of one circuit, in device memory.  Offsets gr, gs in bytes of the
// storage type; amplitudes at `limit` and beyond (padding) load as zero and
// are not stored.
struct ChipSweep {
    const void *sr, *si;  // psi is loaded from here ...
    void *pr, *pi;        // ... and stored here
    void *qr, *qi;        // lambda (reverse sweeps)
    uint64_t limit;
    const TileOp *ops;
    double *part;         // gradient pairs: row r of slot k of tile t at
                          // part[2 ((k tiles + t) kChipRows + r)]
    uint32_t nops, tiles;
    uint32_t width;       // workgroups of the circuit (they stride over its tiles)
    uint32_t flags;
    int8_t spos[16];
    int8_t tin[16];
    uint64_t tg[8], gr[16], gs[16];
};

// lambda = H psi and the energy's level-1 pairs of one circuit (blocks of 4096
// amplitudes; a smaller state is one block).
struct ChipIsing {
    const void *re, *im;
    void *lr, *li;
    uint64_t N;
    double *part;
    uint32_t blocks;
    int32_t n;
};

// out[dst] = the sum of n pairs.
struct ChipSum {
    const double *part;
    uint32_t n, dst;
};

// Launches on the library stream: `count` descriptors, of at most `width`
// workgroups (blocks) each; `lds` pads the workgroups' LDS (a cap on how many
// are resident).  Reverse sweeps and H psi take FP64 states.
int launch_chip_sweeps(int prec, bool reverse, const ChipSweep *d, uint32_t count, uint32_t width,
                       size_t lds);
int launch_chip_ising(const ChipIsing *d, uint32_t count, uint32_t width, double hx);
int launch_chip_sums(const ChipSum *d, uint32_t count, double *out);

// The sweeps of a circuit of validated ops: forward, or the undoing of its ops
// with their gradients.  Planned without the searches of the single-circuit
// executor (a batch plans thousands of sweeps; these run from the caches).
struct ChipPlan {
    struct Sweep {
        TileDesc desc;
        uint32_t op_begin, op_count, slot_begin, slots;
    };
    std::vector<TileOp> prog;
    std::vector<Sweep> sweeps;
    std::vector<uint32_t> grads;  // op index of every gradient slot
};
int chip_plan(int n, const spz_op *ops, uint64_t n_ops, bool reverse, ChipPlan &out);

// Fills the geometry of one sweep of a plan (everything but the pointers).
void chip_geometry(const ChipPlan::Sweep &s, int n, int prec, ChipSweep &out);

}  // namespace spz
