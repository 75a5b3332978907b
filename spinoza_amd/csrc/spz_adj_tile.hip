// spz_adj_tile.hip -- reverse tile sweeps of the adjoint gradient.
//
// A sweep is a tile sweep (spz_tile_kernel.h) over two states at once: a
// workgroup holds the same 2^12-amplitude tile of psi and of lambda in
// registers, walks the program of inverse gates (planned like any other run;
// RX and RY with one product and one FMA per output, the rest with the
// reference's arithmetic), and for every gate with a parameter first sums
// Im <lambda|G|psi> over its tile.  The sum is compensated from the first pair on: a thread's
// pairs by TwoSum, then 16 lanes with DPP moves, then the rows of 16 lanes in
// LDS; one (S, C) pair per tile and gradient goes out, which a second kernel
// adds with the reduction tree.  (Plain sums and FMA chains round the sum three
// times as much for random terms; the gradients' error against 80-bit
// arithmetic, 13 to 16 qubits and 2 to 8 layers, is that of one compensated
// term per pair: 1.10e-15.)
//
// What bounded it: groups of gates on at most 3 qubits, one read and write of
// psi and lambda each (24 qubits, 10 layers: 80 passes of 259 us for 480
// rotations, plus two tile sweeps per run of CX).  A sweep takes about 50 gates
// in one pass: 15 of 424 us (1.07 GB each, 2.5 TB/s: FP64 issue, three waves
// per SIMD with both states in registers) and 15 forward sweeps; the gradient
// takes 11.0 ms instead of 34.9.
#include "spz_adj_tile.h"
#include "spz_adj_body.h"

namespace spz {

namespace {

template <typename T, int K>
__global__ void __launch_bounds__(1 << (K - 4)) __attribute__((amdgpu_waves_per_eu(3, 3)))
k_adj_tile(const T *sr, const T *si, T *pr, T *pi, T *qr, T *qi, const TileDesc d,
           const TileOp *__restrict__ ops, int slots, double *__restrict__ part)
{
    constexpr int LOGW = K - 4, RB = 4, R = 16, ROWS = (1 << LOGW) / 16;
    __shared__ double lds[1 << K];
    __shared__ double2 sums[kAdjSlots][ROWS];
    const uint32_t tid = threadIdx.x;
    const uint64_t base = insert_zeros((uint64_t)blockIdx.x, d.spos, K);
    uint32_t lt = 0;
#pragma unroll
    for (int i = 0; i < LOGW; i++) lt |= ((tid >> i) & 1u) << d.tin[i];
    const uint64_t gt = lane_offset<LOGW>(tid, d.tg);
    double vr[R], vi[R], ur[R], ui[R];
    {
        const uint64_t at = (base + gt) * sizeof(T);
        const char *a = (const char *)sr + at, *b = (const char *)si + at;
        const char *c = (const char *)qr + at, *e = (const char *)qi + at;
#pragma unroll
        for (int p = 0; p < R; p++) {
            vr[p] = (double)*(const T *)(a + d.gr[p]);
            vi[p] = (double)*(const T *)(b + d.gr[p]);
            ur[p] = (double)*(const T *)(c + d.gr[p]);
            ui[p] = (double)*(const T *)(e + d.gr[p]);
        }
    }
    const Amps s{vr, vi, ur, ui};

    const uint64_t ope = reinterpret_cast<uint64_t>(ops + d.nops);
    for (uint64_t opa = reinterpret_cast<uint64_t>(ops); opa != ope; opa += sizeof(TileOp)) {
        asm volatile("" : "+s"(opa));
        const TileOp cur = fetch_op(opa);
        if (hit(cur.grp & TG_LAYOUT)) {
            LayoutMove<R, LOGW> m;
            lt = m.set(cur.lay, lt, tid, lds);
            m.move(vr);
            m.move(vi);
            m.move(ur);
            m.move(ui);
        }
        Sum g;
        adj_gate<R, RB>(cur, base, lt, s, g);
        if (cur.pad) {  // (a tile or lane whose controls are not met adds zero)
            row_sum(g);
            if ((tid & 15u) == 0) sums[cur.pad - 1][tid >> 4] = make_double2(g.s, g.c);
        }
    }

    uint64_t gsb[K];
#pragma unroll
    for (int b = 0; b < K; b++) gsb[b] = 1ull << d.spos[b];
    {
        const uint64_t at = (base + lane_offset<K>(lt, gsb)) * sizeof(T);
        char *a = (char *)pr + at, *b = (char *)pi + at;
        char *c = (char *)qr + at, *e = (char *)qi + at;
#pragma unroll
        for (int p = 0; p < R; p++) {
            *(T *)(a + d.gs[p]) = (T)vr[p];
            *(T *)(b + d.gs[p]) = (T)vi[p];
            *(T *)(c + d.gs[p]) = (T)ur[p];
            *(T *)(e + d.gs[p]) = (T)ui[p];
        }
    }
    __syncthreads();
    if ((int)tid < slots)  // slots <= kAdjSlots <= threads
        sum_rows(sums[tid], ROWS, part + 2 * ((uint64_t)tid * gridDim.x + blockIdx.x));
}

// Block k adds slot k's pairs.
__global__ void __launch_bounds__(kRT)
k_adj_sum(const double *__restrict__ part, uint64_t tiles, const uint32_t *__restrict__ idx,
          double *__restrict__ grad)
{
    __shared__ double S[kRT], C[kRT];
    const double r = reduce_pairs(part + 2 * (uint64_t)blockIdx.x * tiles, tiles, S, C);
    if (threadIdx.x == 0) grad[idx[blockIdx.x]] = r;
}

}  // namespace

int launch_adj_tile(const spz_state_s *src, spz_state_s *psi, spz_state_s *lam, const TileDesc &d,
                    const TileOp *d_ops, int slots, double *part)
{
    const uint64_t tiles = psi->N >> kAdjK;
    if (tiles == 0 || tiles > (1ull << 31) - 1) return fail(SPZ_ERR_ARG, "tile grid out of range");
    if (slots < 0 || slots > kAdjSlots) return fail(SPZ_ERR_ARG, "too many gradients in a sweep");
    if (psi->prec != SPZ_F64) return fail(SPZ_ERR_ARG, "reverse sweeps take FP64 states");
    const size_t esz = sizeof(double);
    TileDesc db = d;  // register terms as byte offsets
    for (int p = 0; p < 16; p++) {
        db.gr[p] *= esz;
        db.gs[p] *= esz;
    }
    LaunchTimer tm(SPZ_K_ADJOINT, 8.0 * (double)psi->N * (double)esz);
    const dim3 g((unsigned)tiles), b(1 << (kAdjK - 4));
    hipLaunchKernelGGL((k_adj_tile<double, kAdjK>), g, b, 0, rt().stream, (const double *)src->re,
                       (const double *)src->im, (double *)psi->re, (double *)psi->im,
                       (double *)lam->re, (double *)lam->im, db, d_ops, slots, part);
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

int launch_adj_sum(const double *part, uint64_t tiles, const uint32_t *d_idx, int slots,
                   double *grad)
{
    if (slots <= 0) return SPZ_OK;
    hipLaunchKernelGGL(k_adj_sum, dim3(slots), dim3(kRT), 0, rt().stream, part, tiles, d_idx, grad);
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

}  // namespace spz
