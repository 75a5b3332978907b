// spz_chip.hip -- tile sweeps of many circuits per launch, and of circuits
// that fit in one tile.
//
// A circuit is a list of sweeps (spz_tile.h): forward over psi, then lambda =
// H psi, then reverse over psi and lambda with the gradients.  One launch runs
// one sweep of each of its circuits: blockIdx.y picks the circuit's descriptor,
// blockIdx.x its tiles.  A circuit of at most 12 qubits is one tile (padded to
// 2^12 amplitudes), so the whole of it is one forward and one reverse sweep;
// on its own it is the fast path of small states, where a launch per gate cost
// 1.5 us of device time and 3 us of queueing each (9 qubits, 78 gates, 512
// shots: 336 -> 117 us, 49 of them the sweep; a gradient of 11 qubits and 88
// parameters: 837 -> 524 us, 81 and 140 of them the two sweeps).  One workgroup
// is bound by the latency of its instruction stream, about 0.5 us per gate.
//
// The arithmetic is the reference's (RX and RY of the reverse sweeps with one
// FMA per output, see spz_adj_tile.hip); nothing depends on which workgroup
// runs a tile.
#include <algorithm>

#include "spz_adj_body.h"
#include "spz_chip.h"
#include "spz_ising.h"

namespace spz {

namespace {

constexpr int kLogW = kChipK - 4, kRegs = 16;
static_assert(kChipRows == (1 << kLogW) / 16, "one pair per 16 lanes");

// The gate of a forward sweep (the STRICT arithmetic of k_tile).
__device__ __forceinline__ void fwd_gate(const TileOp &cur, uint64_t base, uint32_t lt, double *vr,
                                         double *vi)
{
    if ((base & cur.em) != cur.eo) return;
    const uint32_t g = cur.grp, sel = cur.sel, pm = cur.pm;
    const double *k = cur.c;
    if (hit(g & (TG_PAIR | TG_PAIRP))) {
        if (hit(g & TG_PAIR)) pair_kinds<kRegs, 4, false, false>(g, sel, vr, vi, k, 0);
        if (hit(g & TG_PAIRP))
            if (lane_pass(lt, cur.mlo, cur.mlz))
                pair_kinds<kRegs, 4, true, false>(g, sel, vr, vi, k, pm);
    }
    if (hit(g & (TG_DREG | TG_DREGP | TG_DLANE | TG_DLANEP))) {
        if (hit(g & TG_DREG)) diag_reg_kinds<kRegs, 4, false, false>(g, sel, vr, vi, k, 0);
        if (hit(g & TG_DREGP))
            if (lane_pass(lt, cur.mlo, cur.mlz))
                diag_reg_kinds<kRegs, 4, true, false>(g, sel, vr, vi, k, pm);
        if (hit(g & (TG_DLANE | TG_DLANEP))) {
            const bool bit = cur.dsel == 2 ? (base & cur.ebit) != 0
                                           : ((lt >> cur.dpos) & 1u) != 0;
            if (hit(g & TG_DLANE)) diag_lane_kinds<kRegs, false, false>(g, vr, vi, k, bit, 0);
            if (hit(g & TG_DLANEP))
                if (lane_pass(lt, cur.mlo, cur.mlz))
                    diag_lane_kinds<kRegs, true, false>(g, vr, vi, k, bit, pm);
        }
    }
}

// Reverse sweeps hold two states (three waves per SIMD, as k_adj_tile),
// forward sweeps one (four).
template <typename T, bool REV>
__global__ void __launch_bounds__(1 << kLogW)
__attribute__((amdgpu_waves_per_eu(REV ? 3 : 4, REV ? 3 : 4)))
k_chip(const ChipSweep *__restrict__ sweeps)
{
    __shared__ double lds[1 << kChipK];
    const uint32_t tid = threadIdx.x;
    const ChipSweep &d = sweeps[blockIdx.y];
    if (blockIdx.x >= d.width) return;
    for (uint32_t tile = blockIdx.x; tile < d.tiles; tile += d.width) {
        const uint64_t base = insert_zeros((uint64_t)tile, d.spos, kChipK);
        uint32_t lt = 0;
#pragma unroll
        for (int i = 0; i < kLogW; i++) lt |= ((tid >> i) & 1u) << d.tin[i];
        const uint64_t at = (base + lane_offset<kLogW>(tid, d.tg)) * sizeof(T);
        const uint64_t end = d.limit * sizeof(T);
        double vr[kRegs], vi[kRegs], ur[REV ? kRegs : 1], ui[REV ? kRegs : 1];
        if (d.flags & CHIP_INIT) {
#pragma unroll
            for (int p = 0; p < kRegs; p++) {
                vr[p] = at + d.gr[p] == 0 ? 1.0 : 0.0;
                vi[p] = 0.0;
            }
        } else {
#pragma unroll
            for (int p = 0; p < kRegs; p++) {
                const uint64_t o = at + d.gr[p];
                const bool in = o < end;
                vr[p] = in ? (double)*(const T *)((const char *)d.sr + o) : 0.0;
                vi[p] = in ? (double)*(const T *)((const char *)d.si + o) : 0.0;
            }
        }
        if constexpr (REV) {
#pragma unroll
            for (int p = 0; p < kRegs; p++) {
                const uint64_t o = at + d.gr[p];
                const bool in = o < end;
                ur[p] = in ? (double)*(const T *)((const char *)d.qr + o) : 0.0;
                ui[p] = in ? (double)*(const T *)((const char *)d.qi + o) : 0.0;
            }
        }
        const uint64_t ope = reinterpret_cast<uint64_t>(d.ops + d.nops);
        warm_program<kLogW>(d.ops, d.nops, tid);
        for (uint64_t opa = reinterpret_cast<uint64_t>(d.ops); opa != ope; opa += sizeof(TileOp)) {
            asm volatile("" : "+s"(opa));
            const TileOp cur = fetch_op(opa);
            const uint64_t ahead = touch_next(cur, opa, ope);
            if (hit(cur.grp & TG_LAYOUT)) {
                LayoutMove<kRegs, kLogW> m;
                lt = m.set(cur.lay, lt, tid, lds);
                m.move(vr);
                m.move(vi);
                if constexpr (REV) {
                    m.move(ur);
                    m.move(ui);
                }
            }
            if constexpr (REV) {
                Sum g;
                adj_gate<kRegs, 4>(cur, base, lt, Amps{vr, vi, ur, ui}, g);
                if (cur.pad) {
                    row_sum(g);
                    // straight to memory: no bound on the sweep's gradients, and
                    // 16 KiB of LDS less per workgroup
                    if ((tid & 15u) == 0)
                        reinterpret_cast<double2 *>(d.part)[((uint64_t)(cur.pad - 1) * d.tiles + tile) *
                                                                kChipRows + (tid >> 4)] =
                            make_double2(g.s, g.c);
                }
            } else {
                fwd_gate(cur, base, lt, vr, vi);
            }
            asm volatile("" ::"s"(ahead));
        }
        if (d.flags & CHIP_STORE) {
            uint64_t gsb[kChipK];
#pragma unroll
            for (int b = 0; b < kChipK; b++) gsb[b] = 1ull << d.spos[b];
            const uint64_t to = (base + lane_offset<kChipK>(lt, gsb)) * sizeof(T);
#pragma unroll
            for (int p = 0; p < kRegs; p++) {
                const uint64_t o = to + d.gs[p];
                if (o < end) {
                    *(T *)((char *)d.pr + o) = (T)vr[p];
                    *(T *)((char *)d.pi + o) = (T)vi[p];
                    if constexpr (REV) {
                        *(T *)((char *)d.qr + o) = (T)ur[p];
                        *(T *)((char *)d.qi + o) = (T)ui[p];
                    }
                }
            }
        }
        __syncthreads();  // (the next tile reuses the LDS)
    }
}

template <typename T>
__global__ void __launch_bounds__(kRT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_chip_ising(const ChipIsing *__restrict__ all, double hx)
{
    __shared__ double S[kRT], C[kRT];
    const ChipIsing &d = all[blockIdx.y];
    if (blockIdx.x >= d.blocks) return;
    const T *re = (const T *)d.re, *im = (const T *)d.im;
    T *lr = (T *)d.lr, *li = (T *)d.li;
    double *out = d.part + 2 * (uint64_t)blockIdx.x;
    if (d.N < kRB)
        ising_block<T, true, true>(re, im, lr, li, 0, d.n, d.N, hx, out, S, C);
    else
        ising_block<T, true, false>(re, im, lr, li, blockIdx.x * kRB, d.n, d.N, hx, out, S, C);
}

// One wavefront per sum, four to a workgroup: a TwoSum chain per lane, then
// the halving tree over the lanes.
__global__ void __launch_bounds__(256)
k_chip_sum(const ChipSum *__restrict__ all, uint32_t count, double *__restrict__ out)
{
    const uint32_t i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (i >= count) return;
    const ChipSum d = all[i];
    double s = 0.0, c = 0.0;
    for (uint32_t j = lane; j < d.n; j += 64) {
        double ns, e;
        two_sum(s, d.part[2 * (uint64_t)j], ns, e);
        c = (c + d.part[2 * (uint64_t)j + 1]) + e;
        s = ns;
    }
    for (int h = 32; h >= 1; h >>= 1) {
        const double os = __shfl_down(s, h), oc = __shfl_down(c, h);
        double ns, e;
        two_sum(s, os, ns, e);
        c = (c + oc) + e;
        s = ns;
    }
    if (lane == 0) out[d.dst] = s + c;
}

}  // namespace

int launch_chip_sweeps(int prec, bool reverse, const ChipSweep *d, uint32_t count, uint32_t width,
                       size_t lds)
{
    if (!count || !width) return SPZ_OK;
    if (count > 65535) return fail(SPZ_ERR_ARG, "too many circuits in a launch");
    const dim3 g(width, count), b(1 << kLogW);
    hipStream_t st = rt().stream;
    if (reverse) {
        if (prec != SPZ_F64) return fail(SPZ_ERR_ARG, "reverse sweeps take FP64 states");
        hipLaunchKernelGGL((k_chip<double, true>), g, b, lds, st, d);
    } else if (prec == SPZ_F64) {
        hipLaunchKernelGGL((k_chip<double, false>), g, b, lds, st, d);
    } else {
        hipLaunchKernelGGL((k_chip<float, false>), g, b, lds, st, d);
    }
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

int launch_chip_ising(const ChipIsing *d, uint32_t count, uint32_t width, double hx)
{
    if (!count || !width) return SPZ_OK;
    hipLaunchKernelGGL((k_chip_ising<double>), dim3(width, count), dim3(kRT), 0, rt().stream, d, hx);
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

int launch_chip_sums(const ChipSum *d, uint32_t count, double *out)
{
    if (!count) return SPZ_OK;
    hipLaunchKernelGGL(k_chip_sum, dim3((count + 3) / 4), dim3(256), 0, rt().stream, d, count, out);
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

void chip_geometry(const ChipPlan::Sweep &s, int n, int prec, ChipSweep &out)
{
    const uint64_t esz = prec == SPZ_F64 ? 8 : 4;
    for (int i = 0; i < 16; i++) {
        out.spos[i] = s.desc.spos[i];
        out.tin[i] = s.desc.tin[i];
        out.gr[i] = s.desc.gr[i] * esz;
        out.gs[i] = s.desc.gs[i] * esz;
    }
    for (int i = 0; i < 8; i++) out.tg[i] = s.desc.tg[i];
    out.limit = 1ull << n;
    out.tiles = n > kChipK ? 1u << (n - kChipK) : 1u;
    out.width = out.tiles;
    out.nops = s.op_count;
}

}  // namespace spz
