// spz_adj_body.h -- device code of the reverse sweeps: gate dispatch over the
// registers of psi and lambda with the gradient sums (see spz_adj_tile.hip),
// shared by the single-circuit and the batched kernels.
#pragma once

#include "spz_reduce.h"
#include "spz_tile_kernel.h"

namespace spz {

namespace {

template <int CTRL>
__device__ __forceinline__ double dpp_move(double x)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (uint64_t)(uint32_t)lo | ((uint64_t)(uint32_t)hi << 32));
}

// A compensated sum (S, C).
struct Sum {
    double s = 0.0, c = 0.0;
};

template <int CTRL>
__device__ __forceinline__ void row_step(Sum &g)
{
    const double xs = dpp_move<CTRL>(g.s), xc = dpp_move<CTRL>(g.c);
    double ns, e;
    two_sum(g.s, xs, ns, e);
    g.c = (g.c + xc) + e;
    g.s = ns;
}

// Sum over the 16 lanes of a row.
__device__ __forceinline__ void row_sum(Sum &g)
{
    row_step<0xB1>(g);   // quad_perm [1,0,3,2]
    row_step<0x4E>(g);   // quad_perm [2,3,0,1]
    row_step<0x141>(g);  // row_half_mirror
    row_step<0x140>(g);  // row_mirror
}

// Registers of one tile of psi (r, i) and lambda (u, v).
struct Amps {
    double *r, *i, *u, *v;
};

// The gradient sums are inline assembly like the updates: left to the compiler
// their products are shared between the dispatch's paths, which keeps them and
// copies of the amplitudes alive across the program (4000 spills).

// g += t: (S, C) <- TwoSum(S, t), with t = a0 b0 - a1 b1 + a2 b2 - a3 b3.
__device__ __forceinline__ void grad_4(Sum &g, double a0, double b0, double a1, double b1,
                                       double a2, double b2, double a3, double b3)
{
    double t, x, n;
    asm volatile("v_mul_f64 %0, %5, %6\n\t"
                 "v_fma_f64 %0, -%7, %8, %0\n\t"
                 "v_fma_f64 %0, %9, %10, %0\n\t"
                 "v_fma_f64 %0, -%11, %12, %0\n\t"
                 "v_add_f64 %2, %3, %0\n\t"
                 "v_add_f64 %1, %2, -%3\n\t"
                 "v_add_f64 %0, %0, -%1\n\t"
                 "v_add_f64 %1, %2, -%1\n\t"
                 "v_add_f64 %1, %3, -%1\n\t"
                 "v_add_f64 %0, %1, %0\n\t"
                 "v_add_f64 %4, %4, %0"
                 : "=&v"(t), "=&v"(x), "=&v"(n), "+v"(g.s), "+v"(g.c)
                 : "v"(a0), "v"(b0), "v"(a1), "v"(b1), "v"(a2), "v"(b2), "v"(a3), "v"(b3));
    g.s = n;
}

// g += a0 b0 - a1 b1
__device__ __forceinline__ void grad_2(Sum &g, double a0, double b0, double a1, double b1)
{
    double t, x, n;
    asm volatile("v_mul_f64 %0, %5, %6\n\t"
                 "v_fma_f64 %0, -%7, %8, %0\n\t"
                 "v_add_f64 %2, %3, %0\n\t"
                 "v_add_f64 %1, %2, -%3\n\t"
                 "v_add_f64 %0, %0, -%1\n\t"
                 "v_add_f64 %1, %2, -%1\n\t"
                 "v_add_f64 %1, %3, -%1\n\t"
                 "v_add_f64 %0, %1, %0\n\t"
                 "v_add_f64 %4, %4, %0"
                 : "=&v"(t), "=&v"(x), "=&v"(n), "+v"(g.s), "+v"(g.c)
                 : "v"(a0), "v"(b0), "v"(a1), "v"(b1));
    g.s = n;
}

// Two rotations of real pairs, x' = x c - y s, y' = y c + x s: one product and
// one FMA per output (a rounding less than the reference's two products and a
// sum).  NEG: the second pair by -s.
template <bool NEG>
__device__ __forceinline__ void rot_fma2(double c, double s, double &x0, double &y0, double &x1,
                                         double &y1)
{
    double t0, u0, t1, u1;
#define SPZ_ROT_FMA(N, P)                                                          \
    asm volatile("v_mul_f64 %0, %9, %5\n\t"                                        \
                 "v_mul_f64 %1, %9, %4\n\t"                                        \
                 "v_mul_f64 %2, %9, %7\n\t"                                        \
                 "v_mul_f64 %3, %9, %6\n\t"                                        \
                 "v_fma_f64 %4, %8, %4, -%0\n\t"                                   \
                 "v_fma_f64 %5, %8, %5, %1\n\t"                                    \
                 "v_fma_f64 %6, %8, %6, " N "%2\n\t"                               \
                 "v_fma_f64 %7, %8, %7, " P "%3"                                    \
                 : "=&v"(t0), "=&v"(u0), "=&v"(t1), "=&v"(u1), "+v"(x0), "+v"(y0), \
                   "+v"(x1), "+v"(y1)                                              \
                 : "s"(c), "s"(s))
    if constexpr (NEG) SPZ_ROT_FMA("", "-");
    else SPZ_ROT_FMA("-", "");
#undef SPZ_ROT_FMA
}

template <int R, int AK, int J, bool PRED>
__device__ __forceinline__ void rot_pairs(double *r, double *i, const double *k, uint32_t pm)
{
#pragma unroll
    for (int p = 0; p < R; p++) {
        if (p & (1 << J)) continue;
        const int q = p | (1 << J);
        if (PRED && !((pm >> p) & 1u)) continue;
        if constexpr (AK == AK_RX) rot_fma2<true>(k[0], k[1], r[p], i[q], i[p], r[q]);
        else rot_fma2<false>(k[1], k[0], r[p], r[q], i[p], i[q]);
    }
}

// Gradient terms and inverse of a 2x2 gate on register bit J of both states.
template <int R, int AK, int J, bool PRED>
__device__ __forceinline__ void adj_pair_j(const Amps &s, const double *k, uint32_t pm, Sum &g)
{
    if constexpr (AK == AK_RX || AK == AK_RY) {
#pragma unroll
        for (int p = 0; p < R; p++) {
            if (p & (1 << J)) continue;
            const int q = p | (1 << J);
            if (PRED && !((pm >> p) & 1u)) continue;
            if constexpr (AK == AK_RX)  // Im <l|X|p> = Im(l0* p1) + Im(l1* p0)
                grad_4(g, s.u[p], s.i[q], s.v[p], s.r[q], s.u[q], s.i[p], s.v[q], s.r[p]);
            else  // Im <l|Y|p> = Re(l1* p0) - Re(l0* p1)
                grad_4(g, s.u[q], s.r[p], s.u[p], s.r[q], s.v[q], s.i[p], s.v[p], s.i[q]);
        }
    }
    if constexpr (AK == AK_RX || AK == AK_RY) {
        rot_pairs<R, AK, J, PRED>(s.r, s.i, k, pm);
        rot_pairs<R, AK, J, PRED>(s.u, s.v, k, pm);
    } else {
        pair_j<R, AK, J, PRED, false>(s.r, s.i, k, pm);
        pair_j<R, AK, J, PRED, false>(s.u, s.v, k, pm);
    }
}

template <int R, int RB, int AK, bool PRED>
__device__ __forceinline__ void adj_pair_sel(uint32_t sel, const Amps &s, const double *k,
                                             uint32_t pm, Sum &g)
{
    if (hit(sel & 1u)) adj_pair_j<R, AK, 0, PRED>(s, k, pm, g);
    if (hit(sel & 2u)) adj_pair_j<R, AK, 1, PRED>(s, k, pm, g);
    if (hit(sel & 4u)) adj_pair_j<R, AK, 2, PRED>(s, k, pm, g);
    if (hit(sel & 8u)) adj_pair_j<R, AK, 3, PRED>(s, k, pm, g);
}

template <int R, int RB, bool PRED>
__device__ __forceinline__ void adj_pair_kinds(uint32_t gr, uint32_t sel, const Amps &s,
                                               const double *k, uint32_t pm, Sum &g)
{
    if (hit(gr & (TG_H | TG_X | TG_Y))) {
        if (hit(gr & TG_H)) adj_pair_sel<R, RB, AK_H, PRED>(sel, s, k, pm, g);
        if (hit(gr & TG_X)) adj_pair_sel<R, RB, AK_X, PRED>(sel, s, k, pm, g);
        if (hit(gr & TG_Y)) adj_pair_sel<R, RB, AK_Y, PRED>(sel, s, k, pm, g);
    }
    if (hit(gr & (TG_RX | TG_RY | TG_U))) {
        if (hit(gr & TG_RX)) adj_pair_sel<R, RB, AK_RX, PRED>(sel, s, k, pm, g);
        if (hit(gr & TG_RY)) adj_pair_sel<R, RB, AK_RY, PRED>(sel, s, k, pm, g);
        if (hit(gr & TG_U)) adj_pair_sel<R, RB, AK_U, PRED>(sel, s, k, pm, g);
    }
}

// Diagonal gates with the target on register bit J.  RZ: Im(l0* p0) - Im(l1* p1);
// P: -2 Im(l1* p1).
template <int R, int AK, int J, bool PRED>
__device__ __forceinline__ void adj_diag_j(const Amps &s, const double *k, uint32_t pm, Sum &g)
{
    if constexpr (AK == AK_RZ || AK == AK_PHASE) {
#pragma unroll
        for (int p = 0; p < R; p++) {
            if (PRED && !((pm >> p) & 1u)) continue;
            if (p & (1 << J)) continue;
            const int q = p | (1 << J);
            if constexpr (AK == AK_RZ)  // (no control on the target: q passes with p)
                grad_4(g, s.u[p], s.i[p], s.v[p], s.r[p], s.v[q], s.r[q], s.u[q], s.i[q]);
            else
                grad_2(g, s.v[q], s.r[q], s.u[q], s.i[q]);
        }
        if constexpr (AK == AK_PHASE) {
            g.s = g.s + g.s;
            g.c = g.c + g.c;
        }
    }
    diag_j<R, AK, J, PRED, false>(s.r, s.i, k, pm);
    diag_j<R, AK, J, PRED, false>(s.u, s.v, k, pm);
}

template <int R, int RB, int AK, bool PRED>
__device__ __forceinline__ void adj_diag_sel(uint32_t sel, const Amps &s, const double *k,
                                             uint32_t pm, Sum &g)
{
    if (hit(sel & 1u)) adj_diag_j<R, AK, 0, PRED>(s, k, pm, g);
    if (hit(sel & 2u)) adj_diag_j<R, AK, 1, PRED>(s, k, pm, g);
    if (hit(sel & 4u)) adj_diag_j<R, AK, 2, PRED>(s, k, pm, g);
    if (hit(sel & 8u)) adj_diag_j<R, AK, 3, PRED>(s, k, pm, g);
}

template <int R, int RB, bool PRED>
__device__ __forceinline__ void adj_diag_reg(uint32_t gr, uint32_t sel, const Amps &s,
                                             const double *k, uint32_t pm, Sum &g)
{
    if (hit(gr & TG_NEG)) adj_diag_sel<R, RB, AK_NEG, PRED>(sel, s, k, pm, g);
    if (hit(gr & TG_PHASE)) adj_diag_sel<R, RB, AK_PHASE, PRED>(sel, s, k, pm, g);
    if (hit(gr & TG_RZ)) adj_diag_sel<R, RB, AK_RZ, PRED>(sel, s, k, pm, g);
}

// ... and with the target on a lane bit or outside the tile.
template <int R, int AK, bool PRED>
__device__ __forceinline__ void adj_diag_lane(const Amps &s, const double *k, bool bit,
                                              uint32_t pm, Sum &g)
{
    if constexpr (AK == AK_RZ || AK == AK_PHASE) {
#pragma unroll
        for (int p = 0; p < R; p++) {
            if constexpr (PRED) {
                if ((pm >> p) & 1u) grad_2(g, s.u[p], s.i[p], s.v[p], s.r[p]);
            } else if (p < R / 2) {
                const int q = p + R / 2;
                grad_4(g, s.u[p], s.i[p], s.v[p], s.r[p], s.u[q], s.i[q], s.v[q], s.r[q]);
            }
        }
        const double f = AK == AK_RZ ? (bit ? -1.0 : 1.0) : (bit ? -2.0 : 0.0);
        g.s = g.s * f;
        g.c = g.c * f;
    }
    diag_lane<R, AK, PRED, false>(s.r, s.i, k, bit, pm);
    diag_lane<R, AK, PRED, false>(s.u, s.v, k, bit, pm);
}

template <int R, bool PRED>
__device__ __forceinline__ void adj_diag_lane_kinds(uint32_t gr, const Amps &s, const double *k,
                                                    bool bit, uint32_t pm, Sum &g)
{
    if (hit(gr & TG_NEG)) adj_diag_lane<R, AK_NEG, PRED>(s, k, bit, pm, g);
    if (hit(gr & TG_PHASE)) adj_diag_lane<R, AK_PHASE, PRED>(s, k, bit, pm, g);
    if (hit(gr & TG_RZ)) adj_diag_lane<R, AK_RZ, PRED>(s, k, bit, pm, g);
}

// An LDS change of layout: set() forms the addresses, move() takes one
// register array through it.
template <int R, int LOGW>
struct LayoutMove {
    uint32_t so, sn, ro[R], rn[R];
    char *lb;

    __device__ __forceinline__ uint32_t set(const TileLayout &lay, uint32_t lt, uint32_t tid,
                                            double *lds)
    {
        uint32_t nlt = 0;
#pragma unroll
        for (int i = 0; i < LOGW; i++) nlt |= ((tid >> i) & 1u) << lay.newthr[i];
        so = swz(lt) << 3;
        sn = swz(nlt) << 3;
        asm volatile("" : "+v"(so), "+v"(sn));
        ro[0] = 0;
        rn[0] = 0;
#pragma unroll
        for (int p = 1; p < R; p++) {
            const int j = __builtin_ctz(p);
            ro[p] = ro[p & (p - 1)] ^ lay.rob[j];
            rn[p] = rn[p & (p - 1)] ^ lay.rnb[j];
        }
        lb = reinterpret_cast<char *>(lds);
        return nlt;
    }

    __device__ __forceinline__ void move(double *x) const
    {
        __syncthreads();
#pragma unroll
        for (int p = 0; p < R; p++) *reinterpret_cast<double *>(lb + (so ^ ro[p])) = x[p];
        __syncthreads();
#pragma unroll
        for (int p = 0; p < R; p++) x[p] = *reinterpret_cast<const double *>(lb + (sn ^ rn[p]));
    }
};

// Undo one gate on both states; its gradient terms go to g.
template <int R, int RB>
__device__ __forceinline__ void adj_gate(const TileOp &cur, uint64_t base, uint32_t lt,
                                         const Amps &s, Sum &g)
{
    if ((base & cur.em) != cur.eo) return;
    const uint32_t gr = cur.grp, sel = cur.sel, pm = cur.pm;
    const double *k = cur.c;
    if (hit(gr & (TG_PAIR | TG_PAIRP))) {
        if (hit(gr & TG_PAIR)) adj_pair_kinds<R, RB, false>(gr, sel, s, k, 0, g);
        if (hit(gr & TG_PAIRP))
            if (lane_pass(lt, cur.mlo, cur.mlz))
                adj_pair_kinds<R, RB, true>(gr, sel, s, k, pm, g);
    }
    if (hit(gr & (TG_DREG | TG_DREGP | TG_DLANE | TG_DLANEP))) {
        if (hit(gr & TG_DREG)) adj_diag_reg<R, RB, false>(gr, sel, s, k, 0, g);
        if (hit(gr & TG_DREGP))
            if (lane_pass(lt, cur.mlo, cur.mlz)) adj_diag_reg<R, RB, true>(gr, sel, s, k, pm, g);
        if (hit(gr & (TG_DLANE | TG_DLANEP))) {
            const bool bit = cur.dsel == 2 ? (base & cur.ebit) != 0
                                           : ((lt >> cur.dpos) & 1u) != 0;
            if (hit(gr & TG_DLANE)) adj_diag_lane_kinds<R, false>(gr, s, k, bit, 0, g);
            if (hit(gr & TG_DLANEP))
                if (lane_pass(lt, cur.mlo, cur.mlz))
                    adj_diag_lane_kinds<R, true>(gr, s, k, bit, pm, g);
        }
    }
}

// Add up one slot's row sums (in LDS) into a pair at o.
__device__ __forceinline__ void sum_rows(const double2 *rows, int n, double *o)
{
    double t = 0.0, c = 0.0;
    for (int w = 0; w < n; w++) {
        double ns, e;
        two_sum(t, rows[w].x, ns, e);
        c = (c + rows[w].y) + e;
        t = ns;
    }
    o[0] = t;
    o[1] = c;
}

}  // namespace

}  // namespace spz
