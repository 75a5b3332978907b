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
        asm volatile("" : "+s"(opa));  // (scalar loads off one advancing base, as in k_tile)
        TileOp cur;
        {
            const __attribute__((address_space(4))) uint64_t *w =
                reinterpret_cast<const __attribute__((address_space(4))) uint64_t *>(opa);
            uint64_t x[sizeof(TileOp) / 8];
#pragma unroll
            for (int i = 0; i < (int)(sizeof(TileOp) / 8); i++) x[i] = w[i];
            __builtin_memcpy(&cur, x, sizeof(TileOp));
        }
        const uint32_t gr = cur.grp;
        if (hit(gr & TG_LAYOUT)) {
            uint32_t nlt = 0;
#pragma unroll
            for (int i = 0; i < LOGW; i++) nlt |= ((tid >> i) & 1u) << cur.lay.newthr[i];
            uint32_t so = swz(lt) << 3, sn = swz(nlt) << 3;
            asm volatile("" : "+v"(so), "+v"(sn));
            uint32_t ro[R], rn[R];
            ro[0] = 0;
            rn[0] = 0;
#pragma unroll
            for (int p = 1; p < R; p++) {
                const int j = __builtin_ctz(p);
                ro[p] = ro[p & (p - 1)] ^ cur.lay.rob[j];
                rn[p] = rn[p & (p - 1)] ^ cur.lay.rnb[j];
            }
            char *lb = reinterpret_cast<char *>(lds);
            auto move = [&](double *x) {
                __syncthreads();
#pragma unroll
                for (int p = 0; p < R; p++) *reinterpret_cast<double *>(lb + (so ^ ro[p])) = x[p];
                __syncthreads();
#pragma unroll
                for (int p = 0; p < R; p++)
                    x[p] = *reinterpret_cast<const double *>(lb + (sn ^ rn[p]));
            };
            move(vr);
            move(vi);
            move(ur);
            move(ui);
            lt = nlt;
        }
        Sum g;
        if ((base & cur.em) == cur.eo) {
            const uint32_t sel = cur.sel, pm = cur.pm;
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
                    if (lane_pass(lt, cur.mlo, cur.mlz))
                        adj_diag_reg<R, RB, true>(gr, sel, s, k, pm, g);
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
    if ((int)tid < slots) {  // slots <= kAdjSlots <= threads
        double t = 0.0, c = 0.0;
        for (int w = 0; w < ROWS; w++) {
            double ns, e;
            two_sum(t, sums[tid][w].x, ns, e);
            c = (c + sums[tid][w].y) + e;
            t = ns;
        }
        double *o = part + 2 * ((uint64_t)tid * gridDim.x + blockIdx.x);
        o[0] = t;
        o[1] = c;
    }
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
    const size_t esz = psi->prec == SPZ_F64 ? sizeof(double) : sizeof(float);
    TileDesc db = d;  // register terms as byte offsets
    for (int p = 0; p < 16; p++) {
        db.gr[p] *= esz;
        db.gs[p] *= esz;
    }
    LaunchTimer tm(SPZ_K_ADJOINT, 8.0 * (double)psi->N * (double)esz);
    const dim3 g((unsigned)tiles), b(1 << (kAdjK - 4));
#define SPZ_ADJ(T)                                                                          \
    hipLaunchKernelGGL((k_adj_tile<T, kAdjK>), g, b, 0, rt().stream, (const T *)src->re,      \
                       (const T *)src->im, (T *)psi->re, (T *)psi->im, (T *)lam->re,          \
                       (T *)lam->im, db, d_ops, slots, part)
    if (psi->prec == SPZ_F64) SPZ_ADJ(double);
    else SPZ_ADJ(float);
#undef SPZ_ADJ
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
