// spz_adj_group.hip -- the reverse pass of the adjoint gradient for FP32 storage.
//
// Consecutive ops (taken backwards) whose targets fit in 3 qubits form a group
// that costs one pass over psi and lambda: per element (the 8 amplitudes that
// differ in those qubits) each op adds its gradient term (TwoSum-compensated
// FP64 per thread, a halving tree per block, one more block over the block
// partials, written to a device gradient array) and then applies U_k^dag to
// both states.  Runs of 4 or more parameter-free ops are undone with the fused
// tile executor, once on psi and once on lambda.
//
// FP64 states go back in tile sweeps (spz_adj_tile.hip), which are 3 times as
// fast.  FP32 states keep the groups because these fix where the states are
// rounded to FP32: sweeps round less often and give other gradients (more
// accurate ones, 5e-8 instead of 4e-7), and a caller's results are not to move
// by that.
#include <string.h>

#include <algorithm>
#include <vector>

#include "spz_adj_tile.h"
#include "spz_inplace.h"
#include "spz_internal.h"
#include "spz_tile.h"

namespace spz {

namespace {

constexpr int kT = 256;

enum GradKind { GK_NONE = 0, GK_X = 1, GK_Y = 2, GK_Z = 3, GK_P = 4 };

__device__ __forceinline__ void two_sum_d(double a, double b, double &s, double &e)
{
    double ss = a + b;
    double bb = ss - a;
    double aa = ss - bb;
    e = (a - aa) + (b - bb);
    s = ss;
}

// Im(conj(a) b) for a = (ar, ai), b = (br, bi)
__device__ __forceinline__ double im_cj(double ar, double ai, double br, double bi)
{
    return ar * bi - ai * br;
}
__device__ __forceinline__ double re_cj(double ar, double ai, double br, double bi)
{
    return ar * br + ai * bi;
}

// A reverse-sweep group: up to kGMaxOps consecutive ops (taken in reverse
// order) whose targets lie in a set Q of at most kGMaxQ qubits.  One pass
// visits every element (the 2^|Q| amplitudes that differ only in the Q bits,
// with the common control bits fixed) and applies each op's inverse to both
// psi and lambda, after adding the op's gradient term for that element.
constexpr int kGMaxOps = 8;
constexpr int kGMaxQ = 3;
constexpr int kGPerThread = 4;  // elements per thread

struct GroupOp {
    int32_t ak, gk, tq;       // arithmetic, gradient kind, index of the target in Q
    uint32_t kb;              // one-hot kind bit (TileGroup TG_H ... TG_RZ) of ak
    uint64_t cm, ones;        // control mask and the control bits that must be 1
    double c[8];              // inverse-gate coefficients
};

struct GroupDesc {
    int8_t q[kGMaxQ + 1];  // the qubits of Q
    int32_t nop;
    uint64_t base_ones;    // common controls that must be 1 (fixed in every element)
    GroupOp op[kGMaxOps];
};

__device__ __forceinline__ double grad_term(int gk, double la, double lb, double lc, double ld,
                                            double a, double b, double c, double d)
{
    if (gk == GK_X)  // Im <l|X|p> = Im(l0* p1) + Im(l1* p0)
        return im_cj(la, lb, c, d) + im_cj(lc, ld, a, b);
    if (gk == GK_Y)  // Im <l|Y|p> = Re(l1* p0) - Re(l0* p1)
        return re_cj(lc, ld, a, b) - re_cj(la, lb, c, d);
    if (gk == GK_Z)  // Im <l|Z|p> = Im(l0* p0) - Im(l1* p1)
        return im_cj(la, lb, a, b) - im_cj(lc, ld, c, d);
    return -2.0 * im_cj(lc, ld, c, d);  // P: -2 Im <l|Pi_1|p>
}

// The inverse gate on one pair, in place (the kind is a compile-time constant).
template <int AK>
__device__ __forceinline__ void inv_pair(const double *k, double &a, double &b, double &c, double &d)
{
    if constexpr (AK == AK_H) ip_h(k[0], a, b, c, d);
    else if constexpr (AK == AK_X) { ip_swap(a, c); ip_swap(b, d); }
    else if constexpr (AK == AK_Y) ip_y(a, b, c, d);
    else if constexpr (AK == AK_RX) ip_rx(k[0], k[1], a, b, c, d);
    else if constexpr (AK == AK_RY) ip_ry(k[0], k[1], a, b, c, d);
    else if constexpr (AK == AK_U) ip_u(k, a, b, c, d);
    else if constexpr (AK == AK_NEG) { c = -c; d = -d; }
    else if constexpr (AK == AK_PHASE) ip_phase(k[0], k[1], c, d);
    else { ip_rz<false>(k[0], k[1], a, b); ip_rz<false>(k[2], k[3], c, d); }  // AK_RZ
}

// Apply op (target = Q[TQ]) to the pairs of one element, adding the gradient
// terms of the pairs whose controls are met to (s, e).
template <int M, int TQ, int AK>
__device__ __forceinline__ void group_apply(const GroupOp &op, uint64_t base, const uint64_t *off,
                                            double *ar, double *ai, double *lr, double *li,
                                            double &s, double &e)
{
#pragma unroll
    for (int x = 0; x < (1 << M); x++) {
        if (x & (1 << TQ)) continue;
        const int y = x | (1 << TQ);
        if (((base | off[x]) & op.cm) != op.ones) continue;
        if (op.gk != GK_NONE) {
            const double t = grad_term(op.gk, lr[x], li[x], lr[y], li[y], ar[x], ai[x], ar[y], ai[y]);
            double ns, er;
            two_sum_d(s, t, ns, er);
            s = ns;
            e = e + er;
        }
        inv_pair<AK>(op.c, ar[x], ai[x], ar[y], ai[y]);
        inv_pair<AK>(op.c, lr[x], li[x], lr[y], li[y]);
    }
}

// Dispatch on the op's kind through independent tests of one-hot bits (a
// multi-way branch would merge the register arrays of every path and copy them).
template <int M, int TQ>
__device__ __forceinline__ void group_kinds(const GroupOp &op, uint64_t base, const uint64_t *off,
                                            double *ar, double *ai, double *lr, double *li,
                                            double &s, double &e)
{
    const uint32_t kb = op.kb;
    if (kb & TG_H) group_apply<M, TQ, AK_H>(op, base, off, ar, ai, lr, li, s, e);
    if (kb & TG_X) group_apply<M, TQ, AK_X>(op, base, off, ar, ai, lr, li, s, e);
    if (kb & TG_Y) group_apply<M, TQ, AK_Y>(op, base, off, ar, ai, lr, li, s, e);
    if (kb & TG_RX) group_apply<M, TQ, AK_RX>(op, base, off, ar, ai, lr, li, s, e);
    if (kb & TG_RY) group_apply<M, TQ, AK_RY>(op, base, off, ar, ai, lr, li, s, e);
    if (kb & TG_U) group_apply<M, TQ, AK_U>(op, base, off, ar, ai, lr, li, s, e);
    if (kb & TG_NEG) group_apply<M, TQ, AK_NEG>(op, base, off, ar, ai, lr, li, s, e);
    if (kb & TG_PHASE) group_apply<M, TQ, AK_PHASE>(op, base, off, ar, ai, lr, li, s, e);
    if (kb & TG_RZ) group_apply<M, TQ, AK_RZ>(op, base, off, ar, ai, lr, li, s, e);
}

// partials[(j * gridDim.x + block) * 2 + {0, 1}]: compensated block sum of
// op j's gradient terms (ops without a gradient write nothing).
template <typename T, int M>
__global__ void __launch_bounds__(kT)
k_adj_group(T *__restrict__ pr, T *__restrict__ pi, T *__restrict__ qr, T *__restrict__ qi,
            uint64_t nel, PosList pl, GroupDesc gd, double *__restrict__ partials)
{
    __shared__ double S[kGMaxOps][kT], C[kGMaxOps][kT];
    const int tid = threadIdx.x;
    const int nop = gd.nop;
    for (int j = 0; j < nop; j++) {
        S[j][tid] = 0.0;
        C[j][tid] = 0.0;
    }
    uint64_t off[1 << M];
#pragma unroll
    for (int x = 0; x < (1 << M); x++) {
        uint64_t o = 0;
#pragma unroll
        for (int b = 0; b < M; b++)
            if (x & (1 << b)) o |= 1ull << gd.q[b];
        off[x] = o;
    }
    // blocks stride over chunks of kT * kGPerThread elements
    const uint64_t chunk = (uint64_t)kT * kGPerThread;
    for (uint64_t block0 = (uint64_t)blockIdx.x * chunk; block0 < nel;
         block0 += (uint64_t)gridDim.x * chunk) {
        for (int w = 0; w < kGPerThread; w++) {
            const uint64_t u = block0 + (uint64_t)w * kT + tid;
            if (u >= nel) break;
            const uint64_t base = insert_zeros(u, pl.pos, pl.np) | gd.base_ones;
            double ar[1 << M], ai[1 << M], lr[1 << M], li[1 << M];
#pragma unroll
            for (int x = 0; x < (1 << M); x++) {
                const uint64_t i = base | off[x];
                ar[x] = pr[i]; ai[x] = pi[i]; lr[x] = qr[i]; li[x] = qi[i];
            }
            for (int j = 0; j < nop; j++) {
                const GroupOp &op = gd.op[j];
                double s = S[j][tid], e = C[j][tid];
                const uint32_t tqb = 1u << op.tq;  // one-hot, tested independently
                if (tqb & 1u) group_kinds<M, 0>(op, base, off, ar, ai, lr, li, s, e);
                if constexpr (M > 1) if (tqb & 2u) group_kinds<M, 1>(op, base, off, ar, ai, lr, li, s, e);
                if constexpr (M > 2) if (tqb & 4u) group_kinds<M, 2>(op, base, off, ar, ai, lr, li, s, e);
                S[j][tid] = s;
                C[j][tid] = e;
            }
#pragma unroll
            for (int x = 0; x < (1 << M); x++) {
                const uint64_t i = base | off[x];
                pr[i] = (T)ar[x]; pi[i] = (T)ai[x]; qr[i] = (T)lr[x]; qi[i] = (T)li[x];
            }
        }
    }
    __syncthreads();
    for (int h = kT / 2; h >= 1; h >>= 1) {
        if (tid < h)
            for (int j = 0; j < nop; j++) {
                double ns, e;
                two_sum_d(S[j][tid], S[j][tid + h], ns, e);
                C[j][tid] = (C[j][tid] + C[j][tid + h]) + e;
                S[j][tid] = ns;
            }
        __syncthreads();
    }
    if (tid < nop && gd.op[tid].gk != GK_NONE) {
        const uint64_t k = ((uint64_t)tid * gridDim.x + blockIdx.x) * 2;
        partials[k] = S[tid][0];
        partials[k + 1] = C[tid][0];
    }
}

// Block j reduces op j's nb block partials into grad[idx.i[j]].
struct GradIdx {
    int64_t i[kGMaxOps];
};

__global__ void __launch_bounds__(kT)
k_adj_finish(const double *__restrict__ partials, uint64_t nb, GradIdx idx,
             double *__restrict__ grad)
{
    __shared__ double S[kT], C[kT];
    const int tid = threadIdx.x;
    const double *p = partials + (uint64_t)blockIdx.x * nb * 2;
    double s = 0.0, c = 0.0;
    for (uint64_t j = tid; j < nb; j += kT) {
        double ns, e;
        two_sum_d(s, p[2 * j], ns, e);
        c = (c + p[2 * j + 1]) + e;
        s = ns;
    }
    S[tid] = s;
    C[tid] = c;
    __syncthreads();
    for (int h = kT / 2; h >= 1; h >>= 1) {
        if (tid < h) {
            double ns, e;
            two_sum_d(S[tid], S[tid + h], ns, e);
            C[tid] = (C[tid] + C[tid + h]) + e;
            S[tid] = ns;
        }
        __syncthreads();
    }
    if (tid == 0 && idx.i[blockIdx.x] >= 0) grad[idx.i[blockIdx.x]] = S[0] + C[0];
}

// Blocks of kT threads covering `units` (per_block units each), capped at the
// dispatch limit of 2^32 - 1 work-items (element-wise kernels grid-stride).
inline unsigned blocks_for(uint64_t units, uint64_t per_block)
{
    uint64_t g = (units + per_block - 1) / per_block;
    const uint64_t cap = 0xFFFFFFFFull / kT;
    if (g > cap) g = cap;
    return (unsigned)(g == 0 ? 1 : g);
}

uint32_t kind_bit_of(int ak)
{
    switch (ak) {
    case AK_H: return TG_H;
    case AK_X: return TG_X;
    case AK_Y: return TG_Y;
    case AK_RX: return TG_RX;
    case AK_RY: return TG_RY;
    case AK_U: return TG_U;
    case AK_NEG: return TG_NEG;
    case AK_PHASE: return TG_PHASE;
    case AK_RZ: return TG_RZ;
    default: return 0;
    }
}

bool has_param(int kind)
{
    return kind == SPZ_RX || kind == SPZ_RY || kind == SPZ_RZ || kind == SPZ_P;
}

int grad_kind(int kind)
{
    switch (kind) {
    case SPZ_RX: return GK_X;
    case SPZ_RY: return GK_Y;
    case SPZ_RZ: return GK_Z;
    case SPZ_P: return GK_P;
    default: return GK_NONE;
    }
}

int launch_group(spz_state_s *psi, spz_state_s *lam, int nq, uint64_t nel, const PosList &pl,
                 const GroupDesc &gd, double *partials, unsigned g)
{
    hipStream_t st = rt().stream;
#define SPZ_GRP(M)                                                                                \
    hipLaunchKernelGGL((k_adj_group<float, M>), dim3(g), dim3(kT), 0, st, (float *)psi->re,       \
                       (float *)psi->im, (float *)lam->re, (float *)lam->im, nel, pl, gd, partials)
    if (nq == 1) SPZ_GRP(1);
    else if (nq == 2) SPZ_GRP(2);
    else SPZ_GRP(3);
#undef SPZ_GRP
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

}  // namespace

size_t adj_group_part_bytes(uint64_t N)
{
    const uint64_t per_block = (uint64_t)kT * kGPerThread;
    return ((N / 2 + per_block - 1) / per_block + 1) * 2 * kGMaxOps * sizeof(double);
}

int adjoint_undo_groups(spz_state_s *wk, spz_state_s *lm, const spz_op *ops, uint64_t lo_lim,
                        uint64_t ii, double *part, double *gdev)
{
    const uint64_t per_block = (uint64_t)kT * kGPerThread;
    const double amp = 8.0;
    const bool tiled = wk->n >= 13;  // the fused executor tiles 12 qubits
    constexpr uint64_t kMinRun = 4;
    spz_exec_opts eo;
    memset(&eo, 0, sizeof eo);
    eo.mode = SPZ_EXEC_AUTO;
    // run_lo[k - lo_lim]: first index of the run of parameter-free ops that ends at k
    std::vector<uint64_t> run_lo(ii - lo_lim);
    for (uint64_t k = lo_lim; k < ii; k++)
        run_lo[k - lo_lim] = has_param(ops[k].kind) ? k + 1
                             : k > lo_lim && !has_param(ops[k - 1].kind) ? run_lo[k - 1 - lo_lim]
                                                                         : k;
    while (ii > lo_lim) {
        const uint64_t hi = ii - 1;
        const spz_op &o = ops[hi];
        uint64_t lo = hi;
        if (tiled && !has_param(o.kind) && hi + 1 - run_lo[hi - lo_lim] >= kMinRun) {
            lo = run_lo[hi - lo_lim];
            std::vector<spz_op> inv;
            inv.reserve(hi + 1 - lo);
            for (uint64_t k = hi + 1; k-- > lo;) inv.push_back(inverse_op(ops[k]));
            SPZ_TRY(execute_ops(wk, inv.data(), inv.size(), nullptr, &eo, nullptr));
            SPZ_TRY(execute_ops(lm, inv.data(), inv.size(), nullptr, &eo, nullptr));
            ii = lo;
            continue;
        }
        if (o.kind == SPZ_SWAP) {  // self-inverse, no parameter
            SPZ_TRY(apply_gate(wk, SPZ_SWAP, 0, 0, 0, o.target, o.t1, o.ones, o.zeros));
            SPZ_TRY(apply_gate(lm, SPZ_SWAP, 0, 0, 0, o.target, o.t1, o.ones, o.zeros));
            ii = lo;
            continue;
        }
        // greedy group: ops hi, hi-1, ... while the targets fit in kGMaxQ qubits
        GroupDesc gd;
        memset(&gd, 0, sizeof gd);
        GradIdx gi;
        int nq = 0, ngrad = 0;
        uint64_t qmask = 0, all_ones = ~0ull, all_zeros = ~0ull;
        for (uint64_t k = hi + 1; k-- > lo_lim;) {
            const spz_op &g = ops[k];
            if (g.kind == SPZ_SWAP || gd.nop == kGMaxOps) break;
            if (k != hi && tiled && !has_param(g.kind) && k + 1 - run_lo[k - lo_lim] >= kMinRun)
                break;  // leave a long parameter-free run to the tile executor
            const uint64_t tb = 1ull << g.target;
            if (!(qmask & tb)) {
                if (nq == kGMaxQ) break;
                gd.q[nq++] = (int8_t)g.target;
                qmask |= tb;
            }
            GroupOp &go = gd.op[gd.nop];
            const spz_op inv = inverse_op(g);
            Coef kc;
            SPZ_TRY(make_coef(inv.kind, inv.theta, inv.phi, inv.lambda, &kc));
            go.ak = kc.ak;
            go.kb = kind_bit_of(kc.ak);
            if (!go.kb) return fail(SPZ_ERR_GATE, "adjoint: unsupported arithmetic");
            memcpy(go.c, kc.c, sizeof go.c);
            go.gk = grad_kind(g.kind);
            for (int b = 0; b < nq; b++)
                if (gd.q[b] == g.target) go.tq = b;
            go.cm = g.ones | g.zeros;
            go.ones = g.ones;
            all_ones &= g.ones;
            all_zeros &= g.zeros;
            gi.i[gd.nop] = go.gk != GK_NONE ? (int64_t)k : -1;
            ngrad += go.gk != GK_NONE;
            gd.nop++;
            lo = k;
        }
        // common controls outside Q are fixed positions of every element
        all_ones &= ~qmask;
        all_zeros &= ~qmask;
        gd.base_ones = all_ones;
        PosList pl;
        const int np = build_poslist(qmask | all_ones | all_zeros, &pl);
        const uint64_t nel = wk->N >> np;
        const unsigned g = blocks_for(nel, per_block);
        {
            LaunchTimer tm(SPZ_K_ADJOINT, 2.0 * 2.0 * (double)(nel << nq) * amp);
            SPZ_TRY(launch_group(wk, lm, nq, nel, pl, gd, part, g));
        }
        if (ngrad) {  // one block per op; ops without a gradient write nothing
            hipLaunchKernelGGL(k_adj_finish, dim3(gd.nop), dim3(kT), 0, rt().stream, part,
                               (uint64_t)g, gi, gdev);
            SPZ_HIP(hipGetLastError());
        }
        ii = lo;
    }
    return SPZ_OK;
}

}  // namespace spz
