// spz_kernels.hip -- plain (one gate per HBM pass) kernels for gfx950.
//
// Layout: two arrays re[N], im[N] (FP64 or FP32), N = 2^n.  A gate on target
// t pairs amplitude s0 (bit t clear) with s1 = s0 | 2^t.  The launch maps a
// flat pair index to s0 by inserting zero bits at the ascending positions of
// the target and every control, then OR-ing the controls that must read 1,
// so consecutive lanes touch consecutive addresses whenever the lowest
// inserted position is >= 1 (paired coalesced streams), and each lane then
// moves two consecutive pairs with 2-element vector loads.  Target 0 loads
// the pair itself as one 2-element vector.
//
// Every kernel is a grid-stride loop over "units" so that one launch of
// about 2048 workgroups keeps all 256 CUs busy for any state size.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "spz_reduce.h"

namespace spz {

namespace {

constexpr int kThreads = 256;
static_assert(kThreads == kRT, "the reductions share the kernels' block size");

enum Mode { MODE_VEC = 0, MODE_T0 = 1, MODE_SCALAR = 2 };

// Internal arithmetic kinds for the measurement collapse (k[0] = 1/sqrt(p)).
constexpr int AK_COLLAPSE0 = 20;   // keep |0> * scale, zero |1>
constexpr int AK_COLLAPSE1 = 21;   // keep |1> * scale, zero |0>
constexpr int AK_COLLAPSE1R = 22;  // keep |1> * scale, then X (reset)

template <int AK>
__device__ __forceinline__ void pair_op(const double *k, double &a, double &b, double &c,
                                        double &d)
{
    if constexpr (AK == AK_COLLAPSE0) {
        a = a * k[0]; b = b * k[0]; c = 0.0; d = 0.0;
    } else if constexpr (AK == AK_COLLAPSE1) {
        c = c * k[0]; d = d * k[0]; a = 0.0; b = 0.0;
    } else if constexpr (AK == AK_COLLAPSE1R) {
        a = c * k[0]; b = d * k[0]; c = 0.0; d = 0.0;
    } else {
        pair_update(AK, k, a, b, c, d);
    }
}

template <typename T> struct Vec2;
template <> struct Vec2<double> { using type = double2; };
template <> struct Vec2<float> { using type = float2; };

// Exact grids (one unit per thread) stream HBM markedly faster on MI355X than
// capped grid-stride launches (measured 5.5-6.0 vs 4.8-5.0 TB/s for paired
// streams); the grid-stride loop only engages beyond 2^30 workgroups.
// One unit per thread up to the dispatch limit (a grid of at most 2^32 - 1
// work-items); beyond it the grid-stride loops of the kernels take over.
inline unsigned grid_for(uint64_t units)
{
    uint64_t g = (units + kThreads - 1) / kThreads;
    const uint64_t cap = 0xFFFFFFFFull / kThreads;
    if (g > cap) g = cap;
    if (g == 0) g = 1;
    return (unsigned)g;
}

// Lane width of the plain kernels: 8-byte lanes (one pair per thread) by
// default; SPZ_PLAIN_VEC=1 selects 16-byte lanes (two pairs per thread).
inline bool plain_vec()
{
    static int v = -1;
    if (v < 0) {
        const char *e = getenv("SPZ_PLAIN_VEC");
        v = (e && e[0] == '1') ? 1 : 0;
    }
    return v == 1;
}

// ---------------------------------------------------------------------------
// Pair kernel
// ---------------------------------------------------------------------------
template <typename T, int AK, int MODE>
__global__ void __launch_bounds__(kThreads)
k_pair(T *__restrict__ re, T *__restrict__ im, uint64_t units, int target, uint64_t ones,
       PosList pl, Coef kc)
{
    using V = typename Vec2<T>::type;
    const uint64_t tb = 1ull << target;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; u < units; u += stride) {
        if constexpr (MODE == MODE_VEC) {
            uint64_t s0 = insert_zeros(u << 1, pl.pos, pl.np) | ones;
            uint64_t s1 = s0 | tb;
            V r0 = *reinterpret_cast<const V *>(re + s0);
            V i0 = *reinterpret_cast<const V *>(im + s0);
            V r1 = *reinterpret_cast<const V *>(re + s1);
            V i1 = *reinterpret_cast<const V *>(im + s1);
            double a0 = r0.x, b0 = i0.x, c0 = r1.x, d0 = i1.x;
            double a1 = r0.y, b1 = i0.y, c1 = r1.y, d1 = i1.y;
            pair_op<AK>(kc.c, a0, b0, c0, d0);
            pair_op<AK>(kc.c, a1, b1, c1, d1);
            r0.x = (T)a0; r0.y = (T)a1; i0.x = (T)b0; i0.y = (T)b1;
            r1.x = (T)c0; r1.y = (T)c1; i1.x = (T)d0; i1.y = (T)d1;
            *reinterpret_cast<V *>(re + s0) = r0;
            *reinterpret_cast<V *>(im + s0) = i0;
            *reinterpret_cast<V *>(re + s1) = r1;
            *reinterpret_cast<V *>(im + s1) = i1;
        } else if constexpr (MODE == MODE_T0) {
            uint64_t s0 = insert_zeros(u, pl.pos, pl.np) | ones;
            V r = *reinterpret_cast<const V *>(re + s0);
            V i = *reinterpret_cast<const V *>(im + s0);
            double a = r.x, b = i.x, c = r.y, d = i.y;
            pair_op<AK>(kc.c, a, b, c, d);
            r.x = (T)a; r.y = (T)c; i.x = (T)b; i.y = (T)d;
            *reinterpret_cast<V *>(re + s0) = r;
            *reinterpret_cast<V *>(im + s0) = i;
        } else {
            uint64_t s0 = insert_zeros(u, pl.pos, pl.np) | ones;
            uint64_t s1 = s0 | tb;
            double a = re[s0], b = im[s0], c = re[s1], d = im[s1];
            pair_op<AK>(kc.c, a, b, c, d);
            re[s0] = (T)a; im[s0] = (T)b; re[s1] = (T)c; im[s1] = (T)d;
        }
    }
}

// ---------------------------------------------------------------------------
// Diagonal kernel: visits only amplitudes whose fixed bits match.
// ---------------------------------------------------------------------------
template <typename T, int AK, int MODE>
__global__ void __launch_bounds__(kThreads)
k_diag(T *__restrict__ re, T *__restrict__ im, uint64_t units, int target, uint64_t ones,
       PosList pl, Coef kc)
{
    using V = typename Vec2<T>::type;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; u < units; u += stride) {
        if constexpr (MODE == MODE_VEC) {
            uint64_t j = insert_zeros(u << 1, pl.pos, pl.np) | ones;
            V r = *reinterpret_cast<const V *>(re + j);
            V i = *reinterpret_cast<const V *>(im + j);
            double x0 = r.x, y0 = i.x, x1 = r.y, y1 = i.y;
            diag_update(AK, kc.c, (int)((j >> target) & 1), x0, y0);
            diag_update(AK, kc.c, (int)(((j + 1) >> target) & 1), x1, y1);
            r.x = (T)x0; r.y = (T)x1; i.x = (T)y0; i.y = (T)y1;
            *reinterpret_cast<V *>(re + j) = r;
            *reinterpret_cast<V *>(im + j) = i;
        } else {
            uint64_t j = insert_zeros(u, pl.pos, pl.np) | ones;
            double x = re[j], y = im[j];
            diag_update(AK, kc.c, (int)((j >> target) & 1), x, y);
            re[j] = (T)x; im[j] = (T)y;
        }
    }
}

// ---------------------------------------------------------------------------
// SWAP kernel (gates.rs:1376-1386): exchange |..0_q0..1_q1..> and |..1_q0..0_q1..>
// ---------------------------------------------------------------------------
template <typename T, int MODE>
__global__ void __launch_bounds__(kThreads)
k_swap(T *__restrict__ re, T *__restrict__ im, uint64_t units, int q0, int q1, uint64_t ones,
       PosList pl)
{
    using V = typename Vec2<T>::type;
    const uint64_t b0 = 1ull << q0, b1 = 1ull << q1;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; u < units; u += stride) {
        if constexpr (MODE == MODE_VEC) {
            uint64_t base = insert_zeros(u << 1, pl.pos, pl.np) | ones;
            uint64_t sa = base | b1, sb = base | b0;
            V ra = *reinterpret_cast<const V *>(re + sa);
            V ia = *reinterpret_cast<const V *>(im + sa);
            V rb = *reinterpret_cast<const V *>(re + sb);
            V ib = *reinterpret_cast<const V *>(im + sb);
            *reinterpret_cast<V *>(re + sa) = rb;
            *reinterpret_cast<V *>(im + sa) = ib;
            *reinterpret_cast<V *>(re + sb) = ra;
            *reinterpret_cast<V *>(im + sb) = ia;
        } else {
            uint64_t base = insert_zeros(u, pl.pos, pl.np) | ones;
            uint64_t sa = base | b1, sb = base | b0;
            T r = re[sa], i = im[sa];
            re[sa] = re[sb]; im[sa] = im[sb];
            re[sb] = r; im[sb] = i;
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_fill_basis(T *__restrict__ re, T *__restrict__ im, uint64_t N, uint64_t index)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < N; j += stride) {
        re[j] = (T)(j == index ? 1.0 : 0.0);
        im[j] = (T)0.0;
    }
}

// ---------------------------------------------------------------------------
// Dense block (transform_u): each thread owns one 2^M-amplitude vector.
// Row dot products accumulate in the order of unitary_col_vec_mul
// (gates.rs:1405-1419).
// ---------------------------------------------------------------------------
template <typename T, int M>
__global__ void __launch_bounds__(kThreads)
k_dense(T *__restrict__ re, T *__restrict__ im, uint64_t units, int t, int control,
        const double *__restrict__ ur, const double *__restrict__ ui)
{
    constexpr int D = 1 << M;
    __shared__ double sr[D * D], si[D * D];
    for (int i = threadIdx.x; i < D * D; i += blockDim.x) { sr[i] = ur[i]; si[i] = ui[i]; }
    __syncthreads();
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t lowmask = (1ull << t) - 1ull;
    for (uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; u < units; u += stride) {
        uint64_t base = ((u >> t) << (t + M)) | (u & lowmask);
        if (control >= 0 && !((base >> control) & 1)) continue;
        double vr[D], vi[D];
#pragma unroll
        for (int j = 0; j < D; j++) {
            uint64_t kk = base + ((uint64_t)j << t);
            vr[j] = re[kk]; vi[j] = im[kk];
        }
#pragma unroll
        for (int row = 0; row < D; row++) {
            double dr = 0.0, di = 0.0;
#pragma unroll
            for (int col = 0; col < D; col++) {
                double a = sr[row * D + col], b = si[row * D + col];
                dr += a * vr[col] - b * vi[col];
                di += a * vi[col] + b * vr[col];
            }
            uint64_t kk = base + ((uint64_t)row << t);
            re[kk] = (T)dr; im[kk] = (T)di;
        }
    }
}

// Blocks of 8 amplitudes and more: a workgroup takes 64 vectors, staged in LDS,
// and each of its wavefronts a quarter of the rows (the same additions in the same
// order), with the coefficients in scalar registers.  Bound by one read and write
// of the state and, from m = 4 on, by 2^(m+3) unfused FP64 operations per
// amplitude.  One thread per vector left 1024 wavefronts for a 32-amplitude block
// of 21 qubits, read low blocks at a stride of the vector's length and took every
// coefficient from LDS.  m = 3, 4, 5, then and now: 21 qubits FP64 18-33, 68-84,
// 76-131 us, now 13-15, 17-18, 29-32; 26 qubits 494-824, 1990-2290, 2170-3240 us,
// now 360-400, 395-420, 517-546 (6.0, 5.4, 4.0 TB/s); 27 qubits FP32 0.94-2.1,
// 3.8-5.1, 4.5-5.8 ms, now 0.46-0.49, 0.58, 1.0; 12 qubits 6.2, 23, 44 us, now 6.2,
// 10, 26.
// coef: [wavefront][column][row of the wavefront][re, im] (dense_coefs).
// first: the launch's first workgroup of the whole (dense_dispatch).
template <typename T, int M>
__global__ void __launch_bounds__(kThreads)
k_dense_rows(T *__restrict__ re, T *__restrict__ im, uint64_t first, int t, int control,
             const double *__restrict__ coef)
{
    constexpr int D = 1 << M, ROWS = D / 4, LD = 65;  // (65: low blocks spread over the banks)
    __shared__ T vr[D * LD], vi[D * LD];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint64_t u0 = (first + blockIdx.x) * 64, u = u0 + lane;
    const uint64_t mine = ((u >> t) << (t + M)) | (u & ((1ull << t) - 1ull));
    const bool on = control < 0 || ((mine >> control) & 1);
    if (!__ballot(on)) return;  // the same for all four wavefronts
    // with t < 6 the 64 vectors are one run of memory: local index i holds
    // column (i >> t) % D of vector (i % 2^t) + (i >> (t + M)) 2^t
    auto place = [&](uint32_t i) {
        const uint32_t v = (i & ((1u << t) - 1u)) | ((i >> (t + M)) << t);
        return ((i >> t) & (D - 1)) * LD + v;
    };
    if (t >= 6) {
#pragma unroll
        for (int k = 0; k < ROWS; k++) {
            const uint32_t j = k * 4 + wave;
            const uint64_t g = mine + ((uint64_t)j << t);
            vr[j * LD + lane] = re[g];
            vi[j * LD + lane] = im[g];
        }
    } else {
#pragma unroll
        for (int k = 0; k < ROWS; k++) {
            const uint32_t i = k * kThreads + tid, o = place(i);
            vr[o] = re[(u0 << M) + i];
            vi[o] = im[(u0 << M) + i];
        }
    }
    __syncthreads();
    double dr[ROWS], di[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) dr[r] = di[r] = 0.0;
    const double *c = coef + wave * (2 * ROWS * D);
#pragma unroll 2
    for (int col = 0; col < D; col++, c += 2 * ROWS) {
        const double x = vr[col * LD + lane], y = vi[col * LD + lane];
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const double a = c[2 * r], b = c[2 * r + 1];
            dr[r] += a * x - b * y;
            di[r] += a * y + b * x;
        }
    }
    if (t >= 6) {
        if (!on) return;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const uint64_t g = mine + ((uint64_t)(wave * ROWS + r) << t);
            re[g] = (T)dr[r];
            im[g] = (T)di[r];
        }
        return;
    }
    __syncthreads();
    if (on) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            vr[(wave * ROWS + r) * LD + lane] = (T)dr[r];
            vi[(wave * ROWS + r) * LD + lane] = (T)di[r];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ROWS; k++) {
        const uint32_t i = k * kThreads + tid, o = place(i);
        re[(u0 << M) + i] = vr[o];
        im[(u0 << M) + i] = vi[o];
    }
}

// ---------------------------------------------------------------------------
// Fixed-tree compensated reduction (spz_reduce.h).
// ---------------------------------------------------------------------------
template <typename T, typename T2, int TERM>
__device__ __forceinline__ double term(const T *__restrict__ re, const T *__restrict__ im,
                                       const T2 *__restrict__ re2, const T2 *__restrict__ im2,
                                       uint64_t j, int q0, int q1, int n, double hx)
{
    if constexpr (TERM == TERM_NORM) {
        double x = re[j], y = im[j];
        return x * x + y * y;
    } else if constexpr (TERM == TERM_PROB0) {
        uint64_t lo = j & ((1ull << q0) - 1ull);
        uint64_t a = ((j >> q0) << (q0 + 1)) | lo;
        double x = re[a], y = im[a];
        return x * x + y * y;
    } else if constexpr (TERM == TERM_X) {
        uint64_t p = j ^ (1ull << q0);
        double a = re[j], b = im[j], c = re[p], d = im[p];
        return a * c + b * d;
    } else if constexpr (TERM == TERM_Y) {
        uint64_t p = j ^ (1ull << q0);
        double a = re[j], b = im[j];
        double vr, vi;
        if ((j >> q0) & 1) { vr = -(double)im[p]; vi = re[p]; }
        else { vr = im[p]; vi = -(double)re[p]; }
        return a * vr + b * vi;
    } else if constexpr (TERM == TERM_Z) {
        double a = re[j], b = im[j];
        double vr = a, vi = b;
        if ((j >> q0) & 1) { vr = -vr; vi = -vi; }
        return a * vr + b * vi;
    } else if constexpr (TERM == TERM_ZZ) {
        double x = re[j], y = im[j];
        double w = x * x + y * y;
        return (((j >> q0) ^ (j >> q1)) & 1) ? -w : w;
    } else if constexpr (TERM == TERM_DOT_RE) {
        double a = re[j], b = im[j], c = re2[j], d = im2[j];
        return a * c + b * d;
    } else {  // TERM_DOT_IM: Im(conj(a) b) = a_re*b_im - a_im*b_re
        double a = re[j], b = im[j], c = re2[j], d = im2[j];
        return a * d - b * c;
    }
}

// T2: storage type of the second state (dot products of an FP32 and an FP64
// state are summed in FP64 like the rest).
template <typename T, typename T2, int TERM>
__global__ void __launch_bounds__(kThreads)
k_reduce1(const T *__restrict__ re, const T *__restrict__ im, const T2 *__restrict__ re2,
          const T2 *__restrict__ im2, uint64_t M, int q0, int q1, int n, double hx,
          double *__restrict__ partials)
{
    __shared__ double S[kThreads], C[kThreads];
    const int tid = threadIdx.x;
    const uint64_t base = (uint64_t)blockIdx.x * kRB;
    double s = 0.0, c = 0.0;
#pragma unroll 4
    for (int e = 0; e < kRE; e++) {
        uint64_t j = base + (uint64_t)e * kThreads + tid;
        if (j < M) {
            double x = term<T, T2, TERM>(re, im, re2, im2, j, q0, q1, n, hx);
            double ns, er;
            two_sum(s, x, ns, er);
            s = ns;
            c = c + er;
        }
    }
    S[tid] = s;
    C[tid] = c;
    __syncthreads();
    tree256(S, C);
    if (tid == 0) {
        partials[2 * blockIdx.x] = S[0];
        partials[2 * blockIdx.x + 1] = C[0];
    }
}

// ---------------------------------------------------------------------------
// Dispatch helpers
// ---------------------------------------------------------------------------
template <typename T, int AK>
int pair_dispatch(spz_state_s *s, const Coef &k, int target, uint64_t ones, const PosList &pl,
                  uint64_t npairs, double bytes)
{
    T *re = (T *)s->re, *im = (T *)s->im;
    hipStream_t st = rt().stream;
    LaunchTimer tm(AK >= AK_COLLAPSE0 ? SPZ_K_OTHER : SPZ_K_PAIR, bytes);
    if (plain_vec() && pl.pos[0] >= 1 && npairs >= 2) {
        uint64_t units = npairs >> 1;
        hipLaunchKernelGGL((k_pair<T, AK, MODE_VEC>), dim3(grid_for(units)), dim3(kThreads), 0,
                           st, re, im, units, target, ones, pl, k);
    } else if (target == 0) {
        hipLaunchKernelGGL((k_pair<T, AK, MODE_T0>), dim3(grid_for(npairs)), dim3(kThreads), 0,
                           st, re, im, npairs, target, ones, pl, k);
    } else {
        hipLaunchKernelGGL((k_pair<T, AK, MODE_SCALAR>), dim3(grid_for(npairs)), dim3(kThreads),
                           0, st, re, im, npairs, target, ones, pl, k);
    }
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

template <typename T>
int pair_by_kind(spz_state_s *s, const Coef &k, int target, uint64_t ones, const PosList &pl,
                 uint64_t npairs, double bytes)
{
    switch (k.ak) {
    case AK_H: return pair_dispatch<T, AK_H>(s, k, target, ones, pl, npairs, bytes);
    case AK_X: return pair_dispatch<T, AK_X>(s, k, target, ones, pl, npairs, bytes);
    case AK_Y: return pair_dispatch<T, AK_Y>(s, k, target, ones, pl, npairs, bytes);
    case AK_RX: return pair_dispatch<T, AK_RX>(s, k, target, ones, pl, npairs, bytes);
    case AK_RY: return pair_dispatch<T, AK_RY>(s, k, target, ones, pl, npairs, bytes);
    case AK_U: return pair_dispatch<T, AK_U>(s, k, target, ones, pl, npairs, bytes);
    case AK_MAT: return pair_dispatch<T, AK_MAT>(s, k, target, ones, pl, npairs, bytes);
    case AK_COLLAPSE0: return pair_dispatch<T, AK_COLLAPSE0>(s, k, target, ones, pl, npairs, bytes);
    case AK_COLLAPSE1: return pair_dispatch<T, AK_COLLAPSE1>(s, k, target, ones, pl, npairs, bytes);
    case AK_COLLAPSE1R:
        return pair_dispatch<T, AK_COLLAPSE1R>(s, k, target, ones, pl, npairs, bytes);
    default: return fail(SPZ_ERR_GATE, "pair kernel: unsupported arithmetic kind");
    }
}

template <typename T, int AK>
int diag_dispatch(spz_state_s *s, const Coef &k, int target, uint64_t ones, const PosList &pl,
                  uint64_t namps, double bytes)
{
    T *re = (T *)s->re, *im = (T *)s->im;
    hipStream_t st = rt().stream;
    LaunchTimer tm(SPZ_K_DIAG, bytes);
    if (plain_vec() && (pl.np == 0 || pl.pos[0] >= 1) && namps >= 2) {
        uint64_t units = namps >> 1;
        hipLaunchKernelGGL((k_diag<T, AK, MODE_VEC>), dim3(grid_for(units)), dim3(kThreads), 0,
                           st, re, im, units, target, ones, pl, k);
    } else {
        hipLaunchKernelGGL((k_diag<T, AK, MODE_SCALAR>), dim3(grid_for(namps)), dim3(kThreads),
                           0, st, re, im, namps, target, ones, pl, k);
    }
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

template <typename T>
int diag_by_kind(spz_state_s *s, const Coef &k, int target, uint64_t ones, const PosList &pl,
                 uint64_t namps, double bytes)
{
    switch (k.ak) {
    case AK_NEG: return diag_dispatch<T, AK_NEG>(s, k, target, ones, pl, namps, bytes);
    case AK_PHASE: return diag_dispatch<T, AK_PHASE>(s, k, target, ones, pl, namps, bytes);
    case AK_RZ: return diag_dispatch<T, AK_RZ>(s, k, target, ones, pl, namps, bytes);
    default: return fail(SPZ_ERR_GATE, "diag kernel: unsupported arithmetic kind");
    }
}

inline double amp_bytes(const spz_state_s *s) { return s->prec == SPZ_F64 ? 16.0 : 8.0; }

}  // namespace

int build_poslist(uint64_t mask, PosList *pl)
{
    pl->np = 0;
    for (int q = 0; q < 64; q++)
        if ((mask >> q) & 1) pl->pos[pl->np++] = (int8_t)q;
    for (int i = pl->np; i < 64; i++) pl->pos[i] = 64;
    return pl->np;
}

int launch_pair(spz_state_s *s, const Coef &k, int target, uint64_t ones, uint64_t zeros)
{
    PosList pl;
    uint64_t fixed = ones | zeros | (1ull << target);
    int np = build_poslist(fixed, &pl);
    if (np > s->n) return fail(SPZ_ERR_QUBIT, "more fixed qubits than the state has");
    uint64_t npairs = s->N >> np;
    // read + write both amplitudes of every visited pair
    double bytes = 2.0 * 2.0 * (double)npairs * amp_bytes(s);
    if (s->prec == SPZ_F64) return pair_by_kind<double>(s, k, target, ones, pl, npairs, bytes);
    return pair_by_kind<float>(s, k, target, ones, pl, npairs, bytes);
}

int launch_diag(spz_state_s *s, const Coef &k, int target, uint64_t ones, uint64_t zeros)
{
    PosList pl;
    uint64_t fixed = ones | zeros;
    uint64_t ones2 = ones;
    if (k.ak != AK_RZ) {  // Z and P only touch amplitudes with the target bit set
        fixed |= 1ull << target;
        ones2 |= 1ull << target;
    }
    int np = build_poslist(fixed, &pl);
    if (np > s->n) return fail(SPZ_ERR_QUBIT, "more fixed qubits than the state has");
    uint64_t namps = s->N >> np;
    double bytes = 2.0 * (double)namps * amp_bytes(s);
    if (s->prec == SPZ_F64) return diag_by_kind<double>(s, k, target, ones2, pl, namps, bytes);
    return diag_by_kind<float>(s, k, target, ones2, pl, namps, bytes);
}

int launch_swap(spz_state_s *s, int q0, int q1, uint64_t ones, uint64_t zeros)
{
    PosList pl;
    uint64_t fixed = ones | zeros | (1ull << q0) | (1ull << q1);
    int np = build_poslist(fixed, &pl);
    uint64_t units = s->N >> np;  // pairs of swapped amplitudes
    double bytes = 2.0 * 2.0 * (double)units * amp_bytes(s);
    hipStream_t st = rt().stream;
    LaunchTimer tm(SPZ_K_PAIR, bytes);
    if (s->prec == SPZ_F64) {
        if (plain_vec() && pl.pos[0] >= 1 && units >= 2)
            hipLaunchKernelGGL((k_swap<double, MODE_VEC>), dim3(grid_for(units >> 1)),
                               dim3(kThreads), 0, st, (double *)s->re, (double *)s->im,
                               units >> 1, q0, q1, ones, pl);
        else
            hipLaunchKernelGGL((k_swap<double, MODE_SCALAR>), dim3(grid_for(units)),
                               dim3(kThreads), 0, st, (double *)s->re, (double *)s->im, units, q0,
                               q1, ones, pl);
    } else {
        if (plain_vec() && pl.pos[0] >= 1 && units >= 2)
            hipLaunchKernelGGL((k_swap<float, MODE_VEC>), dim3(grid_for(units >> 1)),
                               dim3(kThreads), 0, st, (float *)s->re, (float *)s->im, units >> 1,
                               q0, q1, ones, pl);
        else
            hipLaunchKernelGGL((k_swap<float, MODE_SCALAR>), dim3(grid_for(units)),
                               dim3(kThreads), 0, st, (float *)s->re, (float *)s->im, units, q0,
                               q1, ones, pl);
    }
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

int launch_collapse(spz_state_s *s, int target, int outcome, int reset, double scale)
{
    Coef k{};
    k.ak = outcome == 0 ? AK_COLLAPSE0 : (reset ? AK_COLLAPSE1R : AK_COLLAPSE1);
    k.c[0] = scale;
    return launch_pair(s, k, target, 0, 0);
}

int launch_fill_basis(spz_state_s *s, uint64_t index)
{
    hipStream_t st = rt().stream;
    LaunchTimer tm(SPZ_K_OTHER, (double)s->N * amp_bytes(s));
    if (s->prec == SPZ_F64)
        hipLaunchKernelGGL((k_fill_basis<double>), dim3(grid_for(s->N)), dim3(kThreads), 0, st,
                           (double *)s->re, (double *)s->im, s->N, index);
    else
        hipLaunchKernelGGL((k_fill_basis<float>), dim3(grid_for(s->N)), dim3(kThreads), 0, st,
                           (float *)s->re, (float *)s->im, s->N, index);
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

// Whether a block runs on k_dense_rows: 8 amplitudes and more, and at least the 64
// vectors of a workgroup.  (Blocks of 4 are at the memory rate with a thread per
// vector, 9-19 us at 21 qubits, and have one row to a wavefront here.)
static bool dense_by_rows(const spz_state_s *s, int m) { return m >= 3 && (s->N >> m) >= 64; }

// The block's matrix (row-major) in the order its kernel reads it.
void dense_coefs(const spz_state_s *s, int m, const double *ur, const double *ui,
                 std::vector<double> &out)
{
    const size_t D = (size_t)1 << m, rows = D / 4;
    out.resize(2 * D * D);
    for (size_t row = 0; row < D; row++)
        for (size_t col = 0; col < D; col++) {
            const double a = ur[row * D + col], b = ui[row * D + col];
            if (dense_by_rows(s, m)) {
                double *o = &out[2 * (((row / rows) * D + col) * rows + row % rows)];
                o[0] = a;
                o[1] = b;
            } else {
                out[row * D + col] = a;
                out[D * D + row * D + col] = b;
            }
        }
}

template <typename T>
static int dense_dispatch(spz_state_s *s, int m, const double *coef, int t, int control)
{
    const uint64_t units = s->N >> m;
    hipStream_t st = rt().stream;
    T *re = (T *)s->re, *im = (T *)s->im;
    const double *ui = coef + ((size_t)1 << (2 * m));
    LaunchTimer tm(SPZ_K_DENSE, 2.0 * (double)s->N * amp_bytes(s));
#define SPZ_DENSE(M)                                                                            \
    hipLaunchKernelGGL((k_dense<T, M>), dim3(grid_for(units)), dim3(kThreads), 0, st, re, im,     \
                       units, t, control, coef, ui)
    // workgroups of 64 vectors, at most 2^23 of them to a launch: 2^31 work-items,
    // where a dispatch takes fewer than 2^32 (a 3-qubit block of 33 qubits has 2^24)
    const uint64_t groups = units / 64, most = 1ull << 23;
#define SPZ_DENSE_ROWS(M)                                                                       \
    for (uint64_t f = 0; f < groups; f += most)                                                   \
        hipLaunchKernelGGL((k_dense_rows<T, M>), dim3((unsigned)std::min(groups - f, most)),       \
                           dim3(kThreads), 0, st, re, im, f, t, control, coef)
    if (dense_by_rows(s, m)) {
        switch (m) {
        case 3: SPZ_DENSE_ROWS(3); break;
        case 4: SPZ_DENSE_ROWS(4); break;
        case 5: SPZ_DENSE_ROWS(5); break;
        default: return fail(SPZ_ERR_ARG, "dense block wider than 5 qubits");
        }
    } else {
        switch (m) {
        case 1: SPZ_DENSE(1); break;
        case 2: SPZ_DENSE(2); break;
        case 3: SPZ_DENSE(3); break;
        case 4: SPZ_DENSE(4); break;
        case 5: SPZ_DENSE(5); break;
        default: return fail(SPZ_ERR_ARG, "dense block wider than 5 qubits");
        }
    }
#undef SPZ_DENSE
#undef SPZ_DENSE_ROWS
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

int launch_dense(spz_state_s *s, int m, const double *coef, int t, int control)
{
    if (s->prec == SPZ_F64) return dense_dispatch<double>(s, m, coef, t, control);
    return dense_dispatch<float>(s, m, coef, t, control);
}

// ---------------------------------------------------------------------------
// Reductions
// ---------------------------------------------------------------------------
template <typename T, typename T2 = T>
static int reduce_launch(const spz_state_s *a, const spz_state_s *b, int term, int q0, int q1,
                         double hx, uint64_t M, uint64_t nb, double *part)
{
    const T *re = (const T *)a->re, *im = (const T *)a->im;
    const T2 *re2 = b ? (const T2 *)b->re : nullptr, *im2 = b ? (const T2 *)b->im : nullptr;
    hipStream_t st = rt().stream;
    dim3 g((unsigned)nb), blk(kThreads);
    int n = a->n;
#define SPZ_RL(TM) hipLaunchKernelGGL((k_reduce1<T, T2, TM>), g, blk, 0, st, re, im, re2, im2, M, q0, q1, n, hx, part)
    if constexpr (!std::is_same<T, T2>::value) {  // mixed precision: dot products only
        if (term == TERM_DOT_RE) SPZ_RL(TERM_DOT_RE);
        else if (term == TERM_DOT_IM) SPZ_RL(TERM_DOT_IM);
        else return fail(SPZ_ERR_ARG, "mixed-precision reduction other than a dot product");
        SPZ_HIP(hipGetLastError());
        return SPZ_OK;
    }
    switch (term) {
    case TERM_NORM: SPZ_RL(TERM_NORM); break;
    case TERM_PROB0: SPZ_RL(TERM_PROB0); break;
    case TERM_X: SPZ_RL(TERM_X); break;
    case TERM_Y: SPZ_RL(TERM_Y); break;
    case TERM_Z: SPZ_RL(TERM_Z); break;
    case TERM_ZZ: SPZ_RL(TERM_ZZ); break;
    case TERM_DOT_RE: SPZ_RL(TERM_DOT_RE); break;
    case TERM_DOT_IM: SPZ_RL(TERM_DOT_IM); break;
    default: return fail(SPZ_ERR_ARG, "unknown reduction term");
    }
#undef SPZ_RL
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

static int reduce_level1(const spz_state_s *a, const spz_state_s *b, int term, int q0, int q1,
                         double hx, uint64_t *nb_out)
{
    uint64_t M = term == TERM_PROB0 ? (a->N >> 1) : a->N;
    uint64_t nb = (M + kRB - 1) / kRB;
    if (nb == 0) nb = 1;
    SPZ_TRY(ensure_partials(nb));
    double per_term = amp_bytes(a) * (term == TERM_X || term == TERM_Y ? 2.0 : 1.0);
    if (term == TERM_DOT_RE || term == TERM_DOT_IM) per_term = amp_bytes(a) + amp_bytes(b);
    LaunchTimer tm(SPZ_K_REDUCE, (double)M * per_term);
    int rc;
    double *part = rt().d_partials;
    if (b && b->prec != a->prec)
        rc = a->prec == SPZ_F64 ? reduce_launch<double, float>(a, b, term, q0, q1, hx, M, nb, part)
                                : reduce_launch<float, double>(a, b, term, q0, q1, hx, M, nb, part);
    else
        rc = a->prec == SPZ_F64 ? reduce_launch<double>(a, b, term, q0, q1, hx, M, nb, part)
                                : reduce_launch<float>(a, b, term, q0, q1, hx, M, nb, part);
    *nb_out = nb;
    return rc;
}

int reduce(const spz_state_s *a, const spz_state_s *b, int term, int q0, int q1, double hx,
           double *out)
{
    uint64_t nb;
    if (term == TERM_ISING) {
        nb = std::max<uint64_t>(a->N / kRB, 1);
        SPZ_TRY(ensure_partials(nb));
        LaunchTimer tm(SPZ_K_REDUCE, (double)a->N * amp_bytes(a));
        SPZ_TRY(ising_level1(a, hx, nullptr, nullptr, rt().d_partials));
    } else {
        SPZ_TRY(reduce_level1(a, b, term, q0, q1, hx, &nb));
    }
    return reduce_finish(rt().d_partials, nb, out);
}

// ---------------------------------------------------------------------------
// Ising energy without allocation (spz_ising_energy_noalloc)
// ---------------------------------------------------------------------------
// The block partials live in a file-scope device array of fixed
// size instead of the grow-only scratch that reduce() allocates: 2^18 blocks
// of 4096 terms (states up to 2^30 amplitudes, 30 qubits), 4 MiB of partial
// pairs.  Host code reaches it only through the address that
// hipGetSymbolAddress returns (the array's name is a host-side stand-in);
// that address is taken once, when the library initialises on its device.
// Every call shares the array; the library lock serialises calls within a
// process, and each call overwrites every pair it reads (no clearing needed).
constexpr uint64_t kStaticBlocks = 1ull << 18;
static __device__ __align__(256) double scratch[2 * kStaticBlocks];
static double *g_static_scratch = nullptr;

int static_scratch_init()
{
    void *p = nullptr;
    SPZ_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_static_scratch = static_cast<double *>(p);
    return SPZ_OK;
}

int ising_energy_noalloc(const spz_state_s *s, double hx, double *out)
{
    if (!g_static_scratch) return fail(SPZ_ERR_ARG, "library not initialised");
    const uint64_t M = s->N;
    const uint64_t nb = (M + kRB - 1) / kRB;
    if (nb > kStaticBlocks)
        return fail(SPZ_ERR_ARG, "state too large for spz_ising_energy_noalloc (at most 2^30 "
                                 "amplitudes; use spz_ising_energy)");
    double *part = g_static_scratch;
    SPZ_TRY(ising_level1(s, hx, nullptr, nullptr, part));
    // the pinned result slots were allocated when the library initialised
    return reduce_finish(part, nb, out);
}

// Level-1 pairs of |psi|^2, one per block of 4096 indices, left in
// rt().d_partials (for sampling).
int norm_level1(const spz_state_s *s, uint64_t *nb)
{
    return reduce_level1(s, nullptr, TERM_NORM, 0, 0, 0.0, nb);
}

}  // namespace spz
