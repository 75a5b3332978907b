// spz_expect.hip -- expectations of many qubits in one pass, and the Ising
// energy and H psi, for states of at least one reduction block (4096
// amplitudes).
//
// A workgroup owns one block of the reduction tree and holds it in registers:
// thread t has amplitudes t + 256 e, e = 0..15.  The partner j ^ 2^q of an
// amplitude is then in another lane of the wavefront (q < 6), in another
// register of the same thread (8 <= q < 12), or in another wavefront or block
// (loaded).  Every term and every addition is the reduction tree's own, in its
// order, so results are bit-identical to one pass per target.
//
// What bounded it: one pass over the state, one second-level launch, one copy
// and one wait per target (23 qubits: 69 passes of 22-28 us and 70 round
// trips for x, y and z).  Now kExpectGroup targets share a pass, all targets of
// a call share one second-level launch per pass and one wait, and results land
// in pinned memory.  x, y and z of all 23 qubits and the energy: 3.08 -> 0.73
// ms; a pass of 8 targets takes 28 us for z (one state read, then additions)
// and 64 us for x or y.
#include <algorithm>

#include "spz_ising.h"

namespace spz {

namespace {

struct Targets {
    int32_t q[kExpectGroup];
    int32_t count;
};

__device__ __forceinline__ double lane_xor(double x, int mask) { return __shfl_xor(x, mask); }

// Block that workgroup i handles: workgroup i runs on XCD i % 8, and each XCD
// takes a contiguous eighth of the blocks, so that the partner blocks of the
// lower block bits are read by the same XCD at about the same time (its L2).
__device__ __forceinline__ uint64_t xcd_block(uint32_t i, uint64_t nb)
{
    return nb >= 8 ? (uint64_t)(i & 7u) * (nb >> 3) + (i >> 3) : i;
}

// One target's terms: p[e] is the partner of amplitude e.
template <char OBS>
__device__ __forceinline__ double expect_term(bool bit, double a, double b, double c, double d)
{
    if constexpr (OBS == 'x') {
        return a * c + b * d;
    } else {  // (Y psi)_1 = i psi_0, (Y psi)_0 = -i psi_1
        const double vr = bit ? -d : d, vi = bit ? c : -c;
        return a * vr + b * vi;
    }
}

template <char OBS, int BIT>
__device__ __forceinline__ void expect_reg(const double *a, const double *b, double &s, double &c)
{
#pragma unroll
    for (int e = 0; e < kRE; e++)
        add_term(s, c, expect_term<OBS>((e & BIT) != 0, a[e], b[e], a[e ^ BIT], b[e ^ BIT]));
}

// Which of j and its partner over q forms the sum of both: for q = 6 and 7 the one
// with the bit clear; for the block bits above 12 in even blocks that one, in odd
// blocks the other, so that both halves of a state, which run on different XCDs
// (xcd_block), have as much to do (qubit 21 of 22 alone, a whole call: 40 us with
// the clear side only, 30 now; 34 when every amplitude formed its own).
__device__ __forceinline__ bool forms_sum(uint64_t j, int q)
{
    const uint64_t odd = q > 12 ? j >> 12 : 0;
    return (((j >> q) ^ odd) & 1) == 0;
}

// G: the most targets of the launch.  One alone needs 4 KiB of LDS instead of 32,
// so more workgroups share a CU (x on qubit 0, a whole call: 23 qubits FP64 42 ->
// 38 us, 25 qubits FP32 76 -> 59), and blocks whose sum the partner forms end at once.
template <typename T, char OBS, int G>
__global__ void __launch_bounds__(kRT)
k_expect(const T *__restrict__ re, const T *__restrict__ im, uint64_t nb, Targets tg,
         double *__restrict__ partials)
{
    __shared__ double S[G][kRT], C[G][kRT];
    const uint32_t tid = threadIdx.x;
    const uint64_t blk = xcd_block(blockIdx.x, nb), base = blk * kRB;
    if constexpr (G == 1 && OBS != 'z')  // (a block whose only sum its partner forms)
        if (tg.q[0] >= 12 && !forms_sum(base, tg.q[0])) return;
    double a[kRE], b[kRE];
#pragma unroll
    for (int e = 0; e < kRE; e++) {
        a[e] = re[base + e * kRT + tid];
        b[e] = im[base + e * kRT + tid];
    }
    if constexpr (OBS == 'z') {
#pragma unroll
        for (int e = 0; e < kRE; e++) a[e] = a[e] * a[e] + b[e] * b[e];
    }
    const int count = G == 1 ? 1 : tg.count;
    for (int t = 0; t < count; t++) {
        const int q = tg.q[t];
        double s = 0.0, c = 0.0;
        if constexpr (OBS == 'z') {  // a (-a) + b (-b) is exactly -(a a + b b)
            if (q >= 8 && q < 12) {
#pragma unroll
                for (int e = 0; e < kRE; e++)
                    add_term(s, c, ((uint32_t)e >> (q - 8)) & 1u ? -a[e] : a[e]);
            } else {
                const bool bit = (((base + tid) >> q) & 1) != 0;
#pragma unroll
                for (int e = 0; e < kRE; e++) add_term(s, c, bit ? -a[e] : a[e]);
            }
        } else if (q < 6) {
            const bool bit = ((tid >> q) & 1u) != 0;
#pragma unroll
            for (int e = 0; e < kRE; e++) {
                const double x = lane_xor(a[e], 1 << q), y = lane_xor(b[e], 1 << q);
                add_term(s, c, expect_term<OBS>(bit, a[e], b[e], x, y));
            }
        } else if (q == 8) {
            expect_reg<OBS, 1>(a, b, s, c);
        } else if (q == 9) {
            expect_reg<OBS, 2>(a, b, s, c);
        } else if (q == 10) {
            expect_reg<OBS, 4>(a, b, s, c);
        } else if (q == 11) {
            expect_reg<OBS, 8>(a, b, s, c);
        } else {
            // An amplitude and its partner have the same X and Y term, so a
            // thread and its partner thread (q = 6, 7: another wavefront),
            // and a block and its partner block, have the same sums: one
            // side (forms_sum) forms them for both.
            const uint64_t j0 = base + tid;
            if (!forms_sum(j0, q)) continue;
            const uint64_t p0 = j0 ^ (1ull << q);
            const bool bit = ((j0 >> q) & 1) != 0;
            T x[kRE], y[kRE];
#pragma unroll
            for (int e = 0; e < kRE; e++) {
                x[e] = re[p0 + e * kRT];
                y[e] = im[p0 + e * kRT];
            }
#pragma unroll
            for (int e = 0; e < kRE; e++)
                add_term(s, c, expect_term<OBS>(bit, a[e], b[e], x[e], y[e]));
            if (q < 8) {
                S[t][tid | (1u << q)] = s;
                C[t][tid | (1u << q)] = c;
            }
        }
        S[t][tid] = s;
        C[t][tid] = c;
    }
    __syncthreads();
    // the halving tree of every target at once
    for (int lh = 7; lh >= 0; lh--) {
        const uint32_t h = 1u << lh;
        for (uint32_t i = tid; i < (uint32_t)count << lh; i += kRT) {
            const uint32_t t = i >> lh, k = i & (h - 1);
            double ns, e;
            two_sum(S[t][k], S[t][k + h], ns, e);
            C[t][k] = (C[t][k] + C[t][k + h]) + e;
            S[t][k] = ns;
        }
        __syncthreads();
    }
    if ((int)tid < count) {
        const int q = tg.q[tid];
        double *p = partials + 2 * (uint64_t)tid * nb;
        if (OBS == 'z' || q < 12 || forms_sum(base, q)) {
            p[2 * blk] = S[tid][0];
            p[2 * blk + 1] = C[tid][0];
            if (OBS != 'z' && q >= 12) {
                const uint64_t other = blk ^ (1ull << (q - 12));
                p[2 * other] = S[tid][0];
                p[2 * other + 1] = C[tid][0];
            }
        }
    }
}

// Block t finishes target t.
__global__ void __launch_bounds__(kRT)
k_finish(const double *__restrict__ partials, uint64_t nb, double *__restrict__ out)
{
    __shared__ double S[kRT], C[kRT];
    const double r = reduce_pairs(partials + 2 * (uint64_t)blockIdx.x * nb, nb, S, C);
    if (threadIdx.x == 0) out[blockIdx.x] = r;
}

// H psi and the energy's level-1 pairs, one block per workgroup (spz_ising.h).
//
// Bound: the partner loads of the qubits above the block (one state read each,
// from L2 where the partner block is in flight on the same XCD, else from the
// memory-side cache): 11 reads of 134 MB at 23 qubits.  Whole calls for the energy
// and for both with H psi, FP64: 23 qubits 190 and 218 us, 24 qubits 390-402 and 445,
// 28 qubits 8.6 and 9.1 ms.  Two waves per SIMD, whose 256 registers hold the block
// and the partners on their way, not three (168): 211 and 245, 430 and 488 us, 8.8
// and 9.3 ms.  One thread per term: 210 and 346, 403 and 730 us, 9.9 and 13.6 ms.
template <typename T, bool STORE>
__global__ void __launch_bounds__(kRT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_ising(const T *__restrict__ re, const T *__restrict__ im, T *__restrict__ lr,
        T *__restrict__ li, uint64_t nb, int n, double hx, double *__restrict__ partials)
{
    __shared__ double S[kRT], C[kRT];
    const uint64_t blk = xcd_block(blockIdx.x, nb);
    ising_block<T, STORE, false>(re, im, lr, li, blk * kRB, n, 0, hx, partials + 2 * blk, S, C);
}

template <typename T, bool STORE>
__global__ void __launch_bounds__(kRT)
k_ising_small(const T *__restrict__ re, const T *__restrict__ im, T *__restrict__ lr,
              T *__restrict__ li, uint64_t N, int n, double hx, double *__restrict__ partials)
{
    __shared__ double S[kRT], C[kRT];
    ising_block<T, STORE, true>(re, im, lr, li, 0, n, N, hx, partials, S, C);
}

template <typename T>
void launch_expect(const spz_state_s *s, char obs, uint64_t nb, const Targets &tg, double *part)
{
    const T *re = (const T *)s->re, *im = (const T *)s->im;
    const dim3 g((unsigned)nb), b(kRT);
    hipStream_t st = rt().stream;
#define SPZ_EX(OBS)                                                                          \
    do {                                                                                     \
        if (tg.count == 1)                                                                     \
            hipLaunchKernelGGL((k_expect<T, OBS, 1>), g, b, 0, st, re, im, nb, tg, part);          \
        else                                                                                 \
            hipLaunchKernelGGL((k_expect<T, OBS, kExpectGroup>), g, b, 0, st, re, im, nb, tg,       \
                               part);                                                        \
    } while (0)
    if (obs == 'x') SPZ_EX('x');
    else if (obs == 'y') SPZ_EX('y');
    else SPZ_EX('z');
#undef SPZ_EX
}

}  // namespace

int reduce_finish_to(const double *part, uint64_t nb, double *pinned)
{
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(kRT), 0, rt().stream, part, nb, pinned);
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

int reduce_finish(const double *part, uint64_t nb, double *out)
{
    SPZ_TRY(reduce_finish_to(part, nb, rt().h_result));
    SPZ_HIP(hipStreamSynchronize(rt().stream));
    *out = rt().h_result[0];
    return SPZ_OK;
}

int expect_many(const spz_state_s *s, char observable, const int32_t *targets, uint64_t n_targets,
                double *out)
{
    const uint64_t nb = s->N / kRB;
    // targets per pass: all kExpectGroup while their pairs take at most 64 MiB
    const uint64_t room = (64ull << 20) / (16 * nb);
    const int group = (int)std::max<uint64_t>(1, std::min<uint64_t>(kExpectGroup, room));
    SPZ_TRY(ensure_partials(nb * std::min<uint64_t>(group, n_targets)));
    const double bytes = (double)s->N * (s->prec == SPZ_F64 ? 16.0 : 8.0);
    for (uint64_t r = 0; r < n_targets; r += kResults) {
        const uint64_t m = std::min<uint64_t>(kResults, n_targets - r);
        for (uint64_t t = 0; t < m; t += group) {
            Targets tg;
            tg.count = (int32_t)std::min<uint64_t>(group, m - t);
            for (int k = 0; k < tg.count; k++) tg.q[k] = targets[r + t + k];
            LaunchTimer tm(SPZ_K_REDUCE, bytes);
            if (s->prec == SPZ_F64) launch_expect<double>(s, observable, nb, tg, rt().d_partials);
            else launch_expect<float>(s, observable, nb, tg, rt().d_partials);
            hipLaunchKernelGGL(k_finish, dim3(tg.count), dim3(kRT), 0, rt().stream,
                               rt().d_partials, nb, rt().h_result + t);
            SPZ_HIP(hipGetLastError());
        }
        SPZ_HIP(hipStreamSynchronize(rt().stream));
        for (uint64_t t = 0; t < m; t++) out[r + t] = rt().h_result[t];
    }
    return SPZ_OK;
}

int ising_level1(const spz_state_s *s, double hx, void *lr, void *li, double *part)
{
    const uint64_t nb = s->N / kRB;
    hipStream_t st = rt().stream;
#define SPZ_IS(T, ST)                                                                              \
    do {                                                                                           \
        if (nb)                                                                                    \
            hipLaunchKernelGGL((k_ising<T, ST>), dim3((unsigned)nb), dim3(kRT), 0, st,               \
                               (const T *)s->re, (const T *)s->im, (T *)lr, (T *)li, nb, s->n, hx,    \
                               part);                                                              \
        else                                                                                       \
            hipLaunchKernelGGL((k_ising_small<T, ST>), dim3(1), dim3(kRT), 0, st,                    \
                               (const T *)s->re, (const T *)s->im, (T *)lr, (T *)li, s->N, s->n, hx,  \
                               part);                                                              \
    } while (0)
    if (s->prec == SPZ_F64) {
        if (lr) SPZ_IS(double, true);
        else SPZ_IS(double, false);
    } else {
        if (lr) SPZ_IS(float, true);
        else SPZ_IS(float, false);
    }
#undef SPZ_IS
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

}  // namespace spz
