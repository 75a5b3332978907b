// spz_reduce.h -- the fixed compensated reduction tree, shared by the kernels
// that sum terms over a state: blocks of 4096 terms in index order, thread t
// of 256 sums terms t, t + 256, ... (16 of them) as a TwoSum pair (S, C), the
// pairs are combined by the halving tree h = 128 .. 1, and the blocks' pairs by
// the same tree once more.
#pragma once

#include "spz_internal.h"

namespace spz {

constexpr int kRT = 256;                          // threads of a reduction block
constexpr int kRE = 16;                           // terms per thread
constexpr uint64_t kRB = (uint64_t)kRT * kRE;     // terms per block

__device__ __forceinline__ void two_sum(double a, double b, double &s, double &e)
{
    double ss = a + b;
    double bb = ss - a;
    double aa = ss - bb;
    e = (a - aa) + (b - bb);
    s = ss;
}

// (s, c) += x
__device__ __forceinline__ void add_term(double &s, double &c, double x)
{
    double ns, er;
    two_sum(s, x, ns, er);
    s = ns;
    c = c + er;
}

__device__ __forceinline__ void tree256(double *S, double *C)
{
    const int tid = threadIdx.x;
    for (int h = kRT / 2; h >= 1; h >>= 1) {
        if (tid < h) {
            double s, e;
            two_sum(S[tid], S[tid + h], s, e);
            C[tid] = (C[tid] + C[tid + h]) + e;
            S[tid] = s;
        }
        __syncthreads();
    }
}

// The second level: thread t of 256 combines pairs t, t + 256, ... of the nb
// block pairs, then the tree.  The result S + C is in thread 0's return value.
// Eight pairs are loaded ahead of the chain that combines them.
__device__ __forceinline__ double reduce_pairs(const double *__restrict__ p, uint64_t nb,
                                               double *S, double *C)
{
    const int tid = threadIdx.x;
    if (nb == 1) return p[0] + p[1];
    double s = 0.0, c = 0.0;
    uint64_t j = tid;
    for (; j + 7 * kRT < nb; j += 8 * kRT) {
        double2 v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = reinterpret_cast<const double2 *>(p)[j + k * kRT];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            double ns, e;
            two_sum(s, v[k].x, ns, e);
            c = (c + v[k].y) + e;
            s = ns;
        }
    }
    for (; j < nb; j += kRT) {
        double ns, e;
        two_sum(s, p[2 * j], ns, e);
        c = (c + p[2 * j + 1]) + e;
        s = ns;
    }
    S[tid] = s;
    C[tid] = c;
    __syncthreads();
    tree256(S, C);
    return S[0] + C[0];
}

// Targets of one pass over the state (spz_expect.hip).
constexpr int kExpectGroup = 8;

// Re <psi|O_t|psi> for every target, O = 'x', 'y' or 'z' (targets in range,
// states of at least 4096 amplitudes).
int expect_many(const spz_state_s *s, char observable, const int32_t *targets, uint64_t n_targets,
                double *out);
// Level-1 pairs of the Ising energy into `part` (one per 4096 amplitudes, or
// one) and, with lr and li, the amplitudes of H psi.
int ising_level1(const spz_state_s *s, double hx, void *lr, void *li, double *part);
// Second level over `nb` pairs into *out (waits for the result), or into a
// pinned slot of rt().h_result without a wait.
int reduce_finish(const double *part, uint64_t nb, double *out);
int reduce_finish_to(const double *part, uint64_t nb, double *pinned);

}  // namespace spz
