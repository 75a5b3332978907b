// spz_ising.h -- H psi and the energy terms of one reduction block, shared by
// the single-circuit and the batched kernels.
#pragma once

#include "spz_reduce.h"

namespace spz {

namespace {

// xr += partner over a qubit held in registers (bit BIT of e).
template <int BIT>
__device__ __forceinline__ void reg_sum(const double *a, const double *b, double *xr, double *xi)
{
#pragma unroll
    for (int e = 0; e < kRE; e++) {
        xr[e] = xr[e] + a[e ^ BIT];
        xi[e] = xi[e] + b[e ^ BIT];
    }
}

// H psi = (sum Z_i Z_{i+1} + hx sum X_i) psi on the block at `base`: the X sum
// of each amplitude runs over the qubits in order; the block's energy terms
// Re conj(psi_j) (H psi)_j go to the pair at `out`.  STORE keeps H psi, and the
// terms then use it as stored.  SMALL: a state of fewer than 4096 amplitudes
// (N), one block whose other amplitudes are zero.  S, C: kRT doubles of LDS.
template <typename T, bool STORE, bool SMALL>
__device__ __forceinline__ void ising_block(const T *__restrict__ re, const T *__restrict__ im,
                                            T *__restrict__ lr, T *__restrict__ li, uint64_t base,
                                            int n, uint64_t N, double hx, double *out, double *S,
                                            double *C)
{
    const uint32_t tid = threadIdx.x;
    double a[kRE], b[kRE], xr[kRE], xi[kRE];
#pragma unroll
    for (int e = 0; e < kRE; e++) {
        const uint64_t j = base + e * kRT + tid;
        a[e] = !SMALL || j < N ? (double)re[j] : 0.0;
        b[e] = !SMALL || j < N ? (double)im[j] : 0.0;
        xr[e] = 0.0;
        xi[e] = 0.0;
    }
    auto far = [&](int q) {
        const uint64_t p0 = (base + tid) ^ (1ull << q);
        // a quarter of the block at a time (half of it measured the same)
#pragma unroll
        for (int h = 0; h < kRE; h += kRE / 4) {
            T x[kRE / 4], y[kRE / 4];
#pragma unroll
            for (int e = 0; e < kRE / 4; e++) {
                const uint64_t p = p0 + (h + e) * kRT;
                x[e] = !SMALL || p < N ? re[p] : (T)0;
                y[e] = !SMALL || p < N ? im[p] : (T)0;
            }
#pragma unroll
            for (int e = 0; e < kRE / 4; e++) {
                xr[h + e] = xr[h + e] + (double)x[e];
                xi[h + e] = xi[h + e] + (double)y[e];
            }
        }
    };
    const int near = SMALL && n < 6 ? n : 6;
#pragma unroll 1
    for (int q = 0; q < near; q++) {
#pragma unroll
        for (int e = 0; e < kRE; e++) {
            xr[e] = xr[e] + __shfl_xor(a[e], 1 << q);
            xi[e] = xi[e] + __shfl_xor(b[e], 1 << q);
        }
    }
    if (!SMALL || n > 6) far(6);
    if (!SMALL || n > 7) far(7);
    if (!SMALL || n > 8) reg_sum<1>(a, b, xr, xi);
    if (!SMALL || n > 9) reg_sum<2>(a, b, xr, xi);
    if (!SMALL || n > 10) reg_sum<4>(a, b, xr, xi);
    if (!SMALL || n > 11) reg_sum<8>(a, b, xr, xi);
    if constexpr (!SMALL) {
#pragma unroll 1
        for (int q = 12; q < n; q++) far(q);
    }
    const uint64_t bonds = (1ull << (n - 1)) - 1;
    double s = 0.0, c = 0.0;
#pragma unroll
    for (int e = 0; e < kRE; e++) {
        const uint64_t j = base + e * kRT + tid;
        // aligned bonds count +1, opposed ones -1: an exact integer
        const int czz = (n - 1) - 2 * __builtin_popcountll((j ^ (j >> 1)) & bonds);
        double vr = (double)czz * a[e] + hx * xr[e];
        double vi = (double)czz * b[e] + hx * xi[e];
        if constexpr (STORE) {
            if (!SMALL || j < N) {
                lr[j] = (T)vr;
                li[j] = (T)vi;
            }
            vr = (double)(T)vr;
            vi = (double)(T)vi;
        }
        if (!SMALL || j < N) add_term(s, c, a[e] * vr + b[e] * vi);
    }
    S[tid] = s;
    C[tid] = c;
    __syncthreads();
    tree256(S, C);
    if (tid == 0) {
        out[0] = S[0];
        out[1] = C[0];
    }
}

}  // namespace

}  // namespace spz
