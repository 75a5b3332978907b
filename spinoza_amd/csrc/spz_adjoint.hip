// spz_adjoint.hip -- adjoint differentiation of E = <psi|H|psi> (no counterpart
// in the reference; built beside the gate path).
//
//   psi_k = U_k ... U_1 psi_0,  lambda_k = U_{k+1}^dag ... U_L^dag H psi_L.
//   For U_k = exp(-i theta G / 2) (RX, RY, RZ with G = X, Y, Z; controls
//   project onto the control subspace), dE/dtheta_k = Im <lambda_k| G~ |psi_k>,
//   and for P(theta) = diag(1, e^{i theta}), dE/dtheta_k = -2 Im <lambda_k|Pi_1~|psi_k>
//   (G~, Pi_1~: the operator restricted to amplitudes whose controls are met).
//
// Reverse sweep.  Both states are undone together in tile sweeps
// (spz_adj_tile.hip; states of at most 12 qubits are one tile and take one
// launch, spz_chip.hip); FP32 states in groups of gates (spz_adj_group.hip).
#include <math.h>
#include <string.h>

#include <algorithm>
#include <memory>
#include <mutex>
#include <vector>

#include "spz_adj_tile.h"
#include "spz_chip.h"
#include "spz_reduce.h"
#include "spz_tile.h"

namespace spz {

int execute_ops(spz_state_s *s, const spz_op *ops, uint64_t n_ops, spz_tracker *trk,
                const spz_exec_opts *opts, uint8_t *outcomes);

static bool has_param(int kind)
{
    return kind == SPZ_RX || kind == SPZ_RY || kind == SPZ_RZ || kind == SPZ_P;
}

// The inverse of one op (gates.rs:78-92): rotations and P negate theta,
// U(theta, phi, lambda)^-1 = U(-theta, -lambda, -phi), the rest are self-inverse.
spz_op inverse_op(const spz_op &o)
{
    spz_op r = o;
    if (has_param(o.kind)) r.theta = -o.theta;
    if (o.kind == SPZ_U) {
        r.theta = -o.theta;
        r.phi = -o.lambda;
        r.lambda = -o.phi;
    }
    return r;
}

namespace {

constexpr int kT = 256;

// max |a - b| over the state, into out[0]: a grid-stride maximum per thread,
// a wavefront shuffle and an LDS step per block, then one integer atomic max
// per block on the (non-negative) double bit patterns.
template <typename T>
__global__ void __launch_bounds__(kT)
k_maxdiff(const T *__restrict__ ar, const T *__restrict__ ai, const T *__restrict__ br,
          const T *__restrict__ bi, uint64_t N, unsigned long long *__restrict__ out)
{
    __shared__ double W[kT / 64];
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    double m = 0.0;
    for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < N; j += stride)
        m = fmax(m, fmax(fabs((double)ar[j] - (double)br[j]), fabs((double)ai[j] - (double)bi[j])));
    for (int off = 32; off >= 1; off >>= 1) m = fmax(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) W[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kT / 64; w++) m = fmax(m, W[w]);
        atomicMax(out, (unsigned long long)__double_as_longlong(m));
    }
}

// Blocks of the drift check: enough to fill the GPU, each striding over the state.
unsigned maxdiff_grid(uint64_t N)
{
    const uint64_t cap = (uint64_t)std::max(rt().cu_count, 1) * 8;
    return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(cap, (N + kT - 1) / kT));
}

// Owns a scratch state; not copyable, so it can live in a vector only
// behind a unique_ptr (a copy would free the state twice).
struct OwnedState {
    spz_state_s *s = nullptr;
    OwnedState() = default;
    OwnedState(const OwnedState &) = delete;
    OwnedState &operator=(const OwnedState &) = delete;
    ~OwnedState() { if (s) spz_state_destroy(s); }
};

// Checkpoint states kept between calls of one shape (allocating and freeing
// them costs a device synchronisation each): given back when a call has
// another shape, and at the end of a call that needs more than kCkptKeep bytes.
constexpr size_t kCkptKeep = (size_t)4 << 30;

struct CkptPool {
    std::vector<std::unique_ptr<OwnedState>> st;
    size_t used = 0;  // by the call that is running

    // The i-th checkpoint of a call (i = 0, 1, ...).
    int get(size_t i, const spz_state_s *like, spz_state_s **out)
    {
        used = i;
        if (!st.empty() && (st[0]->s->n != like->n || st[0]->s->prec != like->prec)) st.clear();
        while (st.size() <= i) {
            auto o = std::make_unique<OwnedState>();
            SPZ_TRY(spz_state_create(like->n, like->prec, &o->s));
            st.push_back(std::move(o));
        }
        *out = st[i]->s;
        used = i + 1;
        return SPZ_OK;
    }

    bool drop_unused()
    {
        if (st.size() <= used) return false;
        st.resize(used);
        return true;
    }

    void trim()
    {
        used = 0;
        if (st.empty()) return;
        const size_t each = (size_t)st[0]->s->N * (st[0]->s->prec == SPZ_F64 ? 16 : 8);
        if (each * st.size() > kCkptKeep) st.clear();
    }
};

// Scratch kept between calls (hipFree synchronises the device, and small
// circuits would otherwise spend most of their time allocating): four
// grow-only arrays that back the two working states (psi copy and lambda,
// viewed with the current shape) and grow-only device buffers.  One lock
// serialises the adjoint calls that share it.
struct AdjScratch {
    std::mutex mu;
    void *arr[4] = {nullptr, nullptr, nullptr, nullptr};  // work re/im, lambda re/im
    size_t arr_cap = 0;
    spz_state_s work, lam;  // views into arr
    void *grad = nullptr, *part = nullptr, *dmax = nullptr;
    size_t grad_cap = 0, part_cap = 0;
    CkptPool ckpts;
    bool in_use = false;  // a call is running

    // Free what no call uses (a running one: checkpoint states beyond its own).
    bool give_back()
    {
        bool any = ckpts.drop_unused();
        if (in_use) return any;
        for (void *&a : arr) drop(&a, any);
        drop(&grad, any);
        drop(&part, any);
        arr_cap = grad_cap = part_cap = 0;
        return any;
    }

    static void drop(void **p, bool &any)
    {
        if (!*p) return;
        (void)hipFree(*p);
        *p = nullptr;
        any = true;
    }

    int reserve_states(int n, int prec)
    {
        const size_t bytes = ((size_t)1 << n) * (prec == SPZ_F64 ? 8 : 4);
        if (bytes > arr_cap) {
            for (void *&a : arr)
                if (a) {
                    SPZ_HIP(hipFree(a));
                    a = nullptr;
                }
            arr_cap = 0;
            for (void *&a : arr)
                if (device_alloc(&a, bytes) != hipSuccess) {
                    for (void *&b : arr)
                        if (b) {
                            (void)hipFree(b);
                            b = nullptr;
                        }
                    return fail(SPZ_ERR_OOM, "adjoint scratch allocation failed");
                }
            arr_cap = bytes;
        }
        return SPZ_OK;
    }

    int states_like(const spz_state_s *s)
    {
        SPZ_TRY(reserve_states(s->n, s->prec));
        work.n = lam.n = s->n;
        work.prec = lam.prec = s->prec;
        work.N = lam.N = s->N;
        work.re = arr[0];
        work.im = arr[1];
        lam.re = arr[2];
        lam.im = arr[3];
        return SPZ_OK;
    }

    static int grow(void **p, size_t *cap, size_t bytes)
    {
        if (bytes <= *cap) return SPZ_OK;
        if (*p) SPZ_HIP(hipFree(*p));
        *p = nullptr;
        *cap = 0;
        if (device_alloc(p, bytes) != hipSuccess)
            return fail(SPZ_ERR_OOM, "adjoint scratch allocation failed");
        *cap = bytes;
        return SPZ_OK;
    }

    int buffers(size_t grad_bytes, size_t part_bytes)
    {
        SPZ_TRY(grow(&grad, &grad_cap, grad_bytes));
        SPZ_TRY(grow(&part, &part_cap, part_bytes));
        if (!dmax) {
            if (device_alloc(&dmax, sizeof(unsigned long long)) != hipSuccess)
                return fail(SPZ_ERR_OOM, "adjoint scratch allocation failed");
        }
        return SPZ_OK;
    }
};

size_t grad_bytes(uint64_t n_ops) { return std::max<uint64_t>(n_ops, 1) * sizeof(double); }

size_t part_bytes(const spz_state_s *s, uint64_t n_ops)
{
    const uint64_t N = s->N;
    if (s->prec == SPZ_F32) return adj_group_part_bytes(N);
    if (N > (1ull << kAdjK)) return adj_part_bytes(N);
    return std::max<uint64_t>(n_ops, 1) * 2 * kChipRows * sizeof(double);
}

AdjScratch &adj_scratch()
{
    static AdjScratch *a = new AdjScratch();  // lives until the process ends
    return *a;
}

}  // namespace

bool adjoint_give_back() { return adj_scratch().give_back(); }

// The ops a differentiated circuit may hold: unitary single-target gates H..U
// (and SWAP where allowed) with 1- and 0-controls; every qubit in range, the
// target (SWAP: both qubits) not a control, no qubit both a 1- and a
// 0-control, and at most max_controls controls.  The single-circuit and the
// batched paths share this check, so a circuit is accepted or rejected the
// same way whichever path runs it.
int validate_adjoint_op(int n, const spz_op &o, uint64_t idx, bool allow_swap, int max_controls)
{
    const bool swap = o.kind == SPZ_SWAP;
    if (o.kind < SPZ_H || o.kind > SPZ_SWAP || (swap && !allow_swap))
        return fail(SPZ_ERR_GATE, "adjoint: op " + std::to_string(idx) + " is not a unitary " +
                                      (allow_swap ? "single-target gate or SWAP"
                                                  : "single-target gate"));
    const uint64_t all = n >= 64 ? ~0ull : (1ull << n) - 1;
    const uint64_t tb = o.target >= 0 && o.target < n ? 1ull << o.target : 0;
    const uint64_t t1b = o.t1 >= 0 && o.t1 < n ? 1ull << o.t1 : 0;
    if (!tb || (swap && (!t1b || t1b == tb)) || ((o.ones | o.zeros) & ~all) ||
        (o.ones & o.zeros) || ((o.ones | o.zeros) & (tb | (swap ? t1b : 0))))
        return fail(SPZ_ERR_QUBIT, "adjoint: op " + std::to_string(idx) +
                                       " has a qubit out of range or used twice");
    if (__builtin_popcountll(o.ones | o.zeros) > max_controls)
        return fail(SPZ_ERR_GATE, "adjoint: op " + std::to_string(idx) + " has more than " +
                                      std::to_string(max_controls) + " controls");
    return SPZ_OK;
}

int adjoint_grad(spz_state_s *s, const spz_op *ops, uint64_t n_ops, double hx, int ckpt_every,
                 double *grad, double *energy, double *drift)
{
    SPZ_TRY(check_state(s));
    if (n_ops && (!ops || !grad)) return fail(SPZ_ERR_ARG, "null ops/grad");
    for (uint64_t i = 0; i < n_ops; i++) SPZ_TRY(validate_adjoint_op(s->n, ops[i], i, true, 64));
    AdjScratch &sc = adj_scratch();
    std::lock_guard<std::mutex> lock(sc.mu);
    struct Running {
        AdjScratch &s;
        explicit Running(AdjScratch &a) : s(a) { s.in_use = true; }
        ~Running()
        {
            s.ckpts.trim();
            s.in_use = false;
        }
    } running(sc);
    // ---- forward pass with checkpoints ---------------------------------------
    std::vector<spz_state_s *> ckpts;
    std::vector<uint64_t> ckpt_at;  // checkpoint j holds psi after op ckpt_at[j]
    spz_exec_opts eo;
    memset(&eo, 0, sizeof eo);
    eo.mode = SPZ_EXEC_AUTO;
    const bool f32 = s->prec == SPZ_F32;
    if (f32 && s->n <= kChipK) {  // FP32: the rounding points stay (spz_adj_group.hip)
        if (s->n <= 10) eo.mode = SPZ_EXEC_PLAIN;
        else eo.tile_qubits = s->n - 1;
    }
    const uint64_t step = ckpt_every > 0 ? (uint64_t)ckpt_every : std::max<uint64_t>(n_ops, 1);
    for (uint64_t done = 0; done < n_ops;) {
        const uint64_t len = std::min<uint64_t>(step, n_ops - done);
        SPZ_TRY(execute_ops(s, ops + done, len, nullptr, &eo, nullptr));
        done += len;
        if (done < n_ops) {
            spz_state_s *c = nullptr;
            SPZ_TRY(sc.ckpts.get(ckpts.size(), s, &c));
            SPZ_TRY(spz_state_copy(c, s));
            ckpts.push_back(c);
            ckpt_at.push_back(done - 1);
        }
    }
    // ---- lambda = H psi, energy (read with the gradients at the end) ----------
    SPZ_TRY(sc.states_like(s));
    SPZ_TRY(sc.buffers(grad_bytes(n_ops), part_bytes(s, n_ops)));
    spz_state_s *const wk = &sc.work, *const lm = &sc.lam;  // psi copy, lambda
    const double amp = s->prec == SPZ_F64 ? 16.0 : 8.0;
    double *const e_out = rt().h_result + (kResults - 1);
    const uint64_t nb = std::max<uint64_t>(s->N / kRB, 1);
    SPZ_TRY(ensure_partials(nb));
    {  // H psi and the energy's first level in one pass
        LaunchTimer tm(SPZ_K_ADJOINT, 2.0 * (double)s->N * amp);
        SPZ_TRY(ising_level1(s, hx, lm->re, lm->im, rt().d_partials));
    }
    SPZ_TRY(reduce_finish_to(rt().d_partials, nb, e_out));
    // ---- reverse sweep -------------------------------------------------------
    SPZ_HIP(hipMemsetAsync(sc.grad, 0, grad_bytes(n_ops), rt().stream));
    SPZ_HIP(hipMemsetAsync(sc.dmax, 0, sizeof(unsigned long long), rt().stream));
    double *gdev = (double *)sc.grad, *part = (double *)sc.part;
    const spz_state_s *src = s;  // holds the current psi (wk once anything was undone)
    for (size_t seg = ckpts.size() + 1; seg-- > 0 && n_ops;) {
        const uint64_t lo = seg ? ckpt_at[seg - 1] + 1 : 0;
        const uint64_t hi = seg < ckpts.size() ? ckpt_at[seg] + 1 : n_ops;
        if (f32) {
            SPZ_TRY(spz_state_copy(wk, const_cast<spz_state_s *>(src)));
            SPZ_TRY(adjoint_undo_groups(wk, lm, ops, lo, hi, part, gdev));
        } else {
            SPZ_TRY(adjoint_undo(src, wk, lm, ops, lo, hi, part, gdev));
        }
        if (!seg) break;
        // wk holds the uncomputed psi: compare it with the checkpoint, go on from that
        const spz_state_s *ck = ckpts[seg - 1];
        if (s->prec == SPZ_F64)
            hipLaunchKernelGGL((k_maxdiff<double>), dim3(maxdiff_grid(s->N)), dim3(kT), 0,
                               rt().stream, (const double *)wk->re, (const double *)wk->im,
                               (const double *)ck->re, (const double *)ck->im, s->N,
                               (unsigned long long *)sc.dmax);
        else
            hipLaunchKernelGGL((k_maxdiff<float>), dim3(maxdiff_grid(s->N)), dim3(kT), 0,
                               rt().stream, (const float *)wk->re, (const float *)wk->im,
                               (const float *)ck->re, (const float *)ck->im, s->N,
                               (unsigned long long *)sc.dmax);
        SPZ_HIP(hipGetLastError());
        src = ck;
    }
    if (n_ops)
        SPZ_HIP(hipMemcpyAsync(grad, gdev, n_ops * sizeof(double), hipMemcpyDeviceToHost,
                               rt().stream));
    unsigned long long mx = 0;
    SPZ_HIP(hipMemcpyAsync(&mx, sc.dmax, sizeof mx, hipMemcpyDeviceToHost, rt().stream));
    SPZ_HIP(hipStreamSynchronize(rt().stream));
    if (energy) *energy = *e_out;
    if (drift) {
        double d;
        memcpy(&d, &mx, sizeof d);
        *drift = d;
    }
    return SPZ_OK;
}

}  // namespace spz

extern "C" int spz_adjoint_grad(spz_state s, const spz_op *ops, uint64_t n_ops, double hx,
                                int ckpt_every, double *grad, double *energy, double *drift)
{
    SPZ_API_LOCK;
    return spz::adjoint_grad(s, ops, n_ops, hx, ckpt_every, grad, energy, drift);
}
