// spz_sample.hip -- inverse-CDF sampling of |psi|^2 (replaces
// reservoir_sampling, core.rs:125-129).
//
// The rule (the oracle restates it): W_b is the compensated partial of block
// b of 4096 indices, P the running sums of W in block order; a uniform u asks
// for x = u P_nb, picks the first block with P_{b+1} > x and then the first j
// of it with P_b + w_0 + ... + w_j > x, all sums in index order.  Both sums are
// chains of dependent additions that fix the rounding, so they cannot be
// reassociated; what is parallel is everything around them.
//
// What bounded it: one thread per uniform walked its block alone, 4096
// dependent loads and additions at memory latency (859 us for 4096 samples of
// 20 qubits, 734 us for 1000 of 17), with the block sums carried to the host
// and back and six allocations around it.  Here the samples are counted into
// their blocks (atomic ranks, one scan, one scatter) and for every 1024 samples
// of a block a workgroup forms the block's 4096 running sums in LDS (loads
// and squares by the whole workgroup, the chain by one lane at the FP64
// addition latency) and answers them by bisection: a running
// sum of non-negative terms never decreases, so the first one above x is
// where the walk stopped.  (A NaN or infinite weight makes the total NaN, no
// sum compares above x, and every sample falls to the last index of positive
// weight, as in the walk.)
#include <string.h>

#include <algorithm>

#include "spz_internal.h"

namespace spz {

namespace {

constexpr int kT = 256;
constexpr uint32_t kBlock = 4096;      // indices per block of the sampling rule
constexpr uint32_t kPiece = 1u << 20;  // uniforms per round (bounds the scratch)
constexpr uint32_t kPer = 1024;        // samples a workgroup picks (4 per thread)
constexpr uint32_t kFew = 64;          // blocks counted in LDS first
constexpr uint64_t kHostBlocks = 1u << 12;  // blocks whose sums the host forms
constexpr uint64_t kHostPiece = 1u << 20;   // ... so many at a time
constexpr uint32_t kDirect = 1u << 14; // samples a call reads and writes in pinned memory

struct SampleMeta {
    int64_t lastnz;    // last block with a positive weight (-1: none)
    double total;      // P_nb
    uint32_t nslots;   // workgroups' worth of samples of this round
    uint32_t pad;
};

struct Slot {
    uint32_t block, start, count;
};

// The running sums of `steps` groups of kStep LDS values, by one lane: ck[i] is
// the sum up to and with group i.  One dependent addition per value, the reads
// one group ahead of it.  Only every kStep-th sum is stored (a store per value
// would double the LDS traffic and make that, not the addition, the pace:
// 12.7 against 5 ns per value); whoever needs one in between adds at most
// kStep terms to the sum before, the same additions in the same order.
constexpr uint32_t kStep = 16;

__device__ __forceinline__ double chain(const double *v, uint32_t steps, double acc, double *ck)
{
    double t[kStep], nx[kStep];
#pragma unroll
    for (uint32_t k = 0; k < kStep; k++) t[k] = v[k];
    for (uint32_t i = 0; i < steps; i++) {
        const uint32_t n = i + 1 < steps ? (i + 1) * kStep : 0;
#pragma unroll
        for (uint32_t k = 0; k < kStep; k++) nx[k] = v[n + k];
#pragma unroll
        for (uint32_t k = 0; k < kStep; k++) acc = acc + t[k];
        ck[i] = acc;
#pragma unroll
        for (uint32_t k = 0; k < kStep; k++) t[k] = nx[k];
    }
    return acc;
}

// P[0..nb] from the level-1 pairs, the total and the last positive block; also
// clears the blocks' sample counts.  One workgroup: the chain over blocks is
// serial, the next chunk's pairs are loaded while it runs.
constexpr int kPT = 1024;
constexpr uint32_t kPC = 2048;  // blocks per chunk

__global__ void __launch_bounds__(kPT)
k_block_prefix(const double *__restrict__ pairs, uint64_t nb, double *__restrict__ P,
               uint32_t *__restrict__ counts, SampleMeta *__restrict__ meta,
               SampleMeta *__restrict__ host_meta)
{
    __shared__ __align__(16) double v[kPC];
    __shared__ double ck[kPC / kStep], carry;
    __shared__ long long last;
    const uint32_t tid = threadIdx.x;
    if (tid == 0) {
        carry = 0.0;
        last = -1;
        P[0] = 0.0;
    }
    double w[kPC / kPT];
    long long mine = -1;
    auto fetch = [&](uint64_t base) {
#pragma unroll
        for (uint32_t e = 0; e < kPC / kPT; e++) {
            const uint64_t b = base + e * kPT + tid;
            w[e] = b < nb ? pairs[2 * b] + pairs[2 * b + 1] : 0.0;
            if (b < nb) counts[b] = 0u;
        }
    };
    fetch(0);
    for (uint64_t base = 0; base < nb; base += kPC) {
        const uint32_t cnt = (uint32_t)(nb - base < kPC ? nb - base : kPC);
#pragma unroll
        for (uint32_t e = 0; e < kPC / kPT; e++) {
            v[e * kPT + tid] = w[e];
            if (w[e] > 0.0) mine = (long long)(base + e * kPT + tid);
        }
        if (base + kPC < nb) fetch(base + kPC);
        __syncthreads();
        const double before = carry;
        __syncthreads();
        if (tid == 0) carry = chain(v, (cnt + kStep - 1) / kStep, before, ck);
        __syncthreads();
#pragma unroll
        for (uint32_t e = 0; e < kPC / kPT; e++) {
            const uint32_t i = e * kPT + tid;
            if (i < cnt) {
                const uint32_t g = i / kStep;
                double acc = g ? ck[g - 1] : before;
                for (uint32_t j = g * kStep; j <= i; j++) acc = acc + v[j];
                P[base + i + 1] = acc;
            }
        }
        __syncthreads();
    }
    if (mine >= 0) atomicMax(&last, mine);
    __syncthreads();
    if (tid == 0) {
        meta->lastnz = last;
        if (host_meta) host_meta->lastnz = last;
        meta->total = carry;
        meta->nslots = 0;
    }
}

// The same for many blocks, whose sums the host forms (block_prefix_on_host): their
// way to pinned memory and back, and the start of a round.
__global__ void __launch_bounds__(kT)
k_block_sums(const double *__restrict__ pairs, uint64_t cnt, double *__restrict__ host_v)
{
    const uint64_t b = (uint64_t)blockIdx.x * kT + threadIdx.x;
    if (b < cnt) host_v[b] = pairs[2 * b] + pairs[2 * b + 1];
}

__global__ void __launch_bounds__(kT)
k_take_sums(const double *__restrict__ host_v, uint64_t cnt, double *__restrict__ P)
{
    const uint64_t b = (uint64_t)blockIdx.x * kT + threadIdx.x;
    if (b < cnt) P[b] = host_v[b];
}

__global__ void __launch_bounds__(kT)
k_sample_begin(uint32_t *__restrict__ counts, uint64_t nb, double *__restrict__ P,
               SampleMeta *__restrict__ meta, SampleMeta *__restrict__ host_meta, SampleMeta m)
{
    const uint64_t b = (uint64_t)blockIdx.x * kT + threadIdx.x;
    if (b < nb) counts[b] = 0u;
    if (b == 0) {
        P[nb] = m.total;
        *meta = m;
        if (host_meta) host_meta->lastnz = m.lastnz;
    }
}

// The block of every uniform, and its rank among the block's samples.  With few
// blocks (kFew) a workgroup counts in LDS and takes its places at once: the
// samples of a state of one block would queue at one address (10000 samples of
// 4 qubits: 243 us a call with an atomic each and one workgroup to pick them, 78
// so and in slots of kPer; 14 qubits 173 -> 108 us).
__global__ void __launch_bounds__(kT)
k_sample_block(const double *__restrict__ P, uint64_t nb, const SampleMeta *__restrict__ meta,
               const double *__restrict__ U, uint32_t k, uint32_t *__restrict__ counts,
               uint32_t *__restrict__ blk, uint32_t *__restrict__ rank)
{
    __shared__ uint32_t mine[kFew], first[kFew];
    const uint32_t s = blockIdx.x * kT + threadIdx.x;
    if (meta->lastnz < 0) return;  // uniform over the grid
    const bool few = nb <= kFew;
    if (few) {
        if (threadIdx.x < kFew) mine[threadIdx.x] = 0u;
        __syncthreads();
    }
    const double x = s < k ? U[s] * meta->total : 0.0;
    uint64_t lo = 0, hi = nb;
    while (lo < hi) {
        const uint64_t mid = lo + (hi - lo) / 2;
        if (P[mid + 1] > x) hi = mid;
        else lo = mid + 1;
    }
    const uint32_t b = (uint32_t)(lo < nb ? lo : (uint64_t)meta->lastnz);
    if (few) {
        const uint32_t r = s < k ? atomicAdd(&mine[b], 1u) : 0u;
        __syncthreads();
        if (threadIdx.x < nb && mine[threadIdx.x])
            first[threadIdx.x] = atomicAdd(&counts[threadIdx.x], mine[threadIdx.x]);
        __syncthreads();
        if (s < k) {
            blk[s] = b;
            rank[s] = first[b] + r;
        }
        return;
    }
    if (s >= k) return;
    blk[s] = b;
    rank[s] = atomicAdd(&counts[b], 1u);
}

// Exclusive scan of the counts (in place: counts[b] becomes the block's first
// position) and the list of the blocks' samples, at most kPer to a slot.  One
// workgroup, `kScan` blocks to a thread at a time: one, and eight where there are
// more blocks than threads (one there took 0.1 ms more for 2^18 blocks).
template <int kScan>
__global__ void __launch_bounds__(kPT)
k_sample_scan(uint32_t *__restrict__ counts, uint64_t nb, Slot *__restrict__ slots,
              SampleMeta *__restrict__ meta)
{
    __shared__ uint32_t ws[kPT / 64], wz[kPT / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t base_s = 0, base_z = 0;
    for (uint64_t b0 = 0; b0 < nb; b0 += kPT * kScan) {
        const uint64_t b = b0 + (uint64_t)tid * kScan;
        uint32_t c[kScan], cs = 0, cz = 0;
#pragma unroll
        for (int i = 0; i < kScan; i++) c[i] = b + i < nb ? counts[b + i] : 0u;
#pragma unroll
        for (int i = 0; i < kScan; i++) {
            cs += c[i];
            cz += (c[i] + kPer - 1) / kPer;
        }
        uint32_t s = cs, z = cz;  // inclusive scans over the wavefront
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t us = __shfl_up(s, d), uz = __shfl_up(z, d);
            if (lane >= (uint32_t)d) {
                s += us;
                z += uz;
            }
        }
        if (lane == 63) {
            ws[wave] = s;
            wz[wave] = z;
        }
        __syncthreads();
        uint32_t os = base_s + s - cs, oz = base_z + z - cz;
        for (uint32_t w = 0; w < kPT / 64; w++) {
            if (w < wave) {
                os += ws[w];
                oz += wz[w];
            }
            base_s += ws[w];
            base_z += wz[w];
        }
#pragma unroll
        for (int i = 0; i < kScan; i++) {
            if (b + i < nb) counts[b + i] = os;
            for (uint32_t at = 0; at < c[i]; at += kPer)
                slots[oz++] = Slot{(uint32_t)(b + i), os + at, min(c[i] - at, kPer)};
            os += c[i];
        }
        __syncthreads();
    }
    if (tid == 0) meta->nslots = base_z;
}

__global__ void __launch_bounds__(kT)
k_sample_order(const uint32_t *__restrict__ starts, const SampleMeta *__restrict__ meta,
               const uint32_t *__restrict__ blk, const uint32_t *__restrict__ rank, uint32_t k,
               uint32_t *__restrict__ order)
{
    const uint32_t s = blockIdx.x * kT + threadIdx.x;
    if (s < k && meta->lastnz >= 0) order[starts[blk[s]] + rank[s]] = s;
}

// A workgroup's samples of one block, `before` the sum of the blocks before it; a
// sample bisects the group sums, then walks its group.  at(i): the i-th sample.
template <typename T, typename At>
__device__ __forceinline__ void
pick_samples(const T *__restrict__ re, const T *__restrict__ im, uint64_t N, uint32_t block,
             double before, double total, uint32_t count, At at, const double *__restrict__ U,
             uint64_t *__restrict__ out)
{
    __shared__ __align__(16) double v[kBlock];
    __shared__ double ck[kBlock / kStep];  // sum up to and with step i
    __shared__ int last;
    const uint32_t tid = threadIdx.x;
    const uint64_t j0 = (uint64_t)block * kBlock;
    const uint32_t cnt = (uint32_t)(N - j0 < kBlock ? N - j0 : kBlock);
    const uint32_t steps = (cnt + kStep - 1) / kStep;
    if (tid == 0) last = -1;
    int mine = -1;
    constexpr uint32_t E = kBlock / kT;
    if (cnt == kBlock) {  // all loads in flight together
        T a[E], b[E];
#pragma unroll
        for (uint32_t e = 0; e < E; e++) {
            a[e] = re[j0 + e * kT + tid];
            b[e] = im[j0 + e * kT + tid];
        }
#pragma unroll
        for (uint32_t e = 0; e < E; e++) {
            const double x = a[e], y = b[e];
            const double w = x * x + y * y;
            v[e * kT + tid] = w;
            if (w > 0.0) mine = (int)(e * kT + tid);
        }
    } else {  // a state smaller than a block: its last step is padded with zeros
        for (uint32_t i = tid; i < steps * kStep; i += kT) {
            double w = 0.0;
            if (i < cnt) {
                const double x = re[j0 + i], y = im[j0 + i];
                w = x * x + y * y;
                if (w > 0.0) mine = (int)i;
            }
            v[i] = w;
        }
    }
    __syncthreads();
    if (mine >= 0) atomicMax(&last, mine);
    if (tid == 0) chain(v, steps, before, ck);
    __syncthreads();
    for (uint32_t i = tid; i < count; i += kT) {
        const uint32_t s = at(i);
        const double x = U[s] * total;
        uint32_t lo = 0, hi = steps;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (ck[mid] > x) hi = mid;
            else lo = mid + 1;
        }
        uint64_t pick;
        if (lo < steps) {
            double acc = lo ? ck[lo - 1] : before;
            uint32_t j = lo * kStep;
            acc = acc + v[j];
            while (!(acc > x)) acc = acc + v[++j];  // (ends at ck[lo] > x at the latest)
            pick = j0 + j;
        } else {
            pick = last >= 0 ? j0 + (uint64_t)last : ~0ull;
        }
        out[s] = pick;
    }
}

// One workgroup per slot.
template <typename T>
__global__ void __launch_bounds__(kT)
k_sample_pick(const T *__restrict__ re, const T *__restrict__ im, uint64_t N,
              const double *__restrict__ P, const SampleMeta *__restrict__ meta,
              const Slot *__restrict__ slots, const uint32_t *__restrict__ order,
              const double *__restrict__ U, uint64_t *__restrict__ out)
{
    if (blockIdx.x >= meta->nslots) return;  // uniform over the workgroup
    const Slot sl = slots[blockIdx.x];
    pick_samples(re, im, N, sl.block, P[sl.block], meta->total, sl.count,
                 [&](uint32_t i) { return order[sl.start + i]; }, U, out);
}

// States of one block (12 qubits and fewer): every sample is of block 0, so there
// is nothing to count or order, and uniforms and results stay in pinned memory.
// One launch instead of five and two copies: a call for 1 to 1000 samples of 9
// qubits 61 -> 28-36 us, 10000 samples 84 -> 40.
template <typename T>
__global__ void __launch_bounds__(kT)
k_sample_one(const T *__restrict__ re, const T *__restrict__ im, uint64_t N,
             const double *__restrict__ pairs, const double *__restrict__ U, uint32_t k,
             SampleMeta *__restrict__ meta, uint64_t *__restrict__ out)
{
    const double total = pairs[0] + pairs[1];
    const bool some = total > 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) meta->lastnz = some ? 0 : -1;
    if (!some) return;
    const uint32_t start = blockIdx.x * kPer;
    pick_samples(re, im, N, 0u, 0.0, total, min(k - start, kPer),
                 [&](uint32_t i) { return start + i; }, U, out);
}

// Device and pinned scratch, grown as needed under the library lock; what is
// over kKeep bytes is given back at the end of the call.
struct Scratch {
    void *dev = nullptr, *host = nullptr;
    size_t dev_cap = 0, host_cap = 0;
};
Scratch g_scr;
constexpr size_t kKeep = 64u << 20;

int reserve(size_t dev_bytes, size_t host_bytes)
{
    if (dev_bytes > g_scr.dev_cap) {
        if (g_scr.dev) SPZ_HIP(hipFree(g_scr.dev));
        g_scr.dev = nullptr;
        g_scr.dev_cap = 0;
        if (device_alloc(&g_scr.dev, dev_bytes) != hipSuccess)
            return fail(SPZ_ERR_OOM, "sampling scratch allocation failed");
        g_scr.dev_cap = dev_bytes;
    }
    if (host_bytes > g_scr.host_cap) {
        if (g_scr.host) SPZ_HIP(hipHostFree(g_scr.host));
        g_scr.host = nullptr;
        g_scr.host_cap = 0;
        if (hipHostMalloc(&g_scr.host, host_bytes, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            g_scr.host = nullptr;
            return fail(SPZ_ERR_OOM, "sampling staging allocation failed");
        }
        g_scr.host_cap = host_bytes;
    }
    return SPZ_OK;
}

size_t up(size_t b) { return (b + 255) & ~(size_t)255; }

int sample_one(const spz_state_s *s, const double *uniforms, uint64_t k, uint64_t *out)
{
    const uint32_t piece = (uint32_t)std::min<uint64_t>(k, kPiece);
    const size_t o_meta = up(piece * 8ull), o_u = o_meta + 256;
    SPZ_TRY(reserve(0, o_u + up(piece * 8ull)));
    char *h = (char *)g_scr.host;
    SampleMeta *meta = (SampleMeta *)(h + o_meta);
    double *U = (double *)(h + o_u);
    uint64_t *picked = (uint64_t *)h;
    hipStream_t st = rt().stream;
    LaunchTimer tm(SPZ_K_OTHER, 0.0);
    for (uint64_t at = 0; at < k; at += piece) {
        const uint32_t m = (uint32_t)std::min<uint64_t>(piece, k - at);
        memcpy(U, uniforms + at, m * sizeof(double));
        const unsigned g = (m + kPer - 1) / kPer;
        if (s->prec == SPZ_F64)
            hipLaunchKernelGGL((k_sample_one<double>), dim3(g), dim3(kT), 0, st,
                               (const double *)s->re, (const double *)s->im, s->N,
                               rt().d_partials, U, m, meta, picked);
        else
            hipLaunchKernelGGL((k_sample_one<float>), dim3(g), dim3(kT), 0, st,
                               (const float *)s->re, (const float *)s->im, s->N,
                               rt().d_partials, U, m, meta, picked);
        SPZ_HIP(hipGetLastError());
        SPZ_HIP(hipStreamSynchronize(st));
        if (meta->lastnz < 0) return fail(SPZ_ERR_PROB, "sampling a zero state");
        memcpy(out + at, picked, m * sizeof(uint64_t));
    }
    return SPZ_OK;
}

// P[0..nb-1] in device memory, the total and the last positive block from the level-1
// pairs in rt().d_partials, the additions by the host in the same order: it makes
// one in 1.2 ns where a lane of the GPU takes 5.5, which pays for the blocks' sums
// crossing the bus twice from kHostBlocks blocks on (one sample, the GPU's lane and
// the host: 23 qubits 95 us both, 24 qubits 130 and 118, 26 360 and 270, 28 1260 and
// 860, 30 5.0 and 3.3 ms, 32 in FP32 15.1 and 8.4).  `v`: pinned, kHostPiece values.
int block_prefix_on_host(uint64_t nb, double *P, double *v, SampleMeta *m)
{
    hipStream_t st = rt().stream;
    double acc = 0.0;
    m->lastnz = -1;
    m->nslots = 0;
    m->pad = 0;
    for (uint64_t at = 0; at < nb; at += kHostPiece) {
        const uint64_t cnt = std::min(kHostPiece, nb - at);
        const dim3 g((unsigned)((cnt + kT - 1) / kT)), t(kT);
        hipLaunchKernelGGL(k_block_sums, g, t, 0, st, rt().d_partials + 2 * at, cnt, v);
        SPZ_HIP(hipGetLastError());
        SPZ_HIP(hipStreamSynchronize(st));
        for (uint64_t b = 0; b < cnt; b++) {
            const double w = v[b];
            v[b] = acc;
            acc = acc + w;
            if (w > 0.0) m->lastnz = (int64_t)(at + b);
        }
        hipLaunchKernelGGL(k_take_sums, g, t, 0, st, v, cnt, P + at);
        SPZ_HIP(hipGetLastError());
    }
    m->total = acc;
    return SPZ_OK;
}

int sample_rounds(const spz_state_s *s, uint64_t nb, const double *uniforms, uint64_t k,
                  uint64_t *out)
{
    const uint32_t piece = (uint32_t)std::min<uint64_t>(k, kPiece);
    const uint64_t slots_max = std::min<uint64_t>(piece, nb + piece / kPer);
    // device layout: out and meta together (one copy back), then the rest
    const size_t o_out = 0, o_meta = up(piece * 8ull), o_u = o_meta + 256;
    const size_t o_blk = o_u + up(piece * 8ull), o_rank = o_blk + up(piece * 4ull);
    const size_t o_ord = o_rank + up(piece * 4ull), o_slot = o_ord + up(piece * 4ull);
    const size_t o_cnt = o_slot + up(slots_max * sizeof(Slot)), o_p = o_cnt + up(nb * 4ull);
    const size_t dev_bytes = o_p + up((nb + 1) * 8ull);
    // few samples: uniforms and results stay in pinned memory, without copies
    // (16 to 20 qubits, one sample 71 -> 65 us, 4096 103 -> 76, 16384 118 -> 106;
    // the picks' scattered stores over the bus catch up with the copies there)
    const bool direct = k <= kDirect;
    const bool on_host = nb >= kHostBlocks;
    const size_t o_stage = direct ? o_u + up(piece * 8ull) : o_u;
    SPZ_TRY(reserve(dev_bytes, o_stage + (on_host ? std::min(nb, kHostPiece) * sizeof(double) : 0)));
    char *d = (char *)g_scr.dev, *h = (char *)g_scr.host;
    SampleMeta *meta = (SampleMeta *)(d + o_meta);
    double *U = (double *)((direct ? h : d) + o_u), *P = (double *)(d + o_p);
    uint32_t *blk = (uint32_t *)(d + o_blk), *rank = (uint32_t *)(d + o_rank),
             *order = (uint32_t *)(d + o_ord), *counts = (uint32_t *)(d + o_cnt);
    Slot *slots = (Slot *)(d + o_slot);
    uint64_t *dout = (uint64_t *)((direct ? h : d) + o_out);
    SampleMeta *host_meta = (SampleMeta *)(h + o_meta);
    hipStream_t st = rt().stream;
    LaunchTimer tm(SPZ_K_OTHER, 0.0);
    SampleMeta first;
    if (on_host) {
        SPZ_TRY(block_prefix_on_host(nb, P, (double *)(h + o_stage), &first));
        if (first.lastnz < 0) return fail(SPZ_ERR_PROB, "sampling a zero state");
    }
    for (uint64_t at = 0; at < k; at += piece) {
        const uint32_t m = (uint32_t)std::min<uint64_t>(piece, k - at);
        // (the previous round was waited for: the staging buffer is free)
        memcpy(direct ? (char *)U : h, uniforms + at, m * sizeof(double));
        if (!direct)
            SPZ_HIP(hipMemcpyAsync(U, h, m * sizeof(double), hipMemcpyHostToDevice, st));
        const unsigned g = (m + kT - 1) / kT;
        if (on_host)
            hipLaunchKernelGGL(k_sample_begin, dim3((unsigned)((nb + kT - 1) / kT)), dim3(kT), 0, st,
                               counts, nb, P, meta, direct ? host_meta : nullptr, first);
        else
            hipLaunchKernelGGL(k_block_prefix, dim3(1), dim3(kPT), 0, st, rt().d_partials, nb, P,
                               counts, meta, direct ? host_meta : nullptr);
        hipLaunchKernelGGL(k_sample_block, dim3(g), dim3(kT), 0, st, P, nb, meta, U, m, counts,
                           blk, rank);
        if (nb <= kPT)
            hipLaunchKernelGGL((k_sample_scan<1>), dim3(1), dim3(kPT), 0, st, counts, nb, slots, meta);
        else
            hipLaunchKernelGGL((k_sample_scan<8>), dim3(1), dim3(kPT), 0, st, counts, nb, slots, meta);
        hipLaunchKernelGGL(k_sample_order, dim3(g), dim3(kT), 0, st, counts, meta, blk, rank, m,
                           order);
        const unsigned gs = (unsigned)std::min<uint64_t>(m, nb + m / kPer);
        if (s->prec == SPZ_F64)
            hipLaunchKernelGGL((k_sample_pick<double>), dim3(gs), dim3(kT), 0, st,
                               (const double *)s->re, (const double *)s->im, s->N, P, meta, slots,
                               order, U, dout);
        else
            hipLaunchKernelGGL((k_sample_pick<float>), dim3(gs), dim3(kT), 0, st,
                               (const float *)s->re, (const float *)s->im, s->N, P, meta, slots,
                               order, U, dout);
        SPZ_HIP(hipGetLastError());
        if (!direct) SPZ_HIP(hipMemcpyAsync(h, d, o_u, hipMemcpyDeviceToHost, st));
        SPZ_HIP(hipStreamSynchronize(st));
        if (host_meta->lastnz < 0)
            return fail(SPZ_ERR_PROB, "sampling a zero state");
        memcpy(out + at, h, m * sizeof(uint64_t));
    }
    return SPZ_OK;
}

}  // namespace

int sample_state(const spz_state_s *s, const double *uniforms, uint64_t k, uint64_t *out)
{
    uint64_t nb;
    SPZ_TRY(norm_level1(s, &nb));
    const int rc = nb == 1 ? sample_one(s, uniforms, k, out) : sample_rounds(s, nb, uniforms, k, out);
    if (rc != SPZ_OK) (void)hipStreamSynchronize(rt().stream);  // the scratch is idle again
    if (g_scr.dev_cap > kKeep) {
        (void)hipFree(g_scr.dev);
        g_scr.dev = nullptr;
        g_scr.dev_cap = 0;
    }
    if (g_scr.host_cap > kKeep) {
        (void)hipHostFree(g_scr.host);
        g_scr.host = nullptr;
        g_scr.host_cap = 0;
    }
    return rc;
}

}  // namespace spz
