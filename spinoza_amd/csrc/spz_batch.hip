// spz_batch.hip -- batched adjoint gradients of many independent circuits
// (no counterpart in the reference).
//
// Circuits up to the switch point are planned as tile sweeps and run level by
// level (spz_chip.hip): one launch takes the k-th sweep of every circuit of a
// chunk, so a launch has a tile of 2^12 amplitudes per workgroup whatever the
// circuits' sizes, a gate costs register arithmetic instead of a pass through
// the caches, and nothing waits inside a kernel.  A chunk is a set of circuits
// with about as many tiles as the GPU holds workgroups; its programs are
// planned and uploaded while the GPU runs the chunk before.  Larger circuits use
// the single-circuit path one at a time.  The switch point is measured by
// spz_batch_autotune.
//
// What bounded it: a persistent kernel that moved every gate's pairs through
// the L2 (one workgroup, or a group of workgroups of one XCD with a barrier
// around every gate that crossed their blocks): 33.3 ms of device time for 128
// circuits of 10 to 18 qubits, 6.7 ms now (whole call 50.8 -> 9.7 ms).  Chunks
// of 192 to 1536 tiles measured within 5% of each other.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <functional>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "spz_chip.h"
#include "spz_reduce.h"

namespace spz {

int adjoint_grad(spz_state_s *s, const spz_op *ops, uint64_t n_ops, double hx, int ckpt_every,
                 double *grad, double *energy, double *drift);
int validate_adjoint_op(int n, const spz_op &o, uint64_t idx, bool allow_swap, int max_controls);

namespace {

constexpr int kMaxControls = 7;
constexpr int kBatchMaxQubits = 20;     // larger circuits fill the GPU on their own
constexpr uint64_t kChunkTiles = 768;   // three reverse workgroups on each of 256 CUs
// A chunk ends at so many ops once every CU has a workgroup, and at 256 MiB of
// program (128 bytes per op) in any case.  (Ended at kChunkOps whatever its tiles,
// long circuits ran one after another: 64 of 10 qubits and 10000 ops 996 ms, now
// 65; 256 of 1000 ops 45 and 21 ms; 128 of 10 to 18 qubits 10.3 and 9.6 ms.)
constexpr uint64_t kChunkOps = 20000, kChunkFull = 256, kChunkMax = 1u << 21;
constexpr int kPlanThreads = 8;
constexpr size_t kKeep = (size_t)1 << 30;  // scratch kept between calls
constexpr size_t kKeepPlans = (size_t)64 << 20;

int g_wg_max_qubits = -1;  // autotuned switch point (-1: not tuned yet)

int switch_point() { return g_wg_max_qubits > 0 ? g_wg_max_qubits : 14; }

// Grow-only device buffers, given back at the end of a call that needed more
// than kKeep bytes of them (a free synchronises the device).
struct Buf {
    void *p = nullptr;
    size_t cap = 0;

    int need(size_t bytes)
    {
        if (bytes <= cap) return SPZ_OK;
        drop();
        if (device_alloc(&p, bytes) != hipSuccess)
            return fail(SPZ_ERR_OOM, "batched adjoint scratch allocation failed");
        cap = bytes;
        return SPZ_OK;
    }
    void drop()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
};

// A chunk's program goes through one of two pinned staging buffers and device
// copies, so that the next chunk is planned while this one runs; `done` is
// recorded after the last kernel that reads the slot.
struct Slot {
    char *host = nullptr, *dev = nullptr;
    size_t cap = 0;
    hipEvent_t done = nullptr;
    bool busy = false;

    int open(size_t bytes)
    {
        if (busy) {
            SPZ_HIP(hipEventSynchronize(done));
            busy = false;
        }
        if (!done) SPZ_HIP(hipEventCreateWithFlags(&done, hipEventDisableTiming));
        if (bytes <= cap) return SPZ_OK;
        drop();
        if (device_alloc((void **)&dev, bytes) != hipSuccess ||
            hipHostMalloc(&host, bytes, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            drop();
            return fail(SPZ_ERR_OOM, "batched adjoint program allocation failed");
        }
        cap = bytes;
        return SPZ_OK;
    }
    void drop()
    {
        if (dev) (void)hipFree(dev);
        if (host) (void)hipHostFree(host);
        dev = host = nullptr;
        cap = 0;
    }
};

// All of it is used under the library lock.
struct Scratch {
    Buf states, parts, out;
    Slot slots[2];
    std::vector<hipEvent_t> events;  // pairs of timing events, one per chunk
    std::vector<ChipPlan> fwd, rev;  // a chunk's plans
    bool in_use = false;             // a call is running

    void drop()  // (the stream was waited for, or the frees wait for it)
    {
        for (Buf *b : {&states, &parts, &out}) b->drop();
        for (Slot &s : slots) {
            s.busy = false;
            s.drop();
        }
    }
    // Plans keep their memory from chunk to chunk and call to call (allocated anew, its
    // page faults cost several threads more than planning small circuits does), at
    // most kKeepPlans of it.
    void trim_plans()
    {
        size_t n = 0;
        for (const auto *v : {&fwd, &rev})
            for (const ChipPlan &p : *v)
                n += p.prog.capacity() * sizeof(TileOp) + p.sweeps.capacity() * sizeof(ChipPlan::Sweep);
        if (n <= kKeepPlans) return;
        fwd = std::vector<ChipPlan>();
        rev = std::vector<ChipPlan>();
    }
    size_t bytes() const
    {
        return states.cap + parts.cap + out.cap + slots[0].cap + slots[1].cap;
    }
};
Scratch &scratch()
{
    static Scratch *s = new Scratch();  // lives until the process ends
    return *s;
}

uint64_t tiles_of(int n) { return n > kChipK ? 1ull << (n - kChipK) : 1ull; }

size_t up(size_t n) { return (n + 255) & ~(size_t)255; }

// The sweep of a circuit without ops: it only writes |0...0>.
ChipPlan::Sweep empty_sweep()
{
    ChipPlan::Sweep s;
    memset(&s, 0, sizeof s);
    for (int i = 0; i < 16; i++) s.desc.spos[i] = (int8_t)(i < kChipK ? i : 64);
    for (int i = 0; i < kChipK - 4; i++) {
        s.desc.tin[i] = (int8_t)i;
        s.desc.tg[i] = 1ull << i;
    }
    for (uint64_t p = 0; p < 16; p++) s.desc.gr[p] = s.desc.gs[p] = p << (kChipK - 4);
    return s;
}

// One rule for both paths (the switch point must not decide whether a circuit
// is accepted): gates H..U, at most kMaxControls controls.
int check_circuit(const spz_batch_circuit &c, const spz_op *ops, uint64_t i)
{
    if (c.n < 1 || c.n > 30 || c.n_ops < 0) return fail(SPZ_ERR_ARG, "bad circuit entry");
    for (int o = 0; o < c.n_ops; o++) {
        const int rc = validate_adjoint_op(c.n, ops[c.op_offset + o], (uint64_t)o, false, kMaxControls);
        if (rc != SPZ_OK) {
            set_error("circuit " + std::to_string(i) + ": " + spz_last_error());
            return rc;
        }
    }
    return SPZ_OK;
}

struct Job {
    uint64_t circuit;   // index in the caller's list
    uint32_t width;     // workgroups it may use
};

// Threads that help the caller with a chunk's host work (plans, then the copies of
// programs and descriptors to pinned memory, each by whoever is free), started when
// they are first wanted and ended with the batch.  1000 circuits of 5 qubits, 10 and
// 40 gates: threads started for every chunk's plans and copies by the caller alone
// took 1.5 and 3.1 ms, this 1.04 and 2.5; 128 of 10 to 18 qubits the same 9.7.
class Crew {
    std::vector<std::thread> pool;
    std::mutex mu;
    std::condition_variable wake, idle;
    std::function<void()> job;
    uint64_t turn = 0;     // of the job that is up
    unsigned places = 0;   // helpers the job still takes
    unsigned working = 0;
    bool stop = false;

    void help()
    {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            wake.wait(lk, [&] { return stop || turn != seen; });
            if (stop) return;
            seen = turn;
            if (!places) continue;
            places--;
            working++;
            lk.unlock();
            job();
            lk.lock();
            if (!--working) idle.notify_one();
        }
    }

public:
    ~Crew()
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
        }
        wake.notify_all();
        for (std::thread &t : pool) t.join();
    }

    // Runs f here and on up to want - 1 helpers; f shares out the work by itself, ends
    // when there is none left, and does not throw.
    void run(uint64_t want, const std::function<void()> &f)
    {
        if (want > 1) {
            try {
                while (pool.size() + 1 < want) pool.emplace_back([this] { help(); });
            } catch (const std::exception &) {
                // no more threads to be had: the ones there are do the work
            }
            {
                std::lock_guard<std::mutex> lk(mu);
                job = f;
                turn++;
                places = (unsigned)std::min<uint64_t>(want - 1, pool.size());
            }
            wake.notify_all();
        }
        f();
        std::unique_lock<std::mutex> lk(mu);
        places = 0;  // (whoever has not started need not)
        idle.wait(lk, [&] { return !working; });
    }
};

uint64_t most_threads(uint32_t count)
{
    const unsigned cores = std::max(1u, std::thread::hardware_concurrency());
    return std::min<uint64_t>({(uint64_t)kPlanThreads, cores, count});
}

// Forward and reverse plans of a chunk's circuits.  Planning costs about half a
// microsecond per circuit and 0.06 to 0.2 us per op in each direction, more than
// the GPU takes for circuits of up to 12 qubits (180 of them: 6.0 ms planned by one
// thread, 0.6 ms of sweeps), so a chunk is planned by several threads once there
// is enough to pay for starting them (20 to 40 us each).
int plan_chunk(Crew &crew, const spz_batch_circuit *circuits, const spz_op *ops, const Job *jobs,
               uint32_t count, std::vector<ChipPlan> &fwd, std::vector<ChipPlan> &rev)
{
    uint64_t nops = 0;
    for (uint32_t c = 0; c < count; c++) nops += (uint64_t)circuits[jobs[c].circuit].n_ops;
    std::atomic<uint32_t> next{0};
    std::atomic<int> status{SPZ_OK};
    const uint64_t cost = count + nops / 4;  // about so many us, both directions
    crew.run(std::min(most_threads(count), cost / 150 + 1), [&]() {
        try {
            for (uint32_t c; status == SPZ_OK && (c = next++) < count;) {
                const spz_batch_circuit &q = circuits[jobs[c].circuit];
                const spz_op *o = ops + q.op_offset;
                int rc = chip_plan(q.n, o, (uint64_t)q.n_ops, false, fwd[c]);
                if (rc == SPZ_OK) rc = chip_plan(q.n, o, (uint64_t)q.n_ops, true, rev[c]);
                if (rc == SPZ_OK && fwd[c].sweeps.empty()) fwd[c].sweeps.push_back(empty_sweep());
                if (rc != SPZ_OK) status = rc;
            }
        } catch (const std::bad_alloc &) {
            status = SPZ_ERR_OOM;
        }
    });
    if (status != SPZ_OK) return fail(status, "batched adjoint: planning failed");
    return SPZ_OK;
}

// Plans, uploads and launches one chunk; energies go to out[circuit slot],
// gradients to out[grad0 + grad_offset + op].
struct Chunk {
    const spz_batch_circuit *circuits;
    const spz_op *ops;
    double hx;
    size_t lds;
    uint64_t grad0;
    Crew &crew;

    int run(const Job *jobs, uint32_t count, uint32_t slot0, Scratch &sc, Slot &slot,
            hipEvent_t begin, hipEvent_t end)
    {
        if (sc.fwd.size() < count) {
            sc.fwd.resize(count);
            sc.rev.resize(count);
        }
        std::vector<ChipPlan> &fwd = sc.fwd, &rev = sc.rev;
        uint64_t amps = 0, pairs = 0, nops = 0;
        size_t nf = 0, nr = 0, ns = 0, lf = 0, lr = 0;
        uint32_t width = 0, blocks = 0;
        SPZ_TRY(plan_chunk(crew, circuits, ops, jobs, count, fwd, rev));
        for (uint32_t c = 0; c < count; c++) {
            const spz_batch_circuit &q = circuits[jobs[c].circuit];
            const uint64_t t = tiles_of(q.n);
            amps += 4 * (t << kChipK);
            pairs += rev[c].grads.size() * t * kChipRows + t;
            nops += fwd[c].prog.size() + rev[c].prog.size();
            nf += fwd[c].sweeps.size();
            nr += rev[c].sweeps.size();
            ns += rev[c].grads.size() + 1;
            lf = std::max(lf, fwd[c].sweeps.size());
            lr = std::max(lr, rev[c].sweeps.size());
            width = std::max(width, jobs[c].width);
            blocks = std::max(blocks, (uint32_t)t);
        }
        SPZ_TRY(sc.states.need(amps * sizeof(double)));
        SPZ_TRY(sc.parts.need(pairs * 2 * sizeof(double)));
        const size_t o_f = up(nops * sizeof(TileOp)), o_i = o_f + up(nf * sizeof(ChipSweep));
        const size_t o_r = o_i + up(count * sizeof(ChipIsing));
        const size_t o_s = o_r + up(nr * sizeof(ChipSweep)), total = o_s + up(ns * sizeof(ChipSum));
        SPZ_TRY(slot.open(total));
        TileOp *hp = (TileOp *)slot.host;
        ChipSweep *hf = (ChipSweep *)(slot.host + o_f), *hr = (ChipSweep *)(slot.host + o_r);
        ChipIsing *hi = (ChipIsing *)(slot.host + o_i);
        ChipSum *hs = (ChipSum *)(slot.host + o_s);
        const TileOp *dp = (const TileOp *)slot.dev;
        // where every circuit's programs, states and sums go, and its descriptors,
        // which are in the order of the levels
        struct Place {
            double *psi, *part;
            uint64_t amps;
            size_t fwd, rev, sum;    // first op, first sum
            size_t fwd_at, rev_at;   // in `order`
        };
        struct Level {
            size_t first;
            uint32_t count;
        };
        std::vector<Place> at(count);
        std::vector<Level> levels_f(lf, {0, 0}), levels_r(lr, {0, 0});
        std::vector<size_t> order(nf + nr);  // a sweep's place among its level's
        {
            double *amp = (double *)sc.states.p, *part = (double *)sc.parts.p;
            size_t op = 0, sum = 0, k = 0;
            for (uint32_t c = 0; c < count; c++) {
                const uint64_t t = tiles_of(circuits[jobs[c].circuit].n);
                at[c] = {amp, part, t << kChipK, op, op + fwd[c].prog.size(), sum, k,
                         k + fwd[c].sweeps.size()};
                for (size_t l = 0; l < fwd[c].sweeps.size(); l++) order[k++] = levels_f[l].count++;
                for (size_t l = 0; l < rev[c].sweeps.size(); l++) order[k++] = levels_r[l].count++;
                op += fwd[c].prog.size() + rev[c].prog.size();
                sum += rev[c].grads.size() + 1;
                amp += 4 * at[c].amps;
                part += 2 * (rev[c].grads.size() * t * kChipRows + t);
            }
            for (auto *ls : {&levels_f, &levels_r}) {
                size_t first = 0;
                for (Level &l : *ls) {
                    l.first = first;
                    first += l.count;
                }
            }
        }
        auto fill = [&](ChipSweep &d, uint32_t c, const ChipPlan::Sweep &s, size_t first_op) {
            memset(&d, 0, sizeof d);
            chip_geometry(s, circuits[jobs[c].circuit].n, SPZ_F64, d);
            const uint64_t A = at[c].amps;
            d.sr = d.pr = at[c].psi;
            d.si = d.pi = at[c].psi + A;
            d.qr = at[c].psi + 2 * A;
            d.qi = at[c].psi + 3 * A;
            d.ops = dp + first_op + s.op_begin;
            d.part = at[c].part + 2 * (size_t)s.slot_begin * d.tiles * kChipRows;
            d.width = jobs[c].width;
            d.flags = CHIP_STORE;
        };
        auto write = [&](uint32_t c) {
            const spz_batch_circuit &q = circuits[jobs[c].circuit];
            const uint64_t t = tiles_of(q.n), A = at[c].amps;
            const ChipPlan &f = fwd[c], &r = rev[c];
            if (!f.prog.empty()) memcpy(hp + at[c].fwd, f.prog.data(), f.prog.size() * sizeof(TileOp));
            if (!r.prog.empty()) memcpy(hp + at[c].rev, r.prog.data(), r.prog.size() * sizeof(TileOp));
            ChipSum *sum = hs + at[c].sum;
            for (size_t k = 0; k < r.grads.size(); k++)
                *sum++ = {at[c].part + 2 * k * t * kChipRows, (uint32_t)(t * kChipRows),
                          (uint32_t)(grad0 + q.grad_offset + r.grads[k])};
            double *ep = at[c].part + 2 * r.grads.size() * t * kChipRows, *psi = at[c].psi;
            *sum = {ep, (uint32_t)t, slot0 + c};
            hi[c] = {psi, psi + A, psi + 2 * A, psi + 3 * A, 1ull << q.n, ep, (uint32_t)t, q.n};
            for (size_t l = 0; l < f.sweeps.size(); l++) {
                ChipSweep &d = hf[levels_f[l].first + order[at[c].fwd_at + l]];
                fill(d, c, f.sweeps[l], at[c].fwd);
                if (l == 0) d.flags |= CHIP_INIT;
            }
            for (size_t l = 0; l < r.sweeps.size(); l++) {
                ChipSweep &d = hr[levels_r[l].first + order[at[c].rev_at + l]];
                fill(d, c, r.sweeps[l], at[c].rev);
                if (l + 1 == r.sweeps.size()) d.flags = 0;  // only its sums are used
            }
        };
        std::atomic<uint32_t> next{0};
        crew.run(std::min(most_threads(count), (uint64_t)total / (256 << 10) + 1), [&]() {
            constexpr uint32_t kAtOnce = 8;
            for (uint32_t c; (c = next.fetch_add(kAtOnce)) < count;)
                for (uint32_t e = std::min(c + kAtOnce, count); c < e; c++) write(c);
        });
        hipStream_t st = rt().stream;
        SPZ_HIP(hipEventRecord(begin, st));
        SPZ_HIP(hipMemcpyAsync(slot.dev, slot.host, total, hipMemcpyHostToDevice, st));
        int rc = SPZ_OK;
        for (const Level &l : levels_f)
            if (rc == SPZ_OK)
                rc = launch_chip_sweeps(SPZ_F64, false, (const ChipSweep *)(slot.dev + o_f) + l.first,
                                        l.count, width, lds);
        if (rc == SPZ_OK)
            rc = launch_chip_ising((const ChipIsing *)(slot.dev + o_i), count, blocks, hx);
        for (const Level &l : levels_r)
            if (rc == SPZ_OK)
                rc = launch_chip_sweeps(SPZ_F64, true, (const ChipSweep *)(slot.dev + o_r) + l.first,
                                        l.count, width, lds);
        if (rc == SPZ_OK)
            rc = launch_chip_sums((const ChipSum *)(slot.dev + o_s), (uint32_t)ns,
                                  (double *)sc.out.p);
        SPZ_HIP(hipEventRecord(end, st));
        SPZ_HIP(hipEventRecord(slot.done, st));
        slot.busy = true;
        return rc;
    }
};

}  // namespace

bool batch_give_back()
{
    Scratch &sc = scratch();
    if (sc.in_use || !sc.bytes()) return false;
    sc.drop();
    return true;
}

}  // namespace spz

using namespace spz;

extern "C" {

int spz_batch_adjoint(const spz_batch_circuit *circuits, uint64_t count, const spz_op *ops,
                      double hx, double *energies, double *grads, const spz_batch_opts *opts,
                      spz_batch_stats *stats)
{
    SPZ_API_LOCK;
    SPZ_TRY(ensure_init());
    if (count == 0) return SPZ_OK;
    if (!circuits || !ops || !energies || !grads) return fail(SPZ_ERR_ARG, "null argument");
    const int wg_max = opts && opts->wg_max_qubits > 0
                           ? opts->wg_max_qubits
                           : switch_point();
    // circuits above gq qubits run on 2^(n - gq) workgroups (at most one per tile)
    const int gq_opt = opts ? opts->group_qubits : 0;
    const int gq = gq_opt < 0 ? 64 : (gq_opt == 0 ? kChipK : std::max(gq_opt, 8));
    std::vector<Job> small;
    std::vector<uint64_t> large;
    int n_group = 0;
    uint64_t gmax = 0;
    for (uint64_t i = 0; i < count; i++) {
        const spz_batch_circuit &c = circuits[i];
        SPZ_TRY(check_circuit(c, ops, i));
        if (c.n > wg_max || c.n > kBatchMaxQubits) {
            large.push_back(i);
            continue;
        }
        const uint64_t wgs = c.n > gq ? 1ull << (c.n - gq) : 1ull;
        small.push_back({i, (uint32_t)std::min(wgs, tiles_of(c.n))});
        n_group += c.n > gq;
        gmax = std::max<uint64_t>(gmax, c.grad_offset + (uint64_t)c.n_ops);
    }
    if (small.size() + gmax >= 0xFFFFFFFFull) return fail(SPZ_ERR_ARG, "too many gradients");
    auto t0 = std::chrono::steady_clock::now();
    std::vector<double> lat(count, 0.0);
    // ---- circuits up to the switch point, largest first: circuits of one size
    // share chunks, and the first chunk keeps the GPU busy longest
    std::stable_sort(small.begin(), small.end(), [&](const Job &x, const Job &y) {
        const spz_batch_circuit &a = circuits[x.circuit], &b = circuits[y.circuit];
        return a.n != b.n ? a.n > b.n : a.n_ops > b.n_ops;
    });
    Scratch &sc = scratch();
    struct InUse {
        bool &flag;
        explicit InUse(bool &f) : flag(f) { flag = true; }
        ~InUse() { flag = false; }
    } in_use(sc.in_use);
    // wg_per_cu > 0 caps the workgroups resident on a CU by padding their LDS
    // (160 KiB per CU, 32 KiB used, at most 64 KiB per workgroup)
    size_t lds = 0;
    if (opts && opts->wg_per_cu > 0) {
        const size_t share = std::min<size_t>(64 << 10, (160u << 10) / (size_t)opts->wg_per_cu);
        lds = share > (32u << 10) ? share - (32u << 10) : 0;
    }
    int rc = SPZ_OK;
    std::vector<size_t> first;  // first job of every chunk
    if (!small.empty()) {
        rc = sc.out.need((small.size() + gmax) * sizeof(double));
        // (the gradients of ops without a parameter stay zero)
        if (rc == SPZ_OK && hipMemsetAsync(sc.out.p, 0, (small.size() + gmax) * sizeof(double),
                                           rt().stream) != hipSuccess)
            rc = fail(SPZ_ERR_HIP, "batched adjoint clear failed");
        Crew crew;
        Chunk ch{circuits, ops, hx, lds, small.size(), crew};
        for (size_t a = 0; rc == SPZ_OK && a < small.size();) {
            size_t b = a;
            uint64_t tiles = 0, nops = 0;
            while (b < small.size()) {
                const spz_batch_circuit &c = circuits[small[b].circuit];
                tiles += tiles_of(c.n);
                nops += 2 * (uint64_t)c.n_ops;
                if (b > a && (tiles > kChunkTiles || nops > kChunkMax ||
                              (nops > kChunkOps && tiles > kChunkFull)))
                    break;
                b++;
            }
            const size_t k = first.size();
            while (rc == SPZ_OK && sc.events.size() < 2 * (k + 1)) {
                hipEvent_t e;
                if (hipEventCreate(&e) != hipSuccess) rc = fail(SPZ_ERR_HIP, "event creation failed");
                else sc.events.push_back(e);
            }
            if (rc == SPZ_OK)
                rc = ch.run(&small[a], (uint32_t)(b - a), (uint32_t)a, sc, sc.slots[k & 1],
                            sc.events[2 * k], sc.events[2 * k + 1]);
            first.push_back(a);
            a = b;
        }
    }
    // ---- larger circuits: the single-circuit path, behind them on the stream ------
    std::stable_sort(large.begin(), large.end(),
                     [&](uint64_t x, uint64_t y) { return circuits[x].n < circuits[y].n; });
    spz_state st = nullptr;
    int st_n = 0;
    for (uint64_t i : large) {
        if (rc != SPZ_OK) break;
        const spz_batch_circuit &c = circuits[i];
        auto a = std::chrono::steady_clock::now();
        if (c.n != st_n) {
            if (st) spz_state_destroy(st);
            st = nullptr;
            st_n = 0;
            rc = spz_state_create(c.n, SPZ_F64, &st);
            if (rc == SPZ_OK) st_n = c.n;
        } else {
            rc = spz_state_set_basis(st, 0);
        }
        if (rc == SPZ_OK)
            rc = adjoint_grad(st, ops + c.op_offset, (uint64_t)c.n_ops, hx, 0,
                              grads + c.grad_offset, &energies[i], nullptr);
        auto b = std::chrono::steady_clock::now();
        lat[i] = std::chrono::duration<double, std::milli>(b - a).count();
    }
    if (st) spz_state_destroy(st);
    // ---- collect -----------------------------------------------------------------
    if (hipStreamSynchronize(rt().stream) != hipSuccess && rc == SPZ_OK)
        rc = fail(SPZ_ERR_HIP, "batched adjoint failed");
    if (rc == SPZ_OK && !small.empty()) {
        std::vector<double> out(small.size() + gmax);
        if (hipMemcpy(out.data(), sc.out.p, out.size() * sizeof(double), hipMemcpyDeviceToHost) !=
            hipSuccess)
            rc = fail(SPZ_ERR_HIP, "batched adjoint download failed");
        for (size_t k = 0; rc == SPZ_OK && k < first.size(); k++) {
            float ms = 0.f;  // a circuit's time is its chunk's
            (void)hipEventElapsedTime(&ms, sc.events[2 * k], sc.events[2 * k + 1]);
            const size_t b = k + 1 < first.size() ? first[k + 1] : small.size();
            for (size_t j = first[k]; j < b; j++) {
                const uint64_t i = small[j].circuit;
                const spz_batch_circuit &c = circuits[i];
                energies[i] = out[j];
                if (c.n_ops)
                    memcpy(grads + c.grad_offset, out.data() + small.size() + c.grad_offset,
                           (size_t)c.n_ops * sizeof(double));
                lat[i] = ms;
            }
        }
    }
    if (sc.bytes() > kKeep) sc.drop();
    sc.trim_plans();
    if (rc != SPZ_OK) return rc;
    auto t1 = std::chrono::steady_clock::now();
    if (stats) {
        std::sort(lat.begin(), lat.end());
        stats->total_ms = std::chrono::duration<double, std::milli>(t1 - t0).count();
        stats->p50_ms = lat[(size_t)(0.50 * (lat.size() - 1))];
        stats->p99_ms = lat[(size_t)(0.99 * (lat.size() - 1))];
        stats->n_small = small.size();
        stats->n_large = large.size();
        stats->wg_max_qubits = wg_max;
        stats->n_group = n_group;
    }
    return SPZ_OK;
}

int spz_batch_autotune(const spz_batch_circuit *circuits, uint64_t count, const spz_op *ops,
                       int *wg_max_qubits)
{
    // For every qubit count present that can run batched: run up to 8 of its
    // circuits batched and one at a time; the switch point is the largest n for
    // which the batch wins.  (Larger circuits take the same path in both runs, so
    // only noise would decide; with none but those the switch point stays.)
    SPZ_API_LOCK;
    SPZ_TRY(ensure_init());
    if (!circuits || !ops) return fail(SPZ_ERR_ARG, "null argument");
    std::vector<int> ns;
    for (uint64_t i = 0; i < count; i++) {
        SPZ_TRY(check_circuit(circuits[i], ops, i));
        if (circuits[i].n <= kBatchMaxQubits) ns.push_back(circuits[i].n);
    }
    std::sort(ns.begin(), ns.end());
    ns.erase(std::unique(ns.begin(), ns.end()), ns.end());
    int best = 0;
    for (int n : ns) {
        std::vector<spz_batch_circuit> pick;
        for (uint64_t i = 0; i < count && pick.size() < 8; i++)
            if (circuits[i].n == n) pick.push_back(circuits[i]);
        uint64_t gsz = 0;
        for (auto &c : pick) gsz = std::max<uint64_t>(gsz, c.grad_offset + c.n_ops);
        std::vector<double> e(std::max<uint64_t>(count, 1)), g(std::max<uint64_t>(gsz, 1));
        spz_batch_opts o;
        memset(&o, 0, sizeof o);
        o.use_graph = 1;
        spz_batch_stats sw, sl;
        for (int pass = 0; pass < 2; pass++) {  // (the first sizes the scratch)
            o.wg_max_qubits = 64;  // batched
            SPZ_TRY(spz_batch_adjoint(pick.data(), pick.size(), ops, 1.0, e.data(), g.data(), &o,
                                      &sw));
            o.wg_max_qubits = n - 1;  // one at a time
            if (n == 1) sl.total_ms = INFINITY;
            else
                SPZ_TRY(spz_batch_adjoint(pick.data(), pick.size(), ops, 1.0, e.data(), g.data(),
                                          &o, &sl));
        }
        if (sw.total_ms <= sl.total_ms) best = n;
    }
    if (!ns.empty()) g_wg_max_qubits = best > 0 ? best : 1;
    if (wg_max_qubits) *wg_max_qubits = switch_point();
    return SPZ_OK;
}

}  // extern "C"
