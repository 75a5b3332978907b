// spz_exec.hip -- QuantumCircuit::execute over an op list (circuit.rs:552-600).
//
// PLAIN  : one launch per gate, in program order (the reference's loop).
// STRICT : runs of consecutive gates are packed into fused tile sweeps
//          without reordering anything, so FP64 results are bit-identical to
//          PLAIN (FP32 storage: a sweep rounds to FP32 once at its store,
//          PLAIN after every gate, so they agree within FP32 rounding).
// AUTO   : like STRICT, but a gate may be pulled ahead of earlier gates it
//          commutes with (disjoint qubits, or qubits on which both act
//          diagonally: Z-type targets and controls), which packs more gates
//          into each sweep; floating-point results then differ from PLAIN only
//          by rounding (the same products in a different order).
//
// States of at most 12 qubits (no tile width asked for) keep program order and
// STRICT arithmetic in AUTO too: a run of more than five ops is one launch
// (spz_chip.hip), a shorter one goes op by op.  (At 11 and 12 qubits sweeps of
// narrower tiles are faster, since they reorder: 96 random gates of 11 qubits 48
// us against 69.  tile_qubits = 10 takes them.)
//
// Measurements and dense blocks end a run and execute on their own.  So do, above
// 12 qubits, SWAPs with controls, and in DENSE5 every SWAP; SWAPs without controls
// are a relabelling inside a sweep (FP32: only among themselves).  States of at
// most 12 qubits take SWAPs, controlled ones too, as three CX.  A SWAP under
// classical control always executes on its own.
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <cmath>
#include <vector>

#include "spz_adj_tile.h"
#include "spz_chip.h"
#include "spz_internal.h"
#include "spz_tile.h"

namespace spz {

namespace {

int exec_one_plain(spz_state_s *s, const spz_op &o, spz_tracker *trk, uint8_t *outcome)
{
    if (outcome) *outcome = 255;
    switch (o.kind) {
    case SPZ_UNITARY: {  // transform_u / c_transform_u (circuit.rs:555-558)
        int control = -1;
        if (o.zeros) return fail(SPZ_ERR_GATE, "dense block with a 0-control");
        if (o.ones) {
            if (__builtin_popcountll(o.ones) != 1)
                return fail(SPZ_ERR_GATE, "dense block with more than one control");
            control = __builtin_ctzll(o.ones);
        }
        return spz_transform_u(s, o.m, o.u_re, o.u_im, o.target, control);
    }
    case SPZ_M: {  // circuit.rs:559-566: measure with reset unless already measured
        if (o.ones || o.zeros) return fail(SPZ_ERR_GATE, "controlled measurement");
        if (o.target < 0 || o.target >= s->n) return fail(SPZ_ERR_QUBIT, "target out of range");
        if (trk && ((trk->measured >> o.target) & 1)) return SPZ_OK;
        uint8_t v = 0;
        SPZ_TRY(measure(s, o.target, 1, -1, o.u, &v));
        if (trk) {
            trk->measured |= 1ull << o.target;
            trk->values &= ~(1ull << o.target);
            trk->values |= (uint64_t)v << o.target;
        }
        if (outcome) *outcome = v;
        return SPZ_OK;
    }
    case SPZ_BITFLIP:  // gates.rs:1365-1374
        if (o.ones || o.zeros) return fail(SPZ_ERR_GATE, "controlled bit-flip noise");
        if (o.target < 0 || o.target >= s->n) return fail(SPZ_ERR_QUBIT, "target out of range");
        if (o.u <= o.theta) return apply_gate(s, SPZ_X, 0, 0, 0, o.target, 0, 0, 0);
        return SPZ_OK;
    default:
        break;
    }
    if (o.kind < SPZ_H || o.kind > SPZ_SWAP) return fail(SPZ_ERR_GATE, "unknown gate kind");
    // Classical control once the single control was measured (circuit.rs:570-578).
    if ((o.flags & SPZ_OPF_CLASSICAL) && o.zeros == 0 && __builtin_popcountll(o.ones) == 1 && trk) {
        int c = __builtin_ctzll(o.ones);
        if ((trk->measured >> c) & 1) {
            if ((trk->values >> c) & 1)
                return apply_gate(s, o.kind, o.theta, o.phi, o.lambda, o.target, o.t1, 0, 0);
            return SPZ_OK;
        }
    }
    return apply_gate(s, o.kind, o.theta, o.phi, o.lambda, o.target, o.t1, o.ones, o.zeros);
}

// A single-target gate of a fusable run.
struct SG {
    int op_index;
    int kind;
    int target;
    uint64_t ones, zeros;
    Coef k;
    bool diag;
    uint64_t nd;  // qubits acted on non-diagonally (the target of a 2x2 gate)
    uint64_t dm;  // qubits acted on diagonally (controls, diagonal targets)
    int64_t grad; // reverse sweeps: index of its gradient (-1: none)
    int t1;       // SPZ_SWAP: the other qubit (nd holds both)
};

bool is_barrier(const spz_op &o)
{
    return o.kind == SPZ_M || o.kind == SPZ_SWAP || o.kind == SPZ_UNITARY || o.kind < SPZ_H ||
           o.kind > SPZ_BITFLIP;
}

// Validate and lower one op of a run to an SG; returns 1 if it is a no-op.
int lower(const spz_state_s *s, const spz_op &o, const spz_tracker *trk, int idx, SG *g)
{
    int kind = o.kind;
    uint64_t ones = o.ones, zeros = o.zeros;
    if (kind == SPZ_BITFLIP) {
        if (ones || zeros) return fail(SPZ_ERR_GATE, "controlled bit-flip noise");
        if (!(o.u <= o.theta)) return -1;  // no flip: nothing to do
        kind = SPZ_X;
    }
    if ((o.flags & SPZ_OPF_CLASSICAL) && zeros == 0 && __builtin_popcountll(ones) == 1 && trk) {
        int c = __builtin_ctzll(ones);
        if ((trk->measured >> c) & 1) {
            if (!((trk->values >> c) & 1)) return -1;
            ones = 0;
        }
    }
    const int t = o.target;
    if (t < 0 || t >= s->n) return fail(SPZ_ERR_QUBIT, "target qubit out of range");
    const uint64_t tb = 1ull << t;
    if ((ones | zeros) & tb) return fail(SPZ_ERR_QUBIT, "target is also a control");
    if (ones & zeros) return fail(SPZ_ERR_QUBIT, "qubit both a 1-control and a 0-control");
    if (s->n < 64 && ((ones | zeros) >> s->n)) return fail(SPZ_ERR_QUBIT, "control out of range");
    g->op_index = idx;
    g->kind = kind;
    g->target = t;
    g->ones = ones;
    g->zeros = zeros;
    SPZ_TRY(make_coef(kind, o.theta, o.phi, o.lambda, &g->k));
    g->diag = is_diagonal(g->k.ak);
    g->nd = g->diag ? 0 : tb;
    g->dm = (ones | zeros) | (g->diag ? tb : 0);
    g->grad = -1;
    g->t1 = -1;
    return SPZ_OK;
}

// An uncontrolled SWAP of a run: nothing to compute, its sweep relabels the two
// qubits (Planner::build).
SG lower_swap(const spz_op &o, int idx)
{
    SG g;
    memset(&g, 0, sizeof g);
    g.op_index = idx;
    g.kind = SPZ_SWAP;
    g.target = o.target;
    g.t1 = o.t1;
    g.k.ak = -1;
    g.nd = (1ull << o.target) | (1ull << o.t1);
    g.grad = -1;
    return g;
}

int env_int(const char *name, int dflt)
{
    const char *e = getenv(name);
    return (e && *e) ? atoi(e) : dflt;
}

// How many of the lowest qubits are always in the tile (at most `most`).
int tile_klo(int most) { return std::max(0, std::min(env_int("SPZ_TILE_KLO", 4), most)); }

struct Sweep {
    bool tile;                 // false: a single gate on the plain path
    int gate;                  // plain: index into the run
    TileDesc desc;
    size_t op_begin, op_count; // range in the program buffer
    size_t slot_begin;         // reverse sweeps: range in the list of gradients
    int slots;
    // fast sweeps: the frame a next tile sweep can take over (Z part and
    // phase; the X part is always applied at the store)
    bool can_carry;
    uint64_t carry_z;
    int carry_w;
};

// One-hot TileGroup bit of an arithmetic kind (0: not a tile kind).  AK_MAT
// comes only from a fast sweep's frame conjugation (lower() never makes it).
uint32_t kind_bit(int ak)
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
    case AK_MAT: return TG_MAT;
    case AK_USH: return TG_USH;
    default: return 0;
    }
}

// A change of register layout inside a sweep: an LDS transpose to any
// layout, or in-wavefront swaps of register-index bits with lane bits 4 and 5
// (v_permlane16/32_swap), which move no data through LDS.
// A few values in place (a tile has at most kTileMaxK bits): planning a small
// circuit is otherwise mostly malloc and free.
template <typename T>
struct Few {
    static constexpr int kMost = 16;
    static_assert(kTileMaxK <= kMost, "a value per tile bit");
    T v[kMost];
    int n = 0;

    Few() = default;
    explicit Few(int count, T x = T()) { assign(count, x); }
    Few(const T *b, const T *e) { while (b != e) push_back(*b++); }
    void assign(int count, T x)
    {
        n = count;
        for (int i = 0; i < n; i++) v[i] = x;
    }
    void push_back(T x) { v[n++] = x; }
    void clear() { n = 0; }
    void erase(T *at)
    {
        std::copy(at + 1, end(), at);
        n--;
    }
    size_t size() const { return (size_t)n; }
    bool empty() const { return n == 0; }
    T *begin() { return v; }
    T *end() { return v + n; }
    const T *begin() const { return v; }
    const T *end() const { return v + n; }
    T &operator[](size_t i) { return v[i]; }
    const T &operator[](size_t i) const { return v[i]; }
    bool operator!=(const Few &o) const { return !std::equal(begin(), end(), o.begin(), o.end()); }
};
using Bits = Few<int>;
using Scores = Few<long>;

struct Change {
    bool lds = true;
    Bits rs;                    // register slot -> local bit after it
    Bits thr;                   // thread-index bit -> local bit after it
    std::vector<std::pair<int, int>> sw;    // (register slot, lane bit), in order
};

void gate_matrix2(const Coef &k, double m[8]);

// Pauli frame of a fast sweep: the registers hold phi, and the state is
// psi = i^w X^x Z^z phi (X^x flips the qubits of x, Z^z negates amplitudes of
// odd parity on z).  Uncontrolled X, Y and Z change only the frame; H, CX and
// CZ run unchanged and carry the frame through (Clifford conjugation); every
// other gate runs conjugated by the frame, which leaves the frame as it is.
// The store applies it (see TileDesc).
struct Frame {
    uint64_t x = 0, z = 0;
    int w = 0;
};

// Coefficients of Z^b X^a G X^a Z^b: gate G seen through a frame with X^a Z^b
// on its target.  Keeps the kind where one covers the result (RX, RY, RZ, U
// under Z; a diagonal stays diagonal), else a general matrix (AK_MAT).
void conj_coef(Coef &k, bool a, bool b)
{
    if (!a && !b) return;
    switch (k.ak) {
    case AK_RX:  // [[c, -is], [-is, c]]: X keeps it, Z negates s
        if (b) k.c[1] = -k.c[1];
        return;
    case AK_RY:  // [[c, -s], [s, c]]: X and Z each negate s
        if (a != b) k.c[0] = -k.c[0];
        return;
    case AK_RZ:
        if (a) {
            std::swap(k.c[0], k.c[2]);
            std::swap(k.c[1], k.c[3]);
        }
        return;
    case AK_PHASE:  // X diag(1, p) X = diag(p, 1)
        if (a) {
            const double pr = k.c[0], pi = k.c[1];
            memset(k.c, 0, sizeof k.c);
            k.ak = AK_RZ;
            k.c[0] = pr; k.c[1] = pi; k.c[2] = 1.0;
        }
        return;
    case AK_NEG:  // X Z X = diag(-1, 1)
        if (a) {
            memset(k.c, 0, sizeof k.c);
            k.ak = AK_RZ;
            k.c[0] = -1.0; k.c[2] = 1.0;
        }
        return;
    case AK_U:  // Z negates the off-diagonal entries; X needs a complex u00
        if (!a) {
            for (int i = 2; i < 6; i++) k.c[i] = -k.c[i];
            return;
        }
        break;
    default:
        break;
    }
    double m[8];
    gate_matrix2(k, m);
    if (a) {  // X G X: rows and columns swapped
        const double r[8] = {m[6], m[7], m[4], m[5], m[2], m[3], m[0], m[1]};
        memcpy(m, r, sizeof r);
    }
    if (b)
        for (int i = 2; i < 6; i++) m[i] = -m[i];
    k.ak = AK_MAT;
    memcpy(k.c, m, sizeof m);
}

// The fast sweeps' rotation and phase forms (shears): a rotation by a, |a| <=
// pi/2, given by (cos a, sin a) with cos a >= 0, becomes (-tan(a/2), sin a).
// RX(theta) and RY(theta) rotate by a = theta/2; a phase e^(ib) (P, and each
// half of a controlled general diagonal) by b.  A larger angle a is a - pi
// and a sign: an uncontrolled RX/RY then runs as -G (sign 1: the caller adds
// a global -1), an uncontrolled P(b) as Z P(b - pi) (sign 2: the caller puts
// a Z on the target after it); a controlled one runs twice at half the angle
// (returns 2).  Other kinds are left as they are (returns 1).
void shear_of(double c, double s, double *k)
{
    k[0] = -s / (1.0 + c);
    k[1] = s;
}

// e^(ia/2), cos >= 0, for e^(ia) = (c, s), a in (-pi, pi]: the larger of
// cos(a/2) and |sin(a/2)| from (1 + c) / 2 or (1 - c) / 2, the other from
// sin a = 2 sin(a/2) cos(a/2), so that neither cancels.
void half_of(double c, double s, double *hc, double *hs)
{
    if (c >= 0.0) {
        const double h = std::sqrt(0.5 * (1.0 + c));
        *hc = h;
        *hs = s / (2.0 * h);
    } else {
        const double q = std::sqrt(0.5 * (1.0 - c));
        *hc = std::fabs(s) / (2.0 * q);
        *hs = std::signbit(s) ? -q : q;
    }
}

int shear_form(Coef &k, bool unc, int *sign)
{
    *sign = 0;
    double c, s;
    switch (k.ak) {
    case AK_RX: c = k.c[0]; s = -k.c[1]; break;
    case AK_RY: c = k.c[1]; s = k.c[0]; break;
    case AK_PHASE: c = k.c[0]; s = k.c[1]; break;
    case AK_RZ: {  // controlled general diagonal: both halves
        double c0 = k.c[0], s0 = k.c[1], c1 = k.c[2], s1 = k.c[3];
        const int reps = (c0 < 0.0 || c1 < 0.0) ? 2 : 1;
        if (reps == 2) {
            half_of(c0, s0, &c0, &s0);
            half_of(c1, s1, &c1, &s1);
        }
        memset(k.c, 0, sizeof k.c);
        shear_of(c0, s0, k.c);
        shear_of(c1, s1, k.c + 2);
        return reps;
    }
    default: return 1;
    }
    int reps = 1;
    if (c < 0.0) {
        if (unc) {
            c = -c;
            s = -s;
            *sign = k.ak == AK_PHASE ? 2 : 1;
        } else {
            half_of(c, s, &c, &s);
            reps = 2;
        }
    }
    memset(k.c, 0, sizeof k.c);
    shear_of(c, s, k.c);
    return reps;
}

// An uncontrolled 2x2 unitary M (U, or a gate the frame turned into a general
// matrix) as e^(i al) P(be) RY(2a) P(de), P(x) = diag(1, e^(ix)): |m00| = cos a,
// |m10| = sin a, a in [0, pi/2], and the phases from whichever entries are
// the larger (so a near-zero sin or cos does not amplify rounding).  For the
// shears both phases must have |angle| <= pi/2: P(de) = Z P(de - pi) and
// Z RY(2a) Z = RY(-2a) turn (be, a, de) into (be + pi, -a, de - pi), and a
// remaining P(be) becomes Z P(be - pi), the Z going on phi after the op
// (*zafter).  k gets AK_USH with (-tan(x/2), sin x) for de, a and be; the
// global phase e^(i al) is returned in (*gr, *gi).
void ush_form(Coef &k, double *gr, double *gi, bool *zafter)
{
    double m[8];
    gate_matrix2(k, m);
    const double ca = std::hypot(m[0], m[1]), sa = std::hypot(m[4], m[5]);
    double ar, ai, br, bi, dr, di;  // e^(i al), e^(i (al + be)), e^(i (al + de))
    if (ca >= sa) {
        ar = m[0] / ca;
        ai = m[1] / ca;
        const double tr = m[6] / ca, ti = m[7] / ca;  // e^(i (al + be + de))
        if (sa > 0.0) {
            br = m[4] / sa;
            bi = m[5] / sa;
        } else {
            br = ar;
            bi = ai;
        }
        const double xr = tr * br + ti * bi, xi = ti * br - tr * bi;  // e^(i de)
        dr = xr * ar - xi * ai;
        di = xr * ai + xi * ar;
    } else {
        br = m[4] / sa;
        bi = m[5] / sa;
        dr = -m[2] / sa;
        di = -m[3] / sa;
        if (ca > 0.0) {
            ar = m[0] / ca;
            ai = m[1] / ca;
        } else {
            ar = 1.0;
            ai = 0.0;
        }
    }
    // e^(i be), e^(i de): the conjugate of e^(i al) taken out
    double ebr = br * ar + bi * ai, ebi = bi * ar - br * ai;
    double edr = dr * ar + di * ai, edi = di * ar - dr * ai;
    double s = sa;
    if (edr < 0.0) {
        edr = -edr;
        edi = -edi;
        ebr = -ebr;
        ebi = -ebi;
        s = -s;
    }
    *zafter = ebr < 0.0;
    if (*zafter) {
        ebr = -ebr;
        ebi = -ebi;
    }
    memset(k.c, 0, sizeof k.c);
    k.ak = AK_USH;
    shear_of(edr, edi, k.c);
    shear_of(ca, s, k.c + 2);
    shear_of(ebr, ebi, k.c + 4);
    *gr = ar;
    *gi = ai;
}

// A stable sort (std::stable_sort allocates).
template <typename Before>
void sort_bits(Bits &v, Before before)
{
    for (size_t i = 1; i < v.size(); i++) {
        const int x = v[i];
        size_t j = i;
        for (; j && before(x, v[j - 1]); j--) v[j] = v[j - 1];
        v[j] = x;
    }
}

struct Planner {
    int n, K, LOGW, RB, klo;
    int improve = 0;  // local-search passes over the tile set (AUTO only)
    bool strict;
    bool fast = false;   // AUTO arithmetic (see launch_tile): H factors carried
    bool swaps = false;  // in-wavefront layout changes when they reach the set
    bool bad = false;
    // Reverse sweeps of the adjoint: every gate runs in a sweep (a single one
    // too), and a sweep takes at most max_grads gates with a gradient.
    int max_grads = 0;
    // Cheap planning (spz_chip.h): every sweep is a tile sweep, the next register
    // bits are simply the best-scored ones.
    bool quick = false;
    // ... and of at most so many gates (0: any number): choosing layouts passes over
    // a sweep's remaining gates at every change, which is quadratic in their
    // number.  Circuits of 8 to 12 qubits are otherwise one sweep: 10000 gates
    // 25 ms and 30000 gates 250 ms a direction, now 6 and 20 ms; a further sweep
    // costs a launch and a pass over the tile, about 10 us for 1024 gates' 500.
    size_t max_gates = 0;
    std::vector<uint32_t> grads;  // the sweeps' gradients, slot by slot
    uint64_t frame_gates = 0;  // gates absorbed into Pauli frames
    uint64_t split_ops = 0;    // second halves of gates run as two half-angle ops
    uint64_t swap_gates = 0;   // SWAPs that a sweep's store carries out
    // The local bits stored to qubits 0..klo-1 by the sweep being built (they end
    // on the low lanes, so that stores are contiguous), and their mask.
    Bits outlow;
    uint32_t outmask = 0;
    std::vector<TileOp> prog;
    std::vector<Sweep> sweeps;

    // What the searches read of a gate, packed (a run's SG records are an order
    // of magnitude larger, and the searches pass over them thousands of times).
    struct Acts {
        uint64_t nd, dm;
    };

    // A gate that a fast sweep absorbs into its frame needs no register slot.
    bool absorbed(const SG &g) const
    {
        return fast && !g.ones && !g.zeros &&
               (g.k.ak == AK_X || g.k.ak == AK_Y || g.k.ak == AK_NEG);
    }
    // Gates that run only with their target on a register bit.
    bool needs_reg(const SG &g) const
    {
        return !g.diag && !absorbed(g) && g.kind != SPZ_SWAP;
    }

    // Choose the tile qubits and the gates of one sweep from `rem` (indices
    // into `run`, in program order).  Returns the chosen gate indices.
    std::vector<int> collect(const std::vector<SG> &run, const std::vector<int> &rem,
                             uint64_t &smask)
    {
        std::vector<int> order;
        order.reserve(std::min<size_t>(rem.size(), 64));
        smask = (klo >= 64) ? ~0ull : ((1ull << klo) - 1);
        int free_slots = K - klo;
        uint64_t bnd = 0, bd = 0;
        const uint64_t all = n >= 64 ? ~0ull : ((1ull << n) - 1);
        for (int idx : rem) {
            const SG &g = run[idx];
            bool ok = !(g.nd & (bnd | bd)) && !(g.dm & bnd);
            const int more = __builtin_popcountll(g.nd & ~smask);
            if (ok && more) {
                if (free_slots >= more) {
                    smask |= g.nd;
                    free_slots -= more;
                } else {
                    ok = false;
                }
            }
            if (ok) {
                order.push_back(idx);
                if (order.size() == max_gates) break;
            } else {
                if (strict) break;
                bnd |= g.nd;
                bd |= g.dm;
                if ((bnd & all) == all) break;
            }
        }
        for (int q = 0; q < n && __builtin_popcountll(smask) < K; q++) smask |= 1ull << q;
        if (!strict && improve > 0 && n > K) improve_set(run, rem, smask, order);
        return order;
    }

    // Gates of `rem` that one sweep over the fixed tile set `smask` can take
    // (program order, skipping past blocked gates); stops once every tile
    // qubit is blocked.  With `out`, also lists them.
    static size_t take_fixed(const std::vector<Acts> &acts, const std::vector<int> &rem,
                             uint64_t smask, std::vector<int> *out)
    {
        uint64_t bnd = 0, bd = 0;
        size_t cnt = 0;
        for (size_t i = 0; i < rem.size(); i++) {
            const Acts &g = acts[i];
            if (!(g.nd & (bnd | bd)) && !(g.dm & bnd) && !(g.nd & ~smask)) {
                cnt++;
                if (out) out->push_back(rem[i]);
            } else {
                bnd |= g.nd;
                bd |= g.dm;
                if ((bnd & smask) == smask) break;
            }
        }
        return cnt;
    }

    static std::vector<Acts> acts_of(const std::vector<SG> &run, const std::vector<int> &rem)
    {
        std::vector<Acts> acts(rem.size());
        for (size_t i = 0; i < rem.size(); i++) acts[i] = {run[rem[i]].nd, run[rem[i]].dm};
        return acts;
    }

    // Local search over the tile set: swap a free tile qubit for a qubit that
    // the next gates target, keep the first swap that lets the sweep take more
    // gates, repeat.  The low klo qubits stay (they make the tile rows contiguous).
    void improve_set(const std::vector<SG> &run, const std::vector<int> &rem, uint64_t &smask,
                     std::vector<int> &order) const
    {
        const uint64_t fixed = (klo >= 64) ? ~0ull : ((1ull << klo) - 1);
        uint64_t cand = 0;  // non-diagonal targets among the next gates
        size_t seen = 0;
        for (int idx : rem) {
            cand |= run[idx].nd;
            if (++seen >= 4 * (size_t)n * 8) break;
        }
        cand &= ~fixed;
        const std::vector<Acts> acts = acts_of(run, rem);
        size_t best = order.size();
        bool moved = false;
        for (int pass = 0; pass < improve; pass++) {
            bool better = false;
            for (int a = 0; a < n && !better; a++) {
                if (!((smask >> a) & 1) || ((fixed >> a) & 1)) continue;
                for (int b = 0; b < n && !better; b++) {
                    if (((smask >> b) & 1) || !((cand >> b) & 1)) continue;
                    const uint64_t m2 = (smask & ~(1ull << a)) | (1ull << b);
                    const size_t c2 = take_fixed(acts, rem, m2, nullptr);
                    if (c2 > best) {
                        best = c2;
                        smask = m2;
                        better = moved = true;
                    }
                }
            }
            if (!better) break;
        }
        if (moved) {
            order.clear();
            take_fixed(acts, rem, smask, &order);
        }
    }

    // Passes a greedy plan of `rem` would make: one per sweep, one half per
    // gate left to the plain path.
    double tail_cost(const std::vector<SG> &run, std::vector<int> rem)
    {
        double cost = 0.0;
        while (!rem.empty()) {
            uint64_t sm;
            const std::vector<int> ord = collect(run, rem, sm);
            if (ord.size() < 2) {
                cost += 0.5;
                rem.erase(rem.begin());
                continue;
            }
            cost += 1.0;
            rem = minus(rem, ord);
        }
        return cost;
    }

    // rem without the gates of ord (ord: a subsequence of rem).
    static std::vector<int> minus(const std::vector<int> &rem, const std::vector<int> &ord)
    {
        std::vector<int> out;
        if (ord.size() == rem.size()) return out;
        out.reserve(rem.size() - ord.size());
        size_t k = 0;
        for (int idx : rem) {
            if (k < ord.size() && ord[k] == idx) { k++; continue; }
            out.push_back(idx);
        }
        return out;
    }

    // End of a run: a greedy plan can leave one gate that no sweep takes, a
    // whole plain pass for one gate.  When about one sweep's worth of gates
    // remains after this sweep and its plan would end that way, the tile sets
    // one swap away from this sweep's are tried, and one whose remainder
    // plans in fewer passes is kept.  Only for states of 2^28 amplitudes and
    // more, where a pass takes milliseconds and this search overlaps the
    // sweeps already queued.
    void endgame(const std::vector<SG> &run, const std::vector<int> &rem, uint64_t &smask,
                 std::vector<int> &order)
    {
        if (strict || improve <= 0 || n < 28 || n <= K) return;
        if (order.size() >= rem.size() || rem.size() - order.size() > order.size()) return;
        const double base = tail_cost(run, minus(rem, order));
        if (base == std::floor(base)) return;  // no plain gate in the tail
        const uint64_t fixed = (klo >= 64) ? ~0ull : ((1ull << klo) - 1);
        uint64_t cand = 0;
        for (int idx : rem) cand |= run[idx].nd;
        cand &= ~fixed;
        const std::vector<Acts> acts = acts_of(run, rem);
        double best = base;
        uint64_t bm = smask;
        std::vector<int> bo;
        for (int a = 0; a < n; a++) {
            if (!((smask >> a) & 1) || ((fixed >> a) & 1)) continue;
            for (int b = 0; b < n; b++) {
                if (((smask >> b) & 1) || !((cand >> b) & 1)) continue;
                const uint64_t m2 = (smask & ~(1ull << a)) | (1ull << b);
                std::vector<int> o2;
                take_fixed(acts, rem, m2, &o2);
                if (o2.size() < 2) continue;
                const double c = tail_cost(run, minus(rem, o2));
                if (c < best) {
                    best = c;
                    bm = m2;
                    bo.swap(o2);
                }
            }
        }
        if (best < base) {
            smask = bm;
            order.swap(bo);
        }
    }

    void emit_layout(const Bits &oldRS, const Bits &RSv,
                     const Bits &thr)
    {
        TileOp op;
        memset(&op, 0, sizeof op);
        op.type = TOP_LAYOUT;
        op.grp = TG_LAYOUT;
        op.eo = 1;  // em = 0: never taken for a gate
        for (int j = 0; j < RB; j++) {
            op.lay.oldreg[j] = (int8_t)oldRS[j];
            op.lay.newreg[j] = (int8_t)RSv[j];
            op.lay.rob[j] = tile_swz(1u << oldRS[j]) << 3;
            op.lay.rnb[j] = tile_swz(1u << RSv[j]) << 3;
        }
        for (int i = 0; i < LOGW; i++) op.lay.newthr[i] = (int8_t)thr[i];
        prog.push_back(op);
    }

    // Register slot j trades its local bit with the one on lane bit tb (4 or 5).
    void emit_swap(int j, int tb, int reg_bit, int lane_bit)
    {
        TileOp op;
        memset(&op, 0, sizeof op);
        op.type = TOP_LAYOUT;
        op.grp = tb == 5 ? TG_SW32 : TG_SW16;
        op.eo = 1;  // never taken for a gate
        op.sel = 1u << j;
        op.mlo = 1u << lane_bit;  // leaves the lane part
        op.mlz = 1u << reg_bit;   // enters it
        prog.push_back(op);
    }

    // Thread layout after an LDS change to register bits rs: lane bits 4 and
    // 5 take the two best-scored free bits (the next register candidates, so
    // that later changes can be swaps); the other free bits fill the thread
    // bits in ascending order, after those that are stored to the low qubits.
    // (lo: bits below it may not go to lanes 4, 5, used for the load layout,
    // whose lanes 0..klo-1 must hold the low bits.)
    Bits thread_layout(const Bits &rs, const Scores *score,
                                   int lo) const
    {
        Bits avail;
        for (int b = 0; b < K; b++)
            if (std::find(rs.begin(), rs.end(), b) == rs.end()) avail.push_back(b);
        Bits thr(LOGW, -1);
        if (swaps && LOGW >= 6 && score) {
            Bits cand;
            for (int b : avail)
                if (b >= lo && (*score)[b] > 0) cand.push_back(b);
            sort_bits(cand, [&](int x, int y) { return (*score)[x] > (*score)[y]; });
            for (int i = 0; i < 2 && i < (int)cand.size(); i++) {
                thr[4 + i] = cand[i];
                avail.erase(std::find(avail.begin(), avail.end(), cand[i]));
            }
        }
        if (!lo)
            sort_bits(avail, [&](int x, int y) {
                return std::find(outlow.begin(), outlow.end(), x) <
                       std::find(outlow.begin(), outlow.end(), y);
            });
        size_t a = 0;
        for (int i = 0; i < LOGW; i++)
            if (thr[i] < 0) thr[i] = avail[a++];
        return thr;
    }

    // Swaps that turn register set rs (slots) into one holding exactly the
    // bits of `want`, if every missing bit sits on lane bit 4 or 5.
    bool swap_path(const Bits &rs, const Bits &thr,
                   const Bits &want, std::vector<std::pair<int, int>> *sw) const
    {
        if (!swaps || LOGW < 6) return false;
        Bits in, out;
        for (int b : want)
            if (std::find(rs.begin(), rs.end(), b) == rs.end()) in.push_back(b);
        for (int j = 0; j < RB; j++)
            if (std::find(want.begin(), want.end(), rs[j]) == want.end()) out.push_back(j);
        if (in.size() != out.size() || in.size() > 2) return false;
        for (size_t i = 0; i < in.size(); i++) {
            const int tb = thr[4] == in[i] ? 4 : thr[5] == in[i] ? 5 : -1;
            if (tb < 0) return false;
            if (sw) sw->push_back({out[i], tb});
        }
        return true;
    }

    void apply_swaps(Bits &rs, Bits &thr,
                     const std::vector<std::pair<int, int>> &sw) const
    {
        for (auto [j, tb] : sw) std::swap(rs[j], thr[tb]);
    }

    // A gate still to run in the sweep: what it acts on, and the local bit that
    // must be in a register for it (0: none).  Gates keep their program order,
    // so one forward pass with masks of what the passed-over gates act on
    // decides everything a dependency graph would: a gate waits for an earlier
    // one when they share a qubit on which at least one acts non-diagonally.
    struct Todo {
        uint64_t nd, dm;
        uint32_t need;
        int at;  // index into `order`
    };

    // Gates that run under register bits rs before the others are stuck (or
    // fewer, once it is certain that they are fewer than `least`).  `all`: the
    // qubits the gates act on.
    static int runs_under(const std::vector<Todo> &todo, uint32_t rs, uint64_t all, int least)
    {
        uint64_t bnd = 0, bd = 0;
        int cnt = 0, spare = (int)todo.size() - least;
        for (const Todo &g : todo) {
            if (!(g.nd & (bnd | bd)) && !(g.dm & bnd) && !(g.need & ~rs)) {
                cnt++;
            } else {
                bnd |= g.nd;
                bd |= g.dm;
                if (--spare < 0 || bnd == all) break;
            }
        }
        return cnt;
    }

    // Register targets still to run, weighted by readiness: a ready gate counts
    // for more than all the waiting ones together, so that the best-scored bit
    // always has a ready gate (a gate that waits never outranks what it waits for).
    void pair_score(const std::vector<Todo> &todo, Scores &score) const
    {
        const long ready_weight = std::max<long>(1000, (long)todo.size() + 1);
        score.assign(K, 0);
        uint64_t bnd = 0, bd = 0;
        for (const Todo &g : todo) {
            if (g.need) {
                const bool ready = !(g.nd & (bnd | bd)) && !(g.dm & bnd);
                score[__builtin_ctz(g.need)] += ready ? ready_weight : 1;
            }
            bnd |= g.nd;
            bd |= g.dm;
        }
    }

    // The RB register bits (from `lo` up) to switch to: every RB-subset of
    // the (up to 8) best-scored bits is tried, and the one under which the
    // most gates run wins (ties: the higher score, then the earlier subset).
    // With a current layout (cur_rs, cur_thr), a set reachable by in-wavefront
    // swaps is charged less than one that needs an LDS transpose (in gates
    // that could have run: a transpose costs about four gates, a swap about
    // half of one).
    Bits best_set(const std::vector<Todo> &todo, const Scores &score, int lo,
                              const Bits *cur_rs = nullptr,
                              const Bits *cur_thr = nullptr) const
    {
        const int left = (int)todo.size();
        Bits bits;
        for (int b = lo; b < K; b++) bits.push_back(b);
        sort_bits(bits, [&](int x, int y) { return score[x] > score[y]; });
        if (quick) {
            Bits out(bits.begin(), bits.begin() + RB);
            std::sort(out.begin(), out.end());
            return out;
        }
        const int T = std::min((int)bits.size(), std::max(RB, 8));
        uint32_t best = 0;
        double best_val = -1e30;
        long best_sc = -1;
        uint64_t all = 0;
        for (const Todo &g : todo) all |= g.nd | g.dm;
        Bits want;
        std::vector<std::pair<int, int>> sw;
        for (uint32_t sub = 0; sub < (1u << T); sub++) {
            if (__builtin_popcount(sub) != RB) continue;
            uint32_t rs = 0;
            long sc = 0;
            for (int i = 0; i < T; i++)
                if ((sub >> i) & 1) {
                    rs |= 1u << bits[i];
                    sc += score[bits[i]];
                }
            // (a count whose value would stay below best_val cannot win: at
            // most 1 is added to it, and without swaps 4 are taken off)
            int cnt = runs_under(todo, rs, all,
                                 (int)std::max(0.0, best_val + (cur_rs && !swaps ? 3.0 : -1.0)));
            // a set that finishes the sweep and keeps the low bits on lanes
            // saves the change back before the store
            if (cnt == left && !(rs & outmask)) cnt++;
            // a set under which nothing runs makes no progress
            if (cnt == 0) continue;
            double val = cnt;
            if (cur_rs && cur_thr) {
                bool swap = false;
                if (swaps) {
                    want.clear();
                    sw.clear();
                    for (int i = 0; i < T; i++)
                        if ((sub >> i) & 1) want.push_back(bits[i]);
                    swap = swap_path(*cur_rs, *cur_thr, want, &sw);
                }
                val -= swap ? 0.5 * (double)sw.size() : 4.0;
            }
            if (val > best_val || (val == best_val && sc > best_sc)) {
                best = rs;
                best_val = val;
                best_sc = sc;
            }
        }
        Bits out;
        if (best_val == -1e30) {
            // nothing runs under any candidate: possible only for the load
            // layout, where every ready target may be a low bit (from lo = 0 the
            // best-scored bit has a ready gate); take the top bits
            for (int i = 0; i < RB && i < (int)bits.size(); i++) out.push_back(bits[i]);
            std::sort(out.begin(), out.end());
            return out;
        }
        for (int b = 0; b < K; b++)
            if ((best >> b) & 1) out.push_back(b);
        return out;
    }

    // Sequence the sweep's gates: the scheduled order itself (strict), or,
    // with reordering allowed, a topological order of the dependency graph
    // that applies every gate the current register layout allows before
    // switching layouts.  Entries >= 0 are gates; -1 marks "apply the next
    // entry of `changes`".  rs_in / thr_in receive the load layout: register
    // bits never among the klo low local bits, which stay on the low lane bits
    // for contiguous loads (with reordering allowed, the register bits with
    // the most ready pair gates, and lane bits 4 and 5 holding the next
    // best-scored bits).
    void sequence(const std::vector<SG> &run, const std::vector<int> &order, const int *lbit,
                  std::vector<int> &seq, std::vector<Change> &changes, Bits &rs_in,
                  Bits &thr_in)
    {
        const int m = (int)order.size();
        seq.reserve(m + m / 2 + 8);
        Bits RS(RB);
        for (int j = 0; j < RB; j++) RS[j] = LOGW + j;
        auto in_rs = [&](int b) {
            for (int j = 0; j < RB; j++)
                if (RS[j] == b) return true;
            return false;
        };
        std::vector<Todo> todo(m);
        for (int a = 0; a < m; a++) {
            const SG &g = run[order[a]];
            todo[a] = {g.nd, g.dm, needs_reg(g) ? 1u << lbit[g.target] : 0u, a};
        }
        Scores score0;
        pair_score(todo, score0);
        if (!strict && K - klo >= RB) RS = best_set(todo, score0, klo);
        Bits THR = thread_layout(RS, &score0, klo);
        rs_in = RS;
        thr_in = THR;
        // move to register bits `nx` (slot order as given): swaps when they
        // reach it, else an LDS transpose whose lane bits 4, 5 get the
        // best-scored free bits
        auto change_to = [&](const Bits &nx, const Scores &score) {
            Change ch;
            if (swap_path(RS, THR, nx, &ch.sw)) {
                ch.lds = false;
                apply_swaps(RS, THR, ch.sw);
            } else {
                // keep bits that stay in place in their old slots
                Bits slotted(RB, -1);
                for (int j = 0; j < RB; j++)
                    if (std::find(nx.begin(), nx.end(), RS[j]) != nx.end()) slotted[j] = RS[j];
                for (int b : nx) {
                    if (std::find(slotted.begin(), slotted.end(), b) != slotted.end()) continue;
                    for (int j = 0; j < RB; j++)
                        if (slotted[j] < 0) { slotted[j] = b; break; }
                }
                RS = slotted;
                THR = thread_layout(RS, &score, 0);
            }
            ch.rs = RS;
            ch.thr = THR;
            seq.push_back(-1);
            changes.push_back(ch);
        };
        if (strict) {
            for (int pos = 0; pos < m; pos++) {
                const SG &g = run[order[pos]];
                if (!g.diag && !in_rs(lbit[g.target])) {
                    Bits nx;
                    Scores score(K, 0);
                    for (int p2 = pos; p2 < m; p2++) {
                        // (scores only place lanes 4 and 5, for swaps)
                        if (!swaps && (int)nx.size() == RB) break;
                        const SG &h = run[order[p2]];
                        if (h.diag) continue;
                        int hb = lbit[h.target];
                        score[hb] += std::max(1, 64 - (p2 - pos));
                        if ((int)nx.size() < RB && std::find(nx.begin(), nx.end(), hb) == nx.end())
                            nx.push_back(hb);
                    }
                    for (int j = 0; j < RB && (int)nx.size() < RB; j++)
                        if (std::find(nx.begin(), nx.end(), RS[j]) == nx.end()) nx.push_back(RS[j]);
                    for (int bb = 0; bb < K && (int)nx.size() < RB; bb++)
                        if (std::find(nx.begin(), nx.end(), bb) == nx.end()) nx.push_back(bb);
                    change_to(nx, score);
                }
                seq.push_back(order[pos]);
            }
            // a first LDS change ahead of every gate that keeps the low bits
            // on lanes becomes the load layout
            if (!seq.empty() && seq[0] == -1 && changes[0].lds) {
                bool low = false;
                for (int b : changes[0].rs) low |= b < klo;
                for (int i = 0; i < klo && i < LOGW; i++) low |= changes[0].thr[i] != i;
                if (!low) {
                    rs_in = changes[0].rs;
                    thr_in = changes[0].thr;
                    seq.erase(seq.begin());
                    changes.erase(changes.begin());
                }
            }
            return;
        }
        std::vector<Todo> stuck;
        Scores score;
        stuck.reserve(m);
        for (;;) {
            // every gate that runs under the current register bits, in order
            uint32_t rs = 0;
            for (int j = 0; j < RB; j++) rs |= 1u << RS[j];
            uint64_t bnd = 0, bd = 0;
            stuck.clear();
            for (const Todo &g : todo) {
                if (!(g.nd & (bnd | bd)) && !(g.dm & bnd) && !(g.need & ~rs)) {
                    seq.push_back(order[g.at]);
                } else {
                    stuck.push_back(g);
                    bnd |= g.nd;
                    bd |= g.dm;
                }
            }
            todo.swap(stuck);
            if (todo.empty()) break;
            // next layout: score target bits of the remaining non-diagonal
            // gates, ready ones first; among the RB-subsets of the best
            // scored bits, take the one under which the most gates run
            // before the next change, less the cost of reaching it
            pair_score(todo, score);
            Bits nx = best_set(todo, score, 0, &RS, &THR);
            change_to(nx, score);
            if ((int)changes.size() > 2 * m + 8) {  // every change runs a gate: cannot happen
                bad = true;
                return;
            }
        }
    }

    // SWAPs move nothing inside a sweep: the gates after one act on the other
    // one of its qubits, and the store puts every local bit where the SWAPs send
    // it (phys[q]: the qubit that holds what is stored to q).  A SWAP by itself
    // is a pass over half the state, or all of it where a low qubit is in it.
    // Fourier transforms, with the SWAPs at the end as passes and in sweeps: 14
    // qubits 113 -> 87 us, 20 qubits 223 -> 187 us, 25 qubits 2.82 -> 1.63 ms, 28
    // qubits 25.0 -> 14.8 ms.
    void relabel(const std::vector<SG> &run, const std::vector<int> &order, int *phys,
                 std::vector<SG> &out)
    {
        auto moved = [&](uint64_t m) {
            uint64_t r = 0;
            for (; m; m &= m - 1) r |= 1ull << phys[__builtin_ctzll(m)];
            return r;
        };
        for (int gi : order) {
            SG g = run[gi];
            if (g.kind == SPZ_SWAP) {
                std::swap(phys[g.target], phys[g.t1]);
                swap_gates++;
                continue;
            }
            g.target = phys[g.target];
            g.ones = moved(g.ones);
            g.zeros = moved(g.zeros);
            g.nd = moved(g.nd);
            g.dm = moved(g.dm);
            out.push_back(g);
        }
    }

    void build(const std::vector<SG> &all, const std::vector<int> &chosen, uint64_t smask)
    {
        int phys[64];
        for (int q = 0; q < 64; q++) phys[q] = q;
        bool swapped = false;
        for (int gi : chosen) swapped |= all[gi].kind == SPZ_SWAP;
        std::vector<SG> relabelled;
        std::vector<int> kept;
        if (swapped) {
            relabel(all, chosen, phys, relabelled);
            kept.resize(relabelled.size());
            for (size_t i = 0; i < kept.size(); i++) kept[i] = (int)i;
        }
        const std::vector<SG> &run = swapped ? relabelled : all;
        const std::vector<int> &order = swapped ? kept : chosen;
        Sweep sw;
        memset(&sw.desc, 0, sizeof sw.desc);
        sw.tile = true;
        sw.gate = -1;
        sw.can_carry = false;
        sw.carry_z = 0;
        sw.carry_w = 0;
        int lbit[64];
        for (int q = 0; q < 64; q++) lbit[q] = -1;
        int i = 0;
        for (int q = 0; q < n; q++)
            if ((smask >> q) & 1) {
                sw.desc.spos[i] = (int8_t)q;
                lbit[q] = i++;
            }
        for (; i < 16; i++) sw.desc.spos[i] = 64;
        memcpy(sw.desc.sout, sw.desc.spos, sizeof sw.desc.sout);
        outlow.clear();
        outmask = 0;
        for (int q = 0; q < n; q++) {
            if (lbit[q] < 0) continue;
            sw.desc.sout[lbit[phys[q]]] = (int8_t)q;
            if (q < klo) {
                outlow.push_back(lbit[phys[q]]);
                outmask |= 1u << lbit[phys[q]];
            }
        }
        sw.op_begin = prog.size();
        sw.slot_begin = grads.size();
        std::vector<int> seq;
        Bits RS, THR;
        std::vector<Change> changes;
        sequence(run, order, lbit, seq, changes, RS, THR);
        // load layout: register bits RS, thread bits THR
        auto reg_offsets = [&](const Bits &rs, const int8_t *qubit, uint64_t *out) {
            for (int p = 0; p < (1 << RB); p++) {
                uint64_t g = 0;
                for (int j = 0; j < RB; j++)
                    if ((p >> j) & 1) g |= 1ull << qubit[rs[j]];
                out[p] = g;
            }
        };
        reg_offsets(RS, sw.desc.spos, sw.desc.gr);
        for (int t = 0; t < LOGW; t++) {
            sw.desc.tin[t] = (int8_t)THR[t];
            sw.desc.tg[t] = 1ull << sw.desc.spos[THR[t]];
        }
        // fast sweeps: uncontrolled H ops leave out their 1/sqrt(2) and
        // uncontrolled diagonals their phase on |0>; both go into one global
        // factor (gre, gim) that the store applies
        size_t hdebt = 0;
        double gre = 1.0, gim = 0.0;
        Frame fr;
        // Consecutive fast sweeps: the previous one stores with only the X
        // part of its frame applied, and this one starts from the rest (its Z
        // part and phase), so the sign work at the store is done once, by
        // the last tile sweep before a plain pass or the end of the run.
        if (fast && !sweeps.empty() && sweeps.back().tile && sweeps.back().can_carry) {
            Sweep &pv = sweeps.back();
            pv.desc.fzl = 0;
            pv.desc.fzr = 0;
            pv.desc.fzg = 0;
            pv.desc.fflags &= ~(TF_SIGN | TF_ODD);
            fr.z = pv.carry_z;
            fr.w = pv.carry_w;
        }
        size_t li_next = 0;
        for (int gi : seq) {
            if (gi < 0) {
                const Change &ch = changes[li_next++];
                if (ch.lds) {
                    if (ch.rs != RS || ch.thr != THR) emit_layout(RS, ch.rs, ch.thr);
                } else {
                    for (auto [j, tb] : ch.sw) {
                        emit_swap(j, tb, RS[j], THR[tb]);
                        std::swap(RS[j], THR[tb]);
                    }
                }
                RS = ch.rs;
                THR = ch.thr;
                continue;
            }
            SG g = run[gi];
            // Pauli frame (fast sweeps): Paulis are absorbed, H / CX / CZ carry
            // the frame (updated below, once the op is out), other gates are
            // conjugated
            enum { KEEP, PUSH_H, PUSH_CX, PUSH_CZ } push = KEEP;
            const uint64_t tb = 1ull << g.target;
            const bool fa = (fr.x & tb) != 0, fb = (fr.z & tb) != 0;
            if (fast) {
                const bool unc = !g.ones && !g.zeros;
                const bool one_ctrl = !g.zeros && g.ones && !(g.ones & (g.ones - 1));
                if (absorbed(g)) {
                    if (g.k.ak == AK_X) {
                        fr.x ^= tb;
                    } else if (g.k.ak == AK_Y) {  // Y = i X Z
                        fr.w += 1 + 2 * fa;
                        fr.x ^= tb;
                        fr.z ^= tb;
                    } else {  // Z
                        fr.w += 2 * fa;
                        fr.z ^= tb;
                    }
                    frame_gates++;
                    continue;
                }
                if (unc && g.k.ak == AK_H) {
                    push = PUSH_H;
                } else if (one_ctrl && g.k.ak == AK_X) {
                    push = PUSH_CX;
                } else if (one_ctrl && g.k.ak == AK_NEG) {
                    push = PUSH_CZ;
                } else {
                    // an X in the frame on a control inverts the condition
                    const uint64_t fl = (g.ones | g.zeros) & fr.x;
                    const uint64_t o2 = (g.ones & ~fl) | (g.zeros & fl);
                    g.zeros = (g.zeros & ~fl) | (g.ones & fl);
                    g.ones = o2;
                    conj_coef(g.k, fa, fb);
                }
            }
            // fast arithmetic: rotations and phases as shears (see
            // shear_form); a controlled one beyond pi/2 runs as two halves
            bool zafter = false;
            int reps = 1;
            if (fast) {
                const bool unc = !g.ones && !g.zeros;
                if (g.k.ak == AK_RZ && unc) {  // d0 to the global factor, d1/d0 on |1>
                    const double d0r = g.k.c[0], d0i = g.k.c[1], d1r = g.k.c[2], d1i = g.k.c[3];
                    const double t = gre * d0r - gim * d0i;
                    gim = gre * d0i + gim * d0r;
                    gre = t;
                    memset(g.k.c, 0, sizeof g.k.c);
                    g.k.ak = AK_PHASE;
                    g.k.c[0] = d1r * d0r + d1i * d0i;
                    g.k.c[1] = d1i * d0r - d1r * d0i;
                }
                if (unc && (g.k.ak == AK_U || g.k.ak == AK_MAT)) {
                    double pr, pi;
                    ush_form(g.k, &pr, &pi, &zafter);
                    const double t = gre * pr - gim * pi;
                    gim = gre * pi + gim * pr;
                    gre = t;
                }
                int sign = 0;
                reps = shear_form(g.k, unc, &sign);
                if (sign == 1) fr.w += 2;     // the op ran as -G: a global -1
                if (sign == 2) zafter = true; // P ran as Z P: Z on phi (after it)
                split_ops += reps - 1;
            }
            for (int rep = 0; rep < reps; rep++) {  // (a split gate: two equal halves)
                TileOp op;
                memset(&op, 0, sizeof op);
                op.ak = g.k.ak;
                for (int j = 0; j < 8; j++) op.c[j] = g.k.c[j];
                const bool uncontrolled = !g.ones && !g.zeros;
                auto slot_of = [&](int b) {
                    for (int j = 0; j < RB; j++)
                        if (RS[j] == b) return j;
                    return -1;
                };
                uint32_t mro = 0, mrz = 0;  // controls on register-index bits (read 1 / 0)
                for (uint64_t ctl = g.ones | g.zeros; ctl; ctl &= ctl - 1) {
                    const int q = __builtin_ctzll(ctl);
                    const bool one = (g.ones >> q) & 1;
                    const int b = lbit[q];
                    if (b < 0) {
                        if (one) op.eo |= 1ull << q;
                        op.em |= 1ull << q;
                        continue;
                    }
                    const int j = slot_of(b);
                    if (j >= 0) {
                        if (one) mro |= 1u << j; else mrz |= 1u << j;
                    } else {
                        if (one) op.mlo |= 1u << b; else op.mlz |= 1u << b;
                    }
                }
                for (uint32_t p = 0; p < (1u << RB); p++)
                    if ((p & mro) == mro && !(p & mrz)) op.pm |= 1u << p;
                const bool pred = (mro | mrz | op.mlo | op.mlz) != 0;
                const uint32_t kbit = kind_bit(op.ak);
                if (!kbit) {
                    bad = true;
                    return;
                }
                op.grp = TG_GATE | kbit;
                if (fast && g.k.ak == AK_H) {
                    if (uncontrolled) hdebt++;
                    else op.grp = (op.grp & ~TG_H) | TG_HS;  // applies its own factor
                }
                if (g.diag) {
                    op.type = TOP_DIAG;
                    const int b = lbit[g.target];
                    if (b < 0) {
                        op.dsel = 2;
                        op.ebit = 1ull << g.target;
                        op.grp |= pred ? TG_DLANEP : TG_DLANE;
                    } else if (slot_of(b) >= 0) {
                        op.dsel = 0;
                        op.dpos = slot_of(b);
                        op.sel = 1u << op.dpos;
                        op.grp |= pred ? TG_DREGP : TG_DREG;
                    } else {
                        op.dsel = 1;
                        op.dpos = b;
                        op.grp |= pred ? TG_DLANEP : TG_DLANE;
                    }
                } else {
                    op.type = TOP_PAIR;
                    const int slot = slot_of(lbit[g.target]);
                    if (slot < 0) {  // sequence() switches layouts before such a gate
                        bad = true;
                        return;
                    }
                    op.sel = 1u << slot;
                    op.grp |= pred ? TG_PAIRP : TG_PAIR;
                }
                if (g.grad >= 0) {
                    grads.push_back((uint32_t)g.grad);
                    op.pad = (uint32_t)(grads.size() - sw.slot_begin);
                }
                prog.push_back(op);
            }
            if (zafter) fr.z ^= tb;  // (on phi: the frame takes it on its right)
            if (push == PUSH_H) {  // H X^a Z^b = (-1)^(ab) X^b Z^a H
                fr.x = (fr.x & ~tb) | (fb ? tb : 0);
                fr.z = (fr.z & ~tb) | (fa ? tb : 0);
                fr.w += 2 * (fa && fb);
            } else if (push == PUSH_CX) {  // X_c -> X_c X_t, Z_t -> Z_c Z_t
                const uint64_t cb = g.ones;
                if (fr.x & cb) fr.x ^= tb;
                if (fb) fr.z ^= cb;
            } else if (push == PUSH_CZ) {  // X_c -> X_c Z_t, X_t -> Z_c X_t
                const uint64_t cb = g.ones;
                const bool xc = (fr.x & cb) != 0;
                fr.w += 2 * (xc && fa);
                if (xc) fr.z ^= tb;
                if (fa) fr.z ^= cb;
            }
        }
        if (fast) {
            const double f = (hdebt & 1) ? std::ldexp(0.70710678118654752440, -(int)(hdebt / 2))
                                         : std::ldexp(1.0, -(int)(hdebt / 2));
            gre *= f;
            gim *= f;
            if (gre != 1.0 || gim != 0.0) {
                sw.desc.gre = gre;
                sw.desc.gim = gim;
                sw.desc.fflags |= TF_PHASE;
            }
        }
        // store layout: the last one, unless it holds a low bit in registers
        // (then those register bits are swapped for unused high bits) or the
        // low lane bits do not hold the low local bits in order
        {
            Bits st = RS;
            uint32_t used = 0;
            for (int b : RS) used |= 1u << b;
            int nb = K - 1;
            for (int j = 0; j < RB; j++) {
                if (!((outmask >> st[j]) & 1)) continue;
                while (nb >= 0 && (((used | outmask) >> nb) & 1)) nb--;
                if (nb < 0) {  // too few other bits: the top RB local bits
                    for (int i = 0; i < RB; i++) st[i] = LOGW + i;
                    break;
                }
                st[j] = nb;
                used |= 1u << nb;
            }
            bool lanes_ok = true;
            for (int i = 0; i < (int)outlow.size() && i < LOGW; i++) lanes_ok &= THR[i] == outlow[i];
            if (st != RS || !lanes_ok) emit_layout(RS, st, thread_layout(st, nullptr, 0));
            reg_offsets(st, sw.desc.sout, sw.desc.gs);
            // the frame, split by where the store layout holds each bit
            if (fr.x & ~smask) {  // frames only flip qubits the sweep targets
                bad = true;
                return;
            }
            uint32_t xl = 0, zl = 0, regm = 0;
            for (int q = 0; q < n; q++) {
                if (lbit[q] < 0) continue;
                if ((fr.x >> q) & 1) xl |= 1u << lbit[q];
                if ((fr.z >> q) & 1) zl |= 1u << lbit[q];
            }
            uint64_t xg = 0;
            for (int j = 0; j < RB; j++) {
                regm |= 1u << st[j];
                if ((xl >> st[j]) & 1) xg |= 1ull << sw.desc.sout[st[j]];
            }
            for (int p = 0; p < (1 << RB); p++) sw.desc.gs[p] ^= xg;
            uint32_t fzr = 0;
            for (int p = 0; p < (1 << RB); p++) {
                uint32_t par = 0;
                for (int j = 0; j < RB; j++) par ^= ((p >> j) & 1) & ((zl >> st[j]) & 1);
                fzr |= par << p;
            }
            const int w = fr.w & 3;
            if (w & 2) fzr ^= (1u << (1 << RB)) - 1;
            sw.desc.fxl = xl & ~regm;
            sw.desc.fzl = zl & ~regm;
            sw.desc.fzr = fzr;
            sw.desc.fzg = fr.z & ~smask;
            if (sw.desc.fzl || sw.desc.fzr || sw.desc.fzg) sw.desc.fflags |= TF_SIGN;
            if (w & 1) sw.desc.fflags |= TF_SIGN | TF_ODD;
            // Without an LDS layout change nothing orders one wavefront's loads
            // before another's stores: where amplitudes are not stored to the
            // place their thread loaded, the kernel waits for all loads first.
            bool lds = false, moved = xl != 0 || swapped;
            for (size_t o = sw.op_begin; o < prog.size(); o++) {
                lds |= (prog[o].grp & TG_LAYOUT) != 0;
                moved |= (prog[o].grp & (TG_SW16 | TG_SW32)) != 0;
            }
            if (moved && !lds) sw.desc.fflags |= TF_SYNC;
            // what a next sweep takes over if this one stores X^x phi only:
            // i^w X^x Z^z = i^(w + 2 |x & z|) Z^z X^x
            sw.can_carry = fast;
            sw.carry_z = 0;
            for (int q = 0; q < n; q++) sw.carry_z |= ((fr.z >> phys[q]) & 1ull) << q;
            sw.carry_w = (fr.w + 2 * __builtin_popcountll(fr.x & fr.z)) & 3;
        }
        sw.op_count = prog.size() - sw.op_begin;
        sw.slots = (int)(grads.size() - sw.slot_begin);
        sw.desc.nops = (int32_t)sw.op_count;
        sweeps.push_back(sw);
    }

    void plan(const std::vector<SG> &run)
    {
        std::vector<int> rem(run.size());
        for (size_t i = 0; i < run.size(); i++) rem[i] = (int)i;
        prog.reserve(run.size() + run.size() / 4 + 8);
        while (!rem.empty()) {
            uint64_t smask;
            std::vector<int> order = collect(run, rem, smask);
            if (order.empty() && (max_grads || quick)) {  // (a tile without a free slot)
                bad = true;
                return;
            }
            if (order.size() >= 2) endgame(run, rem, smask, order);
            if (max_grads) {  // a prefix of the order is a valid sweep
                int left = max_grads;
                size_t keep = 0;
                while (keep < order.size() && (run[order[keep]].grad < 0 || left-- > 0)) keep++;
                order.resize(keep);
            }
            // (two SWAPs alone cost what a sweep costs)
            bool swaps_only = order.size() == 2;
            for (int gi : order) swaps_only &= run[gi].kind == SPZ_SWAP;
            swaps_only &= run[rem[0]].kind == SPZ_SWAP;
            if ((order.size() < 2 || swaps_only) && !max_grads && !quick) {
                // nothing to fuse: the first remaining gate runs on the plain path
                Sweep sw;
                memset(&sw, 0, sizeof sw);
                sw.tile = false;
                sw.gate = rem[0];
                sweeps.push_back(sw);
                rem.erase(rem.begin());
                continue;
            }
            build(run, order, smask);
            rem = minus(rem, order);
        }
    }
};

// Device programs: a ring of two slots, each a pinned host staging buffer, a
// device buffer (both grown as needed) and an event recorded after the last
// sweep that reads it.  A call plans on the host while the GPU may still run
// the previous call's sweeps, and waits only before it overwrites a slot
// whose sweeps have not finished: execute calls return without a device
// synchronisation, in stream order like every other entry point.
struct ProgSlot {
    char *host = nullptr;
    char *dev = nullptr;
    size_t cap = 0;  // bytes
    hipEvent_t done = nullptr;
    bool pending = false;
};
ProgSlot g_slots[2];
int g_slot_next = 0;
std::mutex g_slot_mu;

// Several blocks of bytes into the next slot, each at a 256-byte boundary;
// `at` receives their device addresses.
struct Bytes {
    const void *p;
    size_t n;
};

int reserve_slot(size_t total, ProgSlot **out)
{
    ProgSlot &sl = g_slots[g_slot_next];
    g_slot_next ^= 1;
    if (sl.pending) {
        SPZ_HIP(hipEventSynchronize(sl.done));
        sl.pending = false;
    }
    if (!sl.done) SPZ_HIP(hipEventCreateWithFlags(&sl.done, hipEventDisableTiming));
    if (total > sl.cap) {
        if (sl.dev) SPZ_HIP(hipFree(sl.dev));
        if (sl.host) SPZ_HIP(hipHostFree(sl.host));
        sl.dev = nullptr;
        sl.host = nullptr;
        sl.cap = 0;
        const size_t cap = std::max(total, 4096 * sizeof(TileOp));
        if (device_alloc((void **)&sl.dev, cap) != hipSuccess ||
            hipHostMalloc(&sl.host, cap, hipHostMallocDefault) != hipSuccess)
            return fail(SPZ_ERR_OOM, "tile program allocation failed");
        sl.cap = cap;
    }
    *out = &sl;
    return SPZ_OK;
}

size_t aligned(size_t n) { return (n + 255) & ~(size_t)255; }

int upload(const std::vector<Bytes> &parts, ProgSlot **out, std::vector<char *> *at)
{
    size_t total = 0;
    for (const Bytes &b : parts) total += aligned(b.n);
    ProgSlot *sl;
    SPZ_TRY(reserve_slot(total, &sl));
    size_t o = 0;
    for (const Bytes &b : parts) {
        if (b.n) memcpy(sl->host + o, b.p, b.n);
        at->push_back(sl->dev + o);
        o += aligned(b.n);
    }
    SPZ_HIP(hipMemcpyAsync(sl->dev, sl->host, total, hipMemcpyHostToDevice, rt().stream));
    *out = sl;
    return SPZ_OK;
}

template <typename T>
Bytes bytes_of(const std::vector<T> &v)
{
    return {v.data(), v.size() * sizeof(T)};
}

// Marks a slot busy until the stream passes the point where it goes out of
// scope, on every exit after the upload (an error return included, with the
// copy in flight).
struct Release {
    ProgSlot *sl;
    ~Release()
    {
        if (!sl) return;
        if (hipEventRecord(sl->done, rt().stream) == hipSuccess) sl->pending = true;
        else (void)hipStreamSynchronize(rt().stream);
    }
};

// One gate of a run by itself.
int run_one(spz_state_s *s, const SG &g)
{
    if (g.kind == SPZ_SWAP) return launch_swap(s, g.target, g.t1, 0, 0);
    return g.diag ? launch_diag(s, g.k, g.target, g.ones, g.zeros)
                  : launch_pair(s, g.k, g.target, g.ones, g.zeros);
}

int run_fused(spz_state_s *s, const std::vector<SG> &run, int K, bool strict)
{
    if (run.size() == 1) return run_one(s, run[0]);  // (what its plan would say)
    Planner pl;
    pl.n = s->n;
    pl.K = K;
    pl.LOGW = K - 4;
    pl.RB = 4;
    pl.klo = tile_klo(K);
    pl.improve = env_int("SPZ_TILE_SEARCH", 16);
    pl.strict = strict;
    pl.fast = !strict;
    // In-wavefront lane swaps are off unless asked for: they leave high qubits
    // on lane bits 4 and 5 at load time (four 128-byte runs per wave instead
    // of one 512-byte run), which now costs more than the LDS transposes they
    // save (30 q bench circuit: 7227 against 7190 gates/s without them).
    pl.swaps = env_int("SPZ_TILE_SWAPS", 0) != 0;
    pl.plan(run);
    if (pl.bad) return fail(SPZ_ERR_ARG, "tile planner produced a gate outside the register layout");
    if (pl.fast) {
        // The fast sweeps' global factors are scalars, and every gate in
        // between is linear: a sweep may leave its factor to a later one.
        // Only the last tile sweep of the run applies the product (or an
        // earlier one, once its magnitude leaves [2^-32, 2^32], so that the
        // stored amplitudes stay within 2^32 of the state's).
        size_t last = pl.sweeps.size();
        for (size_t i = 0; i < pl.sweeps.size(); i++)
            if (pl.sweeps[i].tile) last = i;
        double ar = 1.0, ai = 0.0;
        for (size_t i = 0; i < pl.sweeps.size(); i++) {
            if (!pl.sweeps[i].tile) continue;
            TileDesc &d = pl.sweeps[i].desc;
            if (d.fflags & TF_PHASE) {
                const double t = ar * d.gre - ai * d.gim;
                ai = ar * d.gim + ai * d.gre;
                ar = t;
            }
            const double m2 = ar * ar + ai * ai;
            if (i == last || m2 > 0x1p64 || m2 < 0x1p-64) {
                d.gre = ar;
                d.gim = ai;
                if (ar != 1.0 || ai != 0.0) d.fflags |= TF_PHASE;
                else d.fflags &= ~TF_PHASE;
                ar = 1.0;
                ai = 0.0;
            } else {
                d.fflags &= ~TF_PHASE;
            }
        }
    }
    std::lock_guard<std::mutex> lk(g_slot_mu);
    ProgSlot *slot = nullptr;
    std::vector<char *> at;
    if (!pl.prog.empty()) SPZ_TRY(upload({bytes_of(pl.prog)}, &slot, &at));
    Release release{slot};
    const TileOp *d_prog = slot ? (const TileOp *)at[0] : nullptr;
    for (const Sweep &sw : pl.sweeps) {
        if (sw.tile) {
            SPZ_TRY(launch_tile(s, K, sw.desc, d_prog + sw.op_begin, pl.fast));
        } else {
            SPZ_TRY(run_one(s, run[sw.gate]));
        }
    }
    return SPZ_OK;
}

// 2x2 matrix (row-major, interleaved re/im) of a lowered gate.
void gate_matrix2(const Coef &k, double m[8])
{
    for (int i = 0; i < 8; i++) m[i] = 0.0;
    const double *c = k.c;
    switch (k.ak) {
    case AK_H: m[0] = c[0]; m[2] = c[0]; m[4] = c[0]; m[6] = -c[0]; break;
    case AK_X: m[2] = 1.0; m[4] = 1.0; break;
    case AK_Y: m[3] = -1.0; m[5] = 1.0; break;
    case AK_RX: m[0] = c[0]; m[3] = c[1]; m[5] = c[1]; m[6] = c[0]; break;
    case AK_RY: m[0] = c[1]; m[2] = -c[0]; m[4] = c[0]; m[6] = c[1]; break;
    case AK_U:
    case AK_MAT: for (int i = 0; i < 8; i++) m[i] = c[i]; break;
    case AK_NEG: m[0] = 1.0; m[6] = -1.0; break;
    case AK_PHASE: m[0] = 1.0; m[6] = c[0]; m[7] = c[1]; break;
    case AK_RZ: m[0] = c[0]; m[1] = c[1]; m[6] = c[2]; m[7] = c[3]; break;
    default: break;
    }
}

// Fuse runs of gates acting on at most 5 qubits into dense 32x32 blocks.
int run_dense5(spz_state_s *s, const std::vector<SG> &run)
{
    struct Blk {
        int q[5];
        std::vector<int> gates;
        int single;
    };
    // Blocks are formed greedily over the remaining gates in program order:
    // a block takes a gate whose qubits keep it within 5 qubits and that
    // commutes with every gate the block has passed over (the tile planner's
    // rule: a passed gate blocks later gates on its non-diagonal qubits, and
    // non-diagonal action on its diagonal qubits), so a block gathers the
    // gates of a 5-qubit region across layers rather than only a consecutive
    // run.  The taken gates keep their order inside the block; a block of one
    // gate, or a gate on more than 5 qubits, runs on the plain path.
    std::vector<Blk> blocks;
    const uint64_t all = s->n >= 64 ? ~0ull : ((1ull << s->n) - 1);
    std::vector<int> rem(run.size());
    for (size_t i = 0; i < run.size(); i++) rem[i] = (int)i;
    while (!rem.empty()) {
        const SG &g0 = run[rem[0]];
        if (__builtin_popcountll((g0.nd | g0.dm) & all) > 5) {
            Blk b;
            b.single = rem[0];
            blocks.push_back(b);
            rem.erase(rem.begin());
            continue;
        }
        uint64_t Q = 0, bnd = 0, bd = 0;
        std::vector<int> take, left;
        for (size_t r = 0; r < rem.size(); r++) {
            const int idx = rem[r];
            const SG &g = run[idx];
            const uint64_t qs = (g.nd | g.dm) & all;
            const bool ok = !(g.nd & (bnd | bd)) && !(g.dm & bnd) &&
                            __builtin_popcountll(Q | qs) <= 5;
            if (ok) {
                take.push_back(idx);
                Q |= qs;
            } else {
                left.push_back(idx);
                bnd |= g.nd;
                bd |= g.dm;
                if (((bnd | bd) & all) == all) {  // nothing further can pass
                    left.insert(left.end(), rem.begin() + (long)r + 1, rem.end());
                    break;
                }
            }
        }
        rem.swap(left);
        Blk b;
        b.single = -1;
        if (take.size() == 1) {
            b.single = take[0];
        } else {
            int j = 0;
            for (int q = 0; q < s->n && j < 5; q++)
                if ((Q >> q) & 1) b.q[j++] = q;
            for (int q = 0; q < s->n && j < 5; q++)
                if (!((Q >> q) & 1)) { b.q[j++] = q; Q |= 1ull << q; }
            b.gates = take;
        }
        blocks.push_back(b);
    }
    // block matrices: U = G_last ... G_first, embedded in the 5-qubit block
    std::vector<double> f64;
    std::vector<float> f32;
    std::vector<double> U(2 * 32 * 32);
    for (const Blk &b : blocks) {
        if (b.single >= 0) continue;
        for (int i = 0; i < 32 * 32; i++) { U[2 * i] = (i / 32 == i % 32) ? 1.0 : 0.0; U[2 * i + 1] = 0.0; }
        for (int gi : b.gates) {
            const SG &g = run[gi];
            double m[8];
            gate_matrix2(g.k, m);
            int tj = -1;
            uint32_t need1 = 0, need0 = 0;
            for (int j = 0; j < 5; j++) {
                if (b.q[j] == g.target) tj = j;
                if ((g.ones >> b.q[j]) & 1) need1 |= 1u << j;
                if ((g.zeros >> b.q[j]) & 1) need0 |= 1u << j;
            }
            for (uint32_t a0 = 0; a0 < 32; a0++) {
                if ((a0 >> tj) & 1) continue;
                if ((a0 & need1) != need1 || (a0 & need0)) continue;
                const uint32_t a1 = a0 | (1u << tj);
                for (int col = 0; col < 32; col++) {
                    const double xr = U[2 * (a0 * 32 + col)], xi = U[2 * (a0 * 32 + col) + 1];
                    const double yr = U[2 * (a1 * 32 + col)], yi = U[2 * (a1 * 32 + col) + 1];
                    U[2 * (a0 * 32 + col)] = m[0] * xr - m[1] * xi + m[2] * yr - m[3] * yi;
                    U[2 * (a0 * 32 + col) + 1] = m[0] * xi + m[1] * xr + m[2] * yi + m[3] * yr;
                    U[2 * (a1 * 32 + col)] = m[4] * xr - m[5] * xi + m[6] * yr - m[7] * yi;
                    U[2 * (a1 * 32 + col) + 1] = m[4] * xi + m[5] * xr + m[6] * yi + m[7] * yr;
                }
            }
        }
        block5_fragments(U.data(), s->prec, f64, f32);
    }
    // fragments through the program ring: no wait before or after the launches
    std::lock_guard<std::mutex> lk(g_slot_mu);
    ProgSlot *slot = nullptr;
    std::vector<char *> at;
    const bool any = !f64.empty() || !f32.empty();
    if (any) SPZ_TRY(upload({s->prec == SPZ_F64 ? bytes_of(f64) : bytes_of(f32)}, &slot, &at));
    Release release{slot};
    size_t bi = 0;
    const size_t esz = s->prec == SPZ_F64 ? sizeof(double) : sizeof(float);
    for (const Blk &b : blocks) {
        if (b.single >= 0) {
            const SG &g = run[b.single];
            if (g.diag) SPZ_TRY(launch_diag(s, g.k, g.target, g.ones, g.zeros));
            else SPZ_TRY(launch_pair(s, g.k, g.target, g.ones, g.zeros));
            continue;
        }
        SPZ_TRY(launch_block5(s, b.q, at[0] + bi * 4096 * esz));
        bi++;
    }
    return SPZ_OK;
}

}  // namespace

// A dense block (arguments checked): its matrix goes through the program ring, so
// the call neither allocates nor waits.
int run_dense(spz_state_s *s, int m, const double *u_re, const double *u_im, int t, int control)
{
    std::vector<double> coef;
    dense_coefs(s, m, u_re, u_im, coef);
    std::lock_guard<std::mutex> lk(g_slot_mu);
    ProgSlot *slot = nullptr;
    std::vector<char *> at;
    SPZ_TRY(upload({bytes_of(coef)}, &slot, &at));
    Release release{slot};
    return launch_dense(s, m, (const double *)at[0], t, control);
}

// A SWAP as three CX, the middle one with the SWAP's controls.
void swap_as_cx(const spz_op &o, spz_op out[3])
{
    spz_op x;
    memset(&x, 0, sizeof x);
    x.kind = SPZ_X;
    x.target = o.target;
    x.ones = 1ull << o.t1;
    spz_op y = x;
    y.target = o.t1;
    y.ones = o.ones | (1ull << o.target);
    y.zeros = o.zeros;
    out[0] = out[2] = x;
    out[1] = y;
}

// Validated ops as a run on n qubits: forward, or undone from the last to the
// first with the index of each one's gradient (SWAPs as CX).
static int lower_run(int n, const spz_op *ops, uint64_t lo, uint64_t hi, bool reverse,
                     std::vector<SG> &run)
{
    spz_state_s st;  // shape only
    st.n = n;
    st.N = 1ull << n;
    run.clear();
    run.reserve(hi - lo);
    auto add = [&](const spz_op &o, int64_t grad) -> int {
        SG g;
        SPZ_TRY(lower(&st, o, nullptr, (int)run.size(), &g));
        g.grad = grad;
        run.push_back(g);
        return SPZ_OK;
    };
    for (uint64_t i = lo; i < hi; i++) {
        const uint64_t k = reverse ? hi - 1 - (i - lo) : i;
        const spz_op o = reverse ? inverse_op(ops[k]) : ops[k];
        if (o.kind == SPZ_SWAP) {
            spz_op cx[3];
            swap_as_cx(o, cx);
            for (const spz_op &c : cx) SPZ_TRY(add(c, -1));
            continue;
        }
        const bool par = reverse && (o.kind == SPZ_RX || o.kind == SPZ_RY || o.kind == SPZ_RZ ||
                                     o.kind == SPZ_P);
        SPZ_TRY(add(o, par ? (int64_t)k : -1));
    }
    return SPZ_OK;
}

// Lowers ops from *j on into a run, up to the next barrier (*j moves there).
enum class Swaps { BARRIER, AS_CX, RELABEL };
static int collect_run(const spz_state_s *s, const spz_op *ops, uint64_t n_ops,
                       const spz_tracker *trk, Swaps how, uint64_t *j, std::vector<SG> &run);

// Plans a run whose sweeps are all tile sweeps.
static int plan_tiles(Planner &pl, const std::vector<SG> &run, ChipPlan &out)
{
    out.prog.clear();
    out.grads.clear();
    pl.prog.swap(out.prog);  // (their memory is used again)
    pl.grads.swap(out.grads);
    pl.plan(run);
    if (pl.bad) return fail(SPZ_ERR_ARG, "tile planner produced a gate outside the register layout");
    out.sweeps.clear();
    out.sweeps.reserve(pl.sweeps.size());
    for (const Sweep &sw : pl.sweeps)
        out.sweeps.push_back({sw.desc, (uint32_t)sw.op_begin, (uint32_t)sw.op_count,
                              (uint32_t)sw.slot_begin, (uint32_t)sw.slots});
    out.prog.swap(pl.prog);
    out.grads.swap(pl.grads);
    return SPZ_OK;
}

static int plan_chip(int n, const std::vector<SG> &run, bool strict, bool reverse, ChipPlan &out)
{
    Planner pl;
    pl.n = std::max(n, kChipK);  // fewer qubits: the tile's other bits stay |0>
    pl.K = kChipK;
    pl.LOGW = kChipK - 4;
    pl.RB = 4;
    pl.klo = 4;
    pl.strict = strict;
    pl.quick = true;
    if (reverse) pl.max_grads = 1 << 30;
    if (!strict) pl.max_gates = 1024;
    return plan_tiles(pl, run, out);
}

// (spz_chip.h)
int chip_plan(int n, const spz_op *ops, uint64_t n_ops, bool reverse, ChipPlan &out)
{
    std::vector<SG> run;
    SPZ_TRY(lower_run(std::max(n, kChipK), ops, 0, n_ops, reverse, run));
    return plan_chip(n, run, false, reverse, out);
}

// A run on a state of at most kChipK qubits: one launch.  Program order is
// kept, so the amplitudes are bit-identical to one launch per gate (FP32
// storage: rounded once, at the end).
static int run_chip(spz_state_s *s, const std::vector<SG> &run)
{
    ChipPlan cp;
    SPZ_TRY(plan_chip(s->n, run, true, false, cp));
    std::lock_guard<std::mutex> lk(g_slot_mu);
    std::vector<ChipSweep> d(cp.sweeps.size());
    ProgSlot *slot = nullptr;
    SPZ_TRY(reserve_slot(aligned(cp.prog.size() * sizeof(TileOp)) +
                             aligned(d.size() * sizeof(ChipSweep)), &slot));
    Release release{slot};
    const size_t o_d = aligned(cp.prog.size() * sizeof(TileOp));
    for (size_t i = 0; i < d.size(); i++) {
        memset(&d[i], 0, sizeof d[i]);
        chip_geometry(cp.sweeps[i], s->n, s->prec, d[i]);
        d[i].sr = d[i].pr = s->re;
        d[i].si = d[i].pi = s->im;
        d[i].ops = (const TileOp *)slot->dev + cp.sweeps[i].op_begin;
        d[i].flags = CHIP_STORE;
    }
    memcpy(slot->host, cp.prog.data(), cp.prog.size() * sizeof(TileOp));
    memcpy(slot->host + o_d, d.data(), d.size() * sizeof(ChipSweep));
    SPZ_HIP(hipMemcpyAsync(slot->dev, slot->host, o_d + d.size() * sizeof(ChipSweep),
                           hipMemcpyHostToDevice, rt().stream));
    for (size_t i = 0; i < d.size(); i++) {  // (one: every qubit is in the tile)
        LaunchTimer tm(SPZ_K_TILE, 2.0 * (double)s->N * (s->prec == SPZ_F64 ? 16.0 : 8.0));
        SPZ_TRY(launch_chip_sweeps(s->prec, false, (const ChipSweep *)(slot->dev + o_d) + i, 1, 1, 0));
    }
    return SPZ_OK;
}

// (spz_adj_tile.h)
int adjoint_plan(int n, const spz_op *ops, uint64_t lo, uint64_t hi, ChipPlan &out)
{
    std::vector<SG> run;
    SPZ_TRY(lower_run(std::max(n, kChipK), ops, lo, hi, true, run));
    if (n <= kChipK) return plan_chip(n, run, false, true, out);
    Planner pl;
    pl.n = n;
    pl.K = kAdjK;
    pl.LOGW = kAdjK - 4;
    pl.RB = 4;
    pl.klo = tile_klo(kAdjK - 1);  // every gate runs in a sweep: one slot for its target
    pl.improve = env_int("SPZ_TILE_SEARCH", 16);
    pl.strict = false;
    pl.max_grads = kAdjSlots;
    return plan_tiles(pl, run, out);
}

int adjoint_undo(const spz_state_s *src, spz_state_s *psi, spz_state_s *lam, const spz_op *ops,
                 uint64_t lo, uint64_t hi, double *part, double *grad)
{
    ChipPlan cp;
    SPZ_TRY(adjoint_plan(psi->n, ops, lo, hi, cp));
    if (psi->n <= kChipK) {
        std::vector<ChipSweep> d(cp.sweeps.size());
        std::vector<ChipSum> sums;
        const size_t o_d = aligned(cp.prog.size() * sizeof(TileOp));
        const size_t o_s = o_d + aligned(d.size() * sizeof(ChipSweep));
        const size_t total = o_s + aligned(cp.grads.size() * sizeof(ChipSum));
        std::lock_guard<std::mutex> lk(g_slot_mu);
        ProgSlot *slot = nullptr;
        SPZ_TRY(reserve_slot(total, &slot));
        Release release{slot};
        for (size_t i = 0; i < d.size(); i++) {
            memset(&d[i], 0, sizeof d[i]);
            chip_geometry(cp.sweeps[i], psi->n, psi->prec, d[i]);
            d[i].sr = src->re;
            d[i].si = src->im;
            d[i].pr = psi->re;
            d[i].pi = psi->im;
            d[i].qr = lam->re;
            d[i].qi = lam->im;
            d[i].ops = (const TileOp *)slot->dev + cp.sweeps[i].op_begin;
            d[i].part = part + 2 * kChipRows * (size_t)cp.sweeps[i].slot_begin;
            d[i].flags = CHIP_STORE;
            src = psi;
        }
        for (size_t k = 0; k < cp.grads.size(); k++)
            sums.push_back({part + 2 * kChipRows * k, kChipRows, cp.grads[k]});
        memcpy(slot->host, cp.prog.data(), cp.prog.size() * sizeof(TileOp));
        memcpy(slot->host + o_d, d.data(), d.size() * sizeof(ChipSweep));
        if (!sums.empty()) memcpy(slot->host + o_s, sums.data(), sums.size() * sizeof(ChipSum));
        SPZ_HIP(hipMemcpyAsync(slot->dev, slot->host, total, hipMemcpyHostToDevice, rt().stream));
        for (size_t i = 0; i < d.size(); i++) {
            LaunchTimer tm(SPZ_K_ADJOINT, 4.0 * (double)psi->N * (psi->prec == SPZ_F64 ? 16.0 : 8.0));
            SPZ_TRY(launch_chip_sweeps(psi->prec, true, (const ChipSweep *)(slot->dev + o_d) + i, 1,
                                       1, 0));
        }
        return launch_chip_sums((const ChipSum *)(slot->dev + o_s), (uint32_t)sums.size(), grad);
    }
    std::lock_guard<std::mutex> lk(g_slot_mu);
    ProgSlot *slot = nullptr;
    std::vector<char *> at;
    SPZ_TRY(upload({bytes_of(cp.prog), bytes_of(cp.grads)}, &slot, &at));
    Release release{slot};
    const TileOp *d_prog = (const TileOp *)at[0];
    const uint32_t *d_idx = (const uint32_t *)at[1];
    const uint64_t tiles = psi->N >> kAdjK;
    for (const ChipPlan::Sweep &sw : cp.sweeps) {
        SPZ_TRY(launch_adj_tile(src, psi, lam, sw.desc, d_prog + sw.op_begin, sw.slots, part));
        SPZ_TRY(launch_adj_sum(part, tiles, d_idx + sw.slot_begin, sw.slots, grad));
        src = psi;
    }
    return SPZ_OK;
}

int execute_plain(spz_state_s *s, const spz_op *ops, uint64_t n_ops, spz_tracker *trk,
                  uint8_t *outcomes)
{
    for (uint64_t i = 0; i < n_ops; i++) {
        int rc = exec_one_plain(s, ops[i], trk, outcomes ? &outcomes[i] : nullptr);
        if (rc != SPZ_OK) {
            set_error("op " + std::to_string(i) + ": " + spz_last_error());
            return rc;
        }
    }
    return SPZ_OK;
}

// The tile width and low-qubit count an execution uses (options, then the
// SPZ_TILE_K / SPZ_TILE_KLO environment, then 12 and 4).
int tile_width(const spz_exec_opts *opts, int n, int *K_out)
{
    int K = (opts && opts->tile_qubits) ? opts->tile_qubits : env_int("SPZ_TILE_K", 12);
    if (K < 10 || K > 13) return fail(SPZ_ERR_ARG, "tile_qubits must be in [10, 13]");
    if (n < K + 1) K = n - 1;
    *K_out = K;
    return SPZ_OK;
}

// Whether a state takes the one-launch path: at most kChipK qubits, and no
// tile width asked for.
static bool small_path(const spz_exec_opts *opts, int n)
{
    return n <= kChipK && !(opts && opts->tile_qubits) && env_int("SPZ_TILE_K", 0) == 0;
}

// A SWAP that can go into a run: valid, and (its control flags are resolved like
// a gate's) not under classical control.
static bool plain_swap(const spz_op &o, int n)
{
    if (o.kind != SPZ_SWAP || (o.flags & SPZ_OPF_CLASSICAL)) return false;
    if (o.target < 0 || o.target >= n || o.t1 < 0 || o.t1 >= n || o.target == o.t1) return false;
    const uint64_t sw = (1ull << o.target) | (1ull << o.t1), c = o.ones | o.zeros;
    return !(c & sw) && !(o.ones & o.zeros) && !(c >> n);
}

// A run of so few ops goes op by op in small states too: the one launch costs its
// program's copy and a workgroup's start.  3 to 12 qubits, one op 4.2 us and (in
// one launch) 12-13.5, four 12.0 and 14-17, five 14.6 and 14.6-17, six 17.3 and
// 15-19, eight 22.3 and 16-19.6; waited for after each call 12.5 and 21 (one op),
// 22.6 and 23.5 (five), 25 and 24 (six).
constexpr int kShortRun = 5;

// How a run takes SWAPs: one launch as CX, tile sweeps as a relabelling where no
// qubit controls it.
static bool takes_swap(const spz_op &o, int n, Swaps how)
{
    return how != Swaps::BARRIER && plain_swap(o, n) &&
           (how == Swaps::AS_CX || !(o.ones | o.zeros));
}

// The end of the run at `i` if it has at most kShortRun ops, else `i`.
static uint64_t short_run(const spz_op *ops, uint64_t i, uint64_t n_ops, int n, Swaps how)
{
    uint64_t e = i;
    for (; e < n_ops && (!is_barrier(ops[e]) || takes_swap(ops[e], n, how)); e++)
        if (e - i == (uint64_t)kShortRun) return i;
    return e;
}

// Planning only (no device work): how the tile executor would split `ops`.
int plan_info(int n, int prec, const spz_op *ops, uint64_t n_ops, const spz_exec_opts *opts,
              spz_plan_info *out)
{
    if (!out || (n_ops && !ops)) return fail(SPZ_ERR_ARG, "null argument");
    if (n < 1 || n > 40) return fail(SPZ_ERR_QUBIT, "qubit count must be in [1, 40]");
    memset(out, 0, sizeof *out);
    const int mode = opts ? opts->mode : SPZ_EXEC_AUTO;
    if (mode != SPZ_EXEC_AUTO && mode != SPZ_EXEC_STRICT)
        return fail(SPZ_ERR_ARG, "plan statistics cover the tile executors (AUTO, STRICT)");
    int K;
    SPZ_TRY(tile_width(opts, n, &K));
    spz_state_s st;  // shape only: lowering reads n and the precision
    memset(&st, 0, sizeof st);
    st.n = n;
    st.prec = prec;
    st.N = 1ull << n;
    const bool small = small_path(opts, n);
    const Swaps how = small ? Swaps::AS_CX : Swaps::RELABEL;
    uint64_t i = 0;
    while (i < n_ops) {
        const bool barrier = is_barrier(ops[i]) && !takes_swap(ops[i], n, how);
        if (barrier || (K < 10 && !small)) {
            out->plain_gates++;
            i++;
            continue;
        }
        std::vector<SG> run;
        uint64_t j = i;
        SPZ_TRY(collect_run(&st, ops, n_ops, nullptr, how, &j, run));
        if (small) {
            if (j - i <= (uint64_t)kShortRun) {
                out->plain_gates += j - i;
            } else {
                ChipPlan cp;
                SPZ_TRY(plan_chip(n, run, true, false, cp));
                out->sweeps += cp.sweeps.size();
                for (const TileOp &op : cp.prog) {
                    if (op.type == TOP_LAYOUT) out->layouts++;
                    else out->tile_gates++;
                }
            }
            i = j;
            continue;
        }
        Planner pl;
        pl.n = n;
        pl.K = K;
        pl.LOGW = K - 4;
        pl.RB = 4;
        pl.klo = tile_klo(K);
        pl.improve = env_int("SPZ_TILE_SEARCH", 16);
        pl.strict = mode == SPZ_EXEC_STRICT;
        pl.fast = !pl.strict;
        pl.swaps = env_int("SPZ_TILE_SWAPS", 0) != 0;
        pl.plan(run);
        if (pl.bad) return fail(SPZ_ERR_ARG, "tile planner produced a gate outside the register layout");
        out->tile_gates += pl.frame_gates + pl.swap_gates;
        out->tile_gates -= pl.split_ops;
        out->frame_gates += pl.frame_gates;
        for (const Sweep &sw : pl.sweeps) {
            if (!sw.tile) {
                out->plain_gates++;
                continue;
            }
            out->sweeps++;
            for (size_t o = sw.op_begin; o < sw.op_begin + sw.op_count; o++) {
                if (pl.prog[o].type != TOP_LAYOUT) out->tile_gates++;
                else if (pl.prog[o].grp & TG_LAYOUT) out->layouts++;
                else out->lane_swaps++;
            }
        }
        i = j;
    }
    return SPZ_OK;
}

static int collect_run(const spz_state_s *s, const spz_op *ops, uint64_t n_ops,
                       const spz_tracker *trk, Swaps how, uint64_t *j, std::vector<SG> &run)
{
    // FP32 storage rounds at every store: gates keep the sweeps they have with
    // SWAPs as barriers, and only SWAPs share a pass.
    const bool apart = how == Swaps::RELABEL && s->prec == SPZ_F32;
    for (; *j < n_ops; (*j)++) {
        const spz_op &o = ops[*j];
        spz_op cx[3];
        int n = 1;
        if (is_barrier(o)) {
            if (!takes_swap(o, s->n, how)) break;
            if (how == Swaps::RELABEL) {
                if (apart && !run.empty() && run.back().kind != SPZ_SWAP) break;
                run.push_back(lower_swap(o, (int)*j));
                continue;
            }
            swap_as_cx(o, cx);
            n = 3;
        } else {
            if (apart && !run.empty() && run.back().kind == SPZ_SWAP) break;
            cx[0] = o;
        }
        for (int k = 0; k < n; k++) {
            SG g;
            const int rc = lower(s, cx[k], trk, (int)*j, &g);
            if (rc == -1) continue;  // no-op (unflipped noise, classical control read 0)
            if (rc != SPZ_OK) {
                set_error("op " + std::to_string(*j) + ": " + spz_last_error());
                return rc;
            }
            run.push_back(g);
        }
    }
    return SPZ_OK;
}

int execute_ops(spz_state_s *s, const spz_op *ops, uint64_t n_ops, spz_tracker *trk,
                const spz_exec_opts *opts, uint8_t *outcomes)
{
    int mode = opts ? opts->mode : SPZ_EXEC_AUTO;
    if (mode == SPZ_EXEC_PLAIN) return execute_plain(s, ops, n_ops, trk, outcomes);
    if (mode != SPZ_EXEC_AUTO && mode != SPZ_EXEC_STRICT && mode != SPZ_EXEC_DENSE5)
        return fail(SPZ_ERR_ARG, "unknown execution mode");
    const bool dense5 = mode == SPZ_EXEC_DENSE5;
    if (dense5 && s->n < 12) return execute_plain(s, ops, n_ops, trk, outcomes);
    int K;
    SPZ_TRY(tile_width(opts, s->n, &K));
    const bool small = !dense5 && small_path(opts, s->n);
    if (K < 10 && !small) return execute_plain(s, ops, n_ops, trk, outcomes);
    const bool strict = mode == SPZ_EXEC_STRICT;
    const Swaps how = small ? Swaps::AS_CX : dense5 ? Swaps::BARRIER : Swaps::RELABEL;
    if (outcomes)
        for (uint64_t i = 0; i < n_ops; i++) outcomes[i] = 255;
    uint64_t i = 0;
    while (i < n_ops) {
        if (is_barrier(ops[i]) && !takes_swap(ops[i], s->n, how)) {
            int rc = exec_one_plain(s, ops[i], trk, outcomes ? &outcomes[i] : nullptr);
            if (rc != SPZ_OK) {
                set_error("op " + std::to_string(i) + ": " + spz_last_error());
                return rc;
            }
            i++;
            continue;
        }
        if (const uint64_t end = small ? short_run(ops, i, n_ops, s->n, how) : i; end > i) {
            for (; i < end; i++) {
                const int rc = exec_one_plain(s, ops[i], trk, nullptr);
                if (rc != SPZ_OK) {
                    set_error("op " + std::to_string(i) + ": " + spz_last_error());
                    return rc;
                }
            }
            continue;
        }
        std::vector<SG> run;
        uint64_t j = i;
        SPZ_TRY(collect_run(s, ops, n_ops, trk, how, &j, run));
        if (!run.empty())
            SPZ_TRY(small ? run_chip(s, run)
                          : dense5 ? run_dense5(s, run) : run_fused(s, run, K, strict));
        i = j;
    }
    return SPZ_OK;
}

}  // namespace spz

extern "C" int spz_plan_stats(int n, int precision, const spz_op *ops, uint64_t n_ops,
                              const spz_exec_opts *opts, spz_plan_info *out)
{
    return spz::plan_info(n, precision, ops, n_ops, opts, out);
}

