// spz_block.hip -- dense 5-qubit blocks applied with MFMA (gfx950).
//
// A block is a 32x32 complex matrix U on qubits b0..b4.  For every one of the
// 2^(n-5) vectors v (the 32 amplitudes that agree outside the block), out =
// U v, computed as the real product
//     [yr; yi] = [[Ur, -Ui], [Ui, Ur]] [vr; vi]      (64 x 64 times 64 x 16)
// on v_mfma_f64_16x16x4f64 (FP64 storage) or v_mfma_f32_16x16x4f32 (FP32
// storage): 4 output row blocks x 16 k-steps = 64 MFMAs per 16 vectors, 256
// flops per amplitude.
//
// A tile is 2^12 amplitudes: the block qubits, qubits 0..3 (so the tile is a union
// of contiguous 128-byte runs) and the lowest remaining qubits, 128 vectors.  A
// workgroup (512 threads, 8 wavefronts, 16 vectors each) keeps the 64 A fragments
// of the matrix in registers and walks over tiles: the next tile's amplitudes
// travel from memory straight into the other half of its LDS while it contracts
// this one, and results go to memory from the accumulators or, with many low
// qubits in the block, through LDS.
//
// Bound: one read and one write of the state (350 us at 26 qubits FP64) against
// 64 MFMAs per 16 vectors (235 us).  Measured, 26 qubits FP64, 2 GiB of traffic:
// 407-428 us per block (5.1 TB/s), 511-523 us with qubits n-3 and n-2 and two or
// three low ones in the block; 27 qubits FP32 386-472 us; one FP64 tile 11 us.
// Loads through registers into one LDS tile, with two workgroups per CU to
// overlap them, took 511-757 us, 512-601 us and 12.4-16.3 us: each workgroup's
// memory and matrix phases added up.
//
// MFMA lane layout (16x16x4, measured on gfx950): lane i supplies A[i % 16][i / 16]
// and B[i / 16][i % 16] for both types; accumulator slot j of lane i holds
// D[4 (i / 16) + j][i % 16] for f32 but D[4 j + i / 16][i % 16] for f64.
#include <string.h>

#include <algorithm>
#include <vector>

#include "spz_internal.h"

namespace spz {

struct alignas(8) BlockDesc {
    int8_t spos[16];   // tile qubits (ascending), 12 entries
    int8_t bpos[8];    // local positions of the 5 block bits (amplitude index bit a_j)
    int8_t vpos[8];    // local positions of the 7 vector-index bits
    uint64_t bg[5];    // global bit of block bit j
    uint64_t vg[7];    // global bit of vector-index bit j
};

namespace {

constexpr int kBK = 12;             // tile qubits
constexpr int kBT = 512;            // threads: 8 wavefronts of 16 vectors

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <typename T> struct Acc;
template <> struct Acc<double> { using type = v4d; };
template <> struct Acc<float> { using type = v4f; };

__device__ __forceinline__ v4d mfma(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4f mfma(float a, float b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// 16 LDS reads at byte addresses x[s], and the wait for them, in one block: the
// compiler would hold them back until every load to LDS in flight (the next
// tile's, to the other buffer) has landed.
__device__ __forceinline__ void read16(const uint32_t *x, double *v)
{
    asm volatile(
        "ds_read_b64 %0, %16\n\tds_read_b64 %1, %17\n\tds_read_b64 %2, %18\n\t"
        "ds_read_b64 %3, %19\n\tds_read_b64 %4, %20\n\tds_read_b64 %5, %21\n\t"
        "ds_read_b64 %6, %22\n\tds_read_b64 %7, %23\n\tds_read_b64 %8, %24\n\t"
        "ds_read_b64 %9, %25\n\tds_read_b64 %10, %26\n\tds_read_b64 %11, %27\n\t"
        "ds_read_b64 %12, %28\n\tds_read_b64 %13, %29\n\tds_read_b64 %14, %30\n\t"
        "ds_read_b64 %15, %31\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
          "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11]),
          "=&v"(v[12]), "=&v"(v[13]), "=&v"(v[14]), "=&v"(v[15])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]),
          "v"(x[8]), "v"(x[9]), "v"(x[10]), "v"(x[11]), "v"(x[12]), "v"(x[13]), "v"(x[14]),
          "v"(x[15])
        : "memory");
}
__device__ __forceinline__ void read16(const uint32_t *x, float *v)
{
    asm volatile(
        "ds_read_b32 %0, %16\n\tds_read_b32 %1, %17\n\tds_read_b32 %2, %18\n\t"
        "ds_read_b32 %3, %19\n\tds_read_b32 %4, %20\n\tds_read_b32 %5, %21\n\t"
        "ds_read_b32 %6, %22\n\tds_read_b32 %7, %23\n\tds_read_b32 %8, %24\n\t"
        "ds_read_b32 %9, %25\n\tds_read_b32 %10, %26\n\tds_read_b32 %11, %27\n\t"
        "ds_read_b32 %12, %28\n\tds_read_b32 %13, %29\n\tds_read_b32 %14, %30\n\t"
        "ds_read_b32 %15, %31\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
          "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11]),
          "=&v"(v[12]), "=&v"(v[13]), "=&v"(v[14]), "=&v"(v[15])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]),
          "v"(x[8]), "v"(x[9]), "v"(x[10]), "v"(x[11]), "v"(x[12]), "v"(x[13]), "v"(x[14]),
          "v"(x[15])
        : "memory");
}

// Place of the 16-byte unit u of a tile in LDS: its low 3 bits (which 16 bytes
// of a 128-byte line) XORed with two higher groups, so that the strided reads of
// blocks on low qubits spread over the banks.  Its own inverse.
__device__ __forceinline__ uint32_t unit_swz(uint32_t u)
{
    return u ^ (((u >> 3) ^ (u >> 6)) & 7u);
}

typedef __attribute__((address_space(1))) const void *GlobalPtr;
typedef __attribute__((address_space(3))) void *LdsPtr;

// afrag: [r (4)][s (16)][lane (64)] values of the real 64x64 matrix.  FP64: the
// two tile buffers fill 128 KiB of LDS, one workgroup per CU; FP32 two.
// STAGE: results go back through the tile's LDS and leave as 16-byte stores of
// whole lines (see launch_block5).
template <typename T, bool STAGE>
__global__ void __launch_bounds__(kBT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_block5(T *re, T *im, const BlockDesc d, const T *__restrict__ afrag, uint32_t tiles)
{
    using V = typename Acc<T>::type;
    constexpr uint32_t PER = 16 / sizeof(T);              // amplitudes per 16-byte load
    constexpr uint32_t LP = sizeof(T) == 8 ? 1 : 2;       // log2 of that
    constexpr uint32_t ROUNDS = (1u << kBK) / (kBT * PER);  // loads per array and thread
    constexpr uint32_t ARRAY = (1u << kBK) * sizeof(T);   // bytes of one array of a tile
    __shared__ __align__(16) char lds[4 * ARRAY];         // [buffer][re, im]
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;

    // The matrix comes in once per workgroup, to the second tile buffer, and
    // each wavefront takes its fragments from there.
#pragma unroll
    for (uint32_t k = 0; k < ROUNDS; k++)
        __builtin_amdgcn_global_load_lds(
            (GlobalPtr)(reinterpret_cast<const char *>(afrag) + (k * kBT + tid) * 16),
            (LdsPtr)(lds + 2 * ARRAY + (k * kBT + wave * 64) * 16), 16, 0, 0);

    // loads: LDS unit (round, wave, lane) holds the amplitudes whose local index
    // is its swizzled number; their global index has those bits at the tile's
    // qubits (the round's bits are not swizzled)
    uint64_t lg = 0;
    const uint32_t l0 = unit_swz((wave << 6) | lane) << LP;
#pragma unroll
    for (int i = 0; i < 9 + (int)LP; i++)
        if ((l0 >> i) & 1u) lg |= 1ull << d.spos[i];
    auto load = [&](uint32_t tile, uint32_t buf) {
        const uint64_t at = insert_zeros((uint64_t)tile, d.spos, kBK) + lg;
#pragma unroll
        for (uint32_t k = 0; k < ROUNDS; k++) {
            uint64_t g = at;
#pragma unroll
            for (int j = 0; j < (int)(3 - LP); j++)
                if ((k >> j) & 1u) g += 1ull << d.spos[9 + LP + j];
            // (a wavefront's 64 loads of 16 bytes land side by side)
            char *to = lds + buf * 2 * ARRAY + (k * kBT + wave * 64) * 16;
            __builtin_amdgcn_global_load_lds((GlobalPtr)(re + g), (LdsPtr)to, 16, 0, 0);
            __builtin_amdgcn_global_load_lds((GlobalPtr)(im + g), (LdsPtr)(to + ARRAY), 16, 0, 0);
        }
    };

    // this lane's vector, and its B components 4 s + kq (0..31 real, 32..63 imaginary)
    const uint32_t col = lane & 15u, kq = lane >> 4, v = wave * 16 + col;
    uint32_t vl = 0;
    uint64_t out = 0;
#pragma unroll
    for (int j = 0; j < 7; j++)
        if ((v >> j) & 1u) {
            vl |= 1u << d.vpos[j];
            out += d.vg[j];
        }
    // direct stores: component 16 r + 4 j + kq of the vector, the kq part per lane
    if (kq & 1u) out += d.bg[0];
    if (kq & 2u) out += d.bg[1];
    const uint32_t lbase = (uint32_t)(uintptr_t)(LdsPtr)lds;

    const uint32_t step = gridDim.x;  // at most `tiles`
    uint32_t t = blockIdx.x, buf = 0;
    load(t, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    T a[4][16];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int s = 0; s < 16; s++)
            a[r][s] = reinterpret_cast<const T *>(lds + 2 * ARRAY)[(r * 16 + s) * 64 + lane];

    auto contract = [&](uint32_t tile, uint32_t buf) {
        uint32_t x[16];
        T b[16];
#pragma unroll
        for (int s = 0; s < 16; s++) {
            const uint32_t c = (4u * s + kq) & 31u;
            uint32_t l = vl;
#pragma unroll
            for (int j = 0; j < 5; j++) l |= ((c >> j) & 1u) << d.bpos[j];
            x[s] = lbase + (buf * 2 + (s >= 8 ? 1 : 0)) * ARRAY + unit_swz(l >> LP) * 16u +
                   (l & (PER - 1)) * (uint32_t)sizeof(T);
        }
        read16(x, b);
        V acc[4];
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = V{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 16; s++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[r] = mfma(a[r][s], b[s], acc[r]);
        if constexpr (STAGE) {
            // (the wavefront's own vectors: its reads above precede these writes)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t c = (16u * r + 4u * j + kq) & 31u;
                    uint32_t l = vl;
#pragma unroll
                    for (int k = 0; k < 5; k++) l |= ((c >> k) & 1u) << d.bpos[k];
                    const uint32_t o = (buf * 2 + (r >= 2 ? 1 : 0)) * ARRAY +
                                       unit_swz(l >> LP) * 16u + (l & (PER - 1)) * (uint32_t)sizeof(T);
                    *reinterpret_cast<T *>(lds + o) = acc[r][j];
                }
            __syncthreads();
            const uint64_t base = insert_zeros((uint64_t)tile, d.spos, kBK) + lg;
#pragma unroll
            for (uint32_t k = 0; k < ROUNDS; k++) {
                uint64_t g = base;
#pragma unroll
                for (int j = 0; j < (int)(3 - LP); j++)
                    if ((k >> j) & 1u) g += 1ull << d.spos[9 + LP + j];
                const char *from = lds + buf * 2 * ARRAY + (k * kBT + tid) * 16;
                *reinterpret_cast<uint4 *>(re + g) = *reinterpret_cast<const uint4 *>(from);
                *reinterpret_cast<uint4 *>(im + g) = *reinterpret_cast<const uint4 *>(from + ARRAY);
            }
            return;
        }
        const uint64_t at = insert_zeros((uint64_t)tile, d.spos, kBK) + out;
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                uint64_t g = at;
                if (j & 1) g += d.bg[2];
                if (j & 2) g += d.bg[3];
                if (r & 1) g += d.bg[4];
                (r < 2 ? re : im)[g] = acc[r][j];
            }
    };

    // The barrier before each tile ends the reads of the tile before (of the
    // matrix, the first time), so its buffer may be loaded again, and follows
    // the arrival of this one.
    for (; t < tiles; t += step) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tiles - t > step) load(t + step, buf ^ 1u);
        contract(t, buf);
        buf ^= 1u;
    }
}

}  // namespace

// Build the per-lane A fragments of the real 64x64 form of U (32x32 complex,
// row-major interleaved re/im) into out[(r*16+s)*64 + lane].
template <typename T>
static void make_afrag(const double *U, T *out)
{
    for (int r = 0; r < 4; r++)
        for (int s = 0; s < 16; s++)
            for (int lane = 0; lane < 64; lane++) {
                // (f32 accumulators hold row 4 (i / 16) + j: its rows are permuted
                // so that slot j of lane i is component 4 j + i / 16, as in f64)
                const int row = lane & 15;
                const int R = 16 * r + (sizeof(T) == 8 ? row : 4 * (row & 3) + (row >> 2));
                const int C = 4 * s + (lane >> 4);
                const int rr = R & 31, cc = C & 31;
                const double ur = U[2 * (rr * 32 + cc)], ui = U[2 * (rr * 32 + cc) + 1];
                double v;
                if (R < 32) v = C < 32 ? ur : -ui;
                else v = C < 32 ? ui : ur;
                out[(r * 16 + s) * 64 + lane] = (T)v;
            }
}

// Real 64x64 fragments of one block, appended to `out` (4096 values).
void block5_fragments(const double *U, int prec, std::vector<double> &out64,
                      std::vector<float> &out32)
{
    if (prec == SPZ_F64) {
        size_t o = out64.size();
        out64.resize(o + 4096);
        make_afrag<double>(U, out64.data() + o);
    } else {
        size_t o = out32.size();
        out32.resize(o + 4096);
        make_afrag<float>(U, out32.data() + o);
    }
}

// Apply the block whose fragments are at `dfrag` (device) on qubits q[0..4]
// (amplitude index bit j of the block = qubit q[j]).
int launch_block5(spz_state_s *s, const int *q, const void *dfrag)
{
    if (s->n < kBK) return fail(SPZ_ERR_ARG, "dense 5-qubit blocks need at least 12 qubits");
    uint64_t bmask = 0;
    for (int j = 0; j < 5; j++) {
        if (q[j] < 0 || q[j] >= s->n || ((bmask >> q[j]) & 1))
            return fail(SPZ_ERR_QUBIT, "bad block qubits");
        bmask |= 1ull << q[j];
    }
    uint64_t smask = bmask | 0xFull;
    for (int b = 0; b < s->n && __builtin_popcountll(smask) < kBK; b++) smask |= 1ull << b;
    BlockDesc d;
    memset(&d, 0, sizeof d);
    int lbit[64];
    int i = 0;
    for (int b = 0; b < s->n; b++)
        if ((smask >> b) & 1) { d.spos[i] = (int8_t)b; lbit[b] = i++; }
    for (; i < 16; i++) d.spos[i] = 64;
    for (int j = 0; j < 5; j++) d.bpos[j] = (int8_t)lbit[q[j]];
    int nv = 0;
    for (int l = 0; l < kBK; l++) {
        bool isb = false;
        for (int j = 0; j < 5; j++) isb |= d.bpos[j] == l;
        if (!isb) {
            d.vg[nv] = 1ull << d.spos[l];
            d.vpos[nv++] = (int8_t)l;
        }
    }
    for (int j = 0; j < 5; j++) d.bg[j] = 1ull << q[j];
    const uint64_t tiles = s->N >> kBK;
    if (tiles > 0xFFFFFFFFull) return fail(SPZ_ERR_ARG, "state too large for dense 5-qubit blocks");
    // as many workgroups as stay resident (one per CU, FP32 two)
    const uint64_t resident = (uint64_t)std::max(rt().cu_count, 1) * (s->prec == SPZ_F64 ? 1 : 2);
    const unsigned grid = (unsigned)std::min<uint64_t>(tiles, resident);
    const double bytes = 2.0 * (double)s->N * (s->prec == SPZ_F64 ? 16.0 : 8.0);
    LaunchTimer tm(SPZ_K_DENSE, bytes);
    // A store's lanes hold the vector's low bits and two block bits: with more
    // block qubits inside a 128-byte line (qubits 0..3 FP64, 0..4 FP32) it writes
    // parts of lines, and 16-byte stores through LDS are faster.  Measured,
    // direct and staged: 26 qubits FP64, three of them in the line 407-423 and
    // 425-435 us, four 503 and 427 us; 27 qubits FP32, one 421 and 421 us, two
    // 472-496 and 391-460 us, three 648-673 and 414-465 us, five 684 and 386 us.
    const uint64_t line = s->prec == SPZ_F64 ? 0xFull : 0x1Full;
    const bool stage = __builtin_popcountll(bmask & line) >= (s->prec == SPZ_F64 ? 4 : 2);
#define SPZ_B5(T, ST)                                                                           \
    hipLaunchKernelGGL((k_block5<T, ST>), dim3(grid), dim3(kBT), 0, rt().stream, (T *)s->re,      \
                       (T *)s->im, d, (const T *)dfrag, (uint32_t)tiles)
    if (s->prec == SPZ_F64) {
        if (stage) SPZ_B5(double, true);
        else SPZ_B5(double, false);
    } else {
        if (stage) SPZ_B5(float, true);
        else SPZ_B5(float, false);
    }
#undef SPZ_B5
    SPZ_HIP(hipGetLastError());
    return SPZ_OK;
}

}  // namespace spz
