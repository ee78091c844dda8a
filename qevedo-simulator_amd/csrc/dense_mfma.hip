// Fused dense gates, applied as real GEMMs on matrix cores: complex64 with
// K = 5 or 6 targets through v_mfma_f32_16x16x4f32, complex128 with 3 to 6
// through v_mfma_f64_16x16x4f64 (accumulation in the state's precision).
//
// A column is one group of D = 2^K amplitudes the gate mixes (the iteration
// index spread over the non-target, non-control bits, as in k_dense). With
// U = Ur + i Ui the output's parts are real dot products of the column's
// parts with the rows of a 2D x 2D real matrix R, so a block of NC columns is
// the product (2D x 2D) x (2D x NC). R's rows interleave the real and
// imaginary part of each index, so that the four accumulators of a lane
// are two whole amplitudes of one column: they go to memory straight from
// the accumulators, 16 neighbouring columns (128 or 256 bytes) at a time.
// The sums run over the real parts of the column and then the imaginary ones
// in complex64 (the staged block holds them as two planes), over both
// parts of each index in turn in complex128.
//
// A workgroup has one wave per 16 rows of R (8 for K = 6, 1 for K = 3); each
// wave keeps its rows in registers for the whole launch. Blocks of NC columns
// pass through two LDS buffers: while the waves multiply block b, block b + 1
// is in flight from memory, and it is written to the other buffer before the
// one barrier of the iteration.
//
// Bounds at 28 qubits: one pass is 0.79 ms in complex64 and 1.58 ms in
// complex128 at the 5.4 TB/s of a large copy; the products of a 6-qubit gate
// are 0.87 ms at the FP32 matrix peak and 1.75 ms at the FP64 one
// (78.6 TFLOP/s, as the FP64 vector rate), half of that for 5 qubits. Measured
// kernels: K = 6 1.16-1.21 ms and 2.06-2.10 ms (the products, at 72 to 75 and
// 83 to 85 % of their peak), K = 5 0.87-0.92 ms and 1.62-1.80 ms (memory); one
// LDS buffer, outputs through LDS and four barriers per block took 1.32-1.50
// and 0.89-1.19 ms in complex64. At 32 qubits K = 6 takes 18.1-19.7 ms
// (20.2-22.9). 74 registers in complex64 leave room for three workgroups of
// K = 6 on a CU; with 84 there were two (28 qubits: 1.24-1.43 ms).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

#include "dense_mfma.h"

namespace qvd {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

// The 16 x 16 x 4 matrix instruction of a precision. Operand A: lane l holds
// row l % 16, k = l / 16; operand B: column l % 16, k = l / 16. Accumulator
// e of lane l is column l % 16 and row 4 (l / 16) + e in FP32, row
// 4 e + l / 16 in FP64.
template <typename T2> struct Mfma;
template <> struct Mfma<float2> {
    using R = float;
    using V = floatx4;
    static __device__ __forceinline__ V mul(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // Row r of a tile is accumulator `e` of the lanes l with l / 16 = `q`.
    static __device__ __forceinline__ uint32_t q_of(uint32_t r) { return r >> 2; }
    static __device__ __forceinline__ uint32_t e_of(uint32_t r) { return r & 3; }
};
template <> struct Mfma<double2> {
    using R = double;
    using V = doublex4;
    static __device__ __forceinline__ V mul(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t q_of(uint32_t r) { return r & 3; }
    static __device__ __forceinline__ uint32_t e_of(uint32_t r) { return r >> 2; }
};

constexpr int NC = 32;         // columns per block
constexpr int CB = 5;          // column bits of a block
static_assert(NC == 1 << CB, "a block's columns are all values of its column bits");
// Row pitch of a staged block: amplitudes in complex128; in complex64 floats
// of a plane, a multiple of 16 but not of 32, so that the four rows a
// wave reads at once (16 columns each) lie in different banks.
template <typename T2> constexpr int PITCH = sizeof(T2) == 8 ? NC + 16 : NC + 1;
template <typename T2, int K> constexpr int BLOCK = (1 << K) * PITCH<T2>;  // amplitudes of one staged block
constexpr int SLOTS = 3;       // column bases of the block multiplied, loaded and prepared
constexpr int PER = 4;         // amplitudes staged per thread (8 D threads, D x NC amplitudes)

// Where a staged amplitude belongs: its column in the block, its place in the
// buffer and its offset within the column. Each is a sum over the bits of the
// amplitude's number tid + i * threads, so tid's part is a thread's own and i's
// part the same for the workgroup (three registers a thread instead of 16).
struct Place {
    uint64_t off;
    uint32_t col, at;
};
template <int K>
struct Places {
    Place bit[K + 3];  // of each bit of tid
    Place elem[PER];   // of each i
};

__device__ __forceinline__ uint64_t spread(uint64_t x, const uint32_t *pos, uint32_t m) {
    for (uint32_t j = 0; j < m; j++) {
        const uint32_t p = pos[j];
        const uint64_t low = x & ((uint64_t(1) << p) - 1);
        x = ((x >> p) << (p + 1)) | low;
    }
    return x;
}

// v, unknown to the optimiser: what is computed from it is not kept in registers
// across a loop.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <typename T2, int K>
constexpr size_t mfma_lds_bytes() {
    return 2 * sizeof(T2) * (size_t)BLOCK<T2, K> + SLOTS * NC * sizeof(uint64_t);
}

template <typename T2, int K>
__global__ __launch_bounds__(64 << (K - 3)) void k_dense_mfma(T2 *__restrict__ s, const GateDesc d,
                                                              const T2 *__restrict__ mat, const Places<K> p) {
    using M = Mfma<T2>;
    using R = typename M::R;
    using V = typename M::V;
    constexpr int D = 1 << K, THREADS = 8 * D;  // 2D / 16 waves
    constexpr int KS = 2 * D / 4;               // k steps of 4
    static_assert(D * NC == PER * THREADS, "a block is PER amplitudes a thread");
    constexpr uint64_t NONE = ~uint64_t(0);     // a column past the last one
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    T2 *const buf = reinterpret_cast<T2 *>(smem_raw);                       // two blocks
    uint64_t *const colbase = reinterpret_cast<uint64_t *>(buf + 2 * BLOCK<T2, K>);  // SLOTS x NC
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, cl = lane & 15;
    const uint64_t blocks = (d.iterations + NC - 1) / NC;
    uint64_t blk = blockIdx.x;
    if (blk >= blocks) return;  // uniform over the workgroup
    const uint64_t step = gridDim.x;
    auto bases = [&](uint64_t b, uint32_t slot) {
        if (tid < (uint32_t)NC && b < blocks) {
            const uint64_t col = b * NC + tid;
            colbase[slot * NC + tid] = col < d.iterations ? (spread(col, d.ins, d.nins) | d.ctrl_val) : NONE;
        }
    };

    // This wave's rows of R. Row indices pair up as (index of U, part): the
    // lane's accumulators e are index 2q + e / 2 of the wave's 8 and part
    // e % 2. k = 4 ks + q is index k % D, part k / D in complex64, index k / 2,
    // part k % 2 in complex128.
    // Every load is unconditional: where a part was chosen after the load, the
    // compiler branched around each one and waited for it (20 qubits, K = 6:
    // 27.5 us a pass, 14.8 so).
    constexpr bool PLANES = sizeof(T2) == 8;
    R ra[KS];
    {
        const uint32_t jr = wave * 8 + 2 * M::q_of(cl) + (M::e_of(cl) >> 1), im = M::e_of(cl) & 1;
        if constexpr (PLANES) {
#pragma unroll
            for (int ks = 0; ks < KS / 2; ks++) {
                const T2 u = mat[jr * D + 4 * ks + q];
                ra[ks] = im ? u.y : u.x;
                ra[ks + KS / 2] = im ? u.x : -u.y;
            }
        } else {
            const R *const row = reinterpret_cast<const R *>(mat + jr * D + (q >> 1)) + ((q & 1) ^ im);
            const bool neg = (q & 1) > im;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const R v = row[4 * ks];
                ra[ks] = neg ? -v : v;
            }
        }
    }
    // The thread's part of the place of its elements tid + i * THREADS.
    uint32_t c_tid = 0, a_tid = 0;
    uint64_t o_tid = 0;
#pragma unroll
    for (int b = 0; b < K + 3; b++) {
        const uint32_t bit = (tid >> b) & 1;
        c_tid += bit ? p.bit[b].col : 0;
        a_tid += bit ? p.bit[b].at : 0;
        o_tid += bit ? p.bit[b].off : 0;
    }
    // Accumulators 0, 1 are index `wave * 8 + 2 q`, 2 and 3 the next one.
    uint64_t so = 0;
    const uint64_t so_next = d.offsets[1];
#pragma unroll
    for (int t = 1; t < K; t++)
        if (((t < 3 ? 2 * q : wave * 8) >> t) & 1) so += d.offsets[1u << t];

    // Qubit 0 is matrix bit 0: a lane's two amplitudes are neighbours, the
    // first at an even index (16-byte aligned in complex64).
    const bool adjacent = d.offsets[1] == 1;

    bases(blk, 0);
    bases(blk + step, 1);
    __syncthreads();
    T2 pre[PER];
    auto fetch = [&](uint32_t slot) {
        const uint32_t c = opaque(c_tid);
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const uint64_t b = colbase[slot * NC + c + p.elem[i].col];
            pre[i].x = pre[i].y = 0;
            if (b != NONE) pre[i] = s[b + o_tid + p.elem[i].off];
        }
    };
    auto stage = [&](T2 *b) {
        const uint32_t a = opaque(a_tid);
        if constexpr (PLANES) {
            R *const f = reinterpret_cast<R *>(b);
#pragma unroll
            for (int i = 0; i < PER; i++) {
                f[a + p.elem[i].at] = pre[i].x;
                f[BLOCK<T2, K> + a + p.elem[i].at] = pre[i].y;
            }
        } else {
#pragma unroll
            for (int i = 0; i < PER; i++) b[a + p.elem[i].at] = pre[i];
        }
    };
    fetch(0);
    stage(buf);
    __syncthreads();
    uint32_t cur = 0, slot = 0;
    for (;;) {
        const uint64_t next = blk + step;
        const bool more = next < blocks;
        const uint32_t slot1 = slot + 1 == SLOTS ? 0 : slot + 1, slot2 = slot1 + 1 == SLOTS ? 0 : slot1 + 1;
        if (more) fetch(slot1);
        bases(next + step, slot2);
        const R *const cb = reinterpret_cast<const R *>(buf + cur * BLOCK<T2, K>);
        const R *const bp = PLANES ? cb + q * PITCH<T2> + cl : cb + 2 * ((q >> 1) * PITCH<T2> + cl) + (q & 1);
        // k step ks from bp: 4 rows of a plane (the second plane follows the
        // first), or 2 rows of amplitudes.
        constexpr int STEP = 4 * PITCH<T2>, COL = PLANES ? 1 : 2;
        V acc[NC / 16];
#pragma unroll
        for (int g = 0; g < NC / 16; g++) acc[g] = V{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
#pragma unroll
            for (int g = 0; g < NC / 16; g++) acc[g] = M::mul(ra[ks], bp[ks * STEP + COL * 16 * g], acc[g]);
        }
#pragma unroll
        for (int g = 0; g < NC / 16; g++) {
            const uint64_t b = colbase[slot * NC + 16 * g + cl];
            if (b != NONE) {
                T2 o0, o1;
                o0.x = acc[g][0];
                o0.y = acc[g][1];
                o1.x = acc[g][2];
                o1.y = acc[g][3];
                if (sizeof(T2) == 8 && adjacent) {
                    *reinterpret_cast<float4 *>(s + b + so) = make_float4(o0.x, o0.y, o1.x, o1.y);
                } else {
                    s[b + so] = o0;
                    s[b + so + so_next] = o1;
                }
            }
        }
        if (!more) break;
        stage(buf + (cur ^ 1) * BLOCK<T2, K>);
        __syncthreads();
        cur ^= 1;
        slot = slot1;
        blk = next;
    }
}

// The staging order: bit b of an amplitude's number is an index bit of the gate
// or a column bit. The lowest ones follow the qubits they stand for (targets,
// and the lowest free qubits, which the columns of a block span) over a
// 128-byte line, so neighbouring threads load whole lines whichever qubits the
// targets are. Then come the other column bits, then the other index bits: a
// wave writes a few rows of the buffer, not one per thread, whose starts share
// banks in complex64 (targets 0 to 5, 28 qubits, two workgroups per CU: 1434 us a
// pass with a row per thread, 1311 so). A free bit past the last qubit is a column past the last one.
template <typename T2, int K>
Places<K> staging_places(const GateDesc &d) {
    constexpr int LINE = sizeof(T2) == 8 ? 4 : 3;  // bits of an amplitude's place in a line
    Place bits[K + CB];
    int at = 0, f = 0;  // bits and column bits placed
    uint32_t used = 0, fq = 0, ins = 0;  // targets placed, the next free qubit, targets and controls below it
    auto column = [&] {
        bits[at++] = {0, 1u << f, 1u << f};
        f++;
        fq++;
    };
    auto target = [&](int t) {
        bits[at++] = {d.offsets[1 << t], 0, (uint32_t)PITCH<T2> << t};
        used |= 1u << t;
    };
    auto lowest = [&] {  // of the targets left, or -1
        int t = -1;
        for (int k = 0; k < K; k++)
            if (!((used >> k) & 1) && (t < 0 || d.offsets[1 << k] < d.offsets[1 << t])) t = k;
        return t;
    };
    while (at < LINE) {
        for (; ins < d.nins && d.ins[ins] <= fq; ins++) fq += d.ins[ins] == fq;
        const int t = lowest();
        if (t < 0 || (f < CB && (uint64_t(1) << fq) < d.offsets[1 << t])) column();
        else target(t);
    }
    while (f < CB) column();
    for (int t; (t = lowest()) >= 0;) target(t);
    Places<K> p;
    std::copy(bits, bits + K + 3, p.bit);
    for (int i = 0; i < PER; i++) {
        p.elem[i] = {0, 0, 0};
        for (int b = 0; b < 2; b++) {
            const Place &x = bits[K + 3 + b];
            if ((i >> b) & 1) p.elem[i] = {p.elem[i].off + x.off, p.elem[i].col + x.col, p.elem[i].at + x.at};
        }
    }
    return p;
}

// Workgroups launched per CU, given the blocks per CU. K = 6: two are resident
// in complex128 and three in complex64, where an odd number of them leaves the last
// round uneven unless there are many rounds (22 qubits, 8 blocks per CU: two 45 us,
// three 51, six 71; 24 qubits: 103, 106, 119). From 128 blocks per CU on, more
// of them than are resident start as others end, which evens their
// rounds out (26 qubits: two 337 us, six 337; 28: 1264 and 1215; 32: 21.6 and
// 19.7 ms). K = 5 in complex64 is the same from 512 on (28 qubits, 12 per CU 922 us,
// 24 899; 24 qubits: 71 and 84); in complex128 12 are as good (28 qubits: 1.67
// ms, 24 1.69). Fewer targets: many small ones.
template <typename T2, int K>
uint64_t groups_per_cu(uint64_t blocks) {
    if (K == 6) return sizeof(T2) == 8 && blocks >= 128 ? 6 : 2;
    if (K == 5) return sizeof(T2) == 8 && blocks >= 512 ? 24 : 12;
    return 32;
}

template <typename T2, int K>
hipError_t launch_k(T2 *s, const GateDesc &d, const T2 *mat, unsigned cus, hipStream_t st) {
    constexpr size_t lds = mfma_lds_bytes<T2, K>();
    static std::atomic<uint64_t> attr_set{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = uint64_t(1) << (dev & 63);
    if (!(attr_set.load() & bit)) {
        e = hipFuncSetAttribute((const void *)k_dense_mfma<T2, K>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        attr_set.fetch_or(bit);
    }
    const uint64_t blocks = (d.iterations + NC - 1) / NC;
    const unsigned grid = (unsigned)std::min<uint64_t>(blocks, cus * groups_per_cu<T2, K>(blocks / cus));
    k_dense_mfma<T2, K><<<grid, 64 << (K - 3), lds, st>>>(s, d, mat, staging_places<T2, K>(d));
    return hipGetLastError();
}

}  // namespace

template <typename T2>
hipError_t launch_dense_mfma(T2 *s, const GateDesc &d, const T2 *mat, unsigned cus, hipStream_t st) {
    if constexpr (sizeof(T2) == 16) {
        if (d.k == 3) return launch_k<T2, 3>(s, d, mat, cus, st);
        if (d.k == 4) return launch_k<T2, 4>(s, d, mat, cus, st);
    }
    if (d.k == 5) return launch_k<T2, 5>(s, d, mat, cus, st);
    if (d.k == 6) return launch_k<T2, 6>(s, d, mat, cus, st);
    return hipErrorInvalidValue;
}
template hipError_t launch_dense_mfma<float2>(float2 *, const GateDesc &, const float2 *, unsigned, hipStream_t);
template hipError_t launch_dense_mfma<double2>(double2 *, const GateDesc &, const double2 *, unsigned, hipStream_t);

}  // namespace qvd
