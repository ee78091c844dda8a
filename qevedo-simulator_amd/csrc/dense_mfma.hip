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
// Bounds at 28 qubits (2^28 columns x amplitudes): one pass is 0.79 ms in
// complex64 and 1.58 ms in complex128 at the 5.4 TB/s of a large copy; the
// products of a 6-qubit gate are 0.87 ms at the FP32 matrix peak and 1.75 ms
// at the FP64 one (78.6 TFLOP/s, as the FP64 vector rate), half of that for 5
// qubits. Measured, host call included: K = 6 1.23 ms and 2.14 ms (the
// products, at 71 and 82 % of their peak), K = 5 0.95 ms and 1.67-1.84 ms
// (memory). Before, with one LDS buffer, outputs through LDS and four barriers
// per block, FP32 K = 6 took 1.38 ms and K = 5 0.97 ms; complex128 ran on
// vector FMAs with the matrix in LDS: 12.0 ms and 9.1 ms. Blocks of 64
// columns: 1.26 and 2.46 ms. Workgroups per CU: two for K = 6, what its
// registers allow (12: 1.28 ms, each workgroup loading its rows of R again);
// many small ones for the others (K = 5 in FP32: 2 1.04, 3 0.92, 12 0.92 ms).
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

__device__ __forceinline__ uint64_t spread(uint64_t x, const uint32_t *pos, uint32_t m) {
    for (uint32_t j = 0; j < m; j++) {
        const uint32_t p = pos[j];
        const uint64_t low = x & ((uint64_t(1) << p) - 1);
        x = ((x >> p) << (p + 1)) | low;
    }
    return x;
}

template <typename T2, int K>
constexpr size_t mfma_lds_bytes() {
    return 2 * sizeof(T2) * (size_t)BLOCK<T2, K> + SLOTS * NC * sizeof(uint64_t);
}

template <typename T2, int K>
__global__ __launch_bounds__(64 << (K - 3)) void k_dense_mfma(T2 *__restrict__ s, const GateDesc d,
                                                              const T2 *__restrict__ mat) {
    using M = Mfma<T2>;
    using R = typename M::R;
    using V = typename M::V;
    constexpr int D = 1 << K, THREADS = 8 * D;  // 2D / 16 waves
    constexpr int KS = 2 * D / 4;               // k steps of 4
    constexpr int PER = D * NC / THREADS;       // amplitudes staged per thread
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
    constexpr bool PLANES = sizeof(T2) == 8;
    R ra[KS];
    {
        const uint32_t jr = wave * 8 + 2 * M::q_of(cl) + (M::e_of(cl) >> 1), im = M::e_of(cl) & 1;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const uint32_t k = 4 * ks + q;
            const T2 u = mat[jr * D + (PLANES ? k & (D - 1) : k >> 1)];
            ra[ks] = (PLANES ? k >> K : k & 1) == im ? u.x : (im ? u.y : -u.y);
        }
    }
    // Staging order: element e of a block takes its index bits in ascending
    // order of the qubits they stand for (targets, and the lowest free qubits
    // that the columns of a block span), so neighbouring threads load
    // neighbouring amplitudes whichever qubits the targets are. `tq` and `fq`
    // walk both sets; a free bit past the last qubit is a column past the
    // last one.
    uint32_t tbits[K + CB];  // bit i of e: index bit (below K) or K + column bit
    {
        uint32_t f = 0, fq = 0, ins = 0;  // next column bit, its qubit, the inserted (target or control) qubits passed
        uint32_t used = 0;                // targets taken
        for (int i = 0; i < K + CB; i++) {
            while (ins < d.nins && d.ins[ins] <= fq) {  // fq: the next qubit that is no target or control
                if (d.ins[ins] == fq) fq++;
                ins++;
            }
            uint32_t lowest = 0;
            uint64_t lo = ~uint64_t(0);
#pragma unroll
            for (int t = 0; t < K; t++)
                if (!((used >> t) & 1) && d.offsets[1 << t] < lo) {
                    lo = d.offsets[1 << t];
                    lowest = t;
                }
            if (f < (uint32_t)CB && (used == (1u << K) - 1 || (uint64_t(1) << fq) < lo)) {
                tbits[i] = K + f++;
                fq++;
            } else {
                tbits[i] = lowest;
                used |= 1u << lowest;
            }
        }
    }
    uint64_t eo[PER];           // offset of each staged amplitude within its column
    uint32_t ec[PER], ea[PER];  // its column in the block, its place in the buffer
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const uint32_t e = tid + i * THREADS;
        uint32_t jc = 0;
        for (int b = 0; b < K + CB; b++) jc |= ((e >> b) & 1) << tbits[b];
        const uint32_t j = jc & (D - 1);
        ec[i] = jc >> K;
        ea[i] = j * PITCH<T2> + ec[i];
        eo[i] = d.offsets[j];
    }
    const uint64_t so0 = d.offsets[wave * 8 + 2 * q], so1 = d.offsets[wave * 8 + 2 * q + 1];

    // Qubit 0 is matrix bit 0: a lane's two amplitudes are neighbours, the
    // first at an even index (16-byte aligned in complex64).
    const bool adjacent = d.offsets[1] == 1;

    bases(blk, 0);
    bases(blk + step, 1);
    __syncthreads();
    T2 pre[PER];
    auto fetch = [&](uint32_t slot) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const uint64_t b = colbase[slot * NC + ec[i]];
            pre[i].x = pre[i].y = 0;
            if (b != NONE) pre[i] = s[b + eo[i]];
        }
    };
    auto stage = [&](T2 *b) {
        if constexpr (PLANES) {
            R *const f = reinterpret_cast<R *>(b);
#pragma unroll
            for (int i = 0; i < PER; i++) {
                f[ea[i]] = pre[i].x;
                f[BLOCK<T2, K> + ea[i]] = pre[i].y;
            }
        } else {
#pragma unroll
            for (int i = 0; i < PER; i++) b[ea[i]] = pre[i];
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
                    *reinterpret_cast<float4 *>(s + b + so0) = make_float4(o0.x, o0.y, o1.x, o1.y);
                } else {
                    s[b + so0] = o0;
                    s[b + so1] = o1;
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
    const unsigned grid = (unsigned)std::min<uint64_t>(blocks, (uint64_t)cus * (K == 6 ? 2 : K == 5 ? 12 : 32));
    k_dense_mfma<T2, K><<<grid, 64 << (K - 3), lds, st>>>(s, d, mat);
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
