// HIP kernels of the MI355X state-vector engine (gfx950, wave64).
//
// State layout in HBM: 2^n interleaved complex amplitudes (float2 for
// complex64, double2 for complex128) in logical index order; qubit q is bit q
// of the index. Every kernel here is HBM-bound except the in-tile gate
// arithmetic of deep stages.
//
// Compiled with -ffp-contract=off: fused multiply-adds appear only where
// written (fma / fmaf), so the arithmetic is the same on every build.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <atomic>
#include <mutex>

#include "device.h"
#include "kernels.h"

// Constant address space: uniform loads through these pointers are scalar.
#if defined(__HIP_DEVICE_COMPILE__)
#define QVD_CONST __attribute__((address_space(4)))
#else
#define QVD_CONST
#endif

namespace qvd {

// ---------------------------------------------------------------------------
// Complex helpers.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float fmul_add(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmul_add(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename T2> struct Real;
template <> struct Real<float2> { using T = float; };
template <> struct Real<double2> { using T = double; };

// acc += w * x, as four fused multiply-adds.
template <typename T2>
__device__ __forceinline__ void cmac(T2 &acc, const T2 w, const T2 x) {
    acc.x = fmul_add(w.x, x.x, acc.x);
    acc.x = fmul_add(-w.y, x.y, acc.x);
    acc.y = fmul_add(w.x, x.y, acc.y);
    acc.y = fmul_add(w.y, x.x, acc.y);
}

// f * a, with the rounding of the reference's diagonal kernel
// (re = f.re*a.re - f.im*a.im with the second product fused; im likewise,
// src/kernels.rs:464-465).
template <typename T2>
__device__ __forceinline__ T2 cmul_diag(const T2 f, const T2 a) {
    T2 r;
    r.x = fmul_add(-f.y, a.y, f.x * a.x);
    r.y = fmul_add(f.y, a.x, f.x * a.y);
    return r;
}

// Insert a zero bit at each of the ascending positions pos[0..m).
__device__ __forceinline__ uint64_t insert_zeros(uint64_t x, const uint32_t *pos, uint32_t m) {
    for (uint32_t j = 0; j < m; j++) {
        const uint32_t p = pos[j];
        const uint64_t low = x & ((uint64_t(1) << p) - 1);
        x = ((x >> p) << (p + 1)) | low;
    }
    return x;
}

// ---------------------------------------------------------------------------
// Initialisation and conversion.
// ---------------------------------------------------------------------------
template <typename T2>
__global__ void k_init_zero(T2 *__restrict__ s, uint64_t len) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += stride) {
        T2 v;
        v.x = i == 0 ? 1 : 0;
        v.y = 0;
        s[i] = v;
    }
}

// Writes zero over every amplitude whose index has a bit of `stale` set.
template <typename T2>
__global__ void k_zero_stale(T2 *__restrict__ s, uint64_t len, uint64_t stale) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += stride) {
        if (i & stale) {
            T2 v;
            v.x = 0;
            v.y = 0;
            s[i] = v;
        }
    }
}

template <typename T2>
__global__ void k_widen(const T2 *__restrict__ s, double2 *__restrict__ out, uint64_t count) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        const T2 v = s[i];
        out[i] = make_double2((double)v.x, (double)v.y);
    }
}

template <typename T2>
__global__ void k_narrow(const double2 *__restrict__ in, T2 *__restrict__ s, uint64_t count) {
    using T = typename Real<T2>::T;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        const double2 v = in[i];
        T2 o;
        o.x = (T)v.x;
        o.y = (T)v.y;
        s[i] = o;
    }
}

template <typename T2>
__global__ void k_scale(T2 *__restrict__ s, uint64_t len, double factor) {
    using T = typename Real<T2>::T;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += stride) {
        T2 v = s[i];
        v.x = (T)((double)v.x * factor);
        v.y = (T)((double)v.y * factor);
        s[i] = v;
    }
}

// ---------------------------------------------------------------------------
// Full-state ops: one HBM pass each.
// ---------------------------------------------------------------------------

// A dense op on K targets: each thread owns one group of 2^K amplitudes
// (the iteration index spread over the non-target, non-control bits). The
// matrix is the same for every thread. For K <= 2 it sits in scalar registers
// as a whole and enters the FMAs from there. From K = 3 on its rows come from
// LDS, a few at a time: that keeps the registers to what a wave needs (all
// rows unrolled, the compiler holds the matrix and one wave per SIMD is left),
// and a row is there in the time of an LDS read. Rows through the scalar
// cache are waited for one by one (20 qubits, complex64, 4 targets: 12.0 us, 9.1
// so; 18 qubits, complex128, 3 targets: 7.5 and 6.6), and a 6-qubit matrix in
// complex128 does not fit it (24 qubits: 950 us, 648 so). Only the
// 4-qubit gates of complex128 stay there, for the large states they are fused
// for: from LDS 27 qubits with targets 23-26 take 0.94 ms instead of 0.85 and other
// targets the same, while 16 qubits would take 9.3 us instead of 11.8.
//
// A pass is bound by memory up to K = 4 (28 qubits, targets 4-7: 0.78 ms in
// complex64 and 1.60 ms in complex128, a copy of the state taking 0.79 and 1.58).
//
// The matrix is in device memory, or is itself an argument of the launch
// (MatArg; a gate applied by itself needs no copy in front of its pass then).
template <typename T2, int K>
struct MatArg {
    T2 m[1 << (2 * K)];
};
template <typename T2>
__device__ __forceinline__ T2 mat_at(const T2 *mat, int i) {
    return (T2)((const QVD_CONST T2 *)mat)[i];
}
template <typename T2, int K>
__device__ __forceinline__ T2 mat_at(const MatArg<T2, K> &mat, int i) {
    return mat.m[i];
}

template <typename T2>
constexpr bool dense_in_lds(int k) {
    return k >= 3 && !(sizeof(T2) == 16 && k == 4);
}

template <typename T2, int K, typename M>
__global__ __launch_bounds__(256) void k_dense(T2 *__restrict__ s, const GateDesc d, const M mat) {
    constexpr int D = 1 << K;
    constexpr bool LDS = dense_in_lds<T2>(K);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    T2 *const m = reinterpret_cast<T2 *>(smem_raw);
    if (LDS) {
        for (int i = threadIdx.x; i < D * D; i += blockDim.x) m[i] = mat_at(mat, i);
        __syncthreads();
    }
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t it = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; it < d.iterations; it += stride) {
        T2 *const g = s + (insert_zeros(it, d.ins, d.nins) | d.ctrl_val);
        T2 a[D];
#pragma unroll
        for (int j = 0; j < D; j++) a[j] = g[d.offsets[j]];
        // Rows in batches whose matrix elements are 64 registers at most.
        constexpr int FIT = 256 / (D * (int)sizeof(T2));
        constexpr int U = K < 3 ? D : FIT > 1 ? FIT : 1;
#pragma unroll U
        for (int r = 0; r < D; r++) {
            T2 acc;
            acc.x = 0;
            acc.y = 0;
#pragma unroll
            for (int c = 0; c < D; c++) cmac(acc, LDS ? m[r * D + c] : mat_at(mat, r * D + c), a[c]);
            g[d.offsets[r]] = acc;
        }
    }
}

// A diagonal op: amplitude i is multiplied by entries[index of its target
// bits] where every control bit holds.
template <typename T2>
__global__ __launch_bounds__(256) void k_diag(T2 *__restrict__ s, uint64_t len, const uint32_t k,
                                              const DiagTargets t, uint64_t cmask, uint64_t cval,
                                              const T2 *__restrict__ entries) {
    __shared__ T2 e[1 << MAX_GATE_QUBITS];
    for (uint32_t i = threadIdx.x; i < (1u << k); i += blockDim.x) e[i] = entries[i];
    __syncthreads();
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += stride) {
        if ((i & cmask) != cval) continue;
        uint32_t idx = 0;
        for (uint32_t j = 0; j < k; j++) idx |= (uint32_t)((i >> t.q[j]) & 1) << j;
        s[i] = cmul_diag(e[idx], s[i]);
    }
}

// ---------------------------------------------------------------------------
// LDS-tile stages: one HBM pass applies every op of a stage.
//
// A workgroup loads a tile of 2^L amplitudes whose index bits are the
// stage's tile qubits (the lowest `contig` qubits among them, so each HBM
// access is a contiguous run), applies the stage's ops in LDS, and writes
// the tile back. Non-tile qubits are fixed per tile: non-tile controls
// select whether an op runs on the tile at all, and non-tile diagonal targets
// select the entries used.
//
// States smaller than a register tile are one such tile, so one workgroup
// works through the ops and each op's latency counts. The op records and
// matrices of a run of ops are therefore copied to LDS together (a load per
// op was a memory round trip per op), and an op of fewer groups than threads
// deals the rows of its matrix out as well: 12 qubits in complex128, 120 gates
// fused to 4 qubits, 541 -> 91 us. (With 1024 threads in complex128 the 128 VGPRs a
// thread gets leave 64 bytes of it in scratch.)
// ---------------------------------------------------------------------------
constexpr uint32_t STAGE_OPS = 48;             // op records held in LDS
constexpr uint32_t STAGE_COEF_BYTES = 8192;    // their matrices and diagonals
static_assert(STAGE_OPS <= 64, "one lane per op record");
static_assert(sizeof(StageOp) % 4 == 0, "op records are copied by words");

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Spreads x over the bits not set in `taken`.
__device__ __forceinline__ uint32_t spread_around(uint32_t x, uint32_t taken) {
    while (taken) {
        const uint32_t p = __builtin_ctz(taken);
        x = ((x >> p) << (p + 1)) | (x & ((1u << p) - 1));
        taken &= taken - 1;
    }
    return x;
}

// A dense op with rows dealt out: 2^LR threads share a group of 2^K amplitudes,
// each computing 2^(K - LR) rows.
template <typename T2, int K, int LR>
__device__ __forceinline__ void tile_rows(T2 *__restrict__ tile, const T2 *__restrict__ m, const uint32_t (&tb)[K],
                                          uint32_t taken, uint32_t val, uint32_t lg) {
    constexpr int D = 1 << K, RPT = D >> LR;
    const uint32_t sub = threadIdx.x >> lg;
    const bool active = sub < (1u << LR);
    const uint32_t i0 = spread_around(threadIdx.x & ((1u << lg) - 1), taken) | val;
    T2 acc[RPT];
    if (active) {
        T2 a[D];
#pragma unroll
        for (int j = 0; j < D; j++) {
            uint32_t o = 0;
#pragma unroll
            for (int b = 0; b < K; b++)
                if ((j >> b) & 1) o |= tb[b];
            a[j] = tile[i0 | o];
        }
        const T2 *row = m + sub * RPT * D;
#pragma unroll
        for (int r = 0; r < RPT; r++) {
            acc[r].x = 0;
            acc[r].y = 0;
#pragma unroll
            for (int c = 0; c < D; c++) cmac(acc[r], row[r * D + c], a[c]);
        }
    }
    __syncthreads();
    if (active) {
#pragma unroll
        for (int r = 0; r < RPT; r++) {
            const uint32_t j = sub * RPT + r;
            uint32_t o = 0;
#pragma unroll
            for (int b = 0; b < K; b++)
                if ((j >> b) & 1) o |= tb[b];
            tile[i0 | o] = acc[r];
        }
    }
}

template <typename T2, int K, int LOG_THREADS>
__device__ __forceinline__ void tile_dense(T2 *__restrict__ tile, const T2 *__restrict__ m, const StageOp &op,
                                           uint32_t L) {
    constexpr int D = 1 << K;
    uint32_t tb[K];
#pragma unroll
    for (int b = 0; b < K; b++) tb[b] = 1u << uniform(op.tgt[b]);
    const uint32_t taken = uniform(op.taken), val = uniform(op.lc_val);
    const uint32_t lg = L - __builtin_popcount(taken);
    if (lg < LOG_THREADS) {
        const uint32_t lr = LOG_THREADS - lg;
        if (lr == 1) tile_rows<T2, K, 1>(tile, m, tb, taken, val, lg);
        else if (K == 2 || lr == 2) tile_rows<T2, K, K < 2 ? K : 2>(tile, m, tb, taken, val, lg);
        else if (K == 3 || lr == 3) tile_rows<T2, K, K < 3 ? K : 3>(tile, m, tb, taken, val, lg);
        else tile_rows<T2, K, K < 4 ? K : 4>(tile, m, tb, taken, val, lg);
        return;
    }
    for (uint32_t g = threadIdx.x; g < (1u << lg); g += 1u << LOG_THREADS) {
        const uint32_t i0 = spread_around(g, taken) | val;
        T2 a[D];
#pragma unroll
        for (int j = 0; j < D; j++) {
            uint32_t o = 0;
#pragma unroll
            for (int b = 0; b < K; b++)
                if ((j >> b) & 1) o |= tb[b];
            a[j] = tile[i0 | o];
        }
        // Rows one at a time from K = 3 on, their offset rebuilt from r.
        constexpr int U = K < 3 ? D : 1;
#pragma unroll U
        for (int r = 0; r < D; r++) {
            T2 acc;
            acc.x = 0;
            acc.y = 0;
#pragma unroll
            for (int c = 0; c < D; c++) cmac(acc, m[r * D + c], a[c]);
            uint32_t o = 0;
#pragma unroll
            for (int b = 0; b < K; b++) o |= ((r >> b) & 1) ? tb[b] : 0;
            tile[i0 | o] = acc;
        }
    }
}

template <typename T2, int LOG_THREADS>
__device__ __forceinline__ void tile_diag(T2 *__restrict__ tile, const T2 *__restrict__ e, const StageOp &op,
                                          uint32_t L, uint64_t base) {
    const uint32_t k = uniform(op.k), lc_mask = uniform(op.lc_mask), lc_val = uniform(op.lc_val);
    uint32_t gidx = 0, pos[MAX_GATE_QUBITS];
#pragma unroll
    for (uint32_t j = 0; j < MAX_GATE_QUBITS; j++) {
        pos[j] = 0;
        if (j >= k) continue;
        const uint32_t t = uniform(op.tgt[j]);
        if (t & GLOBAL_BIT) gidx |= (uint32_t)((base >> (t & ~GLOBAL_BIT)) & 1) << j;
        else pos[j] = 1u << t;
    }
    const uint32_t tsize = 1u << L;
    for (uint32_t i = threadIdx.x; i < tsize; i += 1u << LOG_THREADS) {
        if ((i & lc_mask) != lc_val) continue;
        uint32_t idx = gidx;
#pragma unroll
        for (uint32_t j = 0; j < MAX_GATE_QUBITS; j++) idx |= (i & pos[j]) ? 1u << j : 0;
        tile[i] = cmul_diag(e[idx], tile[i]);
    }
}

template <typename T2, int LOG_THREADS>
__global__ __launch_bounds__(1 << LOG_THREADS) void k_stage(T2 *__restrict__ s, const StageDesc d,
                                                            const StageOp *__restrict__ ops,
                                                            const T2 *__restrict__ coefs) {
    constexpr uint32_t THREADS = 1u << LOG_THREADS, CMAX = STAGE_COEF_BYTES / sizeof(T2);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    T2 *const tile = reinterpret_cast<T2 *>(smem_raw);
    const uint32_t L = d.L;
    const uint32_t tsize = 1u << L;
    T2 *const mat = tile + tsize;
    StageOp *const lops = reinterpret_cast<StageOp *>(mat + CMAX);
    const uint32_t tid = threadIdx.x;
    const uint32_t lowbits = L < LOG_THREADS ? L : LOG_THREADS;
    uint64_t toff = 0;
    for (uint32_t j = 0; j < lowbits; j++) toff |= (uint64_t)((tid >> j) & 1) << d.local_pos[j];
    const bool active = tid < tsize;
    // Copies the op records from o0 on and the coefficients of as many of them
    // as fit (coefficients lie in op order); returns how many.
    auto load_ops = [&](uint32_t o0) -> uint32_t {
        const uint32_t cnt = d.num_ops - o0 < STAGE_OPS ? d.num_ops - o0 : STAGE_OPS;
        const uint32_t *const src = reinterpret_cast<const uint32_t *>(ops + d.op_off + o0);
        uint32_t *const dst = reinterpret_cast<uint32_t *>(lops);
        for (uint32_t i = tid; i < cnt * (sizeof(StageOp) / 4); i += THREADS) dst[i] = src[i];
        __syncthreads();
        const uint32_t lane = tid & 63, first = uniform(lops[0].coef_off);
        uint32_t end = 0;
        if (lane < cnt) {
            const StageOp &op = lops[lane];
            end = op.coef_off + (1u << (op.kind == OP_DENSE ? 2 * op.k : op.k)) - first;
        }
        const uint32_t fit = (uint32_t)__popcll(__ballot(lane < cnt && end <= CMAX));
        const uint32_t total = uniform(__shfl(end, fit - 1, 64));  // one op always fits
        for (uint32_t i = tid; i < total; i += THREADS) mat[i] = coefs[first + i];
        __syncthreads();
        return fit;
    };
    uint32_t held = load_ops(0);  // the ops [0, held) are in LDS
    for (uint64_t t = blockIdx.x; t < d.num_tiles; t += gridDim.x) {
        uint64_t base = 0;
        for (uint32_t j = 0; j < d.nglob; j++) base |= ((t >> j) & 1) << d.glob_pos[j];
        for (uint32_t m = 0; m < tsize; m += THREADS) {
            uint64_t moff = 0;
            for (uint32_t j = lowbits; j < L; j++) moff |= (uint64_t)((m >> j) & 1) << d.local_pos[j];
            if (!active) continue;
            if (d.from_zero) {
                T2 v;
                v.x = (base | moff | toff) == 0 ? 1 : 0;
                v.y = 0;
                tile[m + tid] = v;
            } else {
                tile[m + tid] = s[base + moff + toff];
            }
        }
        __syncthreads();
        for (uint32_t o0 = 0, cnt; o0 < d.num_ops; o0 += cnt) {
            cnt = held;
            if (held < d.num_ops) cnt = load_ops(o0);
            const uint32_t first = uniform(lops[0].coef_off);
            for (uint32_t o = 0; o < cnt; o++) {
                const StageOp &op = lops[o];
                const uint64_t gm = ((uint64_t)uniform(op.gc_mask >> 32) << 32) | uniform((uint32_t)op.gc_mask);
                const uint64_t gv = ((uint64_t)uniform(op.gc_val >> 32) << 32) | uniform((uint32_t)op.gc_val);
                if ((base & gm) != gv) continue;
                const T2 *const m = mat + (uniform(op.coef_off) - first);
                if (uniform(op.kind) == OP_DENSE) {
                    switch (uniform(op.k)) {
                        case 1: tile_dense<T2, 1, LOG_THREADS>(tile, m, op, L); break;
                        case 2: tile_dense<T2, 2, LOG_THREADS>(tile, m, op, L); break;
                        case 3: tile_dense<T2, 3, LOG_THREADS>(tile, m, op, L); break;
                        case 4: tile_dense<T2, 4, LOG_THREADS>(tile, m, op, L); break;
                        default: break;
                    }
                } else {
                    tile_diag<T2, LOG_THREADS>(tile, m, op, L, base);
                }
                __syncthreads();
            }
            // A skipped op leaves no barrier behind: the next records may be
            // written only when every wave has read these.
            if (held < d.num_ops) __syncthreads();
        }
        for (uint32_t m = 0; m < tsize; m += THREADS) {
            uint64_t moff = 0;
            for (uint32_t j = lowbits; j < L; j++) moff |= (uint64_t)((m >> j) & 1) << d.local_pos[j];
            if (active) s[base + moff + toff] = tile[m + tid];
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// FP64 reductions.
// ---------------------------------------------------------------------------
constexpr int RED_THREADS = 256;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sum of v over the block; the result is valid in thread 0.
__device__ __forceinline__ double block_sum(double v, double *scratch) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) r += scratch[w];
    return r;
}

template <typename T2>
__device__ __forceinline__ double prob(const T2 a) {
    const double re = (double)a.x, im = (double)a.y;
    return re * re + im * im;
}

// Per-block partial sums of |a_i|^2: over all amplitudes, or (HALF) over those
// whose index has bit `qubit` set, which are the only ones it visits.
template <typename T2, bool HALF>
__global__ __launch_bounds__(RED_THREADS) void k_norm(const T2 *__restrict__ s, uint64_t count, uint32_t qubit,
                                                      double *__restrict__ partial) {
    __shared__ double scratch[RED_THREADS / 64];
    double acc = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t bit = HALF ? uint64_t(1) << qubit : 0;
    auto at = [&](uint64_t it) { return HALF ? ((it & ~(bit - 1)) << 1) | bit | (it & (bit - 1)) : it; };
    // U loads in flight per thread, summed in index order.
    constexpr int U = 8;
    for (; i + (U - 1) * stride < count; i += U * stride) {
        T2 a[U];
#pragma unroll
        for (int u = 0; u < U; u++) a[u] = s[at(i + u * stride)];
#pragma unroll
        for (int u = 0; u < U; u++) acc += prob(a[u]);
    }
    for (; i < count; i += stride) acc += prob(s[at(i)]);
    const double r = block_sum(acc, scratch);
    if (threadIdx.x == 0) partial[blockIdx.x] = r;
}

// |a_i|^2 in FP64, in index order.
template <typename T2>
__global__ void k_probabilities(const T2 *__restrict__ s, uint64_t len, double *__restrict__ out) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += stride) out[i] = prob(s[i]);
}

// Pauli strings in groups that share one X part x (qubits with X or Y) and
// differ in their Z parts z[t] (qubits with Z or Y); blockIdx.y names the
// group. With v_j = conj(a_j) a_(j ^ x), a string's value is
// i^popcount(x & z) times the sum over j of (-1)^popcount((j ^ x) & z) v_j. The
// terms of j and j ^ x differ only in the sign of the part that the factor i^..
// makes imaginary: the other part counts twice and that one cancels. So for
// x != 0 only the j without x's highest bit are visited, each amplitude is
// read once, and only the part that stays is summed: the imaginary one where
// popcount(x & z) is odd. Per block and string the sum goes to
// partial[(string - first) * blocks + block]. KT >= a group's strings (a power of two, so
// a group of few strings does not pay for PAULI_TERMS).
//
// Bound by memory (one read of the state per group): 30 qubits in complex64,
// one string 1.6 ms; reading both amplitudes of every j and summing both
// parts took 2.8 ms for a string with X on every qubit.
template <typename T2, int KT>
__global__ __launch_bounds__(RED_THREADS) void k_expect_pauli(const T2 *__restrict__ s, uint64_t len,
                                                              const PauliGroup *__restrict__ groups,
                                                              const uint64_t *__restrict__ zs, uint32_t first,
                                                              double *__restrict__ partial) {
    __shared__ double scratch[RED_THREADS / 64];
    const PauliGroup g = groups[blockIdx.y];
    double sum[KT];
    uint64_t z[KT];
#pragma unroll
    for (int t = 0; t < KT; t++) {
        sum[t] = 0;
        z[t] = t < (int)g.nterms ? zs[g.first + t] : 0;
    }
    const uint64_t x = g.x;
    const uint64_t top = x ? uint64_t(1) << (63 - __builtin_clzll(x)) : 0;
    const uint64_t count = x ? len >> 1 : len;
    const uint64_t low = x ? top - 1 : ~uint64_t(0);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    auto index = [&](uint64_t it) { return (it & low) | ((it & ~low) << 1); };
    auto add = [&](uint64_t j, const T2 a, const T2 b) {
        const double ar = a.x, ai = a.y, br = b.x, bi = b.y;
        const double vr = ar * br + ai * bi, vi = ar * bi - ai * br;  // conj(a) b
        const uint64_t k = j ^ x;
#pragma unroll
        for (int t = 0; t < KT; t++) {  // every slot: unused ones have z = 0 and are not written
            const double v = (g.odd >> t) & 1 ? vi : vr;
            sum[t] += (__popcll(k & z[t]) & 1) ? -v : v;
        }
    };
    // U iterations' loads in flight per thread, summed in index order.
    constexpr int U = 4;
    uint64_t it = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; it + (U - 1) * stride < count; it += U * stride) {
        T2 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint64_t j = index(it + u * stride);
            a[u] = s[j];
            b[u] = s[j ^ x];
        }
#pragma unroll
        for (int u = 0; u < U; u++) add(index(it + u * stride), a[u], b[u]);
    }
    for (; it < count; it += stride) {
        const uint64_t j = index(it);
        add(j, s[j], s[j ^ x]);
    }
#pragma unroll
    for (int t = 0; t < KT; t++) {
        const double r = block_sum(sum[t], scratch);
        if (threadIdx.x == 0 && t < (int)g.nterms) partial[(uint64_t)(g.first - first + t) * gridDim.x + blockIdx.x] = r;
    }
}

// out[v] = the sum of row v of partial[rows][m], one block per row: a thread
// per value where one walks them in order costs a memory round trip per few
// values (1024 partial sums: 66 to 90 us, this 3).
__global__ __launch_bounds__(RED_THREADS) void k_sum_rows(const double *__restrict__ partial, uint32_t m,
                                                          double *__restrict__ out) {
    __shared__ double scratch[RED_THREADS / 64];
    const double *const row = partial + (uint64_t)blockIdx.x * m;
    double r = 0;
    for (uint32_t i = threadIdx.x; i < m; i += RED_THREADS) r += row[i];
    r = block_sum(r, scratch);
    if (threadIdx.x == 0) out[blockIdx.x] = r;
}

// The same for the strings of several launches, whose rows differ in length.
__global__ __launch_bounds__(RED_THREADS) void k_sum_paulis(const double *__restrict__ partial, const PauliLaunches l,
                                                            double *__restrict__ out) {
    __shared__ double scratch[RED_THREADS / 64];
    uint32_t i = 0;
    while (i + 1 < l.n && blockIdx.x >= l.at[i + 1].first) i++;
    const uint32_t m = l.at[i].blocks;
    const double *const row = partial + l.at[i].partial + (uint64_t)(blockIdx.x - l.at[i].first) * m;
    double r = 0;
    for (uint32_t j = threadIdx.x; j < m; j += RED_THREADS) r += row[j];
    r = block_sum(r, scratch);
    if (threadIdx.x == 0) out[blockIdx.x] = r;
}

// Per-block max |a-b|, sum |a-b|^2 and sum |b|^2 over two states.
template <typename TA, typename TB>
__global__ __launch_bounds__(RED_THREADS) void k_compare(const TA *__restrict__ a, const TB *__restrict__ b,
                                                         uint64_t len, double *__restrict__ partial) {
    __shared__ double scratch[RED_THREADS / 64];
    __shared__ double mx[RED_THREADS / 64];
    double m = 0, d2 = 0, r2 = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += stride) {
        const TA x = a[i];
        const TB y = b[i];
        const double dr = (double)x.x - (double)y.x, di = (double)x.y - (double)y.y;
        const double dd = dr * dr + di * di;
        d2 += dd;
        m = dd > m ? dd : m;
        r2 += (double)y.x * (double)y.x + (double)y.y * (double)y.y;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double t = __shfl_xor(m, o, 64);
        m = t > m ? t : m;
    }
    if ((threadIdx.x & 63) == 0) mx[threadIdx.x >> 6] = m;
    const double s1 = block_sum(d2, scratch);
    const double s2 = block_sum(r2, scratch);
    if (threadIdx.x == 0) {
        double mm = 0;
        for (int w = 0; w < RED_THREADS / 64; w++) mm = mx[w] > mm ? mx[w] : mm;
        partial[3 * blockIdx.x] = mm;
        partial[3 * blockIdx.x + 1] = s1;
        partial[3 * blockIdx.x + 2] = s2;
    }
}

// <Z_q> and <Z_q Z_q+1> in one pass. A block covers a segment of 2^B
// contiguous amplitudes; per segment it writes 2B sums of p = |a|^2: the total,
// the signed sums of p (-1)^(bit q) (q < B) and of p (-1)^(bit q + bit q+1)
// (q < B-1), value v of segment g at out[v * segments + g]. Bits above B are
// constant in a segment and are resolved by k_expect_combine.
//
// The lanes' sums go through a Walsh-Hadamard transform over the wave's six
// lane bits: afterwards lane l holds the sum over the wave with sign
// (-1)^popcount(lane & l), so lanes 0, 1 << q and 3 << q hold every total,
// single and pair sum of those bits after 6 exchanges (one wave sum per value
// took 6 each: 34 us for a 20-qubit state against 9 now). Signs of the wave
// bits are applied where one thread per value adds up the waves.
constexpr int EZ_TID_BITS = 10;  // bits from the thread index (1024 threads)
constexpr int EZ_MAX_M_BITS = 6; // bits from the per-thread loop

// The descriptor of block b: `one` when there is a single state, else the
// entry i of `descs` with start[i] <= b < start[i + 1] (binary search).
template <typename S>
__device__ __forceinline__ uint32_t find_range(const S *__restrict__ start, uint32_t count, uint64_t b) {
    uint32_t lo = 0, hi = count;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if ((uint64_t)start[mid] <= b) lo = mid;
        else hi = mid;
    }
    return lo;
}

template <typename T2>
__global__ __launch_bounds__(1 << EZ_TID_BITS) void k_expect_segments(const T2 *__restrict__ s_all, ExpDesc one,
                                                         const ExpDesc *__restrict__ descs, uint32_t ndesc,
                                                         const uint64_t *__restrict__ seg_start,
                                                         double *__restrict__ out_all) {
    __shared__ double scratch[(1 << EZ_TID_BITS) / 64][12 + 2 * EZ_MAX_M_BITS];
    ExpDesc d = one;
    uint64_t seg = blockIdx.x;
    if (ndesc > 1) {
        const uint32_t di = find_range(seg_start, ndesc, blockIdx.x);
        d = descs[di];
        seg = blockIdx.x - seg_start[di];
    }
    const T2 *s = s_all + d.state_off;
    double *out = out_all + d.seg_off;
    const uint32_t B = d.B;
    const uint32_t tb = B < EZ_TID_BITS ? B : EZ_TID_BITS;
    const uint32_t mb = B - tb;
    const uint32_t tid = threadIdx.x;
    const bool active = tid < (1u << tb);
    double T = 0, S[EZ_MAX_M_BITS], P[EZ_MAX_M_BITS];  // the thread's total, and its signed sums over loop bits
#pragma unroll
    for (int j = 0; j < EZ_MAX_M_BITS; j++) S[j] = P[j] = 0;
    if (active) {
        const uint64_t base = (seg << B) + tid;
        const uint32_t M = 1u << mb;
        auto add = [&](uint32_t m, double p) {
            T += p;
#pragma unroll
            for (int j = 0; j < EZ_MAX_M_BITS; j++) {
                if ((uint32_t)j < mb) {
                    S[j] += ((m >> j) & 1) ? -p : p;
                    if ((uint32_t)j + 1 < mb) P[j] += (((m >> j) ^ (m >> (j + 1))) & 1) ? -p : p;
                }
            }
        };
        // U loads in flight per thread (M is a power of two, so a multiple
        // of U once it reaches U: the loads need no bounds test, which would
        // put each in a branch of its own and wait for it), then the sums in
        // the order of m.
        constexpr uint32_t U = 8;
        if (M >= U) {
            for (uint32_t m0 = 0; m0 < M; m0 += U) {
                T2 a[U];
#pragma unroll
                for (uint32_t u = 0; u < U; u++) a[u] = s[base + ((uint64_t)(m0 + u) << tb)];
#pragma unroll
                for (uint32_t u = 0; u < U; u++) add(m0 + u, prob(a[u]));
            }
        } else {
            for (uint32_t m = 0; m < M; m++) add(m, prob(s[base + ((uint64_t)m << tb)]));
        }
    }
    // A wave's sums: slot 0 its total, 1 + q lane bit q, 7 + q lane bits q and
    // q + 1, 12 + j loop bit j, 18 + j loop bits j and j + 1.
    const uint32_t lane = tid & 63, wave = tid >> 6;
    constexpr uint32_t SL = 12, PL = SL + EZ_MAX_M_BITS;
    double w = T;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double other = __shfl_xor(w, o, 64);
        w = (lane & o) ? other - w : w + other;
    }
    const uint32_t first = lane & -lane;
    if (lane == 0) scratch[wave][0] = w;
    else if (lane == first) scratch[wave][1 + __builtin_ctz(lane)] = w;
    else if (lane == 3 * first) scratch[wave][7 + __builtin_ctz(lane)] = w;
#pragma unroll
    for (int j = 0; j < EZ_MAX_M_BITS; j++) {
        if ((uint32_t)j < mb) {
            const double v = wave_sum(S[j]);
            if (lane == 0) scratch[wave][SL + j] = v;
            if ((uint32_t)j + 1 < mb) {
                const double u = wave_sum(P[j]);
                if (lane == 0) scratch[wave][PL + j] = u;
            }
        }
    }
    __syncthreads();
    if (tid < 2 * B) {
        uint32_t slot = 0, waves = 0;  // the value's slot, and the wave bits its sign takes
        if (tid == 0) {
        } else if (tid <= B) {
            const uint32_t q = tid - 1;
            if (q < 6) slot = 1 + q;
            else if (q < EZ_TID_BITS) waves = 1u << (q - 6);
            else slot = SL + q - EZ_TID_BITS;
        } else {
            const uint32_t q = tid - 1 - B;
            if (q < 5) slot = 7 + q;
            else if (q == 5) slot = 6, waves = 1;
            else if (q + 1 < EZ_TID_BITS) waves = 3u << (q - 6);
            else if (q + 1 == EZ_TID_BITS) slot = SL, waves = 1u << (EZ_TID_BITS - 7);
            else slot = PL + q - EZ_TID_BITS;
        }
        double r = 0;
        for (uint32_t v = 0; v < (blockDim.x >> 6); v++) {
            const double x = scratch[v][slot];
            r += (__popc(v & waves) & 1) ? -x : x;
        }
        out[(uint64_t)tid * d.nsegs + seg] = r;
    }
}

// Combines the segment sums into z[q] and zz[q]: output w is the sum over the
// segments g of value `idx` with sign (-1)^popcount(g & bits). TPO threads per
// output (64 or the block): with one thread per output the 2^14 segments of a
// 30-qubit state were a serial chain of 2.3 ms; now 20 us.
template <int THREADS, int TPO>
__global__ __launch_bounds__(THREADS) void k_expect_combine(const double *__restrict__ seg_all, ExpDesc one,
                                                            const ExpDesc *__restrict__ descs, uint32_t ndesc,
                                                            const uint32_t *__restrict__ out_start, uint32_t outs,
                                                            double *__restrict__ z, double *__restrict__ zz) {
    static_assert(TPO == 64 || TPO == THREADS, "an output's threads are a wave or the block");
    __shared__ double scratch[THREADS / 64];
    const uint32_t wg = blockIdx.x * (THREADS / TPO) + threadIdx.x / TPO, t = threadIdx.x % TPO;
    ExpDesc d = one;
    uint32_t w = wg;
    if (wg >= outs) return;  // uniform over the output's threads
    if (ndesc > 1) {
        const uint32_t di = find_range(out_start, ndesc, wg);
        d = descs[di];
        w = wg - out_start[di];
    }
    const uint32_t n = d.n, B = d.B;
    uint32_t idx = 0;
    uint64_t bits = 0;
    if (w < n) {
        const uint32_t q = w;
        if (q < B) idx = 1 + q;
        else bits = uint64_t(1) << (q - B);
    } else {
        const uint32_t q = w - n;
        if (q + 1 < B) idx = 1 + B + q;
        else if (q + 1 == B) idx = 1 + q, bits = 1;
        else bits = uint64_t(3) << (q - B);
    }
    const double *const v = seg_all + d.seg_off + (uint64_t)idx * d.nsegs;
    double r = 0;
    for (uint64_t g = t; g < d.nsegs; g += TPO) {
        const double x = v[g];
        r += (__popcll(g & bits) & 1) ? -x : x;
    }
    if constexpr (TPO == 64) r = wave_sum(r);
    else r = block_sum(r, scratch);
    if (t == 0) {
        if (w < n) z[d.z_off + w] = r;
        else zz[d.zz_off + w - n] = r;
    }
}

// Sets amplitude 0 of each state of a batch to 1 (after a zero fill).
template <typename T2>
__global__ void k_set_basis(T2 *__restrict__ s, const uint64_t *__restrict__ offs, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    T2 v;
    v.x = 1;
    v.y = 0;
    s[offs[i]] = v;
}

// Zero-fills n words (a kernel, not a memset: graph-captured memset nodes are
// avoided).
__global__ void k_zero_words(uint32_t *__restrict__ p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------------------
// Measurement collapse (src/measure.rs:68-80): the kept half scaled by
// 1 / sqrt(its probability) in the state's precision, the other half zeroed. The outcome
// follows from P(1) in device memory, so the host need not wait between the
// two passes. FLIP (reset): outcome 1 is followed by an X on the qubit in the
// same pass, with the arithmetic of k_dense on that matrix.
// ---------------------------------------------------------------------------
//
// On large states, where the qubit lies inside a 128-byte line (LINE), a thread
// owns one amplitude and gets its partner's from the lane beside it: with a thread
// per pair, each load takes pieces of a line only (measurements of qubits 0 to 3, 29
// qubits in complex64: 2.60 ms, 2.41 so; 28 qubits 1.31 and 1.21).
template <typename T2, bool FLIP, bool LINE>
__global__ __launch_bounds__(256) void k_collapse(T2 *__restrict__ s, uint64_t len, uint32_t qubit, double uniform,
                                                  const double *__restrict__ p_one, double *__restrict__ p_copy) {
    using T = typename Real<T2>::T;
    double p1 = *p_one;
    if (blockIdx.x == 0 && threadIdx.x == 0) *p_copy = p1;
    p1 = p1 < 0.0 ? 0.0 : p1;  // a NaN stays one, as in the host's clamp
    p1 = 1.0 < p1 ? 1.0 : p1;
    const bool outcome = uniform < p1;
    T2 keep, drop, one;
    keep.x = (T)(1.0 / sqrt(outcome ? p1 : 1.0 - p1));
    keep.y = drop.x = drop.y = one.y = 0;
    one.x = 1;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t bit = uint64_t(1) << qubit;
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if constexpr (LINE) {
        // A pair's two lanes run the same iterations: they differ in a bit below
        // the wave's size, and len and the stride are multiples of twice it.
        const bool up = (first & bit) != 0;
        const T2 f = up == outcome ? keep : drop;
        for (uint64_t i = first; i < len; i += stride) {
            T2 a = cmul_diag(f, s[i]);
            if (FLIP && outcome) {
                T2 b, o = drop;
                b.x = __shfl_xor(a.x, (int)bit, 64);
                b.y = __shfl_xor(a.y, (int)bit, 64);
                cmac(o, up ? one : drop, up ? b : a);
                cmac(o, up ? drop : one, up ? a : b);
                a = o;
            }
            s[i] = a;
        }
        return;
    }
    for (uint64_t it = first; it < len >> 1; it += stride) {
        const uint64_t i0 = ((it & ~(bit - 1)) << 1) | (it & (bit - 1)), i1 = i0 | bit;
        T2 a = cmul_diag(outcome ? drop : keep, s[i0]), b = cmul_diag(outcome ? keep : drop, s[i1]);
        if (FLIP && outcome) {
            T2 o0 = drop, o1 = drop;
            cmac(o0, drop, a);
            cmac(o0, one, b);
            cmac(o1, one, a);
            cmac(o1, drop, b);
            a = o0;
            b = o1;
        }
        s[i0] = a;
        s[i1] = b;
    }
}

// ---------------------------------------------------------------------------
// Two-pass sampling (src/measure.rs:104-174). The reference's summation
// order is kept exactly: each chunk is summed sequentially in index order,
// the prefix over chunks is sequential, and the walk adds probabilities one
// by one; so one lane owns one chunk. Loads are 16-byte vectors.
// ---------------------------------------------------------------------------
// Amplitudes per batch of the one-lane-per-chunk passes: two batches live in
// registers (128 VGPRs of amplitudes).
template <typename T2>
constexpr int chunk_batch() {
    return sizeof(T2) == 8 ? 32 : 16;
}

// Streams one lane's amplitudes [i, end) through visit(batch, first index) in
// batches of U, two at a time in registers: batch b + 1's loads fly while
// batch b is visited. With one lane per chunk and few chunks (2^15 at 30
// qubits, half a wave per SIMD) nothing else covers a batch's memory round
// trip. visit returns false to stop (`stopped` is then set). issued() runs
// right after each batch's loads go out: a store placed there follows the
// loads the next wait is for, so that wait does not include the store (the
// memory counter of loads and stores runs in order). Returns the first index
// not visited; fewer than U amplitudes are left from there unless it stopped.
template <int U, typename T2, typename F, typename G>
__device__ __forceinline__ uint64_t stream_batches(const T2 *__restrict__ s, uint64_t i, uint64_t end, bool &stopped,
                                                   F &&visit, G &&issued) {
    stopped = false;
    if (i + U > end) return i;
    T2 a[U], b[U];
    uint64_t a_at = i;  // a holds [a_at, a_at + U)
#pragma unroll
    for (int j = 0; j < U; j++) a[j] = s[i + j];
    while (i + 2 * U <= end) {
#pragma unroll
        for (int j = 0; j < U; j++) b[j] = s[i + U + j];
        __builtin_amdgcn_sched_barrier(0);  // b's loads go out before a is used
        issued();
        if (!visit(a, i)) {
            stopped = true;
            return i + U;
        }
        i += U;
        // The next batch, or the last whole one (in bounds: i + U <= end):
        // an unconditional load keeps the waits for b exact.
        a_at = i + 2 * U <= end ? i + U : end - U;
#pragma unroll
        for (int j = 0; j < U; j++) a[j] = s[a_at + j];
        __builtin_amdgcn_sched_barrier(0);  // a's loads go out before b is used
        issued();
        if (!visit(b, i)) {
            stopped = true;
            return i + U;
        }
        i += U;
    }
    if (i + U <= end) {
        if (a_at != i) {
#pragma unroll
            for (int j = 0; j < U; j++) a[j] = s[i + j];
        }
        issued();  // between every two visits
        if (!visit(a, i)) stopped = true;
        i += U;
    }
    return i;
}

template <typename T2>
__global__ __launch_bounds__(64) void k_chunk_sums(const T2 *__restrict__ s, uint64_t len, uint64_t chunk,
                                                    uint64_t num_chunks, double *__restrict__ sums) {
    const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= num_chunks) return;
    const uint64_t start = c * chunk;
    const uint64_t end = start + chunk < len ? start + chunk : len;
    double acc = 0;
    constexpr int U = chunk_batch<T2>();
    bool stopped;
    uint64_t i = stream_batches<U>(s, start, end, stopped, [&](const T2(&v)[U], uint64_t) {
#pragma unroll
        for (int j = 0; j < U; j++) acc += prob(v[j]);
        return true;
    }, [] {});
    for (; i < end; i++) acc += prob(s[i]);
    sums[c] = acc;
}

// The sequential prefix over chunk sums (src/measure.rs:120-124): one lane
// adds them one by one. The sums pass through LDS in tiles: while lane 0
// adds up tile k in place, the workgroup's other lanes store tile k-1's
// prefixes and load tile k+1, all coalesced, so the dependent add chain
// waits on LDS only, never on a memory round trip.
constexpr uint32_t PREFIX_THREADS = 256;
constexpr uint32_t PREFIX_TILE = 2048;  // doubles per tile; two tiles of LDS

__global__ __launch_bounds__(PREFIX_THREADS) void k_prefix(const double *__restrict__ sums, uint64_t num_chunks,
                                                          double *__restrict__ prefix) {
    __shared__ double buf[2][PREFIX_TILE];
    constexpr uint32_t PER = PREFIX_TILE / PREFIX_THREADS;
    const uint32_t t = threadIdx.x;
    const uint64_t tiles = (num_chunks + PREFIX_TILE - 1) / PREFIX_TILE;
    if (t == 0) prefix[0] = 0;
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) {
        const uint64_t c = j * PREFIX_THREADS + t;
        buf[0][j * PREFIX_THREADS + t] = c < num_chunks ? sums[c] : 0.0;
    }
    __syncthreads();
    double p = 0;
    for (uint64_t k = 0; k < tiles; k++) {
        double *cur = buf[k & 1], *other = buf[(k + 1) & 1];
        const uint64_t base = k * PREFIX_TILE;
        if (k > 0) {  // tile k-1's prefixes, finished in the last round
#pragma unroll
            for (uint32_t j = 0; j < PER; j++) {
                const uint64_t c = base - PREFIX_TILE + j * PREFIX_THREADS + t;
                prefix[c + 1] = other[j * PREFIX_THREADS + t];
            }
        }
        const bool more = k + 1 < tiles;
        double v[PER];
        if (more) {
#pragma unroll
            for (uint32_t j = 0; j < PER; j++) {
                const uint64_t c = base + PREFIX_TILE + j * PREFIX_THREADS + t;
                v[j] = c < num_chunks ? sums[c] : 0.0;
            }
        }
        if (t == 0) {
            const uint32_t n = num_chunks - base < PREFIX_TILE ? (uint32_t)(num_chunks - base) : PREFIX_TILE;
            uint32_t i = 0;
            for (; i + 16 <= n; i += 16) {
                double x[16];
#pragma unroll
                for (int j = 0; j < 16; j++) x[j] = cur[i + j];
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    p = p + x[j];
                    x[j] = p;
                }
#pragma unroll
                for (int j = 0; j < 16; j++) cur[i + j] = x[j];
            }
            for (; i < n; i++) {
                p = p + cur[i];
                cur[i] = p;
            }
        }
        if (more) {  // the same slots this thread read above
#pragma unroll
            for (uint32_t j = 0; j < PER; j++) other[j * PREFIX_THREADS + t] = v[j];
        }
        __syncthreads();
    }
    const double *last = buf[(tiles - 1) & 1];
    const uint64_t base = (tiles - 1) * PREFIX_TILE;
#pragma unroll
    for (uint32_t j = 0; j < PER; j++) {
        const uint64_t c = base + j * PREFIX_THREADS + t;
        if (c < num_chunks) prefix[c + 1] = last[j * PREFIX_THREADS + t];
    }
}

// targets = sorted uniforms * total, in place. The order survives: for a
// finite total >= 0, rounding u * total is monotone in u, so scaling the
// sorted uniforms gives sort(u * total) exactly.
__global__ void k_targets(double *__restrict__ targets, const double *__restrict__ total_ptr, uint64_t shots) {
    const double total = *total_ptr;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < shots; i += stride)
        targets[i] = targets[i] * total;
}

// bounds[c] = number of targets < prefix[c] (partition_point).
__global__ void k_bounds(const double *__restrict__ prefix, uint64_t num_chunks, const double *__restrict__ targets,
                         uint64_t shots, uint64_t *__restrict__ bounds) {
    const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c > num_chunks) return;
    const double p = prefix[c];
    uint64_t lo = 0, hi = shots;
    while (lo < hi) {
        const uint64_t mid = lo + (hi - lo) / 2;
        if (targets[mid] < p) lo = mid + 1;
        else hi = mid;
    }
    bounds[c] = lo;
}

// The walk (src/measure.rs:143-166) in two kernels. Shot s of chunk c goes
// to the first index i of the chunk whose running sum prefix[c] + p_start +
// ... + p_i, added one by one in index order, exceeds targets[s]; a shot no
// index of the chunk reaches (rounding) goes to the chunk's last nonzero
// probability. Zero probabilities are never such an index: adding +0.0
// leaves the sum (never -0.0) unchanged, and every target of the chunk is at
// least prefix[c]. So the running sum may add them too.
//
// k_walk_marks runs each chunk's running sum, one lane per chunk, with no
// per-shot work, and stores it every 2^mark_bits amplitudes (marks[b] = the
// sum up to the end of the chunk's block b). It stops after the block where
// the sum passes the chunk's largest target, and stores how many blocks it
// walked. k_walk_place then gives every shot a thread of its own: the first
// mark above its target names its block, and the sum resumes from the mark
// before (bit for bit the value the sequential sum had there) over at most
// 2^mark_bits amplitudes. A shot that no index reaches was left over by a
// walk that went to the chunk's end; its thread scans back from the end for
// the last nonzero probability (rare, and cut short by the first nonzero).
template <typename T2>
__global__ __launch_bounds__(64) void k_walk_marks(const T2 *__restrict__ s, uint64_t len, uint64_t chunk,
                                                    uint64_t num_chunks, uint32_t mark_bits,
                                                    const double *__restrict__ prefix,
                                                    const uint64_t *__restrict__ bounds,
                                                    const double *__restrict__ targets, uint64_t shots,
                                                    double *__restrict__ marks, uint32_t *__restrict__ walked) {
    const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= num_chunks) return;
    const uint64_t lo = bounds[c];
    const uint64_t hi = bounds[c + 1] < shots ? bounds[c + 1] : shots;
    if (lo >= hi) return;  // no shot in this chunk: nothing is read
    const double t_last = targets[hi - 1];
    const uint64_t start = c * chunk;
    const uint64_t end = start + chunk < len ? start + chunk : len;
    const uint64_t block_mask = (uint64_t(1) << mark_bits) - 1;
    double *m = marks + (start >> mark_bits);
    double cumulative = prefix[c];
    uint32_t b = 0;
    bool pending = false;  // amplitudes added since the last mark
    // A mark is stored after the next batch's loads go out (see
    // stream_batches): a store before them would make the wait for them wait
    // for the store too, a memory round trip per mark. Marks gather in LDS
    // and leave 16 at a time, a whole 128-byte line per lane: one 8-byte
    // store per mark left lines partly written while the chunk streamed
    // through the caches.
    constexpr uint32_t MG = 16;
    __shared__ double mbuf[64][MG + 1];
    const uint32_t lane = threadIdx.x;
    uint32_t nbuf = 0, flushed = 0;
    bool mark_ready = false;
    double mark = 0;
    auto store_mark = [&] {
        if (mark_ready) {
            mbuf[lane][nbuf++] = mark;
            b++;
            if (nbuf == MG) {
#pragma unroll
                for (uint32_t k = 0; k < MG; k++) m[flushed + k] = mbuf[lane][k];
                flushed += MG;
                nbuf = 0;
            }
        }
        mark_ready = false;
    };
    constexpr int U = chunk_batch<T2>();  // divides 2^mark_bits
    bool stopped;
    uint64_t i = stream_batches<U>(s, start, end, stopped, [&](const T2(&v)[U], uint64_t at) {
#pragma unroll
        for (int j = 0; j < U; j++) cumulative += prob(v[j]);
        if (((at + U - start) & block_mask) == 0 || at + U == end) {
            mark = cumulative;
            mark_ready = true;
            pending = false;
            return !(t_last < cumulative);  // every shot of the chunk lands in a walked block
        }
        pending = true;
        return true;
    }, store_mark);
    store_mark();
    if (!stopped) {  // fewer than U amplitudes left: a state of fewer than U amplitudes
        for (; i < end; i++) {
            cumulative += prob(s[i]);
            pending = true;
        }
        if (pending) {
            mark = cumulative;
            mark_ready = true;
            store_mark();
        }
    }
    for (uint32_t k = 0; k < nbuf; k++) m[flushed + k] = mbuf[lane][k];
    walked[c] = b;
}

// The chunk sums and the walk for states of few chunks, where one lane per
// chunk leaves most of the chip idle and spends 33 cycles an amplitude on
// conversions and products beside the add that the order of summation asks
// for. Here one wave only adds: its lane c runs chunk c's sum over
// probabilities in LDS, one add after the other, while four waves load the
// coming batches (coalesced) and square them. C chunks per workgroup, batches
// of CHAIN_BATCH amplitudes over all of them, two in LDS and one in registers.
// Bound by the latency of the dependent adds: 24 qubits in complex64 (chunks
// of 2^15) 172 us for the sums where one lane per chunk took 454, 201 us for
// the walk where it took 545. The sums and marks are the same bit for bit.
constexpr int CHAIN_THREADS = 64 + 256, CHAIN_BATCH = 2048;

// Workgroup barrier that waits for LDS only: the loads of a coming batch stay
// in flight across it.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // gfx9 encoding: lgkmcnt(0), vmcnt and expcnt not waited
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <typename T2, int C, bool WALK>
__global__ __launch_bounds__(CHAIN_THREADS) void k_chain(const T2 *__restrict__ s, uint64_t clen, uint32_t mark_bits,
                                                         const double *__restrict__ prefix,
                                                         const uint64_t *__restrict__ bounds,
                                                         const double *__restrict__ targets, uint64_t shots,
                                                         double *__restrict__ marks, uint32_t *__restrict__ walked,
                                                         double *__restrict__ sums) {
    constexpr int BATCH = CHAIN_BATCH / C, PITCH = BATCH + 2, PER = CHAIN_BATCH / 256;
    __shared__ __attribute__((aligned(16))) double p[2][C * PITCH];
    __shared__ uint32_t stop[2];
    const uint64_t c0 = (uint64_t)blockIdx.x * C;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const bool serial = __builtin_amdgcn_readfirstlane(tid >> 6) == 0;  // wave 0
    const uint64_t batches = clen / BATCH;
    double acc = 0, t_last = 0;
    bool done = lane >= C;
    uint32_t nb = 0;
    const uint64_t c = c0 + (lane < C ? lane : 0);
    if constexpr (WALK) {
        const uint64_t first = bounds[c0], past = bounds[c0 + C] < shots ? bounds[c0 + C] : shots;
        if (first >= past) return;  // no shot in these chunks (uniform over the workgroup): nothing is read
        if (serial && lane < C) {
            const uint64_t lo = bounds[c], hi = bounds[c + 1] < shots ? bounds[c + 1] : shots;
            done = lo >= hi;
            if (!done) t_last = targets[hi - 1];
            acc = prefix[c];
        }
    }
    double *const m = WALK ? marks + ((c * clen) >> mark_bits) : nullptr;
    const uint64_t mask = (uint64_t(1) << mark_bits) - 1;
    T2 r[PER];
    auto fetch = [&](uint64_t b) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const uint32_t e = i * 256 + (tid - 64);
            r[i] = s[(c0 + e / BATCH) * clen + b * BATCH + e % BATCH];
        }
    };
    auto put = [&](uint64_t b) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const uint32_t e = i * 256 + (tid - 64);
            p[b & 1][(e / BATCH) * PITCH + e % BATCH] = prob(r[i]);
        }
    };
    if (!serial) {
        fetch(0);
        put(0);
        if (batches > 1) fetch(1);
    }
    if (serial) __builtin_amdgcn_s_setprio(3);  // its adds are the critical path
    lds_barrier();
    for (uint64_t b = 0; b < batches; b++) {
        if (!serial) {
            if (b + 1 < batches) put(b + 1);
            if (b + 2 < batches) fetch(b + 2);
        } else if (lane < C) {
            const double2 *const q = reinterpret_cast<const double2 *>(&p[b & 1][lane * PITCH]);
            // 2 U values are added while the next 2 U come from LDS.
            constexpr int U = BATCH >= 128 ? 16 : 8;
            static_assert(BATCH % (4 * U) == 0 && 2 * U <= 64, "a batch is whole steps, and a mark falls on a step's end");
            double2 a[U], n[U];
#pragma unroll
            for (int j = 0; j < U; j++) a[j] = q[j];
            auto add = [&](const double2(&v)[U], uint32_t at) {  // `at`: the values of the batch added afterwards
#pragma unroll
                for (int j = 0; j < U; j++) {
                    acc += v[j].x;
                    acc += v[j].y;
                }
                if constexpr (WALK) {
                    const uint64_t pos = b * BATCH + at;
                    if (!done && ((pos & mask) == 0 || pos == clen)) {
                        m[nb++] = acc;
                        done = t_last < acc;  // every shot of the chunk lands in a walked block
                        if (done || pos == clen) walked[c] = nb;
                    }
                }
            };
            for (uint32_t k = 0; k < BATCH / 2; k += 2 * U) {
#pragma unroll
                for (int j = 0; j < U; j++) n[j] = q[k + U + j];
                __builtin_amdgcn_sched_barrier(0);
                add(a, 2 * (k + U));
                const uint32_t next = k + 2 * U < BATCH / 2 ? k + 2 * U : 0;
#pragma unroll
                for (int j = 0; j < U; j++) a[j] = q[next + j];
                __builtin_amdgcn_sched_barrier(0);
                add(n, 2 * (k + 2 * U));
            }
            if constexpr (WALK) {
                const bool all = __ballot(!done) == 0;
                if (lane == 0) stop[b & 1] = all;
            }
        }
        lds_barrier();
        // Written again only after the next barrier, which needs this read.
        if (WALK && stop[b & 1]) break;
    }
    if (!WALK && serial && lane < C) sums[c] = acc;
}

template <typename T2>
__global__ __launch_bounds__(256) void k_walk_place(const T2 *__restrict__ s, uint64_t len, uint64_t chunk,
                                                     uint64_t num_chunks, uint32_t mark_bits,
                                                     const double *__restrict__ prefix,
                                                     const uint64_t *__restrict__ bounds,
                                                     const double *__restrict__ targets, uint64_t shots,
                                                     const double *__restrict__ marks,
                                                     const uint32_t *__restrict__ walked,
                                                     uint64_t *__restrict__ out) {
    // Shots [bounds[0], bounds[num_chunks]) fall in some chunk: all of them
    // for uniforms in [0, 1).
    const uint64_t first = bounds[0];
    const uint64_t past = bounds[num_chunks] < shots ? bounds[num_chunks] : shots;
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t shot = first + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; shot < past; shot += step) {
        // the chunk: bounds[c] <= shot < bounds[c + 1]
        uint64_t lo = 0, hi = num_chunks;
        while (hi - lo > 1) {
            const uint64_t mid = (lo + hi) >> 1;
            if (bounds[mid] <= shot) lo = mid;
            else hi = mid;
        }
        const uint64_t c = lo;
        const double t = targets[shot];
        const double *m = marks + ((c * chunk) >> mark_bits);
        const uint32_t nb = walked[c];
        // the first walked block whose mark is not <= t (a NaN sum counts as
        // past every target, as no comparison with it succeeds)
        uint32_t a = 0, z = nb;
        while (a < z) {
            const uint32_t mid = (a + z) >> 1;
            if (m[mid] <= t) a = mid + 1;
            else z = mid;
        }
        const uint64_t cend = c * chunk + chunk < len ? c * chunk + chunk : len;
        uint64_t found = 0;
        bool done = false;
        if (a < nb) {
            double cumulative = a == 0 ? prefix[c] : m[a - 1];
            uint64_t i = c * chunk + ((uint64_t)a << mark_bits);
            const uint64_t stop = i + (uint64_t(1) << mark_bits) < cend ? i + (uint64_t(1) << mark_bits) : cend;
            constexpr int U = 8;
            for (; i + U <= stop && !done; i += U) {
                T2 v[U];
#pragma unroll
                for (int j = 0; j < U; j++) v[j] = s[i + j];
#pragma unroll
                for (int j = 0; j < U; j++) {
                    cumulative += prob(v[j]);
                    if (!done && t < cumulative) {
                        found = i + j;
                        done = true;
                    }
                }
            }
            for (; i < stop && !done; i++) {
                cumulative += prob(s[i]);
                if (t < cumulative) {
                    found = i;
                    done = true;
                }
            }
        }
        if (!done) {  // a rounding leftover: the chunk's last nonzero probability (a NaN counts), else its start
            found = c * chunk;
            for (uint64_t i = cend; i-- > c * chunk;)
                if (!(prob(s[i]) == 0.0)) {
                    found = i;
                    break;
                }
        }
        out[shot] = found;
    }
}

// ---------------------------------------------------------------------------
// Host launchers.
// ---------------------------------------------------------------------------
static inline unsigned grid_for(uint64_t work, unsigned threads, unsigned cap = 16384) {
    uint64_t g = (work + threads - 1) / threads;
    if (g == 0) g = 1;
    return (unsigned)(g < cap ? g : cap);
}

template <typename T2>
void launch_init_zero(T2 *s, uint64_t len, hipStream_t st) {
    k_init_zero<T2><<<grid_for(len, 256), 256, 0, st>>>(s, len);
}
template <typename T2>
void launch_zero_stale(T2 *s, uint64_t len, uint64_t stale, hipStream_t st) {
    k_zero_stale<T2><<<grid_for(len, 256), 256, 0, st>>>(s, len, stale);
}
template <typename T2>
void launch_widen(const T2 *s, double2 *out, uint64_t count, hipStream_t st) {
    k_widen<T2><<<grid_for(count, 256), 256, 0, st>>>(s, out, count);
}
template <typename T2>
void launch_narrow(const double2 *in, T2 *s, uint64_t count, hipStream_t st) {
    k_narrow<T2><<<grid_for(count, 256), 256, 0, st>>>(in, s, count);
}
template <typename T2>
void launch_scale(T2 *s, uint64_t len, double factor, hipStream_t st) {
    k_scale<T2><<<grid_for(len, 256), 256, 0, st>>>(s, len, factor);
}

// Dynamic LDS of a k_dense launch: the matrix, or so much that three workgroups
// fit on a CU. On states far beyond the Infinity Cache, three waves per SIMD read and
// write memory in fewer places at a time than eight (28 qubits in complex64, 1
// target 0.81-0.87 ms, so 0.79-0.80; 2 targets 0.80-1.02 and 0.76-0.94; in
// complex128 2 targets 1.62-1.93 and 1.57-1.82). From 1 GiB on that holds
// for every gate; at 512 MiB for threads that hold more than 32 bytes
// (25 qubits in complex128, 2 targets: 183-219 us, so 181-214; 26 qubits in
// complex64, 1 target: 185-198 us, so 197-209). Below, three are too few (25
// qubits in complex64, 1 target: 69 us, 83 so). 4 targets and more in
// complex128 have few waves by their registers.
template <typename T2>
static size_t dense_lds(uint64_t len, uint32_t k) {
    const size_t matrix = dense_in_lds<T2>(k) ? sizeof(T2) << (2 * k) : 0;
    const uint64_t bytes = len * sizeof(T2);
    const bool large = bytes >= (uint64_t(1) << 30) || (bytes >= (uint64_t(1) << 29) && (sizeof(T2) << k) > 32);
    // 52 KiB: LDS is handed out in pieces of 1280 bytes, 128 to a CU.
    return large && k <= (sizeof(T2) == 8 ? 4 : 3) ? std::max<size_t>(matrix, 52 * 1024) : matrix;
}

template <typename T2>
void launch_dense(T2 *s, uint64_t len, const GateDesc &d, const T2 *mat, hipStream_t st) {
    const unsigned grid = grid_for(d.iterations, 256, 65536);
    const size_t lds = dense_lds<T2>(len, d.k);
    switch (d.k) {
        case 1: k_dense<T2, 1, const T2 *><<<grid, 256, lds, st>>>(s, d, mat); break;
        case 2: k_dense<T2, 2, const T2 *><<<grid, 256, lds, st>>>(s, d, mat); break;
        case 3: k_dense<T2, 3, const T2 *><<<grid, 256, lds, st>>>(s, d, mat); break;
        case 4: k_dense<T2, 4, const T2 *><<<grid, 256, lds, st>>>(s, d, mat); break;
        case 5: k_dense<T2, 5, const T2 *><<<grid, 256, lds, st>>>(s, d, mat); break;
        case 6: k_dense<T2, 6, const T2 *><<<grid, 256, lds, st>>>(s, d, mat); break;
        default: break;
    }
}

template <typename T2, int K>
static void dense_arg(T2 *s, uint64_t len, const GateDesc &d, const T2 *mat, hipStream_t st) {
    MatArg<T2, K> m;
    std::copy(mat, mat + (1 << (2 * K)), m.m);
    k_dense<T2, K, MatArg<T2, K>>
        <<<grid_for(d.iterations, 256, 65536), 256, dense_lds<T2>(len, K), st>>>(s, d, m);
}

template <typename T2>
void launch_dense_arg(T2 *s, uint64_t len, const GateDesc &d, const T2 *mat, hipStream_t st) {
    if (d.k == 1) dense_arg<T2, 1>(s, len, d, mat, st);
    else if (d.k == 2) dense_arg<T2, 2>(s, len, d, mat, st);
    else if (d.k == 3) dense_arg<T2, 3>(s, len, d, mat, st);
}

template <typename T2>
void launch_diag(T2 *s, uint64_t len, uint32_t k, const DiagTargets &t, uint64_t cmask, uint64_t cval,
                 const T2 *entries, hipStream_t st) {
    k_diag<T2><<<grid_for(len, 256, 65536), 256, 0, st>>>(s, len, k, t, cmask, cval, entries);
}

template <typename T2>
size_t stage_lds_bytes(uint32_t L) {
    return (sizeof(T2) << L) + STAGE_COEF_BYTES + STAGE_OPS * sizeof(StageOp);
}

template <typename T2, int LOG_THREADS>
static hipError_t stage_launch(T2 *s, const StageDesc &d, const StageOp *ops, const T2 *coefs, unsigned grid,
                               hipStream_t st) {
    const size_t lds = stage_lds_bytes<T2>(d.L);
    if (lds > 64 * 1024) {
        // Once per device: the largest tile's LDS.
        static std::atomic<uint64_t> attr_set{0};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        const uint64_t bit = uint64_t(1) << (dev & 63);
        if (!(attr_set.load() & bit)) {
            e = hipFuncSetAttribute((const void *)k_stage<T2, LOG_THREADS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)stage_lds_bytes<T2>(sizeof(T2) == 8 ? 14 : 13));
            if (e != hipSuccess) return e;
            attr_set.fetch_or(bit);
        }
    }
    k_stage<T2, LOG_THREADS><<<grid, 1u << LOG_THREADS, lds, st>>>(s, d, ops, coefs);
    return hipGetLastError();
}

// A wave for tiles of up to 2^6 amplitudes (its barriers cost nothing), 4 up
// to 2^9, 16 above: one tile's ops are a chain, so the more threads an op has, the
// shorter it is, down to an amplitude or two a thread.
template <typename T2>
hipError_t launch_stage(T2 *s, const StageDesc &d, const StageOp *ops, const T2 *coefs, unsigned grid,
                        hipStream_t st) {
    if (d.L <= 6) return stage_launch<T2, 6>(s, d, ops, coefs, grid, st);
    if (d.L <= 9) return stage_launch<T2, 8>(s, d, ops, coefs, grid, st);
    return stage_launch<T2, 10>(s, d, ops, coefs, grid, st);
}

// One block while the whole sum is a few batches of loads per thread (up to
// 2^13 amplitudes: a second launch would cost more), then 8 amplitudes a
// thread up to 1024 blocks.
template <typename T2>
void launch_norm(const T2 *s, uint64_t len, int qubit, double *partial, double *out, hipStream_t st) {
    const uint64_t count = qubit >= 0 ? len >> 1 : len;
    const unsigned blocks = count <= (1u << 13) ? 1 : (unsigned)std::min<uint64_t>(count >> 11, NORM_BLOCKS);
    double *const to = blocks == 1 ? out : partial;
    if (qubit >= 0) k_norm<T2, true><<<blocks, RED_THREADS, 0, st>>>(s, count, (uint32_t)qubit, to);
    else k_norm<T2, false><<<blocks, RED_THREADS, 0, st>>>(s, count, 0, to);
    if (blocks > 1) k_sum_rows<<<1, RED_THREADS, 0, st>>>(partial, blocks, out);
}

template <typename T2>
void launch_probabilities(const T2 *s, uint64_t len, double *out, hipStream_t st) {
    k_probabilities<T2><<<grid_for(len, 256), 256, 0, st>>>(s, len, out);
}

// Four pairs of amplitudes a thread where the state is small, and enough blocks
// over the groups of a launch to fill the chip where it is large. Launches follow
// one another, so each has to fill it by itself (28 qubits in complex64, a group each
// of 16, 8, 4 and 2 strings and 16 single ones, on low qubits: 13.3 ms with the blocks
// shared out over all 20 groups, 6.1 so). A power of two of them: every block
// then runs the same rounds (31 groups of one string and one of 16: 10.4 ms with 66
// blocks a group, 7.2 with 64).
PauliLaunches pauli_launches(uint64_t len, const std::vector<uint32_t> &widths) {
    auto slots = [](uint32_t w) { return w <= 1 ? 1u : w <= 2 ? 2u : w <= 4 ? 4u : w <= 8 ? 8u : PAULI_TERMS; };
    const uint64_t want = std::max<uint64_t>(1, len / (2 * 4 * RED_THREADS));
    PauliLaunches l;
    uint32_t first = 0;
    for (size_t g = 0; g < widths.size();) {
        PauliLaunch &p = l.at[l.n++];
        p = {slots(widths[g]), (uint32_t)g, 0, first, 0, 0, l.partials};
        for (; g < widths.size() && slots(widths[g]) == p.slots; g++) {
            p.ngroups++;
            p.nterms += widths[g];
        }
        uint64_t cap = 64;
        while (2 * cap * p.ngroups <= 2048) cap *= 2;
        p.blocks = (uint32_t)std::min(want, cap);
        first += p.nterms;
        l.partials += (uint64_t)p.nterms * p.blocks;
    }
    return l;
}

template <typename T2>
void launch_expect_pauli(const T2 *s, uint64_t len, const PauliGroup *groups, const PauliLaunches &launches,
                         const uint64_t *zs, uint32_t nterms, double *partial, double *out, hipStream_t st) {
    bool direct = true;  // a block per group everywhere: its sums are the results
    for (uint32_t i = 0; i < launches.n; i++) direct = direct && launches.at[i].blocks == 1;
    for (uint32_t i = 0; i < launches.n; i++) {
        const PauliLaunch &p = launches.at[i];
        auto go = [&](auto k) {
            k<<<dim3(p.blocks, p.ngroups), RED_THREADS, 0, st>>>(s, len, groups + p.group, zs, p.first,
                                                                 direct ? out + p.first : partial + p.partial);
        };
        if (p.slots == 1) go(k_expect_pauli<T2, 1>);
        else if (p.slots == 2) go(k_expect_pauli<T2, 2>);
        else if (p.slots == 4) go(k_expect_pauli<T2, 4>);
        else if (p.slots == 8) go(k_expect_pauli<T2, 8>);
        else go(k_expect_pauli<T2, PAULI_TERMS>);
    }
    if (!direct) k_sum_paulis<<<nterms, RED_THREADS, 0, st>>>(partial, launches, out);
}

// Segments of 2^16 amplitudes, 64 a thread; a single state of fewer than 24
// qubits takes smaller ones (at least 2^10), so that 256 of them fill the chip.
uint32_t expect_segment_bits(uint32_t n) {
    if (n <= EZ_TID_BITS) return n;
    return std::min<uint32_t>(EZ_TID_BITS + EZ_MAX_M_BITS, n <= EZ_TID_BITS + 8 ? EZ_TID_BITS : n - 8);
}

ExpDesc expect_desc(uint32_t state_qubits, uint32_t n, uint32_t segment_bits) {
    ExpDesc d{};
    d.B = segment_bits;
    d.nsegs = uint64_t(1) << (state_qubits - d.B);
    d.n = n;
    return d;
}

template <typename T2>
void launch_expect_z(const T2 *s, uint32_t n, double *seg_sums, double *z, double *zz, hipStream_t st) {
    const ExpDesc d = expect_desc(n, n, expect_segment_bits(n));
    k_expect_segments<T2><<<(unsigned)d.nsegs, 1 << EZ_TID_BITS, 0, st>>>(s, d, nullptr, 1, nullptr, seg_sums);
    const uint32_t outs = 2 * n - 1;
    // A block per output once a wave would walk more than 4 segments a lane.
    if (d.nsegs > 256) k_expect_combine<512, 512><<<outs, 512, 0, st>>>(seg_sums, d, nullptr, 1, nullptr, outs, z, zz);
    else k_expect_combine<64, 64><<<outs, 64, 0, st>>>(seg_sums, d, nullptr, 1, nullptr, outs, z, zz);
}

template <typename T2>
void launch_expect_batch(const T2 *s, const ExpDesc *descs, uint32_t ndesc, const uint64_t *seg_start,
                         uint64_t total_segs, const uint32_t *out_start, uint32_t total_outs, double *seg_sums,
                         double *z, double *zz, const ExpDesc &first, hipStream_t st) {
    k_expect_segments<T2><<<(unsigned)total_segs, 1 << EZ_TID_BITS, 0, st>>>(s, first, descs, ndesc, seg_start, seg_sums);
    k_expect_combine<256, 64><<<(total_outs + 3) / 4, 256, 0, st>>>(seg_sums, first, descs, ndesc, out_start, total_outs, z, zz);
}

void launch_zero_words(uint32_t *p, uint32_t n, hipStream_t st) {
    k_zero_words<<<(n + 255) / 256, 256, 0, st>>>(p, n);
}

template <typename T2>
void launch_batch_init(T2 *s, uint64_t len, const uint64_t *offs, uint32_t count, hipStream_t st) {
    k_init_zero<T2><<<grid_for(len, 256), 256, 0, st>>>(s, len);  // amplitude 0 of the first state is 1
    k_set_basis<T2><<<(count + 63) / 64, 64, 0, st>>>(s, offs, count);
}

template <typename TA, typename TB>
void launch_compare(const TA *a, const TB *b, uint64_t len, double *partial, unsigned blocks, hipStream_t st) {
    k_compare<TA, TB><<<blocks, RED_THREADS, 0, st>>>(a, b, len, partial);
}
template void launch_compare<float2, float2>(const float2 *, const float2 *, uint64_t, double *, unsigned, hipStream_t);
template void launch_compare<float2, double2>(const float2 *, const double2 *, uint64_t, double *, unsigned, hipStream_t);
template void launch_compare<double2, float2>(const double2 *, const float2 *, uint64_t, double *, unsigned, hipStream_t);
template void launch_compare<double2, double2>(const double2 *, const double2 *, uint64_t, double *, unsigned,
                                               hipStream_t);

uint32_t expect_batch_segment_bits(uint32_t n) { return std::min<uint32_t>(n, EZ_TID_BITS + EZ_MAX_M_BITS); }

template <typename T2>
void launch_collapse(T2 *s, uint64_t len, uint32_t qubit, double uniform, const double *p_one, bool flip,
                     double *p_copy, hipStream_t st) {
    // From 27 qubits on: below, the lines stay in the cache between a thread's pieces and
    // twice the threads cost more (20 qubits: 20.4 us, 23.5).
    if ((sizeof(T2) << qubit) < 128 && len >= (uint64_t(1) << 27)) {
        const unsigned grid = grid_for(len, 256, 65536);
        if (flip) k_collapse<T2, true, true><<<grid, 256, 0, st>>>(s, len, qubit, uniform, p_one, p_copy);
        else k_collapse<T2, false, true><<<grid, 256, 0, st>>>(s, len, qubit, uniform, p_one, p_copy);
        return;
    }
    const unsigned grid = grid_for(len >> 1, 256, 65536);
    if (flip) k_collapse<T2, true, false><<<grid, 256, 0, st>>>(s, len, qubit, uniform, p_one, p_copy);
    else k_collapse<T2, false, false><<<grid, 256, 0, st>>>(s, len, qubit, uniform, p_one, p_copy);
}

// Workspace of the allocation-free sampler. In host code `scratch` names a
// host-side stand-in, not the device array: its device address comes from
// hipGetSymbolAddress, once per device, and only that address is used.
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

hipError_t noalloc_scratch(void **ptr) {
    static std::mutex mu;
    static void *addr[64] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        addr[dev] = p;
    }
    *ptr = addr[dev];
    return hipSuccess;
}

size_t sort_temp_bytes(uint64_t shots) {
    size_t bytes = 0;
    if (hipcub::DeviceRadixSort::SortKeys(nullptr, bytes, (const double *)nullptr, (double *)nullptr, (int)shots) !=
        hipSuccess)
        return 0;
    return bytes;
}

// Chunks per workgroup of k_chain: one workgroup per CU, up to 16 chunks each;
// 0 where one lane per chunk is better: chunks shorter than a batch, and more
// than 4096 of them, which fill the chip.
static int chain_chunks(uint64_t clen, uint64_t nc) {
    if (clen < CHAIN_BATCH || nc > 4096) return 0;
    return nc >= 4096 ? 16 : nc >= 2048 ? 8 : nc >= 1024 ? 4 : nc >= 512 ? 2 : 1;
}

template <typename T2, bool WALK>
static void chain_launch(const T2 *s, uint64_t clen, uint64_t nc, int per, const SampleScratch &w, uint64_t shots,
                         hipStream_t st) {
    const unsigned grid = (unsigned)(nc / per);  // both are powers of two
    auto go = [&](auto k) {
        k<<<grid, CHAIN_THREADS, 0, st>>>(s, clen, w.mark_bits, w.prefix, w.bounds, w.targets, shots, w.marks, w.walked,
                                          w.sums);
    };
    if (per == 16) go(k_chain<T2, 16, WALK>);
    else if (per == 8) go(k_chain<T2, 8, WALK>);
    else if (per == 4) go(k_chain<T2, 4, WALK>);
    else if (per == 2) go(k_chain<T2, 2, WALK>);
    else go(k_chain<T2, 1, WALK>);
}

template <typename T2>
void launch_sample_sums(const T2 *s, uint64_t len, uint64_t chunk, SampleScratch &w, hipStream_t st) {
    const uint64_t nc = (len + chunk - 1) / chunk;
    const uint64_t clen = std::min(chunk, len);
    if (const int per = chain_chunks(clen, nc)) {
        chain_launch<T2, false>(s, clen, nc, per, w, 0, st);
    } else {
        // 64-lane workgroups for the per-chunk kernels, so 2^15 chunks spread over every CU.
        k_chunk_sums<T2><<<grid_for(nc, 64, 1u << 30), 64, 0, st>>>(s, len, chunk, nc, w.sums);
    }
    k_prefix<<<1, PREFIX_THREADS, 0, st>>>(w.sums, nc, w.prefix);
}

hipError_t launch_sort_uniforms(const double *uniforms, uint64_t shots, SampleScratch &w, hipStream_t st) {
    size_t bytes = w.sort_temp_bytes;
    return hipcub::DeviceRadixSort::SortKeys(w.sort_temp, bytes, uniforms, w.targets, (int)shots, 0,
                                             sizeof(double) * 8, st);
}

template <typename T2>
hipError_t launch_sample_walk(const T2 *s, uint64_t len, uint64_t chunk, uint64_t shots, SampleScratch &w,
                              uint64_t *out, hipStream_t st) {
    const uint64_t nc = (len + chunk - 1) / chunk;
    k_targets<<<grid_for(shots, 256), 256, 0, st>>>(w.targets, w.prefix + nc, shots);
    k_bounds<<<grid_for(nc + 1, 256, 1u << 30), 256, 0, st>>>(w.prefix, nc, w.targets, shots, w.bounds);
    const uint64_t clen = std::min(chunk, len);
    if (const int per = chain_chunks(clen, nc))
        chain_launch<T2, true>(s, clen, nc, per, w, shots, st);
    else
        k_walk_marks<T2><<<grid_for(nc, 64, 1u << 30), 64, 0, st>>>(s, len, chunk, nc, w.mark_bits, w.prefix, w.bounds,
                                                                    w.targets, shots, w.marks, w.walked);
    k_walk_place<T2><<<grid_for(shots, 256), 256, 0, st>>>(s, len, chunk, nc, w.mark_bits, w.prefix, w.bounds,
                                                           w.targets, shots, w.marks, w.walked, out);
    return hipGetLastError();
}

#define QVD_INSTANTIATE(T2)                                                                                     \
    template void launch_init_zero<T2>(T2 *, uint64_t, hipStream_t);                                            \
    template void launch_zero_stale<T2>(T2 *, uint64_t, uint64_t, hipStream_t);                                 \
    template void launch_widen<T2>(const T2 *, double2 *, uint64_t, hipStream_t);                               \
    template void launch_narrow<T2>(const double2 *, T2 *, uint64_t, hipStream_t);                              \
    template void launch_scale<T2>(T2 *, uint64_t, double, hipStream_t);                                        \
    template void launch_dense<T2>(T2 *, uint64_t, const GateDesc &, const T2 *, hipStream_t);                  \
    template void launch_dense_arg<T2>(T2 *, uint64_t, const GateDesc &, const T2 *, hipStream_t);              \
    template void launch_diag<T2>(T2 *, uint64_t, uint32_t, const DiagTargets &, uint64_t, uint64_t, const T2 *, \
                                  hipStream_t);                                                                 \
    template size_t stage_lds_bytes<T2>(uint32_t);                                                              \
    template hipError_t launch_stage<T2>(T2 *, const StageDesc &, const StageOp *, const T2 *, unsigned,        \
                                         hipStream_t);                                                          \
    template void launch_norm<T2>(const T2 *, uint64_t, int, double *, double *, hipStream_t);                  \
    template void launch_expect_z<T2>(const T2 *, uint32_t, double *, double *, double *, hipStream_t);         \
    template void launch_probabilities<T2>(const T2 *, uint64_t, double *, hipStream_t);                        \
    template void launch_expect_pauli<T2>(const T2 *, uint64_t, const PauliGroup *, const PauliLaunches &,      \
                                          const uint64_t *, uint32_t, double *, double *, hipStream_t);         \
    template void launch_expect_batch<T2>(const T2 *, const ExpDesc *, uint32_t, const uint64_t *, uint64_t,    \
                                          const uint32_t *, uint32_t, double *, double *, double *, const ExpDesc &, \
                                          hipStream_t);                                                         \
    template void launch_batch_init<T2>(T2 *, uint64_t, const uint64_t *, uint32_t, hipStream_t);              \
    template void launch_collapse<T2>(T2 *, uint64_t, uint32_t, double, const double *, bool, double *, hipStream_t); \
    template void launch_sample_sums<T2>(const T2 *, uint64_t, uint64_t, SampleScratch &, hipStream_t);         \
    template hipError_t launch_sample_walk<T2>(const T2 *, uint64_t, uint64_t, uint64_t, SampleScratch &,       \
                                               uint64_t *, hipStream_t);

QVD_INSTANTIATE(float2)
QVD_INSTANTIATE(double2)

}  // namespace qvd
