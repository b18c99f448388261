// engine.hip -- gfx950 kernels and the C ABI declared in include/dgq_engine.h.
//
// Kernels:
//   sweep_kernel<T,R,W>  one fused block over every tile of a state (or over a
//                        batch of small states, one tile each).  Replaces the
//                        reference's statevec_fusedKernel
//                        (src/cpp/QuEST_gpu_kernel.cu:175-359) and, through the
//                        store permutation, its reorder_data_kernel (:589-636).
//   small_kernel<T>      whole state in LDS, ops in global-index form; for
//                        registers too small for a 64-lane tile (n < 8).
//   prob_stage1/2<T>     P(q=0) for all qubits + total probability
//                        (replaces :656-840 with wave64 reductions).
//   read/write/init      amplitude gather/scatter and state fill.
//
// Layout: 2^n interleaved complex amplitudes; qubit q = bit q of the index.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "dgq_engine.h"

// ----------------------------------------------------------------------------
// error handling
// ----------------------------------------------------------------------------
static thread_local char g_err[512] = "";

static int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

#define HIPC(x)                                                                          \
    do {                                                                                 \
        hipError_t e_ = (x);                                                             \
        if (e_ != hipSuccess)                                                            \
            return fail(DQ_ERR_HIP, "%s failed: %s (%s:%d)", #x, hipGetErrorString(e_), \
                        __FILE__, __LINE__);                                             \
    } while (0)

extern "C" const char *dq_last_error(void) { return g_err; }

// ----------------------------------------------------------------------------
// device helpers
// ----------------------------------------------------------------------------
template <typename T> struct V2;
template <> struct V2<double> { typedef double type __attribute__((ext_vector_type(2))); };
template <> struct V2<float> { typedef float type __attribute__((ext_vector_type(2))); };

// The register tile of one thread: 2^R amplitudes, real and imaginary parts
// as separate scalars.  Every op below updates these registers in place, so
// the tile keeps one register assignment through the op loop.
template <typename T, int R>
struct Regs {
    T re[1 << R];
    T im[1 << R];
};

// Per-phase and per-block records the engine's host code forms for the sweep
// kernels (u32 arrays in the workspace):
//   phase_aux, DQ_PAUX words per phase: [0] byte offset of the phase's device
//     program, [1] its op count; for the exchange from the previous phase into
//     this one, LDS byte offsets under that exchange's swizzle:
//     [DQ_XA + j] / [DQ_XB + j] the uniform part of register index j in the
//     previous / this phase's layout, [DQ_TA + i] / [DQ_TB + i] the part of
//     thread bit i (lane bits 0..5, then wave bits).  Split exchanges (mode
//     1, owned slots) use the same words for their two computed sides, [2] = 1
//     when the exchange needs its middle barrier, and [DQ_TF + i] /
//     [DQ_FJ + j] for the thread's own slots.
//   block_aux, DQ_BAUX words per block: the non-tile qubits as runs of
//     consecutive qubits, [i] = first bit in the tile index | run length << 16,
//     [16 + i] = the run's lowest qubit; runs past the last have length 0.
#define DQ_PAUX 144
#define DQ_XA 8
#define DQ_XB 40
#define DQ_TA 72
#define DQ_TB 81
#define DQ_TF 96
#define DQ_FJ 105
#define DQ_BAUX 32
#define DQ_RUNS 10
#define DQ_BA_PROG 30     // [30] byte offset of the block's device programs, [31] their bytes
#define DQ_WARM_TILES 512 // workgroups that warm the L2 (about the first that run, two per CU)

// Uniform descriptors: read through the constant address space, so that every
// load is a scalar one whether they lie in the workspace or in the kernel's
// arguments.
#define DQ_CONST __attribute__((address_space(4)))
typedef const DQ_CONST dq_block *CBlock;
typedef const DQ_CONST uint32_t *CWords;

// Byte offset of a thread's part of an exchange address: xor of the parts of
// its set thread bits.  The wave bits are wave-uniform (wv is a scalar), so
// their part is formed with scalar selects; each lane bit costs a bit extract
// (0 or all ones), an and and an xor, with no branch.
template <int W>
__device__ __forceinline__ uint32_t thread_part(CWords t, uint32_t lane, uint32_t wv) {
    uint32_t tv[6 + W];
#pragma unroll
    for (int i = 0; i < 6 + W; i++) tv[i] = t[i];
    uint32_t x = 0;
#pragma unroll
    for (int w = 0; w < W; w++) x ^= ((wv >> w) & 1u) ? tv[6 + w] : 0u;
#pragma unroll
    for (int i = 0; i < 6; i++) x ^= (uint32_t)(-(int32_t)((lane >> i) & 1u)) & tv[i];
    return x;
}

// An LDS element at byte offset `off` of the workgroup's LDS.  The sweep
// kernels declare no static LDS (the engine checks their static group
// segment is 0 when it initialises a device), so their dynamic LDS starts at
// address 0 and an offset is the address itself: no base add per access.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(3))) T *lds_at(uint32_t off) {
    return (__attribute__((address_space(3))) T *)(size_t)off;
}

// Re-distribute the tile from the layout of the previous phase to that of
// this one through LDS (each thread writes its 2^R amplitudes, then reads
// 2^R).  Exchange modes (XM):
//  0  whole amplitudes.  An element's LDS slot is its tile index under a
//     linear swizzle the host picks per exchange (xor of the low bits with
//     images of the high bits) so that the lanes served together by the LDS in
//     either layout hit distinct banks; a byte offset is the thread's part xor
//     a uniform part per register index j, from the host's tables (ex = this
//     phase's phase_aux), one vector xor per access.  A barrier leads every
//     exchange after a block's first (other threads may still read the slots).
//  1  real parts, then imaginary parts, through an LDS array of scalars (half
//     the footprint: more workgroups per CU), in owned slots: every position
//     (thread, register index) of a layout has a fixed slot, own[j] for this
//     thread's register j, under one swizzle per block.  Real parts go from
//     the old positions' slots to their new owners (ex's TB / XB parts: the
//     slot of the previous layout's position of each new element), imaginary
//     parts from their old owners to the new positions' slots (TA / XA).  The
//     imaginary read is from the thread's own slots, which the next
//     exchange's real write reuses, so no barrier leads an exchange; the one
//     between the passes (ex[2]) is needed only when the layout change is not
//     a set of pairwise swaps of positions, since only then may a thread
//     write an imaginary part into a slot another thread has yet to read a
//     real part from.
template <int R, int W, int XM, typename T>
__device__ __forceinline__ void exchange(Regs<T, R> &a, CWords ex, bool lead_barrier,
                                         uint32_t lane, uint32_t wv, const uint32_t *own) {
    constexpr int NR = 1 << R;
    const CWords xa = ex + DQ_XA;
    const CWords xb = ex + DQ_XB;
    const uint32_t sa = thread_part<W>(ex + DQ_TA, lane, wv);
    const uint32_t sb = thread_part<W>(ex + DQ_TB, lane, wv);
    if constexpr (XM == 0) {
        if (lead_barrier) __syncthreads();
#pragma unroll
        for (int j = 0; j < NR; j++) {
            auto *q = lds_at<T>(sa ^ xa[j]);
            q[0] = a.re[j];
            q[1] = a.im[j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NR; j++) {
            const auto *q = lds_at<T>(sb ^ xb[j]);
            a.re[j] = q[0];
            a.im[j] = q[1];
        }
    } else {
        (void)lead_barrier;
#pragma unroll
        for (int j = 0; j < NR; j++) *lds_at<T>(own[j]) = a.re[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NR; j++) a.re[j] = *lds_at<T>(sb ^ xb[j]);
        if (ex[2]) __syncthreads();
#pragma unroll
        for (int j = 0; j < NR; j++) *lds_at<T>(sa ^ xa[j]) = a.im[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NR; j++) a.im[j] = *lds_at<T>(own[j]);
    }
}

// What a launch of a single job carries in its arguments: the job, its block
// and the block's block_aux record.
struct SweepOne {
    dq_block blk;
    uint32_t baux[DQ_BAUX];
    dq_job job;
    double *part;  // where the tiles' probability sums go, or null
    // A launch of one tile that brings the descriptors to the device itself (null: they are there)
    const uint4 *src;
    uint4 *dst;
    uint32_t *read;  // pinned: set to `ticket` once src has been read
    uint32_t n16, ticket;
};

// Non-tile qubits of tile number t (t < 2^31) from the block's runs.
__device__ __forceinline__ uint64_t tile_base_runs(CWords ba, uint32_t t) {
    uint64_t base = 0;
#pragma unroll
    for (int i = 0; i < DQ_RUNS; i++) {
        const uint32_t c = ba[i];
        base |= (uint64_t)((t >> (c & 31u)) & ((1u << (c >> 16)) - 1u)) << ba[16 + i];
    }
    return base;
}

// ---- op interpreter --------------------------------------------------------
// The op list of a phase runs in gfx950 assembly generated by gen_ops_asm.py
// (format of the device program and register use documented there).
#include "ops_asm.inc"

// Occupancy target (waves per SIMD) of a sweep instantiation: the register
// tile takes 2^R amplitudes x (2 * sizeof(T) / 4) VGPRs; allow 40 more for
// addresses, coefficients and temporaries.  Split-exchange R = 5 tiles need
// more: 128 VGPRs and 4 spilled in FP32 (104 and none before the FAN op's FP64
// factor and the sums for P(0)), 168 and 7 in FP64 (as before).
template <typename T, int R, int XM>
constexpr int sweep_waves_per_eu() {
    constexpr int amp = (1 << R) * (int)(2 * sizeof(T) / 4);
    constexpr int budget = amp + 40;
    constexpr int w = 512 / budget;
    return w > 8 ? 8 : (w < 1 ? 1 : w);
}

// Non-tile qubits of tile number `t`: its bits deposited into nontile_mask.
__device__ __forceinline__ uint64_t tile_base(uint64_t msk, uint64_t t) {
    uint64_t base = 0;
    while (msk) {
        const int p = __builtin_ctzll(msk);
        base |= (t & 1ull) << p;
        t >>= 1;
        msk &= msk - 1;
    }
    return base;
}

// Element `lane` of the 64 consecutive amplitudes starting at the
// wave-uniform address p: a 32-bit lane byte offset on a scalar base, so the
// access is one global load/store with a scalar address and no 64-bit vector
// address arithmetic.
template <typename P>
__device__ __forceinline__ P lane_ptr(P p, uint32_t lane) {
    return (P)((const __attribute__((address_space(1))) char *)p + lane * (uint32_t)sizeof(*p));
}

// Load a tile into registers: lane l = qubit l, register / wave bits =
// ld_reg / ld_wave.  The wave index wv is wave-uniform (a scalar), so every
// address is "scalar base + lane * sizeof(V)" with no vector math.
template <typename T, int R, int W>
__device__ __forceinline__ void load_tile(Regs<T, R> &a, CBlock blk,
                                          const __attribute__((address_space(1))) typename V2<T>::type *st,
                                          uint64_t base, uint32_t wv, uint32_t lane) {
    using V = typename V2<T>::type;
    constexpr int NR = 1 << R;
    uint64_t lw[W > 0 ? W : 1], wb = 0;
#pragma unroll
    for (int w = 0; w < W; w++) lw[w] = blk->ld_wave[w];
#pragma unroll
    for (int w = 0; w < W; w++) wb |= lw[w] & (0ull - ((wv >> w) & 1u));
    uint64_t qo[R > 0 ? R : 1];
#pragma unroll
    for (int r = 0; r < R; r++) qo[r] = blk->ld_reg[r];
    const uint32_t ik = blk->init_kind;
    if (ik == DQ_INIT_LOAD) {
#pragma unroll
        for (int j = 0; j < NR; j++) {
            uint64_t u = base | wb;
#pragma unroll
            for (int r = 0; r < R; r++)
                if ((j >> r) & 1) u |= qo[r];
            const V v = __builtin_nontemporal_load(lane_ptr(st + u, lane));
            a.re[j] = v.x;
            a.im[j] = v.y;
        }
    } else if (ik == DQ_INIT_CLASSICAL) {
        const uint64_t want = blk->init_index;
#pragma unroll
        for (int j = 0; j < NR; j++) {
            uint64_t u = base | wb;
#pragma unroll
            for (int r = 0; r < R; r++)
                if ((j >> r) & 1) u |= qo[r];
            a.re[j] = ((u | lane) == want) ? T(1) : T(0);
            a.im[j] = T(0);
        }
    } else {
        const T v = (T)blk->init_value;
#pragma unroll
        for (int j = 0; j < NR; j++) { a.re[j] = v; a.im[j] = T(0); }
    }
}

// Store a tile: lane l = qubit l, register / wave bits = st_reg / st_wave.
// (A macro expanded in the kernel body: as a function taking the tile by
// reference, the FP32 instantiations kept part of the tile in scratch.)
#define DQ_STORE_TILE(A, BASE)                                                            \
    do {                                                                                  \
        uint64_t wb_ = 0;                                                                 \
        _Pragma("unroll") for (int w = 0; w < W; w++) wb_ |= blk->st_wave[w] & (0ull - ((wv >> w) & 1u)); \
        uint64_t qo_[R > 0 ? R : 1];                                                      \
        _Pragma("unroll") for (int r = 0; r < R; r++) qo_[r] = blk->st_reg[r];            \
        _Pragma("unroll") for (int j = 0; j < (1 << R); j++) {                            \
            uint64_t u = (BASE) | wb_;                                                    \
            _Pragma("unroll") for (int r = 0; r < R; r++) if ((j >> r) & 1) u |= qo_[r];  \
            typename V2<T>::type v_;                                                      \
            v_.x = (A).re[j];                                                             \
            v_.y = (A).im[j];                                                             \
            __builtin_nontemporal_store(v_, lane_ptr(st + u, lane));                      \
        }                                                                                 \
    } while (0)

// A one-phase block that moves a qubit between wave bits (ld_wave != st_wave)
// stores part of each wave's amplitudes where another wave of the workgroup
// loaded: every load of the tile must be done before the first store.  With
// two or more phases the first LDS exchange already orders them (each wave
// writes its loaded tile to LDS before the exchange barrier).
template <int W>
__device__ __forceinline__ bool store_needs_barrier(CBlock blk) {
    if (blk->phase_count != 1) return false;
    bool x = false;
#pragma unroll
    for (int w = 0; w < W; w++) x |= blk->ld_wave[w] != blk->st_wave[w];
    return x;
}

// The phases of a block on one tile: exchanges through LDS between phases,
// the op program of each phase in the assembly interpreter.  lead: a barrier
// before the first exchange (LDS may still be read for a previous tile).
template <typename T, int R, int W, int XM>
__device__ __forceinline__ void process_tile(Regs<T, R> &a, const dq_phase *__restrict__ ph, uint32_t nph,
                                             CWords pa, const unsigned char *__restrict__ prog,
                                             uint64_t cbase, uint32_t tid, uint32_t wv, bool lead) {
    // owned-slot exchanges: the thread's own slots are the same in every
    // exchange of a block, formed once
    uint32_t own[XM == 1 ? (1 << R) : 1];
    if constexpr (XM == 1) {
        if (nph > 1) {
            const CWords e1 = pa + DQ_PAUX;
            const uint32_t f = thread_part<W>(e1 + DQ_TF, tid & 63u, wv);
#pragma unroll
            for (int j = 0; j < (1 << R); j++) own[j] = f ^ e1[DQ_FJ + j];
        }
    }
    // A wave in an exchange goes ahead of one in an op program (its workgroup waits
    // for it at a barrier), and in FP64 one that forms addresses and issues loads too
    // (sweep_kernel): 4096 samples of a 25-qubit FP64 ansatz 2815 -> 2744 us, 26-qubit FP64
    // Trotter step 1200 -> 1182 us, 28-qubit FP32 grid 15.8 -> 15.6 ms.  Loads first in
    // FP32 as well made a 27-qubit Fourier transform 1% slower.
    for (uint32_t p = 0; p < nph; p++) {
        if (p > 0) {
            __builtin_amdgcn_s_setprio(2);
            exchange<R, W, XM, T>(a, pa + p * DQ_PAUX, p > 1 || lead, tid & 63u, wv, own);
            __builtin_amdgcn_s_setprio(0);
        }
        AsmOps<T, R>::run(a, prog + pa[p * DQ_PAUX], cbase, tid);
    }
}

// Brings a block's device program and exchange tables into this XCD's L2 while
// the tile is still on its way: they are read line by line, each read waiting
// for the one before, and the first workgroups of a launch would wait for
// memory at every line.  With the argument-borne descriptors below, measured
// per sweep before -> now: 17 qubits FP32 R = 3, W = 0 9.6 -> 6.5 us; 16 tiles of
// 12 bits FP32 19.2 -> 12.4 us; one tile of 10 bits with a whole circuit
// 155 -> 71 us; 21 qubits FP64 R = 4, W = 3 38 -> 27 us.  Loading the program's
// lines into the scalar cache as well gained nothing on top.  (Relaxed atomic loads: a plain load whose result
// nothing uses would be dropped.)
__device__ __forceinline__ void warm_lines(const unsigned char *p, uint32_t bytes, uint32_t tid, uint32_t threads) {
    for (uint32_t i = tid * 128u; i < bytes; i += threads * 128u)
        (void)__hip_atomic_load(reinterpret_cast<const uint32_t *>(p + i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Probability sums of a tile as it is stored, from the registers: for every tile bit
// (lane bits, register bits, wave bits) the sum of |a|^2 over the amplitudes with the
// bit 0, then the total, to part[slot * workgroups + workgroup]; prob_stage2 makes P(0)
// of every qubit of them.  A read-out after a flush took a read of the whole state; the
// sums cost 5 FP64 instructions an amplitude and, with the lane and wave sums left
// to one wave each by way of LDS, ~1 KB of LDS traffic a wave.  A 26-qubit FP64 Trotter step
// with P(0) 1377 -> 1201 us, 17 qubits FP32 with their sums added up by the host 229 -> 224 us.
// t: a thread's total, z[r]: its sum with register bit r 0.  Only sums of
// non-negative terms: an exact 0 stays one.
template <int R, int W>
__device__ __forceinline__ void tile_sums(double t, const double *z, double *__restrict__ part, uint32_t lane, uint32_t wv) {
    constexpr int NW = 1 << W, T = 6 + R + W;
    auto *red = lds_at<double>(0);  // [1 + R][wave][lane]
    __syncthreads();                // other waves may still read the last exchange
    red[wv * 64 + lane] = t;
#pragma unroll
    for (int r = 0; r < R; r++) red[((1 + r) * NW + wv) * 64 + lane] = z[r];
    __syncthreads();
    auto column = [&](int v, uint32_t skip) {  // over the waves without bit `skip`
        double a = 0.0;
#pragma unroll
        for (uint32_t w = 0; w < NW; w++) {
            const double x = red[(v * NW + w) * 64 + lane];
            a += (w & skip) ? 0.0 : x;
        }
        return a;
    };
    auto lanes = [&](double a, int from) {
#pragma unroll
        for (int k = 0; k < 6; k++)
            if (k >= from) a += __shfl_xor(a, 1 << k, 64);
        return a;
    };
    auto put = [&](int slot, double a) {
        if (lane == 0) part[(uint64_t)slot * gridDim.x + blockIdx.x] = a;
    };
    for (uint32_t job = wv; job < 1 + R + W; job += NW) {
        if (job == 0) {
            double a = column(0, 0);
#pragma unroll
            for (int q = 0; q < 6; q++) {
                put(q, lanes(a, q + 1));  // lane 0 has bit q 0
                a += __shfl_xor(a, 1 << q, 64);
            }
            put(T, a);
        } else if (job <= R) {
            put(5 + job, lanes(column(job, 0), 0));
        } else {
            put(5 + job, lanes(column(0, 1u << (job - 1 - R)), 0));
        }
    }
}

// Descriptors from pinned host memory to the device, by the only workgroup that reads
// them: a copying kernel before it takes 4 us and another 4 until the next starts.
// The stores are in the L2 (vmcnt 0) before any wave goes on to read them through
// the scalar cache, which has seen none of these lines since the launch began.
// 12-qubit Fourier transform with its amplitudes 42.3 -> 39.7 us a pass.
template <int W>
__device__ __forceinline__ void bring_descriptors(const uint4 *__restrict__ src, uint4 *__restrict__ dst, uint32_t n16, uint32_t *read,
                                                  uint32_t ticket, uint32_t tid) {
    constexpr uint32_t N = 64u << W;
    auto copy = [&](auto rounds) {  // U loads in flight per thread
        constexpr uint32_t U = decltype(rounds)::value;
        for (uint32_t i0 = tid; i0 < n16; i0 += N * U) {
            uint4 v[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++) v[u] = src[std::min(i0 + u * N, n16 - 1)];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                asm volatile("" : "+v"(v[u].x), "+v"(v[u].y), "+v"(v[u].z), "+v"(v[u].w));  // not sunk into the branch
                if (i0 + u * N < n16) dst[i0 + u * N] = v[u];
            }
        }
    };
    if (n16 <= 2 * N) copy(std::integral_constant<uint32_t, 2>());
    else copy(std::integral_constant<uint32_t, 8>());
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    __syncthreads();
    if (tid == 0) __hip_atomic_store(read, ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A launch of one job reads it, its block and block_aux from the kernel's
// arguments (`one`): the tile's addresses are then one memory latency away
// instead of three (argument, job, block).  A batch reads them per job.
// OWN: a launch of one tile that brings its descriptors itself (one.src).
template <typename T, int R, int W, int XM, bool OWN = false>
__global__ void __launch_bounds__(64 << W, (sweep_waves_per_eu<T, R, XM>()))
sweep_kernel(const SweepOne one, const dq_job *__restrict__ jobs, const dq_block *__restrict__ blocks,
             const dq_phase *__restrict__ phases, const unsigned char *__restrict__ prog,
             const uint32_t *__restrict__ phase_aux, const uint32_t *__restrict__ block_aux) {
    using GV = __attribute__((address_space(1))) typename V2<T>::type;
    (void)one;
    if constexpr (sizeof(T) == 8) __builtin_amdgcn_s_setprio(1);
    const auto *ka = (const DQ_CONST SweepOne *)__builtin_amdgcn_kernarg_segment_ptr();
    CBlock blk = &ka->blk;
    CWords ba = ka->baux;
    void *state = ka->job.state;
    uint64_t hi = ka->job.base_hi;
    if (gridDim.y > 1) {
        const auto *job = (const DQ_CONST dq_job *)(uintptr_t)(jobs + blockIdx.y);
        blk = (CBlock)(uintptr_t)(blocks + job->block);
        ba = (CWords)(uintptr_t)(block_aux + job->block * DQ_BAUX);
        state = job->state;
        hi = job->base_hi;
    }
    GV *__restrict__ st = (GV *)(state);
    const uint32_t tid = threadIdx.x;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lane = tid & 63u;
    if constexpr (OWN) {
        bring_descriptors<W>(ka->src, ka->dst, ka->n16, ka->read, ka->ticket, tid);
        // opaque copies: what the pointers lead to was written just now
        asm volatile("" : "+s"(prog), "+s"(phase_aux) : : "memory");
    }
    const uint64_t base = tile_base_runs(ba, blockIdx.x);
    const CWords pa = (CWords)(uintptr_t)(phase_aux + blk->phase_begin * DQ_PAUX);
    if (!OWN && blockIdx.x < DQ_WARM_TILES) {
        warm_lines(prog + ba[DQ_BA_PROG], ba[DQ_BA_PROG + 1], tid, 64u << W);
        if (blk->phase_count > 1)
            warm_lines(reinterpret_cast<const unsigned char *>(phase_aux + blk->phase_begin * DQ_PAUX), blk->phase_count * DQ_PAUX * 4u, tid, 64u << W);
    }
    Regs<T, R> a;
    load_tile<T, R, W>(a, blk, st, base, wv, lane);
    // an opaque copy: knowing the count again after the loop, the compiler
    // would keep a second copy of the tile for blocks of one phase
    uint32_t nph = blk->phase_count;
    asm volatile("" : "+s"(nph));
    if constexpr (sizeof(T) == 8) __builtin_amdgcn_s_setprio(0);
    process_tile<T, R, W, XM>(a, phases + blk->phase_begin, nph, pa, prog, base | hi, tid, wv, false);
    if (store_needs_barrier<W>(blk)) __syncthreads();
    DQ_STORE_TILE(a, base);
    if (gridDim.y == 1 && ka->part) {
        double t = 0.0, z[R];
#pragma unroll
        for (int r = 0; r < R; r++) z[r] = 0.0;
#pragma unroll
        for (int j = 0; j < (1 << R); j++) {
            const double x = (double)a.re[j], y = (double)a.im[j], p = x * x + y * y;
            t += p;
#pragma unroll
            for (int r = 0; r < R; r++)
                if (!((j >> r) & 1)) z[r] += p;
            if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // not every product at once: they would not fit
        }
        // the lane formed anew: kept through the interpreter it would cost a register
        const uint32_t l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        tile_sums<R, W>(t, z, ka->part, l, wv);
    }
}

// Small registers (n <= 13): whole state in LDS, one workgroup per job.  Ops
// are in global-index form: tbit = target qubit, (c_wg, v_wg) = condition
// over the full index.
template <typename T>
__global__ void __launch_bounds__(256)
small_kernel(const dq_job *__restrict__ jobs, const dq_block *__restrict__ blocks,
             const dq_phase *__restrict__ phases, const dq_op *__restrict__ ops) {
    using V = typename V2<T>::type;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    V *s = reinterpret_cast<V *>(lds_raw);
    const dq_job job = jobs[blockIdx.y];
    const dq_block *__restrict__ blk = blocks + job.block;
    V *__restrict__ st = reinterpret_cast<V *>(job.state);
    const uint32_t n = blk->n_qubits;
    const uint32_t N = 1u << n;
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < N; i += blockDim.x) {
        if (blk->init_kind == DQ_INIT_LOAD) s[i] = st[i];
        else if (blk->init_kind == DQ_INIT_CLASSICAL) { s[i].x = (i == blk->init_index) ? T(1) : T(0); s[i].y = T(0); }
        else { s[i].x = (T)blk->init_value; s[i].y = T(0); }
    }
    const dq_phase *__restrict__ ph = phases + blk->phase_begin;
    for (uint32_t p = 0; p < blk->phase_count; p++) {
        for (uint32_t k = 0; k < ph[p].op_count; k++) {
            const dq_op *__restrict__ op = ops + ph[p].op_begin + k;
            const T *__restrict__ m = reinterpret_cast<const T *>(op->m);
            const uint64_t c = op->c_wg, v = op->v_wg, hi = job.base_hi;
            __syncthreads();
            if (op->kind == DQ_OP_MAT || op->kind == DQ_OP_SWAP || op->kind == DQ_OP_RMAT || op->kind == DQ_OP_SHEAR) {
                const uint32_t t = op->tbit, tm = 1u << t;
                for (uint32_t k2 = tid; k2 < N / 2; k2 += blockDim.x) {
                    const uint32_t i0 = ((k2 >> t) << (t + 1)) | (k2 & (tm - 1));
                    const uint32_t i1 = i0 | tm;
                    if (((i0 | hi) & c) != v) continue;
                    const V x = s[i0], y = s[i1];
                    if (op->kind == DQ_OP_SWAP) { s[i0] = y; s[i1] = x; continue; }
                    if (op->kind == DQ_OP_SHEAR) {
                        V nx, ny;
                        nx.x = x.x + m[0] * y.x; nx.y = x.y + m[0] * y.y;
                        ny.x = y.x + m[1] * nx.x; ny.y = y.y + m[1] * nx.y;
                        s[i0] = nx; s[i1] = ny;
                        continue;
                    }
                    V nx, ny;
                    if (op->kind == DQ_OP_RMAT) {
                        nx.x = m[0] * x.x + m[1] * y.x; nx.y = m[0] * x.y + m[1] * y.y;
                        ny.x = m[2] * x.x + m[3] * y.x; ny.y = m[2] * x.y + m[3] * y.y;
                        s[i0] = nx; s[i1] = ny;
                        continue;
                    }
                    nx.x = m[0] * x.x - m[1] * x.y + m[2] * y.x - m[3] * y.y;
                    nx.y = m[0] * x.y + m[1] * x.x + m[2] * y.y + m[3] * y.x;
                    ny.x = m[4] * x.x - m[5] * x.y + m[6] * y.x - m[7] * y.y;
                    ny.y = m[4] * x.y + m[5] * x.x + m[6] * y.y + m[7] * y.x;
                    s[i0] = nx;
                    s[i1] = ny;
                }
            } else {
                for (uint32_t i = tid; i < N; i += blockDim.x) {
                    if (((i | hi) & c) != v) continue;
                    V x = s[i];
                    if (op->kind == DQ_OP_NEG) { x.x = -x.x; x.y = -x.y; s[i] = x; continue; }
                    V y;
                    y.x = m[0] * x.x - m[1] * x.y;
                    y.y = m[0] * x.y + m[1] * x.x;
                    s[i] = y;
                }
            }
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < N; i += blockDim.x) st[i] = s[i];
}

// ----------------------------------------------------------------------------
// probabilities
// ----------------------------------------------------------------------------
// P(0) of every qubit over the amplitudes whose index has given values on a
// set of fixed bits (none for a whole state).  The other bits, in ascending
// order, number the 2^nf amplitudes read; img[f] is the index bit of number
// bit f (one-hot) and `fixed` the value of the fixed bits.
//
// Stage 1: workgroup g sums the numbers [g * 2^cb, (g + 1) * 2^cb), split as
// bits 0..5 lane, the next JB bits a load index j, two wave bits, and up to
// PROB_OUTER bits of a loop.  A wave has its 2^JB loads (1 KiB each in FP64
// when no lane bit is fixed) in flight together.  It writes cb + 1 partial
// sums, slot-major (part[slot * groups + g]): P0 of number bits 0..cb-1, then
// the total.
//
// Bound: HBM for large states (16 * 2^n bytes, read once), latency for small
// ones.  Before, a workgroup always read 2^16 amplitudes one load at a time:
// a 17-qubit state occupied two workgroups.  Measured, both stages back to
// back, before -> now: 17 qubits FP32 73 -> 6.8 us, 23 qubits FP64 141 -> 27 us
// (4.9 TB/s), 26 qubits FP64 245 -> 169 us, 30 qubits FP64 2.97 -> 2.53 ms
// (6.8 TB/s; 16 loads in flight per thread instead of what one loop step gives).
#define PROB_OUTER 8
#define PROB_SLOTS_MAX (8 + 4 + PROB_OUTER + 1)
#define PROB_MAX_QUBITS 40

struct ProbBits {
    uint64_t img[PROB_MAX_QUBITS];
    uint64_t fixed;
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <typename T, int JB>
__global__ void __launch_bounds__(256)
prob_stage1(const typename V2<T>::type *__restrict__ st, const ProbBits pb, int nf, int cb, double *__restrict__ part) {
    using V = typename V2<T>::type;
    constexpr int J = 1 << JB;
    __shared__ double red[4][PROB_SLOTS_MAX];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint64_t base = pb.fixed;
    for (int i = cb; i < nf; i++) base |= ((blockIdx.x >> (i - cb)) & 1u) ? pb.img[i] : 0ull;
    base |= ((w & 1u) ? pb.img[6 + JB] : 0ull) | ((w & 2u) ? pb.img[7 + JB] : 0ull);
    uint64_t lp = 0;
#pragma unroll
    for (int i = 0; i < 6; i++) lp |= ((lane >> i) & 1u) ? pb.img[i] : 0ull;
    uint64_t jm[JB > 0 ? JB : 1];
#pragma unroll
    for (int b = 0; b < JB; b++) jm[b] = pb.img[6 + b];
    uint64_t S = 0;  // the loop's index bits
    for (int i = 8 + JB; i < cb; i++) S |= pb.img[i];
    const uint32_t loops = cb > 8 + JB ? 1u << (cb - 8 - JB) : 1u;
    const bool on = nf >= 8 || (tid >> nf) == 0;  // fewer than 256 amplitudes: the threads that own one
    double tot = 0.0, zj[JB > 0 ? JB : 1], zo[PROB_OUTER];
#pragma unroll
    for (int b = 0; b < JB; b++) zj[b] = 0.0;
#pragma unroll
    for (int b = 0; b < PROB_OUTER; b++) zo[b] = 0.0;
    uint64_t x = 0;
    for (uint32_t it = 0; it < loops; it++) {
        V v[J];
#pragma unroll
        for (int j = 0; j < J; j++) {
            uint64_t u = base | x;
#pragma unroll
            for (int b = 0; b < JB; b++)
                if ((j >> b) & 1) u |= jm[b];
            v[j] = __builtin_nontemporal_load(st + u + lp);
        }
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < J; j++) {
            const double p = on ? (double)v[j].x * (double)v[j].x + (double)v[j].y * (double)v[j].y : 0.0;
            s += p;
#pragma unroll
            for (int b = 0; b < JB; b++)
                if (!((j >> b) & 1)) zj[b] += p;
        }
        tot += s;
#pragma unroll
        for (int b = 0; b < PROB_OUTER; b++)
            if (!((it >> b) & 1u)) zo[b] += s;
        x = ((x | ~S) + 1ull) & S;
    }
    // lane bit q: the lanes with the bit 0, other bits summed (valid in lane 0)
    double t = tot;
#pragma unroll
    for (int q = 0; q < 6; q++) {
        double r = t;
#pragma unroll
        for (int k = q + 1; k < 6; k++) r += __shfl_xor(r, 1 << k, 64);
        if (lane == 0) red[w][q] = r;
        t += __shfl_xor(t, 1 << q, 64);
    }
    if (lane == 0) red[w][PROB_SLOTS_MAX - 1] = t;
#pragma unroll
    for (int b = 0; b < JB; b++) {
        const double r = wave_sum(zj[b]);
        if (lane == 0) red[w][6 + b] = r;
    }
#pragma unroll
    for (int b = 0; b < PROB_OUTER; b++)
        if (8 + JB + b < cb) {
            const double r = wave_sum(zo[b]);
            if (lane == 0) red[w][8 + JB + b] = r;
        }
    __syncthreads();
    const int s = (int)tid;
    if (s <= cb) {
        const int c = PROB_SLOTS_MAX - 1;
        double r;
        if (s == cb) r = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
        else if (s == 6 + JB) r = red[0][c] + red[2][c];
        else if (s == 7 + JB) r = red[0][c] + red[1][c];
        else r = (red[0][s] + red[1][s]) + (red[2][s] + red[3][s]);
        part[(uint64_t)s * gridDim.x + blockIdx.x] = r;
    }
}

// What stage 2 makes of each qubit: bit[q] = its number bit, PROB_FIXED0 /
// PROB_FIXED1 for a fixed one; every result is multiplied by `scale`.
#define PROB_FIXED0 100
#define PROB_FIXED1 101
struct ProbOut {
    uint8_t bit[PROB_MAX_QUBITS];
    double scale;
};

// Stage 2: one workgroup per output q (0..n).  A number bit below cb sums its
// slot; one at or above cb sums the totals of the workgroups whose index bit
// (bit - cb) is 0; q == n and a qubit fixed to 0 sum every total.
template <int NT>
__global__ void __launch_bounds__(NT) prob_stage2(const double *__restrict__ part, uint32_t groups, int n, int cb,
                                                  const ProbOut po, double *__restrict__ out) {
    __shared__ double red[NT / 64];
    const int q = blockIdx.x;
    const uint32_t tid = threadIdx.x;
    const int bit = q == n ? PROB_FIXED0 : po.bit[q];
    const int slot = bit < cb ? bit : cb;
    const uint32_t skip = bit >= cb && bit < PROB_FIXED0 ? 1u << (bit - cb) : 0u;
    const double *__restrict__ src = part + (uint64_t)slot * groups;
    double acc = 0.0;
#pragma unroll 8
    for (uint32_t g = tid; g < groups; g += NT) {
        const double v = src[g];
        acc += (g & skip) ? 0.0 : v;
    }
    acc = wave_sum(acc);
    if ((tid & 63) == 0) red[tid >> 6] = acc;
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int k = NT / 128; k; k /= 2)
#pragma unroll
            for (int i = 0; i < k; i++) red[i] = red[2 * i] + red[2 * i + 1];
        out[q] = bit == PROB_FIXED1 ? 0.0 : po.scale * red[0];
    }
}

// Both stages in one launch of one workgroup of 16 waves, for up to 2^PROB_ONE_BITS
// amplitudes: number bits 0..5 lane, 6..9 wave, 10.. load index.
#define PROB_ONE_BITS 13

template <typename T>
__global__ void __launch_bounds__(1024)
prob_one(const typename V2<T>::type *__restrict__ st, const ProbBits pb, int nf, int n, const ProbOut po,
         double *__restrict__ out) {
    using V = typename V2<T>::type;
    constexpr int JB = PROB_ONE_BITS - 10, J = 1 << JB;
    __shared__ double red[16][6 + JB + 1];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint64_t base = pb.fixed;
#pragma unroll
    for (int i = 0; i < 4; i++) base |= ((w >> i) & 1u) ? pb.img[6 + i] : 0ull;
    uint64_t lp = 0;
#pragma unroll
    for (int i = 0; i < 6; i++) lp |= ((lane >> i) & 1u) ? pb.img[i] : 0ull;
    const bool on = nf >= 10 || (tid >> nf) == 0;
    const int nj = nf > 10 ? nf - 10 : 0;
    V v[J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        uint64_t u = base;  // img is 0 past the last number bit: the loads j >> nj repeat an amplitude
#pragma unroll
        for (int b = 0; b < JB; b++)
            if ((j >> b) & 1) u |= pb.img[10 + b];
        v[j] = st[u + lp];
    }
    double t = 0.0, zj[JB];
#pragma unroll
    for (int b = 0; b < JB; b++) zj[b] = 0.0;
#pragma unroll
    for (int j = 0; j < J; j++) {
        const double p = on && (j >> nj) == 0 ? (double)v[j].x * (double)v[j].x + (double)v[j].y * (double)v[j].y : 0.0;
        t += p;
#pragma unroll
        for (int b = 0; b < JB; b++)
            if (!((j >> b) & 1)) zj[b] += p;
    }
#pragma unroll
    for (int q = 0; q < 6; q++) {  // as in prob_stage1
        double r = t;
#pragma unroll
        for (int k = q + 1; k < 6; k++) r += __shfl_xor(r, 1 << k, 64);
        if (lane == 0) red[w][q] = r;
        t += __shfl_xor(t, 1 << q, 64);
    }
    if (lane == 0) red[w][6 + JB] = t;
#pragma unroll
    for (int b = 0; b < JB; b++) {
        const double r = wave_sum(zj[b]);
        if (lane == 0) red[w][6 + b] = r;
    }
    __syncthreads();
    const int q = (int)tid;
    if (q > n) return;
    const int bit = q == n ? PROB_FIXED0 : po.bit[q];
    const int slot = bit < 6 ? bit : bit >= 10 && bit < PROB_FIXED0 ? bit - 4 : 6 + JB;
    const uint32_t skip = bit >= 6 && bit < 10 ? 1u << (bit - 6) : 0u;
    double acc = 0.0;
#pragma unroll
    for (uint32_t g = 0; g < 16; g++) acc += (g & skip) ? 0.0 : red[g][slot];
    out[q] = bit == PROB_FIXED1 ? 0.0 : po.scale * acc;
}

// The read-out of many states and the comparison split a state in chunks of
// 2^PROB_WG_BITS amplitudes per workgroup.
#define PROB_WG_BITS 16
#define PROB_SLOTS 17

// Device memory of the allocation-free P(0) entry point
// (dq_prob_zero_all_noalloc): per-workgroup partial sums of one chunk of at
// most 2^NA_CHUNK_BITS amplitudes, then NA_CHUNK_BITS + 1 results per chunk
// for up to NA_MAX_QUBITS qubits; 2.2 MiB on every device the library runs on.
#define NA_CHUNK_BITS 30
#define NA_MAX_QUBITS 36
#define NA_PART_DOUBLES ((1u << (NA_CHUNK_BITS - PROB_WG_BITS)) * PROB_SLOTS)  // at least prob_part_bytes(NA_CHUNK_BITS)
#define NA_CHUNK_DOUBLES ((1u << (NA_MAX_QUBITS - NA_CHUNK_BITS)) * (NA_CHUNK_BITS + 1))
static_assert((size_t)NA_PART_DOUBLES * sizeof(double) % 256 == 0, "chunk results stay 256-byte aligned");
static __device__ __align__(256) double scratch[NA_PART_DOUBLES + NA_CHUNK_DOUBLES];

// ----------------------------------------------------------------------------
// read-out of many states of one size: P(0) per qubit, total probability and
// samples drawn by inverse transform over a tree of probability sums
// ----------------------------------------------------------------------------
// Level 1 of the tree holds the sums of |a|^2 over groups of 2^RO_GB
// amplitudes; every higher level sums RO_FAN entries of the level below,
// until a level has at most RO_FAN entries.  A sample walks down from the
// top, reading at most RO_FAN values per level.
#define RO_GB 10
#define RO_FAN_BITS 10
#define RO_FAN (1u << RO_FAN_BITS)
#define RO_GPW 16        // level-1 groups per wave in stage 1
#define RO_MAX_LEVELS 4  // n <= 40

struct RoLevels {
    double *base[RO_MAX_LEVELS];    // level L+1 of state s at base[L] + s * stride[L]
    uint64_t stride[RO_MAX_LEVELS];
    uint64_t count[RO_MAX_LEVELS];  // entries per state
    int nlev;
};

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// Stage 1, grid (ceil(N1 / 64), count), 256 threads.  Wave w of workgroup x
// owns level-1 groups g = 64x + 16w + k (k < 16); lane l reads amplitudes
// g * 2^gb + 64j + l.  Index bits: 0..5 lane, 6..9 j, 10..13 k, 14..15 w,
// 16.. workgroup -- so the 17 partial slots of a workgroup are P0 partials of
// qubits 0..15 and its total, as in prob_stage1, and stage 2 is shared.
template <typename T>
__global__ void __launch_bounds__(256)
readout_stage1(const void *const *__restrict__ states, int n, double *__restrict__ part, uint64_t part_stride,
               double *__restrict__ lvl1, uint64_t lvl1_stride) {
    using V = typename V2<T>::type;
    __shared__ double red[4][PROB_SLOTS];
    const V *__restrict__ st = reinterpret_cast<const V *>(states[blockIdx.y]);
    const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int gb = n < RO_GB ? n : RO_GB;
    const uint64_t n1 = 1ull << (n - gb);
    const uint32_t gsize = 1u << gb;
    double tot = 0.0;
    double zj[4] = {0.0, 0.0, 0.0, 0.0}, zk[4] = {0.0, 0.0, 0.0, 0.0};
    for (uint32_t k = 0; k < RO_GPW; k++) {
        const uint64_t g = (uint64_t)blockIdx.x * (4 * RO_GPW) + w * RO_GPW + k;
        if (g >= n1) break;  // uniform over the wave
        const V *__restrict__ src = st + (g << gb);
        double gs = 0.0;
        if (gsize == (1u << RO_GB)) {
            V v[16];
#pragma unroll
            for (uint32_t j = 0; j < 16; j++) v[j] = __builtin_nontemporal_load(src + (j << 6) + lane);
#pragma unroll
            for (uint32_t j = 0; j < 16; j++) {
                const double p = (double)v[j].x * (double)v[j].x + (double)v[j].y * (double)v[j].y;
                gs += p;
#pragma unroll
                for (int b = 0; b < 4; b++)
                    if (!((j >> b) & 1)) zj[b] += p;
            }
        } else {
            const uint32_t J = gsize >= 64 ? gsize >> 6 : 1;
            for (uint32_t j = 0; j < J; j++) {
                const uint32_t i = (j << 6) + lane;
                if (i >= gsize) continue;
                const V v = src[i];
                const double p = (double)v.x * (double)v.x + (double)v.y * (double)v.y;
                gs += p;
#pragma unroll
                for (int b = 0; b < 4; b++)
                    if (!((j >> b) & 1)) zj[b] += p;
            }
        }
        tot += gs;
#pragma unroll
        for (int b = 0; b < 4; b++)
            if (!((k >> b) & 1)) zk[b] += gs;
        const double s = wave_sum(gs);
        if (lane == 0) lvl1[blockIdx.y * lvl1_stride + g] = s;
    }
    double vals[PROB_SLOTS];
#pragma unroll
    for (int q = 0; q < 6; q++) vals[q] = ((lane >> q) & 1) ? 0.0 : tot;
#pragma unroll
    for (int b = 0; b < 4; b++) vals[6 + b] = zj[b];
#pragma unroll
    for (int b = 0; b < 4; b++) vals[10 + b] = zk[b];
#pragma unroll
    for (int b = 0; b < 2; b++) vals[14 + b] = ((w >> b) & 1) ? 0.0 : tot;
    vals[16] = tot;
#pragma unroll
    for (int s = 0; s < PROB_SLOTS; s++) {
        const double r = wave_sum(vals[s]);
        if (lane == 0) red[w][s] = r;
    }
    __syncthreads();
    if (tid < PROB_SLOTS)
        part[blockIdx.y * part_stride + (uint64_t)blockIdx.x * PROB_SLOTS + tid] =
            (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
}

// Stage 2, grid (n + 1, count): prob_stage2 per state.
__global__ void __launch_bounds__(256) readout_stage2(const double *__restrict__ part, uint64_t part_stride,
                                                      uint32_t ngroups, int n, double *__restrict__ out) {
    __shared__ double red[4];
    const int q = blockIdx.x;
    const uint32_t tid = threadIdx.x;
    const double *__restrict__ pp = part + blockIdx.y * part_stride;
    double acc = 0.0;
    for (uint32_t g = tid; g < ngroups; g += 256) {
        double v;
        if (q == n) v = pp[(uint64_t)g * PROB_SLOTS + 16];
        else if (q < PROB_WG_BITS) v = pp[(uint64_t)g * PROB_SLOTS + q];
        else v = ((g >> (q - PROB_WG_BITS)) & 1) ? 0.0 : pp[(uint64_t)g * PROB_SLOTS + 16];
        acc += v;
    }
    acc = wave_sum(acc);
    if ((tid & 63) == 0) red[tid >> 6] = acc;
    __syncthreads();
    if (tid == 0) out[(uint64_t)blockIdx.y * (n + 1) + q] = (red[0] + red[1]) + (red[2] + red[3]);
}

// One level of the tree: entry e = sum of entries RO_FAN*e .. RO_FAN*e + RO_FAN-1
// of the level below.  Grid (ceil(out_count / 4), count), one wave per entry.
__global__ void __launch_bounds__(256) readout_level(const double *__restrict__ in, uint64_t in_count, uint64_t in_stride,
                                                     double *__restrict__ out, uint64_t out_count, uint64_t out_stride) {
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint64_t e = (uint64_t)blockIdx.x * 4 + w;
    if (e >= out_count) return;  // uniform over the wave; no barrier follows
    const double *__restrict__ src = in + blockIdx.y * in_stride + (e << RO_FAN_BITS);
    const uint64_t lim = in_count - (e << RO_FAN_BITS);
    double s = 0.0;
#pragma unroll
    for (uint32_t j = 0; j < RO_FAN / 64; j++) {
        const uint64_t i = (j << 6) + lane;
        if (i < lim) s += src[i];
    }
    s = wave_sum(s);
    if (lane == 0) out[blockIdx.y * out_stride + e] = s;
}

// Wave-wide pick inside a chunk of len <= 1024 values (lane l holds values
// 16l .. 16l+15): the first index whose running sum exceeds t.  On return t
// holds the remainder inside the picked value.  A target that rounding puts
// at or past the chunk's total picks the last nonzero value.
template <typename F>
__device__ __forceinline__ uint32_t wave_pick(F value, uint32_t len, double &t, uint32_t lane) {
    double v[16];
    double ls = 0.0;
#pragma unroll
    for (uint32_t j = 0; j < 16; j++) {
        const uint32_t i = lane * 16 + j;
        v[j] = i < len ? value(i) : 0.0;
        ls += v[j];
    }
    double inc = ls;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double y = __shfl_up(inc, o, 64);
        if ((int)lane >= o) inc += y;
    }
    double exc = __shfl_up(inc, 1, 64);
    if (lane == 0) exc = 0.0;
    // lane-local choice: the first j past t, else the last nonzero value
    int jsel = -1, jlast = -1;
    double bsel = 0.0, run = exc;
#pragma unroll
    for (int j = 0; j < 16; j++) {
        const double nr = run + v[j];
        if (jsel < 0 && nr > t) { jsel = j; bsel = run; }
        if (v[j] > 0.0) jlast = j;
        run = nr;
    }
    const uint64_t hit = __ballot(inc > t);
    uint32_t L;
    bool clamp;
    if (hit) {
        L = (uint32_t)__builtin_ctzll(hit);
        clamp = __shfl(jsel, L, 64) < 0;
    } else {
        const uint64_t nz = __ballot(ls > 0.0);
        L = nz ? 63u - (uint32_t)__builtin_clzll(nz) : 0u;
        clamp = true;
    }
    const int j = clamp ? __shfl(jlast, L, 64) : __shfl(jsel, L, 64);
    const int jj = j < 0 ? 0 : j;
    double vsel = v[0];
#pragma unroll
    for (int k = 1; k < 16; k++)
        if (k == jj) vsel = v[k];
    vsel = __shfl(vsel, L, 64);
    const double before = __shfl(bsel, L, 64);
    t = clamp ? 0.5 * vsel : t - before;
    return L * 16 + (uint32_t)jj;
}

// One wave per sample, grid (ceil(shots / 4), count).  u[s] in [0, 1); the
// sample is the first amplitude index whose cumulative probability exceeds
// u[s] times the total.
template <typename T>
__global__ void __launch_bounds__(256)
readout_sample(const void *const *__restrict__ states, int n, RoLevels lv, const double *__restrict__ u, uint32_t shots,
               uint64_t *__restrict__ out) {
    using V = typename V2<T>::type;
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t s = blockIdx.x * 4 + w;
    if (s >= shots) return;  // uniform over the wave; no barrier follows
    const uint32_t sid = blockIdx.y;
    const int gb = n < RO_GB ? n : RO_GB;
    const int top = lv.nlev - 1;
    const double *__restrict__ A = lv.base[top] + sid * lv.stride[top];
    const uint32_t tlen = (uint32_t)lv.count[top];
    double tl = 0.0;
#pragma unroll
    for (uint32_t j = 0; j < 16; j++) {
        const uint32_t i = lane * 16 + j;
        if (i < tlen) tl += A[i];
    }
    const double total = wave_sum(tl);
    double t = u[(uint64_t)sid * shots + s] * total;
    uint64_t e0 = 0;  // first entry of the chunk at the current level
    for (int L = top; L >= 0; L--) {
        const double *__restrict__ B = lv.base[L] + sid * lv.stride[L] + e0;
        const uint64_t rem = lv.count[L] - e0;
        const uint32_t len = rem < RO_FAN ? (uint32_t)rem : RO_FAN;
        const uint32_t e = wave_pick([&](uint32_t i) { return B[i]; }, len, t, lane);
        e0 = (e0 + e) << (L > 0 ? RO_FAN_BITS : gb);
    }
    const V *__restrict__ st = reinterpret_cast<const V *>(states[sid]) + e0;
    const uint32_t e = wave_pick(
        [&](uint32_t i) {
            const V a = st[i];
            return (double)a.x * (double)a.x + (double)a.y * (double)a.y;
        },
        1u << gb, t, lane);
    if (lane == 0) out[(uint64_t)sid * shots + s] = e0 + e;
}

// ----------------------------------------------------------------------------
// comparison of two states of one size (any precisions): <a|b>, <a|a>, <b|b>
// and max |a_i - b_i|
// ----------------------------------------------------------------------------
// Bound: HBM, one read of each state.  A thread has 8 amplitudes of either state in
// flight, sums those first and adds the sums to its totals (short chains of
// additions); workgroups are added up to 2^CMP_GROUPS_LOG, from shares of one such
// step.  One amplitude per loop step and 2^16 amplitudes per workgroup left a
// state of up to 16 qubits on one workgroup and large ones waiting
// for loads.  27 qubits FP64, both stages: 741 -> 627 us (5.8 -> 6.9 TB/s).
#define CMP_SLOTS 5
#define CMP_LOADS_LOG 3    // amplitudes of either state in flight per thread
#define CMP_GROUPS_LOG 13

// qubits of a workgroup's share of an n-qubit state (>= 8 + CMP_LOADS_LOG, fewer for a smaller state)
static int cmp_share(int n) { return std::min(n, std::max(8 + CMP_LOADS_LOG, n - CMP_GROUPS_LOG)); }

template <typename TA, typename TB>
__global__ void __launch_bounds__(256)
compare_stage1(const typename V2<TA>::type *__restrict__ a, const typename V2<TB>::type *__restrict__ b, int share,
               double *__restrict__ part) {
    constexpr uint32_t J = 1u << CMP_LOADS_LOG;
    __shared__ double red[4][CMP_SLOTS];
    const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const uint64_t cnt = 1ull << share;
    a += (uint64_t)blockIdx.x << share;
    b += (uint64_t)blockIdx.x << share;
    double re = 0.0, im = 0.0, aa = 0.0, bb = 0.0, mx = 0.0;
    auto step = [&](const typename V2<TA>::type *x, const typename V2<TB>::type *y, uint32_t count) {
        double r = 0.0, i = 0.0, p = 0.0, q = 0.0;
#pragma unroll
        for (uint32_t j = 0; j < count; j++) {
            const double xr = x[j].x, xi = x[j].y, yr = y[j].x, yi = y[j].y;
            r += xr * yr + xi * yi;
            i += xr * yi - xi * yr;
            p += xr * xr + xi * xi;
            q += yr * yr + yi * yi;
            const double dr = xr - yr, di = xi - yi;
            mx = fmax(mx, dr * dr + di * di);
        }
        re += r;
        im += i;
        aa += p;
        bb += q;
    };
    if (cnt >= 256 * J) {  // a multiple of it: both are powers of two
        for (uint64_t i = tid; i < cnt; i += 256 * J) {
            typename V2<TA>::type x[J];
            typename V2<TB>::type y[J];
#pragma unroll
            for (uint32_t j = 0; j < J; j++) {
                x[j] = __builtin_nontemporal_load(a + i + j * 256);
                y[j] = __builtin_nontemporal_load(b + i + j * 256);
            }
            step(x, y, J);
        }
    } else {
        for (uint64_t i = tid; i < cnt; i += 256) {
            const typename V2<TA>::type x = a[i];
            const typename V2<TB>::type y = b[i];
            step(&x, &y, 1);
        }
    }
    double v[CMP_SLOTS] = {wave_sum(re), wave_sum(im), wave_sum(aa), wave_sum(bb), wave_max(mx)};
    if (lane == 0)
        for (int k = 0; k < CMP_SLOTS; k++) red[w][k] = v[k];
    __syncthreads();
    if (tid < CMP_SLOTS) {
        const double r = tid == 4 ? fmax(fmax(red[0][4], red[1][4]), fmax(red[2][4], red[3][4]))
                                  : (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
        part[(uint64_t)tid * gridDim.x + blockIdx.x] = r;
    }
}

// ----------------------------------------------------------------------------
// dense sweeps: FP32 tile in LDS, dense 2^k x 2^k complex blocks on MFMA
// ----------------------------------------------------------------------------
// A dense op on k tile bits is one complex GEMM per tile, rows and the contraction
// index of size K = 2^k, one column per assignment of the other T - k tile bits
// (NC = 2^(T-k) columns): Yr = Ur Xr - Ui Xi, Yi = Ui Xr + Ur Xi.
//
// Each FP32 factor is the sum of three bf16 numbers (8 significant bits each, 24 in
// all), and a real product is the six
// piece products of order up to 2^-16, on v_mfma_f32_32x32x16_bf16 with FP32
// sums: 16 times the rate of v_mfma_f32_32x32x2f32, so 2.7 times for a product.
// The leading products have accumulators of their own (their sums take 2 K / 16
// roundings instead of 2 K), the other five share the second ones.  What is left out is at most
// 3 * 2^-25 of a product's magnitude, less than the rounding of its two FP32 factors.
// Measured over 15 to 25 qubits, depth 20: error against 64 bits 1.9e-7 .. 3.4e-7 (FP32 MFMA
// 7.4e-7 .. 1.3e-6).  25 qubits, depth 20, kernels of a flush with FP32 MFMA -> now: k = 7
// (42 ops in 26 blocks) 13.9 -> 8.5 ms, k = 6 and 5 6.5 and 4.8 ms.  An op of k = 7 runs
// at 1.1-1.3 PFLOP/s of bf16, what a large library product reaches (1.36): clocks
// fall as the run goes on, so vector instructions beside the products cost time too.
//
// bf16 ends at 2^-133 where FP32 goes to 2^-149, so the lower pieces of a factor below
// 2^-110 would lose bits.  Matrices are scaled by 2^DENSE_SCALE_LOG, and so are the
// amplitudes of a tile as it is loaded: the split of an FP32 amplitude is exact, also of
// a denormal one.  Every op then leaves the tile scaled by as much again; that is
// taken off as the tile is stored, or by an op that would go beyond
// DENSE_SCALE_MAX (taken off at every op it cost 4%, so 2%: 25 qubits, depth 10, k = 5, 6
// and 7 3.71 -> 3.84, 4.92 -> 5.08 and 6.09 -> 6.21 ms).  A tile with an
// amplitude of 2^32 or more, which could overflow, is scaled down instead and its scale
// restored by every op.  The scales are powers of two: results are the same
// otherwise.  An infinite amplitude makes its column NaN.
//
// v_mfma_f32_32x32x16_bf16: lane l supplies A[l % 32][8 (l / 32) + i] and
// B[8 (l / 32) + i][l % 32], i = 0..7 in 16 bytes; result register v of lane l is
// C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32].  A matrix is stored as those 16 bytes:
//   [row block of 32][16 contraction indices][real, imaginary][piece][lane][i].
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

#define DENSE_T_MAX 13
#define DENSE_SCALE_LOG 16
#define DENSE_SCALE_MAX 48
#define DENSE_THREADS 256
#define DENSE_COLS 256  // column-table entries per op: 2^(T - k) <= 2^(13 - 5)
#define DENSE_WAVES (DENSE_THREADS / 64)

// The three bf16 pieces of a scaled matrix entry, rounded to nearest even.
static __host__ __device__ inline void split_entry(double x, uint16_t *piece) {
    x *= (double)(1 << DENSE_SCALE_LOG);
    for (int i = 0; i < 3; i++) {
        const float f = (float)x;
        uint32_t u;
        __builtin_memcpy(&u, &f, 4);
        u += 0x7fffu + ((u >> 16) & 1u);
        piece[i] = (uint16_t)(u >> 16);
        u &= 0xffff0000u;
        float h;
        __builtin_memcpy(&h, &u, 4);
        x -= (double)h;
    }
}

// Position of entry (r, c) of a 2^k x 2^k matrix, part 0 / 1 (real / imaginary), in
// 16-bit words; the pieces follow 512 words apart.
static __host__ __device__ inline size_t entry_pos(int k, uint32_t r, uint32_t c, uint32_t part) {
    const uint32_t lane = (r & 31u) | (((c >> 3) & 1u) << 5);
    return ((((size_t)(r >> 5) << (k - 4)) + (c >> 4)) * 6 + part * 3) * 512 + lane * 8 + (c & 7u);
}

// Two FP32 amplitude parts as pairs of bf16 pieces: hi + mid + lo is x exactly.
__device__ __forceinline__ void split_pair(float x0, float x1, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    auto round2 = [](float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, bf2)); };
    hi = round2(x0, x1);
    x0 -= __uint_as_float(hi << 16);
    x1 -= __uint_as_float(hi & 0xffff0000u);
    mid = round2(x0, x1);
    x0 -= __uint_as_float(mid << 16);
    x1 -= __uint_as_float(mid & 0xffff0000u);
    lo = round2(x0, x1);
}

// LDS slot of tile element e: the low 5 bits are xored with bits 5..9 and
// 10..14, spreading power-of-two strides over the 32 banks (a bijection:
// only the low bits change, by a function of the others).
__device__ __forceinline__ uint32_t dswz(uint32_t e) { return e ^ ((e >> 5) & 31u) ^ ((e >> 10) & 31u); }

// One dense op on the tile in LDS.  A work item is RP row blocks of 32 rows by one
// block of 32 columns; at T = 13 every wave has one (k = 5: two).  Per step of 16
// contraction indices a wave reads 16 amplitude parts a lane from the tile, splits them
// and issues 24 MFMAs for each row block.  Waves that share columns (k = 7: two) split them
// each: the vector instructions run while the matrix unit is busy, and operands
// split once into LDS (96 KiB beside the tile) left room for one workgroup per CU, whose
// loads, stores, splits and products then took turns (k = 5 7.0 ms, k = 6 7.5, k = 7 the
// same).  Matrix operands (L2) come two
// units of 24 MFMAs ahead, amplitudes one step.  coloff[c] is column c's tile offset
// (c's bits placed on the tile bits outside the op), a table the host forms per op.
// Deposit and swizzle are linear over GF(2), so an LDS slot is the xor of the column's and
// of sd[b] = dswz(1 << bits[b]) over the set bits b of the matrix index.
template <int KL>
__device__ __forceinline__ void dense_op(float *__restrict__ re, float *__restrict__ im, uint32_t T, const dq_dense_op &op,
                                         const uint4 *__restrict__ mat, const uint32_t *__restrict__ coloff, uint32_t lane,
                                         uint32_t w, float fix) {
    constexpr uint32_t K = 1u << KL, KS = K / 16, RB = K / 32, RP = RB >= 2 ? 2 : 1;
    const uint32_t lc = T - KL - 5, NCB = 1u << lc, items = NCB * (RB / RP);
    uint32_t sd[KL];
#pragma unroll
    for (int b = 0; b < KL; b++) sd[b] = dswz(1u << op.bits[b]);
    auto mma = [](const uint4 &p, const uint4 &q, const v16f &acc) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, p), __builtin_bit_cast(v8bf, q), acc, 0, 0, 0);
    };
    bool first = true;
    for (uint32_t item = w; RB > RP ? first : item < items; item += DENSE_WAVES) {
        const bool busy = item < items;  // uniform over the wave
        const uint32_t cb = item & (NCB - 1), rb = busy ? (item >> lc) * RP : 0;
        const uint4 *__restrict__ ma = mat + (size_t)rb * KS * 6 * 64 + lane;
        uint4 a[2][6];
        auto load_a = [&](uint4 *to, uint32_t s, uint32_t r) {
#pragma unroll
            for (int i = 0; i < 6; i++) to[i] = ma[((r * KS + s) * 6 + i) * 64];
        };
        load_a(a[0], 0, 0);
        load_a(a[1], RP == 2 ? 0 : 1, RP == 2 ? 1 : 0);
        const uint32_t zc = dswz(coloff[cb * 32 + (lane & 31u)]);
        if (first) __syncthreads();  // the tile is complete
        first = false;
        v16f acc[RP][4];  // real, imaginary: the leading products, the others
        if (busy) {
#pragma unroll
            for (uint32_t r = 0; r < RP; r++)
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[r][c][v] = 0.0f;
            const uint32_t zl = zc ^ ((lane >> 5) ? sd[3] : 0u);
            float xr[8], xi[8];
            auto read_x = [&](uint32_t s) {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    uint32_t u = ((i & 1) ? sd[0] : 0u) ^ ((i & 2) ? sd[1] : 0u) ^ ((i & 4) ? sd[2] : 0u);
#pragma unroll
                    for (int b = 4; b < KL; b++) u ^= ((s >> (b - 4)) & 1u) ? sd[b] : 0u;
                    xr[i] = re[zl ^ u];
                    xi[i] = im[zl ^ u];
                }
            };
            read_x(0);
            // with two row blocks a unit's slot is its row block, also in a real loop
            constexpr int UF = RP == 2 ? 1 : KS;
#pragma unroll UF
            for (uint32_t s = 0; s < KS; s++) {
                uint4 br[3], bi[3];
                split_pair(xr[0], xr[1], br[0].x, br[1].x, br[2].x);
                split_pair(xr[2], xr[3], br[0].y, br[1].y, br[2].y);
                split_pair(xr[4], xr[5], br[0].z, br[1].z, br[2].z);
                split_pair(xr[6], xr[7], br[0].w, br[1].w, br[2].w);
                split_pair(xi[0], xi[1], bi[0].x, bi[1].x, bi[2].x);
                split_pair(xi[2], xi[3], bi[0].y, bi[1].y, bi[2].y);
                split_pair(xi[4], xi[5], bi[0].z, bi[1].z, bi[2].z);
                split_pair(xi[6], xi[7], bi[0].w, bi[1].w, bi[2].w);
                if (s + 1 < KS) read_x(s + 1);
#pragma unroll
                for (uint32_t r = 0; r < RP; r++) {
                    __builtin_amdgcn_sched_barrier(0);  // loads stay ahead of the products that cover them
                    uint4 *slot = a[RP == 2 ? r : (s & 1)];
                    const uint4 *ur = slot, *ui = ur + 3;
                    auto neg = [](const uint4 &q) {
                        return make_uint4(q.x ^ 0x80008000u, q.y ^ 0x80008000u, q.z ^ 0x80008000u, q.w ^ 0x80008000u);
                    };
                    v16f &yr = acc[r][0], &yi = acc[r][1], &cr = acc[r][2], &ci = acc[r][3];
                    yr = mma(ur[0], br[0], yr);
                    yi = mma(ui[0], br[0], yi);
#pragma unroll
                    for (int t = 0; t < 5; t++) {  // pieces (p, q) of matrix and amplitude with p + q = 2, then 1
                        const int p = t < 3 ? t : t - 3, q = (t < 3 ? 2 : 1) - p;
                        cr = mma(ur[p], br[q], cr);
                        ci = mma(ui[p], br[q], ci);
                    }
                    const uint4 un[3] = {neg(ui[0]), neg(ui[1]), neg(ui[2])};
                    yr = mma(un[0], bi[0], yr);
                    yi = mma(ur[0], bi[0], yi);
#pragma unroll
                    for (int t = 0; t < 5; t++) {
                        const int p = t < 3 ? t : t - 3, q = (t < 3 ? 2 : 1) - p;
                        cr = mma(un[p], bi[q], cr);
                        ci = mma(ur[p], bi[q], ci);
                    }
                    if (s + 2 / RP < KS) load_a(slot, s + 2 / RP, r);
                }
            }
        }
        if (busy) {
#pragma unroll
            for (uint32_t r = 0; r < RP; r++)
#pragma unroll
                for (int c = 0; c < 2; c++) acc[r][c] += acc[r][c + 2];
            if (fix != 1.0f)  // uniform
#pragma unroll
                for (uint32_t r = 0; r < RP; r++)
#pragma unroll
                    for (int c = 0; c < 2; c++) acc[r][c] *= fix;
        }
        // In place: an item with every row of its columns reads exactly the tile
        // elements it writes; otherwise every wave has to have read them.
        if constexpr (RB > RP) __syncthreads();
        if (!busy) break;
        // Register v of this lane is row 32 (rb + r) + 8 (v / 4) + 4 (lane / 32) + v % 4.
#pragma unroll
        for (uint32_t r = 0; r < RP; r++) {
            uint32_t z = zc ^ ((lane >> 5) ? sd[2] : 0u);
#pragma unroll
            for (int b = 5; b < KL; b++) z ^= (((rb + r) >> (b - 5)) & 1u) ? sd[b] : 0u;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const uint32_t u = z ^ ((v & 1) ? sd[0] : 0u) ^ ((v & 2) ? sd[1] : 0u) ^ ((v & 4) ? sd[3] : 0u) ^ ((v & 8) ? sd[4] : 0u);
                re[u] = acc[r][0][v];
                im[u] = acc[r][1][v];
            }
        }
    }
    if (first) __syncthreads();  // a wave without an item
}

// One dense block over every tile of an FP32 state: grid = tiles, 256 threads.  Two
// workgroups (64 KiB of LDS each at T = 13) share a CU, a wave of either on each SIMD
// with up to 256 VGPRs: one's loads and stores run beside the other's products.
// 40-54 SGPRs spill to VGPR lanes, at k = 6 two VGPRs to memory.
template <int KL>
__global__ void __launch_bounds__(DENSE_THREADS, 2)
dense_kernel(const dq_dense_block *__restrict__ blk, const dq_dense_op *__restrict__ ops, const uint4 *__restrict__ mats,
             const uint32_t *__restrict__ ctab, typename V2<float>::type *__restrict__ st) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    __shared__ uint32_t wave_large[DENSE_WAVES];  // has the wave loaded an amplitude of 2^32 or more?
    const uint32_t T = blk->tile_bits;
    const uint32_t NT = 1u << T;
    float *re = reinterpret_cast<float *>(lds_raw);
    float *im = re + NT;
    const uint32_t tid = threadIdx.x;
    const uint64_t base = tile_base(blk->nontile_mask, blockIdx.x);
    // tile_q read as four words (scalar loads; byte loads would put these
    // uniform values in vector registers)
    const uint32_t *__restrict__ tq32 = reinterpret_cast<const uint32_t *>(blk->tile_q);
    uint32_t tq[4];
#pragma unroll
    for (int k = 0; k < 4; k++) tq[k] = tq32[k];
    uint64_t hq[DENSE_T_MAX];
#pragma unroll
    for (int b = 0; b < DENSE_T_MAX; b++) hq[b] = 1ull << ((tq[b >> 2] >> (8 * (b & 3))) & 0xffu);
    // Element e = tid + 256 i of the tile holds the amplitude whose qubits are
    // e's bits placed on tile_q (bits 0..5 are qubits 0..5).  The placement and
    // the LDS swizzle are linear, so the thread's part (bits 0..7) is formed
    // once and the part of i (bits 8 and up) is a scalar.
    // Bits 6 and 7 of e are the wave index, a scalar: the thread's part of an
    // address is its lane alone (qubits 0..5), a 32-bit offset on a scalar base.
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lane = tid & 63u;
    const uint64_t tg = base | ((wv & 1u) ? hq[6] : 0ull) | ((wv & 2u) ? hq[7] : 0ull);
    const uint32_t tz = dswz(tid);
    // i < NI = 2^(T - 8) (4..32) runs over the tile bits 8 and up, whose qubits
    // are scalars.  Every thread issues 32 loads before using the first;
    // below T = 13 index i stands for element i mod NI, so the extra loads,
    // LDS writes and stores repeat an element with the same value (no branch).
    constexpr int LI = 1 << (DENSE_T_MAX - 8);
    const uint32_t NI = NT / DENSE_THREADS;
    uint64_t hi[DENSE_T_MAX - 8];
#pragma unroll
    for (int b = 8; b < DENSE_T_MAX; b++) hi[b - 8] = T > (uint32_t)b ? hq[b] : 0ull;
    auto gaddr = [&](uint32_t i) {
        uint64_t g = tg;
#pragma unroll
        for (int b = 0; b < DENSE_T_MAX - 8; b++) g |= ((i >> b) & 1u) ? hi[b] : 0ull;
        return g;
    };
    auto power = [](int e) { return __uint_as_float((uint32_t)(127 + e) << 23); };
    bool large;
    {
        typename V2<float>::type v[LI];
#pragma unroll
        for (int i = 0; i < LI; i++) v[i] = __builtin_nontemporal_load(lane_ptr(st + gaddr((uint32_t)i & (NI - 1)), lane));
        float top = 0.0f;
#pragma unroll
        for (int i = 0; i < LI; i++) top = fmaxf(top, fmaxf(fabsf(v[i].x), fabsf(v[i].y)));
        const uint64_t any = __ballot(top >= 0x1p32f);
        if (lane == 0) wave_large[wv] = any != 0;
        __syncthreads();
        uint32_t l = 0;
#pragma unroll
        for (int w = 0; w < DENSE_WAVES; w++) l |= wave_large[w];
        large = __builtin_amdgcn_readfirstlane(l) != 0;
        const float s = large ? power(-DENSE_SCALE_LOG) : power(DENSE_SCALE_LOG);
#pragma unroll
        for (int i = 0; i < LI; i++) {
            const uint32_t z = tz ^ dswz(((uint32_t)i & (NI - 1)) * DENSE_THREADS);
            re[z] = v[i].x * s;
            im[z] = v[i].y * s;
        }
    }
    constexpr size_t msz = (size_t)12 << (2 * KL);  // bytes of a matrix
    const int first = large ? -DENSE_SCALE_LOG : DENSE_SCALE_LOG, most = large ? first : DENSE_SCALE_MAX;
    int scale = first;  // the tile's, as a power of two
    for (uint32_t o = 0; o < blk->op_count; o++) {
        const dq_dense_op op = ops[blk->op_begin + o];
        scale += DENSE_SCALE_LOG;
        const int off = scale > most ? scale - first : 0;
        scale -= off;
        dense_op<KL>(re, im, T, op, mats + op.mat * (msz / 16), ctab + (size_t)(blk->op_begin + o) * DENSE_COLS, lane, wv, power(-off));
    }
    __syncthreads();
    {
        // opaque copies: the addresses are formed again here instead of being kept
        // live through every op
        uint32_t lane2 = lane, tz2 = tz;
        asm volatile("" : "+v"(lane2), "+v"(tz2));
        typename V2<float>::type v[LI];
        const float s = power(-scale);
#pragma unroll
        for (int i = 0; i < LI; i++) {
            const uint32_t z = tz2 ^ dswz(((uint32_t)i & (NI - 1)) * DENSE_THREADS);
            v[i].x = re[z] * s;
            v[i].y = im[z] * s;
        }
#pragma unroll
        for (int i = 0; i < LI; i++) __builtin_nontemporal_store(v[i], lane_ptr(st + gaddr((uint32_t)i & (NI - 1)), lane2));
    }
}

// Matrices of dense ops as products of gates, formed in FP64 and written in the
// MFMA operand order of dense_op.  A column (the image of one basis state) takes
// one wave, 2^k / 64 amplitudes a lane, two columns a wave for k = 5; a gate is a
// 2x2 on one index bit, its partner amplitude a lane exchange away.  Grid
// (2^k / columns per workgroup, matrices).  Latency-bound (a few gates' lane
// exchanges, every matrix at once).  On the host, gate by gate and column by
// column, the 42 matrices of a 25-qubit grid circuit (k = 7) took 14-17 of the
// 28.7-31.8 ms of a flush and were uploaded (11 MB); the flush now takes 14.7 ms.
template <int KL>
__global__ void __launch_bounds__(256)
dense_form(const dq_small_gate *__restrict__ gates, const uint32_t *__restrict__ begin, uint16_t *__restrict__ mats) {
    constexpr int J = KL == 7 ? 2 : 1;      // amplitudes per lane
    constexpr int CW = KL == 5 ? 2 : 1;     // columns per wave
    constexpr uint32_t LN = 64 / CW;        // lanes per column
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t i0 = lane & (LN - 1);
    const uint32_t c = (blockIdx.x * 4 + w) * CW + lane / LN;
    double re[J], im[J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        re[j] = i0 + LN * j == c ? 1.0 : 0.0;
        im[j] = 0.0;
    }
    const uint32_t g1 = begin[blockIdx.y + 1];
    for (uint32_t g = begin[blockIdx.y]; g < g1; g++) {
        const dq_small_gate *__restrict__ G = gates + g;
        const uint32_t tm = G->tmask, cm = G->cmask;
        double u[8];
#pragma unroll
        for (int i = 0; i < 8; i++) u[i] = G->u[i];
        if (G->diag) {
#pragma unroll
            for (int j = 0; j < J; j++)
                if (((i0 + LN * j) & cm) == cm) {
                    const double r = re[j], x = im[j];
                    re[j] = u[0] * r - u[1] * x;
                    im[j] = u[0] * x + u[1] * r;
                }
            continue;
        }
        double pr[J], pi[J];
#pragma unroll
        for (int j = 0; j < J; j++) {
            if (tm < LN) {
                pr[j] = __shfl_xor(re[j], (int)tm, 64);
                pi[j] = __shfl_xor(im[j], (int)tm, 64);
            } else {
                pr[j] = re[J - 1 - j];
                pi[j] = im[J - 1 - j];
            }
        }
#pragma unroll
        for (int j = 0; j < J; j++) {
            const uint32_t i = i0 + LN * j;
            const bool hi = (i & tm) != 0;
            const double r0 = hi ? pr[j] : re[j], m0 = hi ? pi[j] : im[j];
            const double r1 = hi ? re[j] : pr[j], m1 = hi ? im[j] : pi[j];
            const double ar = hi ? u[4] : u[0], ai = hi ? u[5] : u[1], br = hi ? u[6] : u[2], bi = hi ? u[7] : u[3];
            if ((i & cm) == cm) {
                re[j] = ar * r0 - ai * m0 + br * r1 - bi * m1;
                im[j] = ar * m0 + ai * r0 + br * m1 + bi * r1;
            }
        }
    }
    uint16_t *__restrict__ D = mats + (size_t)blockIdx.y * ((size_t)6 << (2 * KL));
    auto put = [&](uint32_t r, uint32_t part, double v) {
        uint16_t piece[3];
        split_entry(v, piece);
        uint16_t *__restrict__ d = D + entry_pos(KL, r, c, part);
        d[0] = piece[0];
        d[512] = piece[1];
        d[1024] = piece[2];
    };
#pragma unroll
    for (int j = 0; j < J; j++) {
        put(i0 + LN * j, 0, re[j]);
        put(i0 + LN * j, 1, im[j]);
    }
}

// out = {re <a|b>, im <a|b>, <a|a>, <b|b>, max |a_i - b_i|}: one workgroup per slot.
__global__ void __launch_bounds__(256) compare_stage2(const double *__restrict__ part, uint32_t ngroups, double *__restrict__ out) {
    __shared__ double red[4];
    const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int k = blockIdx.x;
    const double *__restrict__ src = part + (uint64_t)k * ngroups;
    double v = 0.0;
#pragma unroll 8
    for (uint32_t g = tid; g < ngroups; g += 256) v = k == 4 ? fmax(v, src[g]) : v + src[g];
    v = k == 4 ? wave_max(v) : wave_sum(v);
    if (lane == 0) red[w] = v;
    __syncthreads();
    if (tid == 0)
        out[k] = k == 4 ? sqrt(fmax(fmax(red[0], red[1]), fmax(red[2], red[3]))) : (red[0] + red[1]) + (red[2] + red[3]);
}

// ----------------------------------------------------------------------------
// amplitude gather / scatter / fill
// ----------------------------------------------------------------------------
// The qubit map travels in the arguments: a staged upload of it took longer
// than the kernel.
struct QubitMap {
    uint8_t l2p[40];
};

template <typename T>
__global__ void read_kernel(const typename V2<T>::type *__restrict__ st, int n, const QubitMap map,
                            uint64_t start, uint64_t count, double *__restrict__ out) {
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    const uint64_t li = start + k;
    uint64_t pi = 0;
    for (int q = 0; q < n; q++) pi |= ((li >> q) & 1ull) << map.l2p[q];
    const typename V2<T>::type v = st[pi];
    out[2 * k] = (double)v.x;
    out[2 * k + 1] = (double)v.y;
}

template <typename T>
__global__ void write_kernel(typename V2<T>::type *__restrict__ st, uint64_t start, uint64_t count,
                             const double *__restrict__ re, const double *__restrict__ im) {
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    typename V2<T>::type v;
    v.x = (T)re[k];
    v.y = (T)im[k];
    st[start + k] = v;
}

// grid-stride: a launch may not exceed 2^32 threads (n >= 32 states)
template <typename T>
__global__ void fill_kernel(typename V2<T>::type *__restrict__ st, uint64_t N, int kind, uint64_t index, double value) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += stride) {
        typename V2<T>::type v;
        v.x = (kind == DQ_INIT_CLASSICAL) ? (i == index ? T(1) : T(0)) : (T)value;
        v.y = T(0);
        __builtin_nontemporal_store(v, st + i);
    }
}

// ----------------------------------------------------------------------------
// permutation of a register's qubits, in place
// ----------------------------------------------------------------------------
// An involution of the index bits swaps amplitudes in pairs.  A workgroup takes
// the tile of a value u of the non-tile bits and the tile of u's image, and
// writes each where the other was: any involution is one pass over the state.
// Any permutation is the product of two involutions, so two passes; one that
// moves only tile bits is one (u is its own image, the tile permutes itself).
// A tile is closed under the involution and holds the low LB index bits and
// their images, so reads and writes both go in runs of 2^LB amplitudes.
//
// Bound: HBM, one read and one write of the state.  Sweeps of one tile each,
// which move at most 7 or 8 qubits besides the low 6, took three or four passes
// for a 25- to 28-qubit register.  Measured, before -> now: reversal of 27 qubits FP32
// 1.13 ms (3 passes) -> 0.64 ms (1 pass, 3.3 TB/s), the map of a 28-qubit FP32 grid circuit 2.37 ->
// 1.91 ms (2 passes of 4.5 TB/s), of a 25-qubit FP64 ansatz 0.80 -> 0.42 ms.
// LB = 5 in FP64, 6 in FP32: 512-byte runs (256-byte runs were 15-25% slower).
// Two tiles of 2^TB amplitudes fill 64 KiB; an FP64 tile of a state whose bits all
// pair off cannot reach 11 bits and takes the 10-bit instance (half of a larger
// one's threads would have nothing to load).
constexpr int perm_low_bits(int prec) { return prec == DQ_F64 ? 5 : 6; }
#define PERM_TB_MAX 12
#define PERM_GRID_X 16  // workgroup index bits in x, the rest in y (one dimension holds less than 2^32 threads)

struct PermArgs {
    int tb, nu;                 // tile bits, non-tile bits
    uint8_t tile[PERM_TB_MAX];  // index bit of tile bit b, ascending
    uint8_t inv[PERM_TB_MAX];   // the tile bit whose value goes to tile bit b
    uint8_t pos[40], img[40];   // non-tile bits: index bit, and its image's
};

// LDS slot of tile element e: linear, spreads power-of-two strides over 128 bytes.
template <typename T> __device__ __forceinline__ uint32_t perm_slot(uint32_t e) {
    constexpr int B = sizeof(T) == 8 ? 3 : 4;
    constexpr uint32_t M = (1u << B) - 1u;
    return e ^ ((e >> B) & M) ^ ((e >> (2 * B)) & M) ^ ((e >> (3 * B)) & M);
}

template <typename T, int TB, int NT>
__global__ void __launch_bounds__(NT, 4)
permute_kernel(typename V2<T>::type *__restrict__ st, const PermArgs pa) {
    using V = typename V2<T>::type;
    constexpr int E = (1 << TB) / NT;
    constexpr int LT = NT == 512 ? 9 : 8;  // thread bits
    static_assert(NT == 1 << LT, "threads are a power of two");
    __shared__ V lds[2][1 << TB];
    const uint32_t group = blockIdx.x | (blockIdx.y << PERM_GRID_X);
    uint64_t u = 0, w = 0;
    for (int i = 0; i < pa.nu; i++) {
        const uint64_t b = (group >> i) & 1u;
        u |= b << pa.pos[i];
        w |= b << pa.img[i];
    }
    if (w < u) return;  // its image's workgroup does both
    const bool pair = w != u;
    const uint32_t tid = threadIdx.x, size = 1u << pa.tb;
    // Element e = tid + NT i: its offset, and the slot of the element that goes
    // there.  Both are linear in the bits of e: a thread's part and a uniform one of i.
    uint64_t lp = 0;
    uint32_t lf = 0;
#pragma unroll
    for (int b = 0; b < LT; b++) {
        const uint32_t x = b < pa.tb ? (tid >> b) & 1u : 0u;
        lp |= (uint64_t)x << pa.tile[b];
        lf |= x << pa.inv[b];
    }
    lf = perm_slot<T>(lf);
    const uint32_t ls = perm_slot<T>(tid);
    uint64_t ui[E];
    uint32_t fi[E];
#pragma unroll
    for (int i = 0; i < E; i++) {
        ui[i] = 0;
        fi[i] = 0;
#pragma unroll
        for (int b = LT; b < TB; b++)
            if ((i >> (b - LT)) & 1) {
                ui[i] |= 1ull << pa.tile[b];
                fi[i] |= 1u << pa.inv[b];
            }
    }
    V a[E], c[E];
#pragma unroll
    for (int i = 0; i < E; i++)
        if (tid + (uint32_t)i * NT < size) {
            a[i] = __builtin_nontemporal_load(st + (u | ui[i]) + lp);
            if (pair) c[i] = __builtin_nontemporal_load(st + (w | ui[i]) + lp);
        }
#pragma unroll
    for (int i = 0; i < E; i++)
        if (tid + (uint32_t)i * NT < size) {
            const uint32_t s = ls ^ perm_slot<T>((uint32_t)i * NT);
            lds[0][s] = a[i];
            if (pair) lds[1][s] = c[i];
        }
    __syncthreads();  // both tiles are read before either is written
#pragma unroll
    for (int i = 0; i < E; i++)
        if (tid + (uint32_t)i * NT < size) {
            const uint32_t s = lf ^ perm_slot<T>(fi[i]);
            __builtin_nontemporal_store(lds[0][s], st + (w | ui[i]) + lp);
            if (pair) __builtin_nontemporal_store(lds[1][s], st + (u | ui[i]) + lp);
        }
}

// ----------------------------------------------------------------------------
// kernel table
// ----------------------------------------------------------------------------
typedef void (*sweep_fn)(const SweepOne, const dq_job *, const dq_block *, const dq_phase *, const unsigned char *, const uint32_t *,
                         const uint32_t *);

template <typename T>
struct SweepTable {
    sweep_fn fn[2][DQ_MAX_REG_BITS + 1][DQ_MAX_WAVE_BITS + 1];
    sweep_fn own[2][DQ_MAX_REG_BITS + 1][DQ_MAX_WAVE_BITS + 1];  // of the shapes that 10 to 13 qubits take in one tile
    SweepTable() {
        memset(fn, 0, sizeof fn);
        memset(own, 0, sizeof own);
#define DQ_INST(R_, W_)                                                                  \
    fn[0][R_][W_] = sweep_kernel<T, R_, W_, 0>;                                          \
    fn[1][R_][W_] = sweep_kernel<T, R_, W_, 1>;
        DQ_INST(1, 0) DQ_INST(2, 0) DQ_INST(3, 0) DQ_INST(4, 0) DQ_INST(5, 0)
        DQ_INST(2, 1) DQ_INST(3, 1) DQ_INST(4, 1) DQ_INST(5, 1)
        DQ_INST(2, 2) DQ_INST(3, 2) DQ_INST(4, 2) DQ_INST(5, 2)
        DQ_INST(3, 3) DQ_INST(4, 3)
        // 14-bit tiles (k = 8) for FP32 only: 32 float amplitudes per thread
        // and a 64 KiB split exchange; the FP64 tile would not fit the registers
        if constexpr (std::is_same<T, float>::value) { DQ_INST(5, 3) }
#undef DQ_INST
#define DQ_OWN(R_, W_)                                   \
    own[0][R_][W_] = sweep_kernel<T, R_, W_, 0, true>;   \
    own[1][R_][W_] = sweep_kernel<T, R_, W_, 1, true>;
        DQ_OWN(3, 1) DQ_OWN(3, 2) DQ_OWN(3, 3) DQ_OWN(4, 3)
#undef DQ_OWN
    }
};

static SweepTable<double> g_tab64;
static SweepTable<float> g_tab32;

// Exchange mode of a tile shape (see exchange): split exchanges (1) for every
// FP32 tile and for FP64 tiles of 12+ bits; half the LDS per workgroup lets
// more FP32 workgroups share a CU (measured 18% faster on 30-qubit FP32
// circuits).  DGQ_SPLIT_EXCHANGE: 0 whole amplitudes everywhere, 1 split
// everywhere, unset the default.
static int g_split_mode = -1;
static int exchange_mode(int prec, int R, int W, int T) {
    (void)R;
    (void)W;
    if (g_split_mode < 0) {
        const char *e = getenv("DGQ_SPLIT_EXCHANGE");
        g_split_mode = e ? atoi(e) : 2;
    }
    if (g_split_mode == 0) return 0;
    if (g_split_mode == 1) return 1;
    return (prec == DQ_F32 || T >= 12) ? 1 : 0;
}

static sweep_fn lookup(int prec, int R, int W, int xm, bool own = false) {
    if (R < 0 || R > DQ_MAX_REG_BITS || W < 0 || W > DQ_MAX_WAVE_BITS || xm < 0 || xm > 1) return nullptr;
    if (own) return prec == DQ_F64 ? g_tab64.own[xm][R][W] : g_tab32.own[xm][R][W];
    return prec == DQ_F64 ? g_tab64.fn[xm][R][W] : g_tab32.fn[xm][R][W];
}

static size_t elem_bytes(int prec) { return prec == DQ_F64 ? 16 : 8; }

// bytes per LDS element of an exchange in mode xm
static uint32_t exchange_elem_bytes(int prec, int xm) {
    return xm == 0 ? (uint32_t)elem_bytes(prec) : (uint32_t)elem_bytes(prec) / 2;
}

// ----------------------------------------------------------------------------
// staging of descriptors: a pool of pinned host buffers.  An upload takes a
// buffer whose last copy has completed, so a stream with a long queue never
// holds up uploads on other streams; the pool grows to kStageMax buffers before
// a caller waits.
//
// Up to kStageKernelBytes a kernel of one workgroup makes the copy and, once it
// has read the buffer, stores the upload's number into it.  An event recorded
// after the copy instead costs the stream 4.5 us before its next kernel starts
// (two launches and a wait: 12.9 us, with an event between them 17.4 us).  The
// compiler keeps stage_copy's array in LDS and waits for each of its up to four
// loads a thread, so 64 KiB take up to four latencies of the host link one after
// another (bring_descriptors has its loads in flight together); longer uploads go
// through the copy engine and an event.
// ----------------------------------------------------------------------------
namespace {
struct StageSlot {
    void *host = nullptr;  // kStageHeader bytes with the number of the last upload read, then the data
    size_t cap = 0;        // of data
    uint32_t ticket = 0;   // number of the slot's last upload
    bool by_event = false; // that upload is guarded by ev, not by its number
    hipEvent_t ev = nullptr;
};
// Host memory of the staging and result protocols, which work while kernels run: the
// host polls words that a kernel stores before it ends, and rewrites a buffer that an
// earlier kernel has read without a wait for that kernel's stream.  Both need coherent
// memory; without the flag the runtime and its environment decide.
hipError_t shared_host_alloc(void **p, size_t bytes) { return hipHostMalloc(p, bytes, hipHostMallocPortable | hipHostMallocCoherent); }

constexpr unsigned kStageMax = 64;
constexpr size_t kStageHeader = 256;
constexpr size_t kStageKernelBytes = 64 * 1024;
constexpr unsigned kStageThreads = 1024;
constexpr std::chrono::seconds kStageWait(60);
std::mutex g_stage_mu;
StageSlot g_stage[kStageMax];
unsigned g_stage_used = 0;
unsigned g_stage_next = 0;
int g_device = -1;
int g_num_cus = 256;
// Address of the allocation-free read-out's `scratch` array on each device
// (hipGetSymbolAddress at dq_device_init; null until then).
constexpr int kMaxDevices = 64;
double *g_scratch_dev[kMaxDevices] = {};
}  // namespace

__global__ void __launch_bounds__(kStageThreads)
stage_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, uint32_t n16, uint32_t *read, uint32_t ticket) {
    constexpr uint32_t U = kStageKernelBytes / 16 / kStageThreads;
    uint4 v[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        const uint32_t i = threadIdx.x + u * kStageThreads;
        if (i < n16) v[u] = src[i];
    }
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        const uint32_t i = threadIdx.x + u * kStageThreads;
        if (i < n16) dst[i] = v[u];
    }
    __syncthreads();  // every thread has what it read: its stores were issued
    if (threadIdx.x == 0) __hip_atomic_store(read, ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A launch with an error code of its own: hipGetLastError also reports what an earlier
// call left, and a staging buffer is in use if the kernel that reads it was launched.
template <typename T> struct Same { using type = T; };
template <typename... A>
static hipError_t launch(void (*f)(A...), dim3 grid, dim3 block, size_t lds, void *stream, typename Same<A>::type... a) {
    void *args[] = {(void *)&a...};
    return hipLaunchKernel((const void *)f, grid, block, args, lds, (hipStream_t)stream);
}

// 1: the slot's last upload has been read, 0: not yet, -1: error (set)
static int stage_free(const StageSlot &c) {
    if (!c.host) return 1;
    if (!c.by_event) return __atomic_load_n((const uint32_t *)c.host, __ATOMIC_ACQUIRE) == c.ticket;
    const hipError_t e = hipEventQuery(c.ev);
    if (e == hipSuccess) return 1;
    if (e == hipErrorNotReady) {
        (void)hipGetLastError();
        return 0;
    }
    fail(DQ_ERR_HIP, "hipEventQuery failed: %s", hipGetErrorString(e));
    return -1;
}

// A slot whose last upload has been read, with room for `bytes`; lk holds g_stage_mu.
// With every slot in flight, waits for the first that comes free, without the lock:
// uploads of other threads go on.  After kStageWait it waits for the device instead,
// which ends with an error if an upload can no longer be read.
static int stage_pick(std::unique_lock<std::mutex> &lk, size_t bytes, StageSlot *&out) {
    StageSlot *slot = nullptr;
    std::chrono::steady_clock::time_point until{};
    bool waited = false;
    for (;;) {
        for (unsigned k = 0; k < g_stage_used && !slot; k++) {
            StageSlot &c = g_stage[(g_stage_next + k) % g_stage_used];
            const int f = stage_free(c);
            if (f < 0) return DQ_ERR_HIP;
            if (f) slot = &c;
        }
        if (slot) break;
        if (g_stage_used < kStageMax) {
            slot = &g_stage[g_stage_used];
            HIPC(hipEventCreateWithFlags(&slot->ev, hipEventDisableTiming));
            g_stage_used++;
            break;
        }
        const auto now = std::chrono::steady_clock::now();
        if (until == std::chrono::steady_clock::time_point{}) until = now + kStageWait;
        if (now < until) {
            lk.unlock();
            std::this_thread::sleep_for(std::chrono::microseconds(20));
            lk.lock();
            continue;
        }
        if (waited) return fail(DQ_ERR_HIP, "stage_upload: an earlier upload never completed");
        waited = true;
        until = {};
        lk.unlock();
        const hipError_t e = hipDeviceSynchronize();
        lk.lock();
        if (e != hipSuccess) return fail(DQ_ERR_HIP, "hipDeviceSynchronize failed: %s", hipGetErrorString(e));
    }
    g_stage_next = (unsigned)(slot - g_stage) + 1;
    StageSlot &s = *slot;
    out = slot;
    if (s.cap < bytes) {
        if (s.host) HIPC(hipHostFree(s.host));
        s.host = nullptr;
        s.cap = 0;
        size_t cap = kStageKernelBytes;
        while (cap < bytes) cap *= 2;
        HIPC(shared_host_alloc(&s.host, kStageHeader + cap));
        s.cap = cap;
        s.ticket = 0;
        s.by_event = false;
        memset(s.host, 0, kStageHeader);
    }
    return DQ_OK;
}

// An upload cannot be part of a graph: its replays would read the staging buffer
// again after it went to other uploads.
static int stage_capture(void *stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    HIPC(hipStreamIsCapturing((hipStream_t)stream, &status));
    return status == hipStreamCaptureStatusNone ? DQ_OK : fail(DQ_ERR_UNSUPPORTED, "descriptors cannot be uploaded while their stream is captured");
}

// Puts up to kStageKernelBytes in a slot for a kernel that reads it itself and then
// stores the ticket to the slot's first word; stage_undo if that kernel is not launched.
static int stage_fill(const std::vector<unsigned char> &src, StageSlot *&slot, void *stream) {
    int rc = stage_capture(stream);
    if (rc) return rc;
    std::unique_lock<std::mutex> lk(g_stage_mu);
    rc = stage_pick(lk, src.size(), slot);
    if (rc) return rc;
    memcpy((unsigned char *)slot->host + kStageHeader, src.data(), src.size());
    slot->ticket++;
    slot->by_event = false;
    return DQ_OK;
}

static void stage_undo(StageSlot *slot) {
    std::lock_guard<std::mutex> lk(g_stage_mu);
    slot->ticket--;
}

static int stage_upload(void *d_dst, const std::vector<unsigned char> &src, void *stream) {
    int rc = stage_capture(stream);
    if (rc) return rc;
    std::unique_lock<std::mutex> lk(g_stage_mu);
    StageSlot *slot = nullptr;
    rc = stage_pick(lk, src.size(), slot);
    if (rc) return rc;
    StageSlot &s = *slot;
    unsigned char *data = (unsigned char *)s.host + kStageHeader;
    memcpy(data, src.data(), src.size());
    if (src.size() <= kStageKernelBytes && src.size() % 16 == 0 && (uintptr_t)d_dst % 16 == 0) {
        s.ticket++;
        s.by_event = false;
        const hipError_t e = launch(stage_copy, dim3(1), dim3(kStageThreads), 0, stream, (const uint4 *)data, (uint4 *)d_dst,
                                    (uint32_t)(src.size() / 16), (uint32_t *)s.host, s.ticket);
        if (e != hipSuccess) {
            s.ticket--;  // nothing was enqueued: the slot is free
            return fail(DQ_ERR_HIP, "stage_copy: %s", hipGetErrorString(e));
        }
        return DQ_OK;
    }
    HIPC(hipMemcpyAsync(d_dst, data, src.size(), hipMemcpyHostToDevice, (hipStream_t)stream));
    s.by_event = true;
    HIPC(hipEventRecord(s.ev, (hipStream_t)stream));
    return DQ_OK;
}

// ----------------------------------------------------------------------------
// results of synchronous read-outs: pinned host slots that kernels write to
// directly, one per call in progress.  A copy of 200 bytes to a caller's pageable
// memory took 12.6 us on top of the kernel before it (24 us for 64 KiB); a kernel
// that stores its results to pinned memory takes no longer than one that stores
// them to the device.  At most kResultMax slots are ever allocated; a call that
// finds none free, or needs a larger one, copies from the device as before.
//
// The caller need not wait for the stream either: a slot is handed out with
// every word set to kUnwritten, and each word is ready once it holds anything
// else.  A word is stored once, by a thread that has read its inputs, so when
// all of them have arrived nothing the kernels read is in use any more.  What else a
// kernel writes may still be on its way: a sweep that writes tile sums has issued the
// stores of its state by then, not completed them.  Work on the same stream is ordered
// after it; another stream needs an event or a wait for this one.  Launch
// and wait for a kernel that stores one word 10.9 -> 5.4 us, 8192 words 11.8 -> 8.5 us.
// A wait longer than kResultPoll goes on as a wait for the stream, which also ends it
// where a result is that very word (no operation makes it: a signalling NaN) or
// a kernel failed.
// ----------------------------------------------------------------------------
namespace {
constexpr int kResultMax = 16;
constexpr size_t kResultBytes = 128 * 1024;
constexpr uint64_t kUnwritten = 0x7ff4dead00beef01ull;
constexpr std::chrono::microseconds kResultPoll(1000);
std::mutex g_result_mu;
void *g_result[kResultMax] = {};
bool g_result_taken[kResultMax] = {};
}  // namespace

extern "C" void *dq_result_acquire(size_t bytes) {
    if (bytes > kResultBytes) return nullptr;
    void *slot = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_result_mu);
        for (int i = 0; i < kResultMax && !slot; i++) {
            if (g_result_taken[i]) continue;
            if (!g_result[i] && shared_host_alloc(&g_result[i], kResultBytes) != hipSuccess) {
                (void)hipGetLastError();
                g_result[i] = nullptr;
                return nullptr;
            }
            g_result_taken[i] = true;
            slot = g_result[i];
        }
    }
    if (slot) std::fill_n((uint64_t *)slot, (bytes + 7) / 8, kUnwritten);
    return slot;
}

extern "C" void dq_result_release(void *slot) {
    if (!slot) return;
    std::lock_guard<std::mutex> lk(g_result_mu);
    for (int i = 0; i < kResultMax; i++)
        if (g_result[i] == slot) g_result_taken[i] = false;
}

extern "C" int dq_result_wait(const void *slot, void *out, size_t bytes, void *stream) {
    if (!slot || !out || bytes % 8 || bytes > kResultBytes) return fail(DQ_ERR_ARG, "dq_result_wait: bad arguments");
    const uint64_t *word = (const uint64_t *)slot;
    const size_t n = bytes / 8;
    uint64_t *to = (uint64_t *)out;
    std::chrono::steady_clock::time_point until{};
    for (size_t i = 0; i < n; i++) {
        uint64_t v;
        for (uint32_t spin = 0; (v = __atomic_load_n(word + i, __ATOMIC_ACQUIRE)) == kUnwritten; spin++) {
            __builtin_ia32_pause();
            if (spin % 64) continue;
            const auto now = std::chrono::steady_clock::now();
            if (until == std::chrono::steady_clock::time_point{}) until = now + kResultPoll;
            if (now < until) continue;
            HIPC(hipStreamSynchronize((hipStream_t)stream));
            memcpy(out, slot, bytes);
            return DQ_OK;
        }
        to[i] = v;
    }
    return DQ_OK;
}

namespace {
// Where a read-out of `bytes` writes: a result slot, or `fallback` on the device.
struct ResultSlot {
    void *host;
    void *dst;
    hipStream_t stream;
    bool waited = false;
    ResultSlot(size_t bytes, void *fallback, void *s) : host(dq_result_acquire(bytes)), dst(host ? host : fallback), stream((hipStream_t)s) {}
    ~ResultSlot() {
        if (host && !waited) (void)hipStreamSynchronize(stream);  // an error came before: kernels may still store to it
        dq_result_release(host);
    }
    ResultSlot(const ResultSlot &) = delete;
    ResultSlot &operator=(const ResultSlot &) = delete;
    // Waits for the results of the kernels enqueued on the stream and hands them over.
    int collect(void *out, size_t bytes) {
        waited = true;
        if (host) return dq_result_wait(host, out, bytes, stream);
        HIPC(hipMemcpyAsync(out, dst, bytes, hipMemcpyDeviceToHost, stream));
        HIPC(hipStreamSynchronize(stream));
        return DQ_OK;
    }
};
}  // namespace

// ----------------------------------------------------------------------------
// C ABI: plumbing
// ----------------------------------------------------------------------------
extern "C" int dq_device_init(int device) {
    if (device < 0 || device >= kMaxDevices) return fail(DQ_ERR_ARG, "dq_device_init: device %d out of range", device);
    HIPC(hipSetDevice(device));
    if (!g_scratch_dev[device]) {
        // each device holds its own copy of `scratch`; host code uses this
        // address, never the array's name (a host-side stand-in)
        void *p = nullptr;
        HIPC(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_dev[device] = (double *)p;
    }
    if (g_device != device) {
        // allow the large LDS tiles (up to 128 KiB) on every sweep instantiation
        for (int sp = 0; sp < 2; sp++)
            for (int R = 0; R <= DQ_MAX_REG_BITS; R++)
                for (int W = 0; W <= DQ_MAX_WAVE_BITS; W++) {
                    for (const void *fn : {(const void *)g_tab64.fn[sp][R][W], (const void *)g_tab32.fn[sp][R][W],
                                           (const void *)g_tab64.own[sp][R][W], (const void *)g_tab32.own[sp][R][W]}) {
                        if (!fn) continue;
                        HIPC(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 131072));
                        // the exchange addresses LDS by offset from 0 (lds_at): no static LDS allowed
                        hipFuncAttributes fa;
                        HIPC(hipFuncGetAttributes(&fa, fn));
                        if (fa.sharedSizeBytes != 0)
                            return fail(DQ_ERR_UNSUPPORTED, "sweep kernel (R=%d, W=%d) has %zu bytes of static LDS", R, W,
                                        (size_t)fa.sharedSizeBytes);
                    }
                }
        {
            hipDeviceProp_t prop;
            HIPC(hipGetDeviceProperties(&prop, device));
            g_num_cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
        }
        HIPC(hipFuncSetAttribute((const void *)small_kernel<double>, hipFuncAttributeMaxDynamicSharedMemorySize, 131072));
        HIPC(hipFuncSetAttribute((const void *)small_kernel<float>, hipFuncAttributeMaxDynamicSharedMemorySize, 131072));
        HIPC(hipFuncSetAttribute((const void *)dense_kernel<5>, hipFuncAttributeMaxDynamicSharedMemorySize, 131072));
        HIPC(hipFuncSetAttribute((const void *)dense_kernel<6>, hipFuncAttributeMaxDynamicSharedMemorySize, 131072));
        HIPC(hipFuncSetAttribute((const void *)dense_kernel<7>, hipFuncAttributeMaxDynamicSharedMemorySize, 131072));
        g_device = device;
    }
    return DQ_OK;
}

extern "C" int dq_device_info(char *name, size_t name_len, int *num_cus, size_t *total_mem, size_t *free_mem) {
    int dev = 0;
    HIPC(hipGetDevice(&dev));
    hipDeviceProp_t p;
    HIPC(hipGetDeviceProperties(&p, dev));
    if (name && name_len) snprintf(name, name_len, "%s", p.gcnArchName);
    if (num_cus) *num_cus = p.multiProcessorCount;
    size_t fr = 0, tot = 0;
    HIPC(hipMemGetInfo(&fr, &tot));
    if (total_mem) *total_mem = tot;
    if (free_mem) *free_mem = fr;
    return DQ_OK;
}

extern "C" int dq_malloc(void **ptr, size_t bytes) {
    if (!ptr) return fail(DQ_ERR_ARG, "dq_malloc: null out pointer");
    hipError_t e = hipMalloc(ptr, bytes ? bytes : 16);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();  // a caller may go on (smaller request, other memory): do not leave the error pending
        return fail(DQ_ERR_NOMEM, "dq_malloc: out of device memory (%zu bytes)", bytes);
    }
    HIPC(e);
    return DQ_OK;
}
extern "C" int dq_free(void *ptr) { HIPC(hipFree(ptr)); return DQ_OK; }
extern "C" int dq_host_alloc(void **ptr, size_t bytes) {
    hipError_t e = hipHostMalloc(ptr, bytes ? bytes : 16, hipHostMallocDefault);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();  // the paging executor falls back to pageable memory: clear the pending error
        return fail(DQ_ERR_NOMEM, "dq_host_alloc: out of pinned memory (%zu bytes)", bytes);
    }
    HIPC(e);
    return DQ_OK;
}
extern "C" int dq_host_free(void *ptr) { HIPC(hipHostFree(ptr)); return DQ_OK; }
extern "C" int dq_stream_create(void **stream) {
    hipStream_t s;
    HIPC(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *stream = (void *)s;
    return DQ_OK;
}
extern "C" int dq_stream_destroy(void *stream) { HIPC(hipStreamDestroy((hipStream_t)stream)); return DQ_OK; }
extern "C" int dq_stream_sync(void *stream) { HIPC(hipStreamSynchronize((hipStream_t)stream)); return DQ_OK; }
extern "C" int dq_device_sync(void) { HIPC(hipDeviceSynchronize()); return DQ_OK; }
extern "C" int dq_memcpy_async(void *dst, const void *src, size_t bytes, int kind, void *stream) {
    hipMemcpyKind k = kind == DQ_H2D ? hipMemcpyHostToDevice : kind == DQ_D2H ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice;
    HIPC(hipMemcpyAsync(dst, src, bytes, k, (hipStream_t)stream));
    return DQ_OK;
}
extern "C" int dq_event_create(void **ev) {
    hipEvent_t e;
    HIPC(hipEventCreate(&e));
    *ev = (void *)e;
    return DQ_OK;
}
extern "C" int dq_event_destroy(void *ev) { HIPC(hipEventDestroy((hipEvent_t)ev)); return DQ_OK; }
extern "C" int dq_event_record(void *ev, void *stream) { HIPC(hipEventRecord((hipEvent_t)ev, (hipStream_t)stream)); return DQ_OK; }
extern "C" int dq_event_elapsed_ms(void *a, void *b, float *ms) {
    HIPC(hipEventSynchronize((hipEvent_t)b));
    HIPC(hipEventElapsedTime(ms, (hipEvent_t)a, (hipEvent_t)b));
    return DQ_OK;
}
extern "C" int dq_stream_wait_event(void *stream, void *ev) {
    HIPC(hipStreamWaitEvent((hipStream_t)stream, (hipEvent_t)ev, 0));
    return DQ_OK;
}

// ----------------------------------------------------------------------------
// C ABI: kernels
// ----------------------------------------------------------------------------
static inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Upper bound of the device program built from n_ops descriptors in n_phases
// phases: at most kOpBytes per descriptor.  A complex matrix in FP64 behind
// a workgroup-condition op takes 128, a FAN op 16 and 32 per term.  A register
// table of 2^R entries takes 16 + 16 * 2^R bytes, emitted once per assignment
// of at most two folded workgroup bits, each copy behind a 32-byte condition:
// 2240 at R = 5.  The planner's tables span 1 + 2^R / 4 descriptors (9 x 320);
// one made of plain phases folds only the bits whose copies fit what its own
// descriptors bring (ProgBuilder::build).  Shears fused with it take 16 * R
// in each copy, what the first of them brings (4 x 80).  Plus an END op
// per phase, and padding so the interpreter's fixed-size header loads stay in
// the buffer.
static constexpr size_t kOpBytes = 320;
static size_t prog_bound(uint32_t n_phases, uint32_t n_ops) { return n_ops * kOpBytes + (size_t)n_phases * 16 + 256; }

extern "C" size_t dq_apply_ws_bytes(uint32_t n_blocks, uint32_t n_phases, uint32_t n_ops, uint32_t n_jobs) {
    return align_up(n_blocks * sizeof(dq_block), 256) + align_up(n_phases * sizeof(dq_phase), 256) +
           align_up(n_ops * sizeof(dq_op), 256) + align_up(n_jobs * sizeof(dq_job), 256) +
           align_up((size_t)n_phases * DQ_PAUX * sizeof(uint32_t), 256) +
           align_up((size_t)n_blocks * DQ_BAUX * sizeof(uint32_t), 256) + align_up(prog_bound(n_phases, n_ops), 256);
}

// Images g[b] < 2^L of the index bits b >= L such that, for as many of the given
// sets of bits (masks) as possible, the images of a set's bits are linearly
// independent (the image of a bit b < L is the bit itself).  Bits in no set get 0.
// A depth-first search, the bits in most sets first, tries kSwizzleTries images; if
// it finds no choice that serves every set, each bit in turn takes the image that
// spoils the fewest.  Sets that recur are looked at once, and an image only
// against the sets its bit is in, in fixed buffers: over 4423 blocks of 10 to 30
// qubits 12 -> 1.3 us a block, 17 qubits of an ansatz in 29 blocks 88 -> 17 us of a pass of
// 319.  The 27 of them that cannot be served took 1.2 ms each and ended with no
// images at all, 1676 sets with conflicts that are now 106: an ansatz of 12 qubits in
// one tile FP32 R = 3, W = 3 took 900 us a flush, now 119 us.
constexpr int kSwizzleTries = 1000;
constexpr int kSwizzleSets = 256;  // distinct sets looked at; later ones may conflict

static void pick_images(const uint32_t *masks, uint32_t n, int L, uint32_t *g) {
    memset(g, 0, 32 * sizeof(uint32_t));
    const uint32_t low = (1u << L) - 1u;
    uint32_t set[kSwizzleSets], times[kSwizzleSets], all = 0;
    int n_sets = 0;
    for (uint32_t i = 0; i < n; i++) {
        if (!(masks[i] & ~low)) continue;
        int k = 0;
        while (k < n_sets && set[k] != masks[i]) k++;
        if (k == kSwizzleSets) continue;
        if (k == n_sets) {
            set[n_sets] = masks[i];
            times[n_sets++] = 0;
            all |= masks[i] & ~low;
        }
        times[k]++;
    }
    int vars[32], in[32] = {}, nv = 0;
    for (uint32_t u = all; u; u &= u - 1) vars[nv++] = __builtin_ctz(u);
    for (int v = 0; v < nv; v++)
        for (int k = 0; k < n_sets; k++) in[vars[v]] += (set[k] >> vars[v]) & 1u;
    std::stable_sort(vars, vars + nv, [&](int a, int b) { return in[a] > in[b]; });
    // are the images of the bits of x that have one independent of each other and of x's low bits?
    auto ok = [&](uint32_t x, uint32_t have) {
        uint32_t base[32];
        int r = 0;
        for (uint32_t u = x & have; u; u &= u - 1) {
            uint32_t v = g[__builtin_ctz(u)] & low & ~x;
            for (int k = 0; k < r; k++) v = std::min(v, v ^ base[k]);
            if (!v) return false;
            base[r++] = v;
        }
        return true;
    };
    uint32_t cand[32];  // single bits first
    int nc = 0;
    for (int i = 0; i < L; i++) cand[nc++] = 1u << i;
    for (uint32_t c = 1; c <= low; c++)
        if (c & (c - 1)) cand[nc++] = c;
    int next[32] = {}, tries = 0, i = 0;
    uint32_t have = 0;
    while (i >= 0 && i < nv && tries < kSwizzleTries) {
        const int b = vars[i];
        have &= ~(1u << b);
        if (next[i] == nc) {
            next[i--] = 0;
            continue;
        }
        g[b] = cand[next[i]++];
        tries++;
        bool good = true;
        for (int k = 0; k < n_sets && good; k++)
            if ((set[k] >> b) & 1u) good = ok(set[k], have | (1u << b));
        if (good) {
            have |= 1u << b;
            i++;
        }
    }
    if (i == nv) return;
    have = 0;
    for (int pass = 0; pass < 2; pass++)
        for (int v = 0; v < nv; v++) {
            const int b = vars[v];
            have |= 1u << b;
            uint32_t best = 0, least = ~0u;
            for (int c = 0; c < nc; c++) {
                g[b] = cand[c];
                uint32_t spoilt = 0;
                for (int k = 0; k < n_sets; k++)
                    if (((set[k] >> b) & 1u) && !ok(set[k], have)) spoilt += times[k];
                if (spoilt < least) {
                    least = spoilt;
                    best = cand[c];
                }
            }
            g[b] = best;
        }
}

// LDS swizzle of one exchange: tile index x -> x ^ (xor of g[b] over the set
// bits b >= L of x), g[b] < 2^L.  The LDS serves 128 bytes a clock, i.e. the
// 2^L lanes whose lane bits 0..L-1 vary (2^L = 128 / element bytes); they hit
// distinct banks iff the images of their L tile bits (bit b itself for b < L,
// else g[b]) are linearly independent, in the writing layout A and in the
// reading layout B.
static void pick_swizzle(const dq_phase &A, const dq_phase &B, int L, uint32_t *g) {
    uint32_t masks[2] = {0, 0};
    for (int l = 0; l < L; l++) {
        masks[0] |= A.lane_t[l];
        masks[1] |= B.lane_t[l];
    }
    pick_images(masks, 2, L, g);
}

// Owned-slot exchanges (split mode 1).  A position of a layout is (thread,
// register index) as the bit vector lane bits 0..5, wave bits, register bits;
// every position has a fixed LDS slot, the position under a swizzle that xors
// images g[b] < 2^L of its high bits b >= L into its low L bits.  The bit of a
// tile bit's position in a phase's layout:
static int pos_bit(const dq_phase &P, uint32_t x, int R, int W) {
    for (int l = 0; l < 6; l++)
        if (P.lane_t[l] == x) return l;
    for (int w = 0; w < W; w++)
        if (P.wave_t[w] == x) return 6 + w;
    for (int r = 0; r < R; r++)
        if (P.reg_t[r] == x) return 6 + W + r;
    return -1;
}

// The tile bit at position bit b of a layout.
static uint32_t tile_bit_at(const dq_phase &P, int b, int W) {
    if (b < 6) return P.lane_t[b];
    if (b < 6 + W) return P.wave_t[b - 6];
    return P.reg_t[b - 6 - W];
}

// One swizzle for all exchanges of a block (consecutive exchanges share the
// slots of the layout between them).  A thread's own slots differ only in its
// lane bits among the 2^L lanes the LDS serves together, so they never
// conflict; the computed sides are the real read (the previous layout's
// positions of the lanes' new elements) and the imaginary write (the next
// layout's positions of their old ones): the images of the lanes' low L bits
// are to be independent on both sides of every exchange.
static void pick_owned_swizzle(const dq_phase *ph, uint32_t nph, int R, int W, int L, uint32_t *g) {
    std::vector<uint32_t> masks;
    masks.reserve(2 * nph);
    for (uint32_t p = 1; p < nph; p++) {
        const dq_phase &A = ph[p - 1], &B = ph[p];
        uint32_t m1 = 0, m2 = 0;
        for (int l = 0; l < L; l++) {
            const int b1 = pos_bit(A, B.lane_t[l], R, W), b2 = pos_bit(B, A.lane_t[l], R, W);
            if (b1 >= 0) m1 |= 1u << b1;
            if (b2 >= 0) m2 |= 1u << b2;
        }
        masks.push_back(m1);
        masks.push_back(m2);
    }
    pick_images(masks.data(), (uint32_t)masks.size(), L, g);
}

// Tables of the owned-slot exchange from layout A to layout B (phase_aux of
// B): [DQ_TF] / [DQ_FJ] the thread's own slots, [DQ_TB] / [DQ_XB] the real
// read (slot of the A-position of B's element), [DQ_TA] / [DQ_XA] the
// imaginary write (slot of the B-position of A's element), [2] = 1 unless the
// layout change is a set of pairwise swaps of position bits.
static bool owned_tables(const dq_phase &A, const dq_phase &B, int R, int W, int L, const uint32_t *g, uint32_t es,
                         uint32_t *pa) {
    const int T = 6 + W + R;
    auto sig = [&](int b) { return ((1u << b) ^ (b >= L ? g[b] : 0u)) * es; };
    int to_b[32], to_a[32];  // position bit of A -> of B, and back
    for (int b = 0; b < T; b++) {
        to_b[b] = pos_bit(B, tile_bit_at(A, b, W), R, W);
        to_a[b] = pos_bit(A, tile_bit_at(B, b, W), R, W);
        if (to_b[b] < 0 || to_a[b] < 0) return false;
    }
    bool swaps = true;
    for (int b = 0; b < T; b++) swaps &= to_b[to_b[b]] == b;
    pa[2] = swaps ? 0u : 1u;
    for (int l = 0; l < 6; l++) {
        pa[DQ_TF + l] = sig(l);
        pa[DQ_TB + l] = sig(to_a[l]);
        pa[DQ_TA + l] = sig(to_b[l]);
    }
    for (int w = 0; w < W; w++) {
        pa[DQ_TF + 6 + w] = sig(6 + w);
        pa[DQ_TB + 6 + w] = sig(to_a[6 + w]);
        pa[DQ_TA + 6 + w] = sig(to_b[6 + w]);
    }
    for (uint32_t j = 0; j < (1u << R); j++) {
        uint32_t f = 0, xb = 0, xa = 0;
        for (int r = 0; r < R; r++)
            if ((j >> r) & 1) {
                f ^= sig(6 + W + r);
                xb ^= sig(to_a[6 + W + r]);
                xa ^= sig(to_b[6 + W + r]);
            }
        pa[DQ_FJ + j] = f;
        pa[DQ_XB + j] = xb;
        pa[DQ_XA + j] = xa;
    }
    return true;
}

// Swizzled tile index of x under images g (bits b >= L).
static uint32_t swizzle_host(uint32_t x, const uint32_t *g, int L) {
    uint32_t y = x;
    for (uint32_t m = x >> L; m; m &= m - 1) y ^= g[L + __builtin_ctz(m)];
    return y;
}

// block_aux record of a block: its non-tile qubits as runs (see block_aux).
static bool block_runs(const dq_block &b, uint32_t *out) {
    memset(out, 0, DQ_BAUX * sizeof(uint32_t));
    uint64_t m = b.nontile_mask;
    uint32_t in = 0;
    int i = 0;
    while (m) {
        if (i == DQ_RUNS) return false;
        const int pos = __builtin_ctzll(m);
        int len = 0;
        while (pos + len < 64 && ((m >> (pos + len)) & 1)) len++;
        out[i] = in | ((uint32_t)len << 16);
        out[16 + i] = (uint32_t)pos;
        in += (uint32_t)len;
        m &= ~(((len == 64) ? ~0ull : ((1ull << len) - 1)) << pos);
        i++;
    }
    return in <= 31;
}

// Device program of one phase (format and op codes in gen_ops_asm.py /
// ops_asm.inc): register conditions resolved into op variants or masks,
// consecutive unconditioned shears on distinct register bits merged into one
// op, unconditioned diagonal ops folded into the table of their run and that
// table fused with the shears after it, a WG op in front of each op with a
// workgroup condition, END last.
namespace {
// Codes of the device ops for one R, looked up once.  Searching the table by
// name for every op, and a heap block for every table, took most of a flush's
// host time: the programs of a 30-qubit circuit (2426 ops in 106 phases)
// 512 -> 104 us, of a 17-qubit one (507 ops in 94 phases) 100 -> 30 us.
struct OpCodes {
    const DevOpCode *tab;
    int n;
    int END, WG, SHEARS, TABLE_FULL, TABLE_GEN, TSH_FULL, TSH_GEN, FAN;
    int TABLE_HALF[DQ_MAX_REG_BITS], TSH_HALF[DQ_MAX_REG_BITS], MAT[DQ_MAX_REG_BITS], SWAP[DQ_MAX_REG_BITS], RMAT[DQ_MAX_REG_BITS];
    int FM_ALL, FM_B[DQ_MAX_REG_BITS][2];
    struct Cond {  // variants of a conditioned op: every register, one bit, two bits (r1 < r2), a mask
        int all, gen, b[DQ_MAX_REG_BITS][2], bb[DQ_MAX_REG_BITS][DQ_MAX_REG_BITS][2][2];
    } NEG, PHASE;
    int find(const char *name, int p0 = -1, int p1 = -1, int p2 = -1, int p3 = -1) const {
        for (int c = 0; c < n; c++)
            if (!strcmp(tab[c].name, name) && tab[c].p[0] == p0 && tab[c].p[1] == p1 && tab[c].p[2] == p2 && tab[c].p[3] == p3)
                return c;
        return -1;
    }
    void find_cond(Cond &d, const std::string &name, int R) const {
        d.all = find((name + "_ALL").c_str());
        d.gen = find((name + "_GEN").c_str());
        for (int r = 0; r < R; r++)
            for (int v = 0; v < 2; v++) {
                d.b[r][v] = find((name + "_B").c_str(), r, v);
                for (int r2 = r + 1; r2 < R; r2++)
                    for (int v2 = 0; v2 < 2; v2++) d.bb[r][r2][v][v2] = find((name + "_BB").c_str(), r, r2, v, v2);
            }
    }
    explicit OpCodes(int R) {
        tab = dev_ops(R, n);
        END = find("END");
        WG = find("WG");
        SHEARS = find("SHEARS");
        TABLE_FULL = find("TABLE_FULL");
        TABLE_GEN = find("TABLE_GEN");
        TSH_FULL = find("TSH_FULL");
        TSH_GEN = find("TSH_GEN");
        FAN = find("FAN");
        FM_ALL = find("FM_ALL");
        for (int r = 0; r < R; r++) {
            TABLE_HALF[r] = find("TABLE_HALF", r);
            TSH_HALF[r] = find("TSH_HALF", r);
            MAT[r] = find("MAT", r);
            SWAP[r] = find("SWAP", r);
            RMAT[r] = find("RMAT", r);
            for (int v = 0; v < 2; v++) FM_B[r][v] = find("FM_B", r, v);
        }
        find_cond(NEG, "NEG", R);
        find_cond(PHASE, "PHASE", R);
    }
    static const OpCodes &of(int R) {
        static const OpCodes all[DQ_MAX_REG_BITS] = {OpCodes(1), OpCodes(2), OpCodes(3), OpCodes(4), OpCodes(5)};
        return all[R - 1];
    }
};
static_assert(DQ_MAX_REG_BITS == 5, "OpCodes::of lists every R");

struct ProgBuilder {
    int prec, R, NR, ncodes;
    size_t ts;
    const OpCodes &cd;
    const DevOpCode *tab;
    std::vector<unsigned char> &out;
    bool gather;       // phases of one register condition become one FAN op
    bool bad = false;  // an op with no code (never sent to the device)
    ProgBuilder(int prec_, int R_, std::vector<unsigned char> &o, bool gather_ = true)
        : prec(prec_), R(R_), NR(1 << R_), ts(prec_ == DQ_F64 ? 8 : 4), cd(OpCodes::of(R_)), out(o), gather(gather_) {
        tab = cd.tab;
        ncodes = cd.n;
    }
    size_t size(int c) const { return (size_t)(prec == DQ_F64 ? tab[c].size64 : tab[c].size32); }
    // one op into `v`: header then coefficient bytes, zero padded to its size
    void encode(std::vector<unsigned char> &v, int c, uint32_t mask, uint32_t cthr, uint32_t vthr, const void *coef,
                size_t nbytes) {
        if (c < 0 || c >= ncodes || nbytes + 16 > size(c)) {
            bad = true;
            return;
        }
        const size_t at = v.size();
        v.resize(at + size(c), 0);
        const uint32_t hdr[4] = {(uint32_t)c, mask, cthr, vthr};
        memcpy(v.data() + at, hdr, 16);
        if (nbytes) memcpy(v.data() + at + 16, coef, nbytes);
    }
    void emit(const std::vector<unsigned char> &op, uint64_t c_wg, uint64_t v_wg) {
        if (c_wg) {
            const uint64_t cond[2] = {c_wg, v_wg};
            encode(out, cd.WG, 0, 0, (uint32_t)op.size(), cond, 16);
        }
        out.insert(out.end(), op.begin(), op.end());
    }
    // register indices (pair ops: lower indices) satisfying (j & c) == v
    uint32_t jmask(uint32_t c, uint32_t v, int pair_bit) const {
        uint32_t m = 0;
        for (int j = 0; j < NR; j++) {
            if (pair_bit >= 0 && ((j >> pair_bit) & 1)) continue;
            if (((uint32_t)j & c) == v) m |= 1u << j;
        }
        return m;
    }
    // NEG / PHASE variant for the register condition (c, v)
    static int cond_variant(const OpCodes::Cond &d, uint32_t c, uint32_t v) {
        const int pc = __builtin_popcount(c);
        if (pc == 0) return d.all;
        if (pc == 1) {
            const int r = __builtin_ctz(c);
            return d.b[r][(v >> r) & 1];
        }
        if (pc == 2) {
            const int r1 = __builtin_ctz(c), r2 = 31 - __builtin_clz(c);
            return d.bb[r1][r2][(v >> r1) & 1][(v >> r2) & 1];
        }
        return d.gen;
    }
    // Value i of op o's coefficient array, in double.
    double val(const dq_op &o, int i) const {
        if (prec == DQ_F64) {
            double v;
            memcpy(&v, reinterpret_cast<const unsigned char *>(o.m) + 8 * i, 8);
            return v;
        }
        float v;
        memcpy(&v, reinterpret_cast<const unsigned char *>(o.m) + 4 * i, 4);
        return (double)v;
    }
    // A diagonal over the register index, in double.
    struct Diag {
        double re[1 << DQ_MAX_REG_BITS], im[1 << DQ_MAX_REG_BITS];
        Diag() { clear(); }
        void clear() {
            std::fill(re, re + (1 << DQ_MAX_REG_BITS), 1.0);
            std::fill(im, im + (1 << DQ_MAX_REG_BITS), 0.0);
        }
        void mul(int j, double fr, double fi) {
            const double r = re[j] * fr - im[j] * fi, i = re[j] * fi + im[j] * fr;
            re[j] = r;
            im[j] = i;
        }
        void mul_cond(int NR, uint32_t c, uint32_t v, double fr, double fi) {
            for (int j = 0; j < NR; j++)
                if (((uint32_t)j & c) == v) mul(j, fr, fi);
        }
    };
    // A table op (or, with shear slots, a table+shears op) for the diagonal
    // d over the register index: HALF when every factor that is not 1
    // has one register bit set, FULL when at least 3/4 of them are not 1, GEN
    // (a mask of the factors to apply) otherwise.  False if every factor is 1.
    bool encode_table(std::vector<unsigned char> &op, const Diag &d, const unsigned char *slots, uint32_t shear_mask) {
        unsigned char body[(2 << DQ_MAX_REG_BITS) * 8 + 2 * DQ_MAX_REG_BITS * 8];
        size_t len = 0;
        uint32_t ne1 = 0;  // factors that are not exactly 1 in the state precision
        for (int e = 0; e < NR; e++) {
            const bool one = prec == DQ_F64 ? d.re[e] == 1.0 && d.im[e] == 0.0 : (float)d.re[e] == 1.0f && (float)d.im[e] == 0.0f;
            if (!one) ne1 |= 1u << e;
        }
        if (!ne1) return false;
        int half = -1;
        for (int r = 0; r < R && half < 0; r++)
            if ((ne1 & ~jmask(1u << r, 1u << r, -1)) == 0) half = r;
        int c;
        uint32_t gen = 0;
        if (half >= 0) {
            c = slots ? cd.TSH_HALF[half] : cd.TABLE_HALF[half];
        } else if (4 * __builtin_popcount(ne1) >= 3 * NR) {
            c = slots ? cd.TSH_FULL : cd.TABLE_FULL;
        } else {
            gen = ne1;
            c = slots ? cd.TSH_GEN : cd.TABLE_GEN;
        }
        for (int e = 0; e < NR; e++) {
            if (half >= 0 && !((e >> half) & 1)) continue;
            if (prec == DQ_F64) {
                const double f[2] = {d.re[e], d.im[e]};
                memcpy(body + len, f, 16);
            } else {
                const float f[2] = {(float)d.re[e], (float)d.im[e]};
                memcpy(body + len, f, 8);
            }
            len += 2 * ts;
        }
        if (slots) {
            memcpy(body + len, slots, 2 * (size_t)R * ts);
            encode(op, c, shear_mask, gen, 0, body, len + 2 * (size_t)R * ts);
        } else {
            encode(op, c, gen, 0, 0, body, len);
        }
        return true;
    }
    // Diagonal ops commute, so every diagonal op without a lane or workgroup
    // condition in a run of diagonal ops that holds a table is multiplied into
    // that run's table; the table is emitted before the next non-diagonal op,
    // fused with it when that op is a run of unconditioned shears.
    // NEG / PHASE ops of such a run whose only condition is one workgroup bit
    // (controlled-Z or controlled phases with a qubit outside the tile) are
    // folded too, for up to kWgFoldBits distinct bits: the table is emitted
    // once per assignment of those bits, each copy guarded by its assignment
    // and holding the factors that apply there.  A workgroup runs exactly one
    // copy and skips the others, so the conditioned factors cost no vector
    // instruction.
    static constexpr int kWgFoldBits = 2;  // the program size bound (prog_bound) assumes at most 2
    struct WgDiag {
        uint64_t c_wg, v_wg;
        uint32_t c_reg, v_reg;
        double fr, fi;
    };
    static constexpr size_t kFanTerm = 32;  // bytes
    // NEG / PHASE ops of a diagonal run with a lane or workgroup condition, kept
    // by register condition (0: none, 1 + 2 r + v: bit r = v) until the run ends.
    std::vector<const dq_op *> held[1 + 2 * DQ_MAX_REG_BITS];
    static bool can_hold(const dq_op &o) {
        return (o.c_thr || o.c_wg) && __builtin_popcountll(o.c_wg) <= 1 && __builtin_popcount(o.c_reg) <= 1;
    }
    void emit_single(const dq_op &o) {
        std::vector<unsigned char> op;
        if (o.kind == DQ_OP_NEG)
            encode(op, cond_variant(cd.NEG, o.c_reg, o.v_reg), jmask(o.c_reg, o.v_reg, -1), o.c_thr, o.v_thr, nullptr, 0);
        else
            encode(op, cond_variant(cd.PHASE, o.c_reg, o.v_reg), jmask(o.c_reg, o.v_reg, -1), o.c_thr, o.v_thr, o.m, 2 * ts);
        emit(op, o.c_wg, o.v_wg);
    }
    // The held ops of one register condition: a FAN op where that takes fewer
    // vector instructions (a complex product of 4 on every selected register, and
    // 6 a term, against 4 or, for a sign, 2 on every selected register and 2 a
    // term; half of those with a workgroup condition are skipped).  A 27-qubit
    // Fourier transform in FP32 ran 254 phases of 16 or 32 registers each.
    void emit_held(uint32_t &n_out) {
        for (int g = 0; g < 1 + 2 * R; g++) {
            auto &h = held[g];
            if (h.empty()) continue;
            const int regs = g ? NR / 2 : NR;
            double one = 0.0, fan = 4.0 * regs;
            for (const dq_op *o : h) {
                const double c = (o->kind == DQ_OP_NEG ? 2.0 : 4.0) * regs + 2.0;
                one += o->c_wg ? 0.5 * c : c;
                fan += o->c_wg ? 3.0 : 6.0;
            }
            if (h.size() < 2 || fan >= one) {
                for (const dq_op *o : h) emit_single(*o);
                n_out += (uint32_t)h.size();
                h.clear();
                continue;
            }
            const size_t at = out.size(), tb = kFanTerm;
            out.resize(at + 16 + h.size() * tb, 0);
            unsigned char *w = out.data() + at;
            const uint32_t apply = (uint32_t)(g ? cd.FM_B[(g - 1) / 2][(g - 1) & 1] : cd.FM_ALL);
            const uint32_t hdr[4] = {(uint32_t)cd.FAN, apply, 0, (uint32_t)(16 + h.size() * tb)};
            memcpy(w, hdr, 16);
            w += 16;
            for (size_t i = 0; i < h.size(); i++, w += tb) {
                const dq_op &o = *h[i];
                uint32_t c[2] = {o.c_thr | (o.v_thr << 16), 0};
                if (o.c_wg) c[1] = (uint32_t)__builtin_ctzll(o.c_wg) | 0x100u | (o.v_wg ? 0x200u : 0u);
                if (i + 1 == h.size()) c[1] |= 0x400u;
                memcpy(w, c, 8);
                const double f[2] = {o.kind == DQ_OP_NEG ? -1.0 : val(o, 0), o.kind == DQ_OP_NEG ? 0.0 : val(o, 1)};
                memcpy(w + 16, f, 16);
            }
            h.clear();
            n_out++;
        }
    }
    void build(const dq_op *ops, uint32_t count, uint32_t &n_out) {
        n_out = 0;
        std::vector<unsigned char> op;
        const size_t nslot = 2 * (size_t)R * ts;  // bytes of the shear slots
        Diag tab_;
        bool pending = false;  // tab_ holds a table not yet emitted
        std::vector<WgDiag> wgd;  // workgroup-conditioned factors of the pending table
        uint64_t wg_bits = 0;     // their workgroup bits
        size_t from = 0;          // descriptors that the table of the current run is made of
        auto is_diag = [](const dq_op &o) {
            return o.kind == DQ_OP_NEG || o.kind == DQ_OP_PHASE || o.kind == DQ_OP_DIAGR;
        };
        auto flush = [&](const unsigned char *slots, uint32_t shear_mask) {
            if (pending && wg_bits) {
                const int nb = __builtin_popcountll(wg_bits);
                for (uint32_t a = 0; a < (1u << nb); a++) {
                    uint64_t val = 0, m = wg_bits;  // assignment a deposited on the bits
                    for (int i = 0; m; i++, m &= m - 1)
                        if ((a >> i) & 1) val |= m & (~m + 1);
                    Diag v = tab_;
                    for (const WgDiag &d : wgd)
                        if ((val & d.c_wg) == d.v_wg) v.mul_cond(NR, d.c_reg, d.v_reg, d.fr, d.fi);
                    op.clear();
                    if (!encode_table(op, v, slots, shear_mask)) {
                        if (!slots) continue;  // nothing to do for these workgroups
                        op.clear();
                        encode(op, cd.SHEARS, shear_mask, 0, 0, slots, nslot);
                    }
                    emit(op, wg_bits, val);
                    n_out++;
                }
            } else {
                op.clear();
                const bool any = pending && encode_table(op, tab_, slots, shear_mask);
                if (any || slots) {
                    if (!any) {
                        op.clear();
                        encode(op, cd.SHEARS, shear_mask, 0, 0, slots, nslot);
                    }
                    emit(op, 0, 0);
                    n_out++;
                }
            }
            if (pending) tab_.clear();
            pending = false;
            wgd.clear();
            wg_bits = 0;
        };
        // a NEG / PHASE with one workgroup-bit condition, folded into the pending table
        // where the copies that a new bit makes fit the bytes of prog_bound
        auto fold_wg = [&](const dq_op &o, double fr, double fi) {
            if (o.c_thr || __builtin_popcountll(o.c_wg) != 1) return false;
            const int nb = __builtin_popcountll(wg_bits | o.c_wg);
            if (nb > kWgFoldBits || ((32 + 16 + 2 * NR * ts) << nb) > kOpBytes * (from + 1)) return false;
            from++;
            wgd.push_back({o.c_wg, o.v_wg, o.c_reg, o.v_reg, fr, fi});
            wg_bits |= o.c_wg;
            pending = true;
            return true;
        };
        auto hold = [&](const dq_op &o) {
            if (!gather || !can_hold(o)) return false;
            held[o.c_reg ? 1 + 2 * __builtin_ctz(o.c_reg) + (o.v_reg ? 1 : 0) : 0].push_back(&o);
            return true;
        };
        bool fold_run = false;  // the current run of diagonal ops holds an unconditioned table
        bool in_run = false;
        for (uint32_t k = 0; k < count; k++) {
            const dq_op &o = ops[k];
            const unsigned char *m = reinterpret_cast<const unsigned char *>(o.m);
            if (is_diag(o) && !in_run) {
                fold_run = false;
                from = 0;
                double plain = 0.0;  // vector instructions of the run's unconditioned ops, each on its own
                for (uint32_t k2 = k; k2 < count && is_diag(ops[k2]); k2 += ops[k2].kind == DQ_OP_DIAGR ? 1 + ops[k2].tbit : 1) {
                    const dq_op &d = ops[k2];
                    if (!d.c_thr && !d.c_wg) from += d.kind == DQ_OP_DIAGR ? 1 + d.tbit : 1;
                    if (d.kind == DQ_OP_DIAGR) fold_run |= !d.c_wg;
                    else if (!d.c_thr && !d.c_wg) plain += (d.kind == DQ_OP_NEG ? 2.0 : 4.0) * (NR >> __builtin_popcount(d.c_reg));
                }
                if (gather && plain > 4.0 * NR) fold_run = true;  // a table of their own takes less
            }
            in_run = is_diag(o);
            if (!in_run) emit_held(n_out);
            op.clear();
            switch (o.kind) {
                case DQ_OP_SHEAR: {
                    // merge the run of unconditioned shears on distinct bits
                    unsigned char slots[2 * DQ_MAX_REG_BITS * 8] = {};
                    uint32_t mask = 0;
                    uint32_t k2 = k;
                    while (k2 < count && ops[k2].kind == DQ_OP_SHEAR && !ops[k2].c_wg && !((mask >> ops[k2].tbit) & 1)) {
                        mask |= 1u << ops[k2].tbit;
                        memcpy(slots + 2 * ops[k2].tbit * ts, ops[k2].m, 2 * ts);
                        k2++;
                    }
                    if (k2 == k) {  // a shear with a workgroup condition: on its own
                        flush(nullptr, 0);
                        op.clear();
                        mask = 1u << o.tbit;
                        memcpy(slots + 2 * o.tbit * ts, o.m, 2 * ts);
                        encode(op, cd.SHEARS, mask, 0, 0, slots, nslot);
                        emit(op, o.c_wg, o.v_wg);
                        n_out++;
                        continue;
                    }
                    flush(slots, mask);
                    k = k2 - 1;
                    continue;
                }
                case DQ_OP_DIAGR: {
                    if (!o.c_wg) {
                        for (int e = 0; e < NR; e++) {
                            const dq_op &d = ops[k + 1 + e / 4];
                            tab_.mul(e, val(d, 2 * (e % 4)), val(d, 2 * (e % 4) + 1));
                        }
                        pending = true;
                    } else {  // a table under a workgroup condition: its own op (it commutes with the pending one)
                        Diag w;
                        for (int e = 0; e < NR; e++) {
                            const dq_op &d = ops[k + 1 + e / 4];
                            w.re[e] = val(d, 2 * (e % 4));
                            w.im[e] = val(d, 2 * (e % 4) + 1);
                        }
                        if (encode_table(op, w, nullptr, 0)) {
                            emit(op, o.c_wg, o.v_wg);
                            n_out++;
                        }
                    }
                    k += o.tbit;
                    continue;
                }
                case DQ_OP_NEG:
                    if (fold_run && !o.c_thr && !o.c_wg) {
                        tab_.mul_cond(NR, o.c_reg, o.v_reg, -1.0, 0.0);
                        pending = true;
                        continue;
                    }
                    if (fold_run && o.c_wg && fold_wg(o, -1.0, 0.0)) continue;
                    if (hold(o)) continue;
                    emit_single(o);
                    n_out++;
                    continue;
                case DQ_OP_PHASE:
                    if (fold_run && !o.c_thr && !o.c_wg) {
                        tab_.mul_cond(NR, o.c_reg, o.v_reg, val(o, 0), val(o, 1));
                        pending = true;
                        continue;
                    }
                    if (fold_run && o.c_wg && fold_wg(o, val(o, 0), val(o, 1))) continue;
                    if (hold(o)) continue;
                    emit_single(o);
                    n_out++;
                    continue;
                case DQ_OP_MAT:
                    flush(nullptr, 0);
                    op.clear();
                    encode(op, cd.MAT[o.tbit], jmask(o.c_reg, o.v_reg, (int)o.tbit), o.c_thr, o.v_thr, m, 8 * ts);
                    break;
                case DQ_OP_SWAP:
                    flush(nullptr, 0);
                    op.clear();
                    encode(op, cd.SWAP[o.tbit], jmask(o.c_reg, o.v_reg, (int)o.tbit), o.c_thr, o.v_thr, nullptr, 0);
                    break;
                case DQ_OP_RMAT:
                    flush(nullptr, 0);
                    op.clear();
                    encode(op, cd.RMAT[o.tbit], 0, 0, 0, m, 4 * ts);
                    break;
                default:
                    continue;
            }
            emit(op, o.c_wg, o.v_wg);
            n_out++;
        }
        emit_held(n_out);
        flush(nullptr, 0);
        op.clear();
        encode(op, cd.END, 0, 0, 0, nullptr, 0);
        out.insert(out.end(), op.begin(), op.end());
    }
    // Walk a built program: every code in range, sizes chaining to END at the
    // end of the buffer (the interpreter jumps through a table on the code).
    bool check(size_t begin) const {
        size_t at = begin;
        while (at + 16 <= out.size()) {
            uint32_t c;
            memcpy(&c, out.data() + at, 4);
            if (c >= (uint32_t)ncodes) return false;
            if (c == (uint32_t)cd.END) return at + size(c) == out.size();
            if (c >= (uint32_t)cd.FM_ALL) return false;  // reached through a FAN's header only
            uint32_t fan[4];
            memcpy(fan, out.data() + at, 16);
            if (c == (uint32_t)cd.FAN) {  // whole terms, the last one marked: the handler's loop ends there
                const size_t tb = kFanTerm;
                if (fan[1] < (uint32_t)cd.FM_ALL || fan[1] >= (uint32_t)ncodes || fan[3] <= 16 || (fan[3] - 16) % tb ||
                    at + fan[3] > out.size())
                    return false;
                uint32_t last;
                memcpy(&last, out.data() + at + fan[3] - tb + 4, 4);
                if (!(last & 0x400u)) return false;
                at += fan[3];
            } else {
                at += size(c);
            }
        }
        return false;
    }
};
}  // namespace

static int build_program(int prec, int reg_bits, const dq_op *ops, uint32_t n_ops, unsigned char *out, size_t cap, size_t *len,
                         bool gather) {
    if ((prec != DQ_F32 && prec != DQ_F64) || reg_bits < 1 || reg_bits > DQ_MAX_REG_BITS || !len || (n_ops && !ops))
        return fail(DQ_ERR_ARG, "dq_build_program: bad arguments");
    std::vector<unsigned char> prog;
    ProgBuilder pb(prec, reg_bits, prog, gather);
    uint32_t n_out = 0;
    pb.build(ops, n_ops, n_out);
    if (pb.bad || !pb.check(0)) return fail(DQ_ERR_ARG, "dq_build_program: op not expressible as a device op");
    *len = prog.size();
    if (out) {
        if (cap < prog.size()) return fail(DQ_ERR_ARG, "dq_build_program: %zu bytes needed", prog.size());
        memcpy(out, prog.data(), prog.size());
    }
    return DQ_OK;
}

// The device program of one phase's ops, built on the host (no GPU needed): lets
// the program encoding be checked against the op semantics on any host.
extern "C" int dq_build_program(int prec, int reg_bits, const dq_op *ops, uint32_t n_ops, unsigned char *out,
                                size_t cap, size_t *len) {
    return build_program(prec, reg_bits, ops, n_ops, out, cap, len, false);
}

extern "C" int dq_build_program_gathered(int prec, int reg_bits, const dq_op *ops, uint32_t n_ops, unsigned char *out,
                                         size_t cap, size_t *len) {
    return build_program(prec, reg_bits, ops, n_ops, out, cap, len, true);
}

extern "C" int dq_init_state(void *state, int n, int prec, int kind, uint64_t index, double value, void *stream) {
    if (!state || n < 1 || n > 40 || (prec != DQ_F32 && prec != DQ_F64)) return fail(DQ_ERR_ARG, "dq_init_state: bad arguments");
    if (kind != DQ_INIT_CLASSICAL && kind != DQ_INIT_PLUS) return fail(DQ_ERR_ARG, "dq_init_state: bad kind %d", kind);
    const uint64_t N = 1ull << n;
    const uint64_t want = (N + 255) / 256;
    const unsigned blocks = (unsigned)(want < (1ull << 20) ? want : (1ull << 20));
    if (prec == DQ_F64)
        hipLaunchKernelGGL(fill_kernel<double>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (V2<double>::type *)state, N, kind, index, value);
    else
        hipLaunchKernelGGL(fill_kernel<float>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (V2<float>::type *)state, N, kind, index, value);
    HIPC(hipGetLastError());
    return DQ_OK;
}

static bool onehot64(uint64_t x) { return x && !(x & (x - 1)); }

// Host-side check of every descriptor against the grid and buffers it
// implies: each workgroup reads and writes exactly the 2^T amplitudes of its
// own tile, every LDS index is below 2^T, every op index is in range.
static int validate_block(const dq_block &b, const dq_phase *phases, uint32_t n_phases, const dq_op *ops, uint32_t n_ops) {
    const int n = (int)b.n_qubits;
    if (n < 1 || n > 40) return fail(DQ_ERR_ARG, "block: n_qubits %d out of range", n);
    if (b.phase_count < 1 || b.phase_begin >= n_phases || b.phase_count > n_phases - b.phase_begin)
        return fail(DQ_ERR_ARG, "block: phase range out of bounds");
    for (uint32_t p = 0; p < b.phase_count; p++) {
        const dq_phase &ph = phases[b.phase_begin + p];
        if (ph.op_begin > n_ops || ph.op_count > n_ops - ph.op_begin) return fail(DQ_ERR_ARG, "phase: op range out of bounds");
        for (uint32_t k = 0; k < ph.op_count; k++) {
            const dq_op &o = ops[ph.op_begin + k];
            if (o.c_thr > 0xFFFFu || o.v_thr > 0xFFFFu || (o.v_thr & ~o.c_thr) || (o.v_reg & ~o.c_reg) ||
                (o.v_wg & ~o.c_wg))
                return fail(DQ_ERR_ARG, "op: condition values outside their masks");
            if ((o.kind == DQ_OP_SHEAR || o.kind == DQ_OP_RMAT || o.kind == DQ_OP_DIAGR) && (o.c_reg || o.c_thr))
                return fail(DQ_ERR_ARG, "op: kind %u takes no register or lane condition", o.kind);
            if (o.kind == DQ_OP_DIAGR) {
                if (b.reg_bits == 0 || o.tbit != ((1u << b.reg_bits) + 3) / 4 || k + o.tbit >= ph.op_count)
                    return fail(DQ_ERR_ARG, "phase: register-diagonal table out of bounds");
                k += o.tbit;
            } else if (o.kind == DQ_OP_MAT || o.kind == DQ_OP_SWAP || o.kind == DQ_OP_RMAT || o.kind == DQ_OP_SHEAR) {
                if (b.reg_bits ? o.tbit >= b.reg_bits : o.tbit >= b.n_qubits)
                    return fail(DQ_ERR_ARG, "op: target bit %u out of range", o.tbit);
            } else if (o.kind != DQ_OP_NEG && o.kind != DQ_OP_PHASE) {
                return fail(DQ_ERR_ARG, "op: unknown kind %u", o.kind);
            }
        }
    }
    if (b.reg_bits == 0) {  // small-state form
        if ((int)b.tile_bits != n || n > 13) return fail(DQ_ERR_ARG, "small block: tile_bits must equal n <= 13");
        return DQ_OK;
    }
    const int T = (int)b.tile_bits, R = (int)b.reg_bits, W = (int)b.wave_bits;
    if (R > DQ_MAX_REG_BITS || W > DQ_MAX_WAVE_BITS || T != 6 + R + W || T > n || T > DQ_MAX_TILE_BITS)
        return fail(DQ_ERR_ARG, "block: tile shape T=%d R=%d W=%d n=%d", T, R, W, n);
    const uint64_t full = (1ull << n) - 1;
    for (int end = 0; end < 2; end++) {
        const uint64_t *rg = end ? b.st_reg : b.ld_reg;
        const uint64_t *wv = end ? b.st_wave : b.ld_wave;
        uint64_t m = 0x3Full;
        int cnt = 6;
        for (int r = 0; r < R; r++) { if (!onehot64(rg[r])) return fail(DQ_ERR_ARG, "block: register mask not one-hot"); m |= rg[r]; cnt++; }
        for (int w = 0; w < W; w++) { if (!onehot64(wv[w])) return fail(DQ_ERR_ARG, "block: wave mask not one-hot"); m |= wv[w]; cnt++; }
        if (__builtin_popcountll(m) != cnt || (m & b.nontile_mask) || ((m | b.nontile_mask) != full))
            return fail(DQ_ERR_ARG, "block: tile and non-tile qubit masks inconsistent");
    }
    for (uint32_t p = 0; p < b.phase_count; p++) {
        const dq_phase &ph = phases[b.phase_begin + p];
        uint32_t m = 0;
        int cnt = 0;
        auto add = [&](uint32_t x) { m |= x; cnt++; return x && !(x & (x - 1)) && x < (1u << T); };
        bool ok = true;
        for (int r = 0; r < R; r++) ok &= add(ph.reg_t[r]);
        for (int w = 0; w < W; w++) ok &= add(ph.wave_t[w]);
        for (int l = 0; l < 6; l++) ok &= add(ph.lane_t[l]);
        if (!ok || m != (1u << T) - 1 || __builtin_popcount(m) != cnt)
            return fail(DQ_ERR_ARG, "phase %u: layout is not a permutation of the tile bits", p);
    }
    return DQ_OK;
}

static int apply_blocks(int prec, const dq_block *blocks, uint32_t n_blocks, const dq_phase *phases, uint32_t n_phases,
                        const dq_op *ops, uint32_t n_ops, const dq_job *jobs, const uint32_t *job_begin, uint32_t n_launch,
                        double *part, void *d_ws, size_t ws_bytes, void *stream) {
    if (prec != DQ_F32 && prec != DQ_F64) return fail(DQ_ERR_ARG, "dq_apply_blocks: bad precision %d", prec);
    if (n_launch == 0) return DQ_OK;
    if (!blocks || !phases || !jobs || !job_begin || !d_ws) return fail(DQ_ERR_ARG, "dq_apply_blocks: null argument");
    const uint32_t n_jobs = job_begin[n_launch];
    const size_t need = dq_apply_ws_bytes(n_blocks, n_phases, n_ops, n_jobs);
    if (need > ws_bytes) return fail(DQ_ERR_ARG, "dq_apply_blocks: workspace %zu < %zu bytes", ws_bytes, need);
    for (uint32_t i = 0; i < n_blocks; i++) {
        int rc = validate_block(blocks[i], phases, n_phases, ops, n_ops);
        if (rc) return rc;
    }
    for (uint32_t j = 0; j < n_jobs; j++)
        if (jobs[j].block >= n_blocks || !jobs[j].state) return fail(DQ_ERR_ARG, "job %u: bad block or state", j);
    for (uint32_t j = 0; j < n_jobs; j++)
        if (jobs[j].base_hi & ((1ull << blocks[jobs[j].block].n_qubits) - 1))
            return fail(DQ_ERR_ARG, "job %u: base_hi overlaps the piece's own qubits", j);
    for (uint32_t l = 0; l < n_launch; l++) {
        if (job_begin[l + 1] <= job_begin[l]) return fail(DQ_ERR_ARG, "launch %u: empty job range", l);
        const dq_block &b0 = blocks[jobs[job_begin[l]].block];
        for (uint32_t j = job_begin[l]; j < job_begin[l + 1]; j++) {
            const dq_block &b = blocks[jobs[j].block];
            if (b.n_qubits != b0.n_qubits || b.reg_bits != b0.reg_bits || b.wave_bits != b0.wave_bits || b.tile_bits != b0.tile_bits)
                return fail(DQ_ERR_ARG, "launch %u: jobs differ in shape", l);
        }
        if (b0.reg_bits && !lookup(prec, b0.reg_bits, b0.wave_bits,
                                   exchange_mode(prec, (int)b0.reg_bits, (int)b0.wave_bits, (int)b0.tile_bits)))
            return fail(DQ_ERR_UNSUPPORTED, "no sweep kernel for R=%d W=%d", b0.reg_bits, b0.wave_bits);
    }

    // per phase of a sweep block: its device program and exchange offsets
    // (phase_aux); per block: the runs of its non-tile qubits (block_aux)
    std::vector<uint32_t> paux((size_t)n_phases * DQ_PAUX, 0), baux((size_t)n_blocks * DQ_BAUX, 0);
    std::vector<int> prog_r(n_phases, -1);
    std::vector<uint32_t> prog_es(n_phases, 0);
    std::vector<unsigned char> prog;
    for (uint32_t i = 0; i < n_blocks; i++) {
        const dq_block &b = blocks[i];
        if (b.reg_bits == 0) continue;
        if (!block_runs(b, baux.data() + (size_t)i * DQ_BAUX))
            return fail(DQ_ERR_UNSUPPORTED, "block %u: non-tile qubits in more than %d runs", i, DQ_RUNS);
        const int bxm = exchange_mode(prec, (int)b.reg_bits, (int)b.wave_bits, (int)b.tile_bits);
        const uint32_t es = exchange_elem_bytes(prec, bxm);
        uint32_t *ba = baux.data() + (size_t)i * DQ_BAUX;
        ba[DQ_BA_PROG] = (uint32_t)prog.size();
        uint32_t gown[32];
        if (bxm == 1) {
            if (b.tile_bits != 6 + b.wave_bits + b.reg_bits)
                return fail(DQ_ERR_ARG, "block %u: tile of %u bits is not 6 + %u + %u", i, b.tile_bits, b.wave_bits, b.reg_bits);
            const int Lo = es == 4 ? 5 : (es == 8 ? 4 : 3);
            pick_owned_swizzle(phases + b.phase_begin, b.phase_count, (int)b.reg_bits, (int)b.wave_bits, Lo, gown);
        }
        for (uint32_t p = b.phase_begin; p < b.phase_begin + b.phase_count; p++) {
            uint32_t *pa = paux.data() + (size_t)p * DQ_PAUX;
            if (prog_r[p] != (int)b.reg_bits || prog_es[p] != es) {
                if (prog_r[p] >= 0) return fail(DQ_ERR_ARG, "phase %u shared by blocks of different tile shapes", p);
                prog_r[p] = (int)b.reg_bits;
                prog_es[p] = es;
                pa[0] = (uint32_t)prog.size();
                ProgBuilder pb(prec, (int)b.reg_bits, prog);
                const size_t start = prog.size();
                pb.build(ops + phases[p].op_begin, phases[p].op_count, pa[1]);
                if (pb.bad || !pb.check(start)) return fail(DQ_ERR_ARG, "phase %u: op not expressible as a device op", p);
            }
            if (p == b.phase_begin) continue;  // no exchange into a block's first phase
            // the exchange from phase p - 1: its swizzle and offset tables
            const dq_phase &A = phases[p - 1], &B = phases[p];
            const int L = es == 4 ? 5 : (es == 8 ? 4 : 3);
            if (bxm == 1) {
                uint32_t t[DQ_PAUX];
                memcpy(t, pa, sizeof t);
                if (!owned_tables(A, B, (int)b.reg_bits, (int)b.wave_bits, L, gown, es, t))
                    return fail(DQ_ERR_ARG, "phase %u: layouts of the exchange do not place the same tile bits", p);
                // a phase shared with an earlier block must get the same tables
                bool filled = false;
                for (int k = 2; k < DQ_PAUX; k++) filled |= pa[k] != 0;
                if (filled && memcmp(t + 2, pa + 2, (DQ_PAUX - 2) * sizeof(uint32_t)))
                    return fail(DQ_ERR_ARG, "phase %u: shared by blocks with different exchange slots", p);
                memcpy(pa, t, sizeof t);
                continue;
            }
            uint32_t g[32];
            pick_swizzle(A, B, L, g);
            for (uint32_t j = 0; j < (1u << b.reg_bits); j++) {
                uint32_t xa = 0, xb = 0;
                for (uint32_t r = 0; r < b.reg_bits; r++)
                    if ((j >> r) & 1) {
                        xa ^= swizzle_host(A.reg_t[r], g, L) * es;
                        xb ^= swizzle_host(B.reg_t[r], g, L) * es;
                    }
                pa[DQ_XA + j] = xa;
                pa[DQ_XB + j] = xb;
            }
            for (int l = 0; l < 6; l++) {
                pa[DQ_TA + l] = swizzle_host(A.lane_t[l], g, L) * es;
                pa[DQ_TB + l] = swizzle_host(B.lane_t[l], g, L) * es;
            }
            for (uint32_t w = 0; w < b.wave_bits; w++) {
                pa[DQ_TA + 6 + w] = swizzle_host(A.wave_t[w], g, L) * es;
                pa[DQ_TB + 6 + w] = swizzle_host(B.wave_t[w], g, L) * es;
            }
        }
        ba[DQ_BA_PROG + 1] = (uint32_t)prog.size() - ba[DQ_BA_PROG];  // 0 when the phases are an earlier block's
    }
    if (prog.size() + 256 > prog_bound(n_phases, n_ops)) return fail(DQ_ERR_ARG, "dq_apply_blocks: device program overflow");

    // pack and upload what the kernels read: the sweep kernels run the device
    // programs, only small_kernel reads op descriptors
    bool small = false;
    for (uint32_t i = 0; i < n_blocks; i++) small |= blocks[i].reg_bits == 0;
    const uint32_t up_ops = small ? n_ops : 0;
    size_t off_b = 0, off_p = align_up(n_blocks * sizeof(dq_block), 256);
    size_t off_o = off_p + align_up(n_phases * sizeof(dq_phase), 256);
    size_t off_j = off_o + align_up(up_ops * sizeof(dq_op), 256);
    size_t off_pa = off_j + align_up(n_jobs * sizeof(dq_job), 256);
    size_t off_ba = off_pa + align_up((size_t)n_phases * DQ_PAUX * sizeof(uint32_t), 256);
    size_t off_pg = off_ba + align_up((size_t)n_blocks * DQ_BAUX * sizeof(uint32_t), 256);
    std::vector<unsigned char> buf(align_up(off_pg + prog.size() + 256, 16), 0);  // + the interpreter's read-ahead
    memcpy(buf.data() + off_b, blocks, n_blocks * sizeof(dq_block));
    memcpy(buf.data() + off_p, phases, n_phases * sizeof(dq_phase));
    if (up_ops) memcpy(buf.data() + off_o, ops, up_ops * sizeof(dq_op));
    memcpy(buf.data() + off_j, jobs, n_jobs * sizeof(dq_job));
    if (n_phases) memcpy(buf.data() + off_pa, paux.data(), paux.size() * sizeof(uint32_t));
    memcpy(buf.data() + off_ba, baux.data(), baux.size() * sizeof(uint32_t));
    if (!prog.empty()) memcpy(buf.data() + off_pg, prog.data(), prog.size());
    // one sweep of one tile: its workgroup brings them itself
    bool own = n_launch == 1 && n_jobs == 1 && buf.size() <= kStageKernelBytes && (uintptr_t)d_ws % 16 == 0;
    if (own) {
        const dq_block &b = blocks[jobs[0].block];
        own = b.reg_bits && b.n_qubits == b.tile_bits &&
              lookup(prec, b.reg_bits, b.wave_bits, exchange_mode(prec, (int)b.reg_bits, (int)b.wave_bits, (int)b.tile_bits), true);
    }
    StageSlot *slot = nullptr;
    int rc = own ? stage_fill(buf, slot, stream) : stage_upload(d_ws, buf, stream);
    if (rc) return rc;
    struct Undo {
        StageSlot *slot;
        ~Undo() { if (slot) stage_undo(slot); }
    } undo{slot};
    unsigned char *d = (unsigned char *)d_ws;
    const dq_block *d_blocks = (const dq_block *)(d + off_b);
    const dq_phase *d_phases = (const dq_phase *)(d + off_p);
    const dq_op *d_ops = (const dq_op *)(d + off_o);
    const dq_job *d_jobs = (const dq_job *)(d + off_j);
    const uint32_t *d_paux = (const uint32_t *)(d + off_pa);
    const uint32_t *d_baux = (const uint32_t *)(d + off_ba);
    const unsigned char *d_prog = d + off_pg;

    for (uint32_t l = 0; l < n_launch; l++) {
        const uint32_t j0 = job_begin[l], nj = job_begin[l + 1] - j0;
        const dq_block &b0 = blocks[jobs[j0].block];
        const int n = b0.n_qubits;
        if (b0.reg_bits == 0) {
            const size_t lds = ((size_t)1 << n) * elem_bytes(prec);
            if (prec == DQ_F64)
                hipLaunchKernelGGL(small_kernel<double>, dim3(1, nj), dim3(256), lds, (hipStream_t)stream, d_jobs + j0, d_blocks, d_phases, d_ops);
            else
                hipLaunchKernelGGL(small_kernel<float>, dim3(1, nj), dim3(256), lds, (hipStream_t)stream, d_jobs + j0, d_blocks, d_phases, d_ops);
        } else {
            bool multi = false;
            for (uint32_t j = j0; j < j0 + nj; j++) multi |= blocks[jobs[j].block].phase_count > 1;
            const int xm = exchange_mode(prec, (int)b0.reg_bits, (int)b0.wave_bits, (int)b0.tile_bits);
            size_t lds = multi ? ((size_t)1 << b0.tile_bits) * exchange_elem_bytes(prec, xm) : 0;
            const bool sums = part && l == n_launch - 1;
            if (sums) lds = std::max(lds, ((size_t)(1 + b0.reg_bits) * 64 * sizeof(double)) << b0.wave_bits);
            if (lds > 131072) return fail(DQ_ERR_UNSUPPORTED, "tile of %d bits needs %zu bytes of LDS", b0.tile_bits, lds);
            const uint64_t tiles = 1ull << (n - b0.tile_bits);
            if (tiles > 0x7fffffffull || nj > 65535 || ((tiles << (6 + b0.wave_bits)) >> 32))
                return fail(DQ_ERR_UNSUPPORTED, "grid too large (at most 2^32 threads per launch)");
            sweep_fn fn = lookup(prec, b0.reg_bits, b0.wave_bits, xm, slot != nullptr);
            if (!fn) return fail(DQ_ERR_UNSUPPORTED, "no sweep kernel for R=%u W=%u exchange mode %d", b0.reg_bits, b0.wave_bits, xm);
            SweepOne one;
            one.blk = b0;
            memcpy(one.baux, baux.data() + (size_t)jobs[j0].block * DQ_BAUX, sizeof one.baux);
            one.job = jobs[j0];
            one.part = sums ? part : nullptr;
            one.src = slot ? (const uint4 *)((unsigned char *)slot->host + kStageHeader) : nullptr;
            one.dst = (uint4 *)d_ws;
            one.read = slot ? (uint32_t *)slot->host : nullptr;
            one.n16 = (uint32_t)(buf.size() / 16);
            one.ticket = slot ? slot->ticket : 0;
            HIPC(launch(fn, dim3((unsigned)tiles, nj), dim3(64u << b0.wave_bits), lds, stream, one, d_jobs + j0, d_blocks, d_phases,
                        d_prog, d_paux, d_baux));
            undo.slot = nullptr;  // the kernel reads it
        }
        HIPC(hipGetLastError());
    }
    return DQ_OK;
}

extern "C" int dq_apply_blocks(int prec, const dq_block *blocks, uint32_t n_blocks, const dq_phase *phases,
                               uint32_t n_phases, const dq_op *ops, uint32_t n_ops, const dq_job *jobs,
                               const uint32_t *job_begin, uint32_t n_launch, void *d_ws, size_t ws_bytes, void *stream) {
    return apply_blocks(prec, blocks, n_blocks, phases, n_phases, ops, n_ops, jobs, job_begin, n_launch, nullptr, d_ws, ws_bytes, stream);
}

// ---- P(0) of every qubit from the sums of the last sweep -------------------------
// Up to kPartHost tiles write their sums to a result slot and the host adds them up: a
// launch less (4-5 us).  From kPartMax tiles on (their sums take 16 MiB) the state
// is read again.
constexpr uint32_t kPartHost = 32, kPartMax = 1u << 17;

extern "C" size_t dq_block_sums_bytes(const dq_block *b) {
    if (!b || b->reg_bits == 0 || b->n_qubits > PROB_MAX_QUBITS || b->tile_bits > b->n_qubits) return 0;
    const uint32_t log = b->n_qubits - b->tile_bits;
    if (log >= 32 || (1u << log) > kPartMax) return 0;
    return ((size_t)(b->tile_bits + 1) << log) * sizeof(double);
}

extern "C" int dq_block_sums_on_host(const dq_block *b) {
    return dq_block_sums_bytes(b) && (1u << (b->n_qubits - b->tile_bits)) <= kPartHost;
}

extern "C" int dq_apply_blocks_sums(int prec, const dq_block *blocks, uint32_t n_blocks, const dq_phase *phases,
                                    uint32_t n_phases, const dq_op *ops, uint32_t n_ops, const dq_job *jobs,
                                    const uint32_t *job_begin, uint32_t n_launch, double *sums, size_t sums_bytes, void *d_ws,
                                    size_t ws_bytes, void *stream) {
    if (!blocks || !jobs || !job_begin || !sums || n_launch == 0) return fail(DQ_ERR_ARG, "dq_apply_blocks_sums: null argument");
    const dq_job &last = jobs[job_begin[n_launch - 1]];
    if (job_begin[n_launch] - job_begin[n_launch - 1] != 1 || last.block >= n_blocks)
        return fail(DQ_ERR_ARG, "dq_apply_blocks_sums: the last launch must have one job");
    const size_t need = dq_block_sums_bytes(blocks + last.block);
    if (!need || sums_bytes < need) return fail(DQ_ERR_ARG, "dq_apply_blocks_sums: sums of %zu bytes", sums_bytes);
    return apply_blocks(prec, blocks, n_blocks, phases, n_phases, ops, n_ops, jobs, job_begin, n_launch, sums, d_ws, ws_bytes, stream);
}

// prob_stage2 on the host.
static void prob_add(const double *part, uint32_t groups, int n, int cb, const ProbOut &po, double *out) {
    for (int q = 0; q <= n; q++) {
        const int bit = q == n ? PROB_FIXED0 : po.bit[q];
        const double *src = part + (size_t)std::min(bit, cb) * groups;
        const uint32_t skip = bit >= cb && bit < PROB_FIXED0 ? 1u << (bit - cb) : 0u;
        double a = 0.0;
        for (uint32_t g = 0; g < groups; g++)
            if (!(g & skip)) a += src[g];
        out[q] = bit == PROB_FIXED1 ? 0.0 : po.scale * a;
    }
}

extern "C" int dq_prob_of_sums(const dq_block *b, const double *sums, double *out, double *d_out, void *stream) {
    const size_t bytes = dq_block_sums_bytes(b);
    if (!bytes || !sums || !out) return fail(DQ_ERR_ARG, "dq_prob_of_sums: bad arguments");
    const int n = (int)b->n_qubits, T = (int)b->tile_bits;
    const uint32_t groups = 1u << (n - T);
    ProbOut po;
    memset(&po, 0, sizeof po);
    po.scale = 1.0;
    int outside = T;
    for (int q = 0; q < n; q++) {
        const uint64_t m = 1ull << q;
        int bit = q < 6 ? q : -1;
        for (uint32_t r = 0; r < b->reg_bits; r++)
            if (b->st_reg[r] == m) bit = 6 + (int)r;
        for (uint32_t w = 0; w < b->wave_bits; w++)
            if (b->st_wave[w] == m) bit = 6 + (int)(b->reg_bits + w);
        if (b->nontile_mask & m) bit = outside++;
        if (bit < 0) return fail(DQ_ERR_ARG, "dq_prob_of_sums: qubit %d is in no place", q);
        po.bit[q] = (uint8_t)bit;
    }
    if (dq_block_sums_on_host(b)) {
        std::vector<double> v(bytes / sizeof(double));
        const int rc = dq_result_wait(sums, v.data(), bytes, stream);
        if (rc) return rc;
        prob_add(v.data(), groups, n, T, po, out);
        return DQ_OK;
    }
    if (!d_out) return fail(DQ_ERR_ARG, "dq_prob_of_sums: null output");
    ResultSlot res((n + 1) * sizeof(double), d_out, stream);
    hipStream_t s = (hipStream_t)stream;
    if (groups > 8192) hipLaunchKernelGGL(prob_stage2<1024>, dim3(n + 1), dim3(1024), 0, s, sums, groups, n, T, po, (double *)res.dst);
    else hipLaunchKernelGGL(prob_stage2<256>, dim3(n + 1), dim3(256), 0, s, sums, groups, n, T, po, (double *)res.dst);
    HIPC(hipGetLastError());
    return res.collect(out, (n + 1) * sizeof(double));
}

// Split of 2^nf amplitudes over prob_stage1's workgroups: cb bits each, 2^JB
// loads in flight per thread.  Small states spread over up to 256 workgroups
// (one per CU) before a thread takes a second amplitude; from 2^20 amplitudes
// a thread has 16 loads in flight and workgroups are added up to 2^PROB_GROUPS,
// from where the loop inside a workgroup grows.
#define PROB_GROUPS 13
constexpr int kProbHostBits = 18;
struct ProbSplit {
    int cb, jb;
    uint32_t groups;
};
static ProbSplit prob_split(int nf) {
    ProbSplit p;
    p.jb = nf <= 16 ? 0 : std::min(nf - 16, 4);
    int outer = nf - 8 - p.jb - PROB_GROUPS;
    outer = std::max(0, std::min(outer, PROB_OUTER));
    p.cb = std::min(nf, 8 + p.jb + outer);
    p.groups = 1u << (nf - p.cb);
    return p;
}

// bytes of per-workgroup partial sums of prob_stage1
static size_t prob_part_bytes(int nf) {
    const ProbSplit p = prob_split(nf);
    return align_up((size_t)p.groups * (p.cb + 1) * sizeof(double), 256);
}

extern "C" size_t dq_prob_ws_bytes(int n) { return prob_part_bytes(n) + 64 * sizeof(double); }

// The number bits of a state's free qubits and what stage 2 makes of every qubit.
static int prob_bits(int n, uint64_t fixed_mask, uint64_t fixed_value, double scale, ProbBits &pb, ProbOut &po) {
    memset(&pb, 0, sizeof pb);
    memset(&po, 0, sizeof po);
    pb.fixed = fixed_value;
    po.scale = scale;
    int f = 0;
    for (int q = 0; q < n; q++) {
        const uint64_t b = 1ull << q;
        if (fixed_mask & b) {
            po.bit[q] = (fixed_value & b) ? PROB_FIXED1 : PROB_FIXED0;
        } else {
            po.bit[q] = (uint8_t)f;
            pb.img[f++] = b;
        }
    }
    return f;
}

static int prob_sums(const void *state, int prec, const ProbBits &pb, int nf, const ProbSplit &p, double *part, hipStream_t stream) {
#define DQ_PROB1(T_, JB_)                                                                          \
    hipLaunchKernelGGL((prob_stage1<T_, JB_>), dim3(p.groups), dim3(256), 0, stream, (const V2<T_>::type *)state, pb, nf, \
                       p.cb, part)
#define DQ_PROB1J(T_)                          \
    switch (p.jb) {                            \
        case 0: DQ_PROB1(T_, 0); break;        \
        case 1: DQ_PROB1(T_, 1); break;        \
        case 2: DQ_PROB1(T_, 2); break;        \
        case 3: DQ_PROB1(T_, 3); break;        \
        default: DQ_PROB1(T_, 4); break;       \
    }
    if (prec == DQ_F64) {
        DQ_PROB1J(double)
    } else {
        DQ_PROB1J(float)
    }
#undef DQ_PROB1J
#undef DQ_PROB1
    HIPC(hipGetLastError());
    return DQ_OK;
}

static int prob_launch(const void *state, int n, int prec, uint64_t fixed_mask, uint64_t fixed_value, double scale,
                       double *d_out, void *d_ws, size_t ws_bytes, hipStream_t stream) {
    if (!state || !d_out || !d_ws || n < 1 || n > PROB_MAX_QUBITS || (prec != DQ_F32 && prec != DQ_F64))
        return fail(DQ_ERR_ARG, "dq_prob_zero_all: bad arguments");
    if ((fixed_mask >> n) || (fixed_value & ~fixed_mask)) return fail(DQ_ERR_ARG, "dq_prob_zero_all: bad fixed bits");
    ProbBits pb;
    ProbOut po;
    const int nf = prob_bits(n, fixed_mask, fixed_value, scale, pb, po);
    if (ws_bytes < prob_part_bytes(nf)) return fail(DQ_ERR_ARG, "dq_prob_zero_all_async: workspace too small");
    const ProbSplit p = prob_split(nf);
    // One launch where a workgroup's 8 loads per thread cover the state: the second
    // launch takes longer (3.5 us) than what more workgroups would save.
    if (nf <= PROB_ONE_BITS) {
        if (prec == DQ_F64)
            hipLaunchKernelGGL(prob_one<double>, dim3(1), dim3(1024), 0, stream, (const V2<double>::type *)state, pb, nf, n, po, d_out);
        else
            hipLaunchKernelGGL(prob_one<float>, dim3(1), dim3(1024), 0, stream, (const V2<float>::type *)state, pb, nf, n, po, d_out);
        HIPC(hipGetLastError());
        return DQ_OK;
    }
    double *part = (double *)d_ws;
    const int rc = prob_sums(state, prec, pb, nf, p, part, stream);
    if (rc) return rc;
    hipLaunchKernelGGL(prob_stage2<256>, dim3(n + 1), dim3(256), 0, stream, part, p.groups, n, p.cb, po, d_out);
    HIPC(hipGetLastError());
    return DQ_OK;
}

extern "C" int dq_prob_zero_all_async(const void *state, int n, int prec, double *d_out, void *d_ws, size_t ws_bytes, void *stream) {
    return prob_launch(state, n, prec, 0, 0, 1.0, d_out, d_ws, ws_bytes, (hipStream_t)stream);
}

extern "C" int dq_prob_zero_all_fixed(const void *state, int n, int prec, uint64_t fixed_mask, uint64_t fixed_value,
                                      double scale, double *out, void *d_ws, size_t ws_bytes, void *stream) {
    if (!out) return fail(DQ_ERR_ARG, "dq_prob_zero_all: null output");
    if (n < 1 || n > PROB_MAX_QUBITS) return fail(DQ_ERR_ARG, "dq_prob_zero_all: bad arguments");
    if (ws_bytes < dq_prob_ws_bytes(n)) return fail(DQ_ERR_ARG, "dq_prob_zero_all: workspace too small");
    const size_t part_bytes = prob_part_bytes(n);
    double *d_out = (double *)((unsigned char *)d_ws + part_bytes);
    if (!state || !d_ws || (prec != DQ_F32 && prec != DQ_F64)) return fail(DQ_ERR_ARG, "dq_prob_zero_all: bad arguments");
    if ((fixed_mask >> n) || (fixed_value & ~fixed_mask)) return fail(DQ_ERR_ARG, "dq_prob_zero_all: bad fixed bits");
    ProbBits pb;
    ProbOut po;
    const int nf = prob_bits(n, fixed_mask, fixed_value, scale, pb, po);
    if (fixed_mask && nf <= kProbHostBits) {
        // (Whole states are summed as dq_prob_zero_all_noalloc does, to the same bits.)  Up to 64 workgroups write their sums to a result slot and the host adds them up: no
        // second launch (4.5 us), and up to 2^13 amplitudes no single workgroup (4.8
        // against 7.6 us).  23 qubits measured one after another 603 -> 541 us.
        ProbSplit p;
        p.cb = std::min(nf, std::max(8, nf - 6));
        p.jb = std::max(0, p.cb - 8);
        p.groups = 1u << (nf - p.cb);
        const size_t bytes = (size_t)p.groups * (p.cb + 1) * sizeof(double);
        ResultSlot res(bytes, nullptr, stream);
        if (res.host) {
            int rc = prob_sums(state, prec, pb, nf, p, (double *)res.host, (hipStream_t)stream);
            std::vector<double> v(bytes / sizeof(double));
            if (!rc) rc = res.collect(v.data(), bytes);
            if (rc) return rc;
            prob_add(v.data(), p.groups, n, p.cb, po, out);
            return DQ_OK;
        }
    }
    ResultSlot res((n + 1) * sizeof(double), d_out, stream);
    const int rc = prob_launch(state, n, prec, fixed_mask, fixed_value, scale, (double *)res.dst, d_ws, part_bytes, (hipStream_t)stream);
    if (rc) return rc;
    return res.collect(out, (n + 1) * sizeof(double));
}

extern "C" int dq_prob_zero_all(const void *state, int n, int prec, double *out, void *d_ws, size_t ws_bytes, void *stream) {
    return dq_prob_zero_all_fixed(state, n, prec, 0, 0, 1.0, out, d_ws, ws_bytes, stream);
}

// ---- P(0) of every qubit without allocation or workspace --------------------
// For callers that may not allocate device memory (code under stream capture,
// serving loops): the partial sums live in a file-scope device array.  A
// state is reduced in chunks of at most 2^NA_CHUNK_BITS amplitudes, each by
// prob_stage1/prob_stage2 (for n <= NA_CHUNK_BITS exactly the launches of
// dq_prob_zero_all_async); prob_combine sums the chunks' results.  The
// array `scratch` (defined with the P(0) kernels) holds the partial sums of
// one chunk, then the results of every chunk.

// out[q] for q < n and the total out[n] from nchunks chunk results of
// NA_CHUNK_BITS + 1 doubles each (chunk c = amplitudes with index bits
// NA_CHUNK_BITS.. equal to c); one thread per output, chunks summed in order.
__global__ void __launch_bounds__(64) prob_combine(const double *__restrict__ chunks, uint32_t nchunks, int n,
                                                   double *__restrict__ out) {
    const int q = threadIdx.x;
    if (q > n) return;
    constexpr int S = NA_CHUNK_BITS + 1;
    double acc = 0.0;
    for (uint32_t c = 0; c < nchunks; c++) {
        if (q < NA_CHUNK_BITS) acc += chunks[(uint64_t)c * S + q];
        else if (q == n || !((c >> (q - NA_CHUNK_BITS)) & 1u)) acc += chunks[(uint64_t)c * S + NA_CHUNK_BITS];
    }
    out[q] = acc;
}

extern "C" int dq_prob_zero_all_noalloc(const void *state, int n, int prec, double *d_out, void *stream) {
    if (!state || !d_out || n < 1 || (prec != DQ_F32 && prec != DQ_F64))
        return fail(DQ_ERR_ARG, "dq_prob_zero_all_noalloc: bad arguments");
    if (n > NA_MAX_QUBITS)
        return fail(DQ_ERR_ARG, "dq_prob_zero_all_noalloc: %d qubits, above its limit of %d", n, NA_MAX_QUBITS);
    int dev = -1;
    HIPC(hipGetDevice(&dev));
    double *scr = (dev >= 0 && dev < kMaxDevices) ? g_scratch_dev[dev] : nullptr;
    if (!scr) return fail(DQ_ERR_ARG, "dq_prob_zero_all_noalloc: dq_device_init(%d) has not been called", dev);
    if (n <= NA_CHUNK_BITS)
        return dq_prob_zero_all_async(state, n, prec, d_out, scr, (size_t)NA_PART_DOUBLES * sizeof(double), stream);
    double *chunk_res = scr + NA_PART_DOUBLES;
    const uint32_t nchunks = 1u << (n - NA_CHUNK_BITS);
    const size_t amp_bytes = prec == DQ_F64 ? 16 : 8;
    for (uint32_t c = 0; c < nchunks; c++) {
        const void *piece = (const unsigned char *)state + ((size_t)c << NA_CHUNK_BITS) * amp_bytes;
        const int rc = dq_prob_zero_all_async(piece, NA_CHUNK_BITS, prec, chunk_res + (size_t)c * (NA_CHUNK_BITS + 1), scr,
                                              (size_t)NA_PART_DOUBLES * sizeof(double), stream);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(prob_combine, dim3(1), dim3(64), 0, (hipStream_t)stream, chunk_res, nchunks, n, d_out);
    HIPC(hipGetLastError());
    return DQ_OK;
}

// ---- read-out of many states ------------------------------------------------
namespace {
struct RoPlan {
    int gb = 0;
    uint64_t wgs = 0;  // stage-1 workgroups per state
    RoLevels lv;
    size_t off_ptr = 0, off_u = 0, off_part = 0, off_lvl[RO_MAX_LEVELS] = {0, 0, 0, 0}, total = 0;
};

RoPlan ro_plan(int n, uint32_t count, uint32_t shots) {
    RoPlan p;
    memset(&p.lv, 0, sizeof p.lv);
    p.gb = n < RO_GB ? n : RO_GB;
    const uint64_t n1 = 1ull << (n - p.gb);
    p.wgs = (n1 + 4 * RO_GPW - 1) / (4 * RO_GPW);
    size_t off = 0;
    p.off_ptr = off;
    off += align_up((size_t)count * sizeof(void *), 256);
    p.off_u = off;
    off += align_up((size_t)count * shots * sizeof(double), 256);
    p.off_part = off;
    off += align_up((size_t)count * p.wgs * PROB_SLOTS * sizeof(double), 256);
    uint64_t c = n1;
    int L = 0;
    for (;;) {
        p.lv.count[L] = c;
        p.lv.stride[L] = c;
        p.off_lvl[L] = off;
        off += align_up((size_t)count * c * sizeof(double), 256);
        L++;
        if (c <= RO_FAN) break;
        c = (c + RO_FAN - 1) >> RO_FAN_BITS;
    }
    p.lv.nlev = L;
    p.total = off;
    return p;
}
}  // namespace

extern "C" size_t dq_readout_ws_bytes(int n, uint32_t count, uint32_t shots) {
    if (n < 1 || n > 40 || count == 0) return 0;
    return ro_plan(n, count, shots).total;
}

extern "C" int dq_readout_many(int prec, int n, const void *const *states, uint32_t count, const double *u,
                               uint32_t shots, double *d_p0, uint64_t *d_shots, void *d_ws, size_t ws_bytes,
                               void *stream) {
    if ((prec != DQ_F32 && prec != DQ_F64) || n < 1 || n > 40 || !states || count == 0 || count > 65535)
        return fail(DQ_ERR_ARG, "dq_readout_many: bad arguments");
    if (shots > (1u << 24)) return fail(DQ_ERR_ARG, "dq_readout_many: at most 2^24 samples per state");
    if (shots && (!u || !d_shots)) return fail(DQ_ERR_ARG, "dq_readout_many: samples need u and d_shots");
    for (uint32_t i = 0; i < count; i++)
        if (!states[i]) return fail(DQ_ERR_ARG, "dq_readout_many: state %u is null", i);
    for (uint64_t i = 0; i < (uint64_t)count * shots; i++)
        if (!(u[i] >= 0.0 && u[i] < 1.0)) return fail(DQ_ERR_ARG, "dq_readout_many: u[%llu] not in [0, 1)", (unsigned long long)i);
    const RoPlan p = ro_plan(n, count, shots);
    if (!d_ws || ws_bytes < p.total) return fail(DQ_ERR_ARG, "dq_readout_many: workspace %zu < %zu bytes", ws_bytes, p.total);
    if (p.wgs > 0x7fffffffull) return fail(DQ_ERR_UNSUPPORTED, "dq_readout_many: grid too large");
    // state pointers and uniforms travel in one staged copy
    std::vector<unsigned char> buf(p.off_part - p.off_ptr, 0);
    memcpy(buf.data(), states, (size_t)count * sizeof(void *));
    if (shots) memcpy(buf.data() + (p.off_u - p.off_ptr), u, (size_t)count * shots * sizeof(double));
    unsigned char *d = (unsigned char *)d_ws;
    int rc = stage_upload(d + p.off_ptr, buf, stream);
    if (rc) return rc;
    const void *const *d_states = (const void *const *)(d + p.off_ptr);
    double *part = (double *)(d + p.off_part);
    RoLevels lv = p.lv;
    for (int L = 0; L < lv.nlev; L++) lv.base[L] = (double *)(d + p.off_lvl[L]);
    const uint64_t part_stride = p.wgs * PROB_SLOTS;
    hipStream_t s = (hipStream_t)stream;
    if (prec == DQ_F64)
        hipLaunchKernelGGL(readout_stage1<double>, dim3((unsigned)p.wgs, count), dim3(256), 0, s, d_states, n, part,
                           part_stride, lv.base[0], lv.stride[0]);
    else
        hipLaunchKernelGGL(readout_stage1<float>, dim3((unsigned)p.wgs, count), dim3(256), 0, s, d_states, n, part,
                           part_stride, lv.base[0], lv.stride[0]);
    HIPC(hipGetLastError());
    if (d_p0) {
        hipLaunchKernelGGL(readout_stage2, dim3(n + 1, count), dim3(256), 0, s, part, part_stride, (uint32_t)p.wgs, n, d_p0);
        HIPC(hipGetLastError());
    }
    if (!shots) return DQ_OK;
    for (int L = 1; L < lv.nlev; L++) {
        hipLaunchKernelGGL(readout_level, dim3((unsigned)((lv.count[L] + 3) / 4), count), dim3(256), 0, s,
                           lv.base[L - 1], lv.count[L - 1], lv.stride[L - 1], lv.base[L], lv.count[L], lv.stride[L]);
        HIPC(hipGetLastError());
    }
    const double *d_u = (const double *)(d + p.off_u);
    if (prec == DQ_F64)
        hipLaunchKernelGGL(readout_sample<double>, dim3((shots + 3) / 4, count), dim3(256), 0, s, d_states, n, lv, d_u,
                           shots, d_shots);
    else
        hipLaunchKernelGGL(readout_sample<float>, dim3((shots + 3) / 4, count), dim3(256), 0, s, d_states, n, lv, d_u,
                           shots, d_shots);
    HIPC(hipGetLastError());
    return DQ_OK;
}

// ---- comparison of two states -------------------------------------------------
extern "C" size_t dq_compare_ws_bytes(int n) {
    if (n < 1 || n > 40) return 0;
    return align_up(((size_t)1 << (n - cmp_share(n))) * CMP_SLOTS * sizeof(double), 256);
}

template <typename TA, typename TB>
static void launch_compare(const void *a, const void *b, int share, unsigned groups, double *part, hipStream_t s) {
    hipLaunchKernelGGL((compare_stage1<TA, TB>), dim3(groups), dim3(256), 0, s, (const typename V2<TA>::type *)a,
                       (const typename V2<TB>::type *)b, share, part);
}

extern "C" int dq_compare_states(const void *a, int prec_a, const void *b, int prec_b, int n, double *d_out,
                                 void *d_ws, size_t ws_bytes, void *stream) {
    const bool pa = prec_a == DQ_F32 || prec_a == DQ_F64, pb = prec_b == DQ_F32 || prec_b == DQ_F64;
    if (!a || !b || !d_out || !pa || !pb || n < 1 || n > 40) return fail(DQ_ERR_ARG, "dq_compare_states: bad arguments");
    if (!d_ws || ws_bytes < dq_compare_ws_bytes(n)) return fail(DQ_ERR_ARG, "dq_compare_states: workspace too small");
    const int share = cmp_share(n);
    const uint64_t groups = 1ull << (n - share);
    double *part = (double *)d_ws;
    hipStream_t s = (hipStream_t)stream;
    if (prec_a == DQ_F64 && prec_b == DQ_F64) launch_compare<double, double>(a, b, share, (unsigned)groups, part, s);
    else if (prec_a == DQ_F64) launch_compare<double, float>(a, b, share, (unsigned)groups, part, s);
    else if (prec_b == DQ_F64) launch_compare<float, double>(a, b, share, (unsigned)groups, part, s);
    else launch_compare<float, float>(a, b, share, (unsigned)groups, part, s);
    HIPC(hipGetLastError());
    hipLaunchKernelGGL(compare_stage2, dim3(CMP_SLOTS), dim3(256), 0, s, part, (uint32_t)groups, d_out);
    HIPC(hipGetLastError());
    return DQ_OK;
}

// ---- dense sweeps -------------------------------------------------------------
namespace {
size_t dense_mat_bytes(int k) { return (size_t)12 << (2 * k); }  // three pieces of two parts
size_t dense_lds_bytes(uint32_t T) { return (size_t)8 << T; }
}  // namespace

extern "C" size_t dq_dense_ws_bytes(int k, uint32_t n_blocks, uint32_t n_ops, uint32_t n_mats) {
    if (k < 5 || k > 7) return 0;
    return align_up(n_blocks * sizeof(dq_dense_block), 256) + align_up(n_ops * sizeof(dq_dense_op), 256) +
           align_up((size_t)n_mats * dense_mat_bytes(k), 256) +
           align_up((size_t)n_ops * DENSE_COLS * sizeof(uint32_t), 256);
}

// Host-side check of dense blocks and ops against the kernel's grid and tile.
static int validate_dense(int k, const dq_dense_block *blocks, uint32_t n_blocks, const dq_dense_op *ops, uint32_t n_ops,
                          uint32_t n_mats) {
    for (uint32_t i = 0; i < n_blocks; i++) {
        const dq_dense_block &b = blocks[i];
        const uint32_t n = b.n_qubits, T = b.tile_bits;
        if (n < 6 || n > 40 || T > DENSE_T_MAX || T > n || (int)T < k + 5)
            return fail(DQ_ERR_ARG, "dense block %u: need k + 5 <= T <= min(n, 13) (n=%u T=%u k=%d)", i, n, T, k);
        uint64_t m = 0;
        for (uint32_t t = 0; t < T; t++) {
            if (t < 6 && b.tile_q[t] != t) return fail(DQ_ERR_ARG, "dense block %u: tile bits 0..5 must be qubits 0..5", i);
            if (b.tile_q[t] >= n || ((m >> b.tile_q[t]) & 1)) return fail(DQ_ERR_ARG, "dense block %u: bad tile qubits", i);
            m |= 1ull << b.tile_q[t];
        }
        if ((m | b.nontile_mask) != ((n == 64) ? ~0ull : ((1ull << n) - 1)) || (m & b.nontile_mask))
            return fail(DQ_ERR_ARG, "dense block %u: tile and non-tile masks inconsistent", i);
        if ((uint64_t)b.op_begin + b.op_count > n_ops) return fail(DQ_ERR_ARG, "dense block %u: op range", i);
        for (uint32_t o = b.op_begin; o < b.op_begin + b.op_count; o++) {
            for (int j = 0; j < k; j++)
                if (ops[o].bits[j] >= T || (j && ops[o].bits[j] <= ops[o].bits[j - 1]))
                    return fail(DQ_ERR_ARG, "dense op %u: bits must be ascending tile bits", o);
            if (ops[o].mat >= n_mats) return fail(DQ_ERR_ARG, "dense op %u: matrix index", o);
        }
        if (n - T > 31) return fail(DQ_ERR_UNSUPPORTED, "dense block %u: grid too large", i);
    }
    return DQ_OK;
}

// Per op: column c's tile offset, c's bits placed on the block's tile bits
// outside the op (in ascending order).
static int dense_columns(int k, const dq_dense_block *blocks, uint32_t n_blocks, const dq_dense_op *ops, uint32_t n_ops,
                         uint32_t *ct) {
    std::vector<int> op_T(n_ops, -1);
    for (uint32_t i = 0; i < n_blocks; i++) {
        const uint32_t T = blocks[i].tile_bits;
        for (uint32_t o = blocks[i].op_begin; o < blocks[i].op_begin + blocks[i].op_count; o++) {
            if (op_T[o] >= 0 && op_T[o] != (int)T) return fail(DQ_ERR_ARG, "dense op %u: in blocks of different tiles", o);
            op_T[o] = (int)T;
            uint32_t used = 0, cb[DENSE_T_MAX];
            for (int j = 0; j < k; j++) used |= 1u << ops[o].bits[j];
            int nc = 0;
            for (uint32_t b = 0; b < T; b++)
                if (!((used >> b) & 1u)) cb[nc++] = b;
            for (uint32_t c = 0; c < (1u << nc); c++) {
                uint32_t v = 0;
                for (int b = 0; b < nc; b++) v |= ((c >> b) & 1u) << cb[b];
                ct[(size_t)o * DENSE_COLS + c] = v;
            }
        }
    }
    return DQ_OK;
}

static int dense_launch(int k, const dq_dense_block *blocks, uint32_t n_blocks, const dq_dense_block *d_blocks,
                        const dq_dense_op *d_ops, const uint4 *d_mats, const uint32_t *d_ct, void *state, hipStream_t s) {
    auto *st = (typename V2<float>::type *)state;
    for (uint32_t i = 0; i < n_blocks; i++) {
        const dq_dense_block &b = blocks[i];
        const unsigned grid = 1u << (b.n_qubits - b.tile_bits);
        const size_t lds = dense_lds_bytes(b.tile_bits);
        if (k == 5) hipLaunchKernelGGL(dense_kernel<5>, dim3(grid), dim3(DENSE_THREADS), lds, s, d_blocks + i, d_ops, d_mats, d_ct, st);
        else if (k == 6) hipLaunchKernelGGL(dense_kernel<6>, dim3(grid), dim3(DENSE_THREADS), lds, s, d_blocks + i, d_ops, d_mats, d_ct, st);
        else hipLaunchKernelGGL(dense_kernel<7>, dim3(grid), dim3(DENSE_THREADS), lds, s, d_blocks + i, d_ops, d_mats, d_ct, st);
        HIPC(hipGetLastError());
    }
    return DQ_OK;
}

extern "C" int dq_apply_dense(int k, const dq_dense_block *blocks, uint32_t n_blocks, const dq_dense_op *ops,
                              uint32_t n_ops, const double *mats, uint32_t n_mats, void *state, void *d_ws,
                              size_t ws_bytes, void *stream) {
    if (k < 5 || k > 7) return fail(DQ_ERR_ARG, "dq_apply_dense: k must be 5, 6 or 7");
    if (!blocks || !state || !d_ws || (n_ops && !ops) || (n_mats && !mats))
        return fail(DQ_ERR_ARG, "dq_apply_dense: null argument");
    const size_t need = dq_dense_ws_bytes(k, n_blocks, n_ops, n_mats);
    if (ws_bytes < need) return fail(DQ_ERR_ARG, "dq_apply_dense: workspace %zu < %zu bytes", ws_bytes, need);
    int rc = validate_dense(k, blocks, n_blocks, ops, n_ops, n_mats);
    if (rc) return rc;
    // upload: blocks | ops | matrices in MFMA operand order | column tables
    const size_t ob = align_up(n_blocks * sizeof(dq_dense_block), 256);
    const size_t mo = ob + align_up(n_ops * sizeof(dq_dense_op), 256);
    const uint32_t K = 1u << k;
    const size_t co = mo + align_up((size_t)n_mats * dense_mat_bytes(k), 256);
    std::vector<unsigned char> buf(co + (size_t)n_ops * DENSE_COLS * sizeof(uint32_t), 0);
    memcpy(buf.data(), blocks, n_blocks * sizeof(dq_dense_block));
    if (n_ops) memcpy(buf.data() + ob, ops, n_ops * sizeof(dq_dense_op));
    for (uint32_t mi = 0; mi < n_mats; mi++) {
        const double *U = mats + ((size_t)mi << (2 * k)) * 2;
        uint16_t *D = reinterpret_cast<uint16_t *>(buf.data() + mo + mi * dense_mat_bytes(k));
        for (uint32_t r = 0; r < K; r++)
            for (uint32_t c = 0; c < K; c++)
                for (uint32_t part = 0; part < 2; part++) {
                    uint16_t piece[3];
                    split_entry(U[2 * ((size_t)r * K + c) + part], piece);
                    for (int i = 0; i < 3; i++) D[entry_pos(k, r, c, part) + 512 * i] = piece[i];
                }
    }
    rc = dense_columns(k, blocks, n_blocks, ops, n_ops, reinterpret_cast<uint32_t *>(buf.data() + co));
    if (rc) return rc;
    rc = stage_upload(d_ws, buf, stream);
    if (rc) return rc;
    unsigned char *d = (unsigned char *)d_ws;
    return dense_launch(k, blocks, n_blocks, (const dq_dense_block *)d, (const dq_dense_op *)(d + ob), (const uint4 *)(d + mo),
                        (const uint32_t *)(d + co), state, (hipStream_t)stream);
}

namespace {
// Workspace of dq_apply_dense_gates: what is uploaded (blocks | ops | column
// tables | gates | first gate of each matrix), then the matrices.
struct DenseGatesWs {
    size_t ops, cols, gates, begin, upload, mats, total;
};
DenseGatesWs dense_gates_ws(int k, uint32_t n_blocks, uint32_t n_ops, uint32_t n_mats, uint32_t n_gates) {
    DenseGatesWs w;
    w.ops = align_up(n_blocks * sizeof(dq_dense_block), 256);
    w.cols = w.ops + align_up(n_ops * sizeof(dq_dense_op), 256);
    w.gates = w.cols + align_up((size_t)n_ops * DENSE_COLS * sizeof(uint32_t), 256);
    w.begin = w.gates + align_up((size_t)n_gates * sizeof(dq_small_gate), 256);
    w.upload = w.begin + ((size_t)n_mats + 1) * sizeof(uint32_t);
    w.mats = align_up(w.upload, 256);
    w.total = w.mats + (size_t)n_mats * dense_mat_bytes(k);
    return w;
}
}  // namespace

extern "C" size_t dq_dense_gates_ws_bytes(int k, uint32_t n_blocks, uint32_t n_ops, uint32_t n_mats, uint32_t n_gates) {
    if (k < 5 || k > 7) return 0;
    return dense_gates_ws(k, n_blocks, n_ops, n_mats, n_gates).total;
}

extern "C" int dq_apply_dense_gates(int k, const dq_dense_block *blocks, uint32_t n_blocks, const dq_dense_op *ops,
                                    uint32_t n_ops, const dq_small_gate *gates, const uint32_t *gate_begin, uint32_t n_mats,
                                    void *state, void *d_ws, size_t ws_bytes, void *stream) {
    if (k < 5 || k > 7) return fail(DQ_ERR_ARG, "dq_apply_dense_gates: k must be 5, 6 or 7");
    if (!blocks || !state || !d_ws || !gate_begin || (n_ops && !ops)) return fail(DQ_ERR_ARG, "dq_apply_dense_gates: null argument");
    for (uint32_t i = 0; i < n_mats; i++)
        if (gate_begin[i + 1] < gate_begin[i]) return fail(DQ_ERR_ARG, "dq_apply_dense_gates: gate ranges not ascending");
    const uint32_t n_gates = gate_begin[n_mats];
    if (n_gates && !gates) return fail(DQ_ERR_ARG, "dq_apply_dense_gates: null argument");
    for (uint32_t i = 0; i < n_gates; i++) {
        const dq_small_gate &g = gates[i];
        const bool one = g.tmask && !(g.tmask & (g.tmask - 1));
        if (((g.tmask | g.cmask) >> k) || (g.tmask & g.cmask) || g.diag > 1 || (g.diag ? g.tmask != 0 : !one))
            return fail(DQ_ERR_ARG, "dq_apply_dense_gates: gate %u: bad bits", i);
    }
    const DenseGatesWs w = dense_gates_ws(k, n_blocks, n_ops, n_mats, n_gates);
    if (ws_bytes < w.total) return fail(DQ_ERR_ARG, "dq_apply_dense_gates: workspace %zu < %zu bytes", ws_bytes, w.total);
    int rc = validate_dense(k, blocks, n_blocks, ops, n_ops, n_mats);
    if (rc) return rc;
    std::vector<unsigned char> buf(align_up(w.upload, 16), 0);  // the matrices begin at the next 256
    memcpy(buf.data(), blocks, n_blocks * sizeof(dq_dense_block));
    if (n_ops) memcpy(buf.data() + w.ops, ops, n_ops * sizeof(dq_dense_op));
    rc = dense_columns(k, blocks, n_blocks, ops, n_ops, reinterpret_cast<uint32_t *>(buf.data() + w.cols));
    if (rc) return rc;
    if (n_gates) memcpy(buf.data() + w.gates, gates, n_gates * sizeof(dq_small_gate));
    memcpy(buf.data() + w.begin, gate_begin, ((size_t)n_mats + 1) * sizeof(uint32_t));
    rc = stage_upload(d_ws, buf, stream);
    if (rc) return rc;
    unsigned char *d = (unsigned char *)d_ws;
    hipStream_t s = (hipStream_t)stream;
    const auto *d_gates = (const dq_small_gate *)(d + w.gates);
    const auto *d_begin = (const uint32_t *)(d + w.begin);
    unsigned char *d_mats = d + w.mats;
    for (uint32_t m0 = 0; m0 < n_mats; m0 += 65535u) {
        const uint32_t nm = std::min(n_mats - m0, 65535u);
        const uint32_t *gb = d_begin + m0;
        uint16_t *dm = (uint16_t *)(d_mats + (size_t)m0 * dense_mat_bytes(k));
        if (k == 5) hipLaunchKernelGGL(dense_form<5>, dim3(4, nm), dim3(256), 0, s, d_gates, gb, dm);
        else if (k == 6) hipLaunchKernelGGL(dense_form<6>, dim3(16, nm), dim3(256), 0, s, d_gates, gb, dm);
        else hipLaunchKernelGGL(dense_form<7>, dim3(32, nm), dim3(256), 0, s, d_gates, gb, dm);
        HIPC(hipGetLastError());
    }
    return dense_launch(k, blocks, n_blocks, (const dq_dense_block *)d, (const dq_dense_op *)(d + w.ops), (const uint4 *)d_mats,
                        (const uint32_t *)(d + w.cols), state, s);
}

// ---- permutation of qubits ----------------------------------------------------
namespace {
// One launch for the permutation `dest` of the index bits, if it is one: moving
// tile bits only, or an involution.  False otherwise (nothing filled).
bool perm_args(int n, const int *dest, int prec, PermArgs &pa) {
    const int lb = perm_low_bits(prec), tmax = prec == DQ_F64 ? 11 : 12;
    memset(&pa, 0, sizeof pa);
    uint64_t moved = 0, low = n < lb ? (1ull << n) - 1 : (1ull << lb) - 1;
    bool swaps = true;
    for (int p = 0; p < n; p++) {
        if (dest[p] != p) moved |= 1ull << p;
        swaps &= dest[dest[p]] == p;
    }
    uint64_t tile = low;
    if (__builtin_popcountll(low | moved) <= tmax) {
        tile |= moved;
    } else {
        if (!swaps) return false;
        for (int p = 0; p < lb; p++) tile |= 1ull << dest[p];
    }
    // fill up with the lowest other bits (with their images)
    for (int p = 0; p < n; p++) {
        const uint64_t add = ((1ull << p) | (1ull << dest[p])) & ~tile;
        if (add && __builtin_popcountll(tile | add) <= tmax) tile |= add;
    }
    int at[64];
    for (int p = 0; p < n; p++)
        if ((tile >> p) & 1) {
            at[p] = pa.tb;
            pa.tile[pa.tb++] = (uint8_t)p;
        } else {
            pa.pos[pa.nu] = (uint8_t)p;
            pa.img[pa.nu++] = (uint8_t)dest[p];
        }
    // the value at tile bit b of the new index is that of bit inv: element e takes
    // the amplitude whose index has bit inv[b] = bit b of e
    for (int p = 0; p < n; p++)
        if ((tile >> p) & 1) pa.inv[at[dest[p]]] = (uint8_t)at[p];
    return true;
}
}  // namespace

extern "C" int dq_permute_launches(int n, int prec, const int *dest) {
    if (!dest || n < 1 || n > 40 || (prec != DQ_F32 && prec != DQ_F64)) return fail(DQ_ERR_ARG, "dq_permute_qubits: bad arguments");
    uint64_t seen = 0;
    bool same = true;
    for (int p = 0; p < n; p++) {
        if (dest[p] < 0 || dest[p] >= n || ((seen >> dest[p]) & 1)) return fail(DQ_ERR_ARG, "dq_permute_qubits: not a permutation");
        seen |= 1ull << dest[p];
        same &= dest[p] == p;
    }
    if (same) return 0;
    PermArgs pa;
    return perm_args(n, dest, prec, pa) ? 1 : 2;
}

extern "C" int dq_permute_qubits(void *state, int n, int prec, const int *dest, void *stream) {
    if (!state) return fail(DQ_ERR_ARG, "dq_permute_qubits: bad arguments");
    const int launches = dq_permute_launches(n, prec, dest);
    if (launches <= 0) return launches;
    int step[2][40];
    if (launches == 1) {
        memcpy(step[0], dest, (size_t)n * sizeof(int));
    } else {
        // every cycle c0 -> c1 -> ... of length k: first c_i <-> c_-i, then c_j <-> c_(1-j)
        bool done[40] = {};
        for (int p = 0; p < n; p++) {
            if (done[p]) continue;
            int c[40], k = 0;
            for (int x = p; !done[x]; x = dest[x]) {
                done[x] = true;
                c[k++] = x;
            }
            for (int i = 0; i < k; i++) {
                step[0][c[i]] = c[(k - i) % k];
                step[1][c[i]] = c[(k + 1 - i) % k];
            }
        }
    }
    PermArgs pa[2];
    for (int l = 0; l < launches; l++)
        if (!perm_args(n, step[l], prec, pa[l]) || pa[l].nu > 31)
            return fail(DQ_ERR_UNSUPPORTED, "dq_permute_qubits: no launch for %d qubits", n);
    for (int l = 0; l < launches; l++) {
        const int gx = std::min(pa[l].nu, PERM_GRID_X);
        const dim3 grid(1u << gx, 1u << (pa[l].nu - gx));
        hipStream_t s = (hipStream_t)stream;
        if (prec == DQ_F32)
            hipLaunchKernelGGL((permute_kernel<float, 12, 512>), grid, dim3(512), 0, s, (V2<float>::type *)state, pa[l]);
        else if (pa[l].tb == 11)
            hipLaunchKernelGGL((permute_kernel<double, 11, 512>), grid, dim3(512), 0, s, (V2<double>::type *)state, pa[l]);
        else
            hipLaunchKernelGGL((permute_kernel<double, 10, 256>), grid, dim3(256), 0, s, (V2<double>::type *)state, pa[l]);
        HIPC(hipGetLastError());
    }
    return DQ_OK;
}

extern "C" int dq_event_query(void *ev) {
    if (!ev) return fail(DQ_ERR_ARG, "dq_event_query: null event");
    const hipError_t e = hipEventQuery((hipEvent_t)ev);
    if (e == hipSuccess) return 0;
    if (e == hipErrorNotReady) {
        (void)hipGetLastError();  // not an error: keep it out of the next launch check
        return 1;
    }
    return fail(DQ_ERR_HIP, "hipEventQuery: %s", hipGetErrorString(e));
}

extern "C" int dq_event_sync(void *ev) {
    if (!ev) return fail(DQ_ERR_ARG, "dq_event_sync: null event");
    HIPC(hipEventSynchronize((hipEvent_t)ev));
    return DQ_OK;
}

extern "C" int dq_read_amps(const void *state, int n, int prec, const int *l2p, uint64_t start, uint64_t count,
                            double *out, void *d_ws, size_t ws_bytes, void *stream) {
    if (!state || !out || n < 1 || n > 40 || (prec != DQ_F32 && prec != DQ_F64)) return fail(DQ_ERR_ARG, "dq_read_amps: bad arguments");
    const uint64_t N = 1ull << n;
    if (start > N || count > N - start) return fail(DQ_ERR_ARG, "dq_read_amps: range out of bounds");
    if (count == 0) return DQ_OK;
    QubitMap map;
    memset(&map, 0, sizeof map);
    for (int q = 0; q < n; q++) {
        const int p = l2p ? l2p[q] : q;
        if (p < 0 || p >= n) return fail(DQ_ERR_ARG, "dq_read_amps: bad qubit map");
        map.l2p[q] = (uint8_t)p;
    }
    const size_t bytes = count * 2 * sizeof(double);
    const size_t need = align_up(64 * sizeof(int), 256) + bytes;
    if (!d_ws || ws_bytes < need) return fail(DQ_ERR_ARG, "dq_read_amps: workspace %zu < %zu bytes", ws_bytes, need);
    ResultSlot res(bytes, (unsigned char *)d_ws + align_up(64 * sizeof(int), 256), stream);
    const unsigned blocks = (unsigned)((count + 255) / 256);
    if (prec == DQ_F64)
        hipLaunchKernelGGL(read_kernel<double>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (const V2<double>::type *)state, n, map, start, count, (double *)res.dst);
    else
        hipLaunchKernelGGL(read_kernel<float>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (const V2<float>::type *)state, n, map, start, count, (double *)res.dst);
    HIPC(hipGetLastError());
    return res.collect(out, bytes);
}

extern "C" int dq_write_amps(void *state, int n, int prec, uint64_t start, uint64_t count, const double *re,
                             const double *im, void *d_ws, size_t ws_bytes, void *stream) {
    if (!state || !re || !im || n < 1 || n > 40 || (prec != DQ_F32 && prec != DQ_F64)) return fail(DQ_ERR_ARG, "dq_write_amps: bad arguments");
    const uint64_t N = 1ull << n;
    if (start > N || count > N - start) return fail(DQ_ERR_ARG, "dq_write_amps: range out of bounds");
    if (count == 0) return DQ_OK;
    const size_t half = align_up(count * sizeof(double), 256);
    if (!d_ws || ws_bytes < 2 * half) return fail(DQ_ERR_ARG, "dq_write_amps: workspace too small");
    double *d_re = (double *)d_ws;
    double *d_im = (double *)((unsigned char *)d_ws + half);
    HIPC(hipMemcpyAsync(d_re, re, count * sizeof(double), hipMemcpyHostToDevice, (hipStream_t)stream));
    HIPC(hipMemcpyAsync(d_im, im, count * sizeof(double), hipMemcpyHostToDevice, (hipStream_t)stream));
    const unsigned blocks = (unsigned)((count + 255) / 256);
    if (prec == DQ_F64)
        hipLaunchKernelGGL(write_kernel<double>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (V2<double>::type *)state, start, count, d_re, d_im);
    else
        hipLaunchKernelGGL(write_kernel<float>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                           (V2<float>::type *)state, start, count, d_re, d_im);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize((hipStream_t)stream));
    return DQ_OK;
}
