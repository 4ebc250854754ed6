// Batched unlinked partitions (IQ-TREE's PhyloSuperTree loop over partitions,
// tree/phylosupertree.cpp:662-734): a traversal is one launch per kernel (4 and 20 states
// each have their own; a small FP32 batch of both is one launch), and every work item is
// one workgroup's patterns of one partition.  Each partition keeps its own model, P(t),
// slots, scale counters and fixed-order reduction, so its result is bit-identical to
// running it alone.
#include "dev_dna.h"
#include "dev_f32.h"
#include "dev_f64.h"
#include "dev_f64_cat.h"

namespace plk {
namespace {
using namespace dev;

__global__ void __launch_bounds__(256) k_batch_pmatrix_f64(const KParams *params, const PJob *jobs) {
    const PJob j = load_uniform(jobs + blockIdx.x);
    const KParams P = load_uniform(params + j.pad);
    pmatrix_f64_body(P, j);
}

__device__ __forceinline__ void pmatrix_f32_job(const KParams *params, const PJob *job) {
    const PJob j = load_uniform(job);
    const KParams P = load_uniform(params + j.pad);
    switch (P.n) {
        case 4: pmatrix_f32_body<4>(P, j); break;
        case 20: pmatrix_f32_body<20>(P, j); break;
        default: break;
    }
}

__global__ void __launch_bounds__(256) k_batch_pmatrix_f32(const KParams *params, const PJob *jobs) {
    pmatrix_f32_job(params, jobs + blockIdx.x);
}

// One kernel per state count: a kernel with both bodies takes the registers and LDS of the
// larger one for every item.  TURNS (gridDim < nitems): workgroup g takes items g, g + grid, ...
// (the host orders items by decreasing cost, so the static stride is a longest-first schedule).
// Otherwise a workgroup has one item and no loop, out of which the compiler would hoist the
// constants of exp and log into registers that stay taken through the op list: FP64 20 states
// 209 registers against 167, 4 states 175 against 125.
template <bool TURNS, typename F>
__device__ __forceinline__ void each_item(const KParams *params, const BatchItem *items, int nitems, F &&f) {
    for (int i = blockIdx.x; i < nitems; i += gridDim.x) {
        const BatchItem it = load_uniform(items + i);
        const KParams P = load_uniform(params + it.part);
        f(P, it.tile);
        if (!TURNS) return;
        __syncthreads();
    }
}

template <int N, bool TURNS>
__global__ void __launch_bounds__(256) k_batch_traverse_f64(const KParams *params, const BatchItem *items, int nitems) {
    each_item<TURNS>(params, items, nitems, [&](const KParams &P, int tile) {
        traverse_f64_body<N, MODE_LOGL>(P, tile);
    });
}

// one thread per (job, category, state); batched partitions have at most four categories
template <int FORM>
__device__ __forceinline__ void pmatrix_dna_thread(const KParams *params, const PJob *jobs, int njobs, int idx) {
    if (idx >= njobs * 16) return;
    const PJob j = jobs[idx >> 4];
    const KParams &P = params[j.pad];
    const int c = (idx >> 2) & 3, i = idx & 3;
    if (c >= P.ncat) return;
    dna_real<FORM> *M = (dna_real<FORM> *)P.mats + (int64_t)j.op * P.mat_stride + j.side * dna_side_len(FORM, 1);
    dna_pmat<FORM>(P, c, i, j.len, M, j.leaf ? M + dna_p_len(FORM) : nullptr);
}

template <int FORM>
__global__ void __launch_bounds__(256) k_batch_pmatrix_dna(const KParams *params, const PJob *jobs, int njobs) {
    pmatrix_dna_thread<FORM>(params, jobs, njobs, blockIdx.x * 256 + threadIdx.x);
}

// FP32 P(t) of both data types: nother workgroups, a job each, then those of the ndna jobs at
// the head of the list
__global__ void __launch_bounds__(256) k_batch_pmatrix_f32_both(const KParams *params, const PJob *jobs, int ndna, int nother) {
    if ((int)blockIdx.x < nother) pmatrix_f32_job(params, jobs + ndna + blockIdx.x);
    else pmatrix_dna_thread<1>(params, jobs, ndna, (blockIdx.x - nother) * 256 + threadIdx.x);
}

template <int FORM, bool SAFE, bool TURNS>
__global__ void __launch_bounds__(256) k_batch_traverse_dna(const KParams *params, const BatchItem *items, int nitems) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    each_item<TURNS>(params, items, nitems, [&](const KParams &P, int tile) {
        traverse_dna_body<FORM, 1, MODE_LOGL, false, SAFE>(P, tile, 0, P.nops, smem);
    });
}

// the 20-state partitions of the matrix-core form: an item is one workgroup's patterns
template <int PG, bool TURNS>
__global__ void __launch_bounds__(256, 2) k_batch_traverse_f64_cat(const KParams *params, const BatchItem *items, int nitems) {
    each_item<TURNS>(params, items, nitems, [&](const KParams &P, int tile) {
        traverse_f64_cat_body<MODE_LOGL, PG>(P, tile);
    });
}

template <int N, bool TURNS>
__global__ void __launch_bounds__(256) k_batch_traverse_f32(const KParams *params, const BatchItem *items, int nitems) {
    each_item<TURNS>(params, items, nitems, [&](const KParams &P, int tile) {
        if constexpr (N == 4) traverse_f32_valu_body<4, MODE_LOGL>(P, tile);
        else traverse_f32_mfma_body<N, MODE_LOGL>(P, tile);
    });
}

// FP32, both data types (batch_traverse_f32_both)
__global__ void __launch_bounds__(256) k_batch_traverse_f32_both(const KParams *params, const BatchItem *items, int nitems) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    each_item<false>(params, items, nitems, [&](const KParams &P, int tile) {
        if (P.n == 20) traverse_f32_mfma_body<20, MODE_LOGL>(P, tile);
        else traverse_dna_body<1, 1, MODE_LOGL, false, false>(P, tile, 0, P.nops, smem);
    });
}

// df/ddf of many branches of one alignment in one launch: item = (branch, tile); each
// branch has its own KParams (branch ends, length, reduction buffers) and theta is not
// stored.  Same arithmetic as the single-branch kernels, so results are identical.  One
// kernel per state count (see above; with all three in one, every count ran with the
// 61-state body's 512 registers, spills and 72 KB of LDS).
template <int N>
__global__ void __launch_bounds__(256) k_multi_derivs_f64(const KParams *params, const BatchItem *items) {
    const BatchItem it = load_uniform(items + blockIdx.x);
    const KParams P = load_uniform(params + it.part);
    traverse_f64_body<N, MODE_THETA, false, false, false>(P, it.tile);
}

template <int N>
__global__ void __launch_bounds__(256) k_multi_derivs_f32(const KParams *params, const BatchItem *items) {
    const BatchItem it = load_uniform(items + blockIdx.x);
    const KParams P = load_uniform(params + it.part);
    theta_f32_body<N>(P, it.tile);
}

// Many-branch Newton: item = (branch, tile); one launch = one derivative evaluation of
// every unfinished branch at its device-held iterate (with the logL there), then that
// branch's minimizeNewton step in the workgroup finishing its reduction.  A finished
// branch's items return at once.  (A branch's state is written only by its last
// workgroup, after all of its items have read it.)
template <int N, bool F32>
__global__ void __launch_bounds__(256) k_multi_newton(const KParams *params, const BatchItem *items, NewtonState *states) {
    const BatchItem it = load_uniform(items + blockIdx.x);
    NewtonState *st = states + it.part;
    if (st->done) return;
    KParams P = load_uniform(params + it.part);
    P.br_len = st->rts;
    bool last;
    if constexpr (F32) last = theta_f32_body<N, true>(P, it.tile);
    else last = traverse_f64_body<N, MODE_THETA, true, false, false>(P, it.tile);
    if (last && threadIdx.x == 0) newton_record(*st, P.result[0], P.result[1], P.result[2]);
}

template <int N>
void multi_newton_n(bool f32, int ncw, const KParams *params, const BatchItem *items, int nitems, NewtonState *states,
                    hipStream_t s) {
    if (f32) hipLaunchKernelGGL((k_multi_newton<N, true>), dim3(nitems), dim3(64 * ncw), 0, s, params, items, states);
    else hipLaunchKernelGGL((k_multi_newton<N, false>), dim3(nitems), dim3(64 * ncw), 0, s, params, items, states);
}

template <int N>
void multi_derivs_n(bool f32, int ncw, const KParams *params, const BatchItem *items, int nitems, hipStream_t s) {
    if (f32) hipLaunchKernelGGL((k_multi_derivs_f32<N>), dim3(nitems), dim3(64 * ncw), 0, s, params, items);
    else hipLaunchKernelGGL((k_multi_derivs_f64<N>), dim3(nitems), dim3(64 * ncw), 0, s, params, items);
}

}  // namespace

hipError_t multi_newton(int prec, int n, int ncw, const KParams *params, const BatchItem *items, int nitems,
                        NewtonState *states, hipStream_t s) {
    if (nitems <= 0) return hipSuccess;
    const bool f32 = prec == PLK_FP32;
    switch (n) {
        case 4: multi_newton_n<4>(f32, ncw, params, items, nitems, states, s); break;
        case 20: multi_newton_n<20>(f32, ncw, params, items, nitems, states, s); break;
        case 61: multi_newton_n<61>(f32, ncw, params, items, nitems, states, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t multi_derivs(int prec, int n, int ncw, const KParams *params, const BatchItem *items, int nitems, hipStream_t s) {
    if (nitems <= 0) return hipSuccess;
    const bool f32 = prec == PLK_FP32;
    switch (n) {
        case 4: multi_derivs_n<4>(f32, ncw, params, items, nitems, s); break;
        case 20: multi_derivs_n<20>(f32, ncw, params, items, nitems, s); break;
        case 61: multi_derivs_n<61>(f32, ncw, params, items, nitems, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t batch_pmatrix_dna(int prec, const KParams *params, const PJob *jobs, int njobs, hipStream_t s) {
    if (njobs <= 0) return hipSuccess;
    const dim3 grid((njobs * 16 + 255) / 256);
    if (prec == PLK_FP64) hipLaunchKernelGGL(k_batch_pmatrix_dna<0>, grid, dim3(256), 0, s, params, jobs, njobs);
    else hipLaunchKernelGGL(k_batch_pmatrix_dna<1>, grid, dim3(256), 0, s, params, jobs, njobs);
    return hipGetLastError();
}

hipError_t batch_pmatrix(int prec, const KParams *params, const PJob *jobs, int njobs, hipStream_t s) {
    if (njobs <= 0) return hipSuccess;
    if (prec == PLK_FP64) hipLaunchKernelGGL(k_batch_pmatrix_f64, dim3(njobs), dim3(256), 0, s, params, jobs);
    else hipLaunchKernelGGL(k_batch_pmatrix_f32, dim3(njobs), dim3(256), 0, s, params, jobs);
    return hipGetLastError();
}

hipError_t batch_pmatrix_f32_both(const KParams *params, const PJob *jobs, int ndna, int njobs, hipStream_t s) {
    const int nother = njobs - ndna;
    const dim3 grid(nother + (ndna * 16 + 255) / 256);
    hipLaunchKernelGGL(k_batch_pmatrix_f32_both, grid, dim3(256), 0, s, params, jobs, ndna, nother);
    return hipGetLastError();
}

hipError_t batch_traverse_f32_both(const KParams *params, const BatchItem *items, int nitems, size_t lds, hipStream_t s) {
    if (lds + kBothLds > 160 * 1024) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(k_batch_traverse_f32_both, dim3(nitems), dim3(256), lds, s, params, items, nitems);
    return hipGetLastError();
}

template <bool TURNS>
static void batch_traverse_t(bool f32, int group, const KParams *params, const BatchItem *items, int nitems, dim3 g,
                             size_t lds, hipStream_t s) {
    const dim3 b(256);
    switch (group) {
        case BATCH_MC: hipLaunchKernelGGL((k_batch_traverse_f64_cat<2, TURNS>), g, b, 0, s, params, items, nitems); break;
        case BATCH_MC1: hipLaunchKernelGGL((k_batch_traverse_f64_cat<1, TURNS>), g, b, 0, s, params, items, nitems); break;
        case BATCH_DNA:
            if (f32) hipLaunchKernelGGL((k_batch_traverse_dna<1, false, TURNS>), g, b, lds, s, params, items, nitems);
            else hipLaunchKernelGGL((k_batch_traverse_dna<0, false, TURNS>), g, b, lds, s, params, items, nitems);
            break;
        case BATCH_DNA_SAFE:
            hipLaunchKernelGGL((k_batch_traverse_dna<0, true, TURNS>), g, b, lds, s, params, items, nitems);
            break;
        case BATCH_20:
            if (f32) hipLaunchKernelGGL((k_batch_traverse_f32<20, TURNS>), g, b, 0, s, params, items, nitems);
            else hipLaunchKernelGGL((k_batch_traverse_f64<20, TURNS>), g, b, 0, s, params, items, nitems);
            break;
        default:
            if (f32) hipLaunchKernelGGL((k_batch_traverse_f32<4, TURNS>), g, b, 0, s, params, items, nitems);
            else hipLaunchKernelGGL((k_batch_traverse_f64<4, TURNS>), g, b, 0, s, params, items, nitems);
    }
}

hipError_t batch_traverse(int prec, int group, const KParams *params, const BatchItem *items, int nitems, int grid,
                          size_t lds, hipStream_t s) {
    if (nitems <= 0) return hipSuccess;
    if (lds > kDnaLdsMax) return hipErrorInvalidConfiguration;
    const bool f32 = prec == PLK_FP32;
    if (grid <= 0 || grid >= nitems) batch_traverse_t<false>(f32, group, params, items, nitems, dim3(nitems), lds, s);
    else batch_traverse_t<true>(f32, group, params, items, nitems, dim3(grid), lds, s);
    return hipGetLastError();
}

}  // namespace plk
