// FP64 kernels for gfx950: thin __global__ wrappers over the bodies in dev_f64.h.
#include <algorithm>

#include "dev_f64.h"
#include "dev_f64_cat.h"
#include "dev_f64_codon.h"

namespace plk {
namespace {
using namespace dev;

// one workgroup per (job, category)
__global__ void __launch_bounds__(256) k_pmatrix_f64(KParams P, const PJob *__restrict__ jobs) {
    pmatrix_f64_body(P, jobs[blockIdx.x / P.ncat], blockIdx.x % P.ncat);
}

// Occupancy floor: the 20-state partial/logL kernels are held to 128 VGPRs (4 waves per
// SIMD, a few bytes of spill), so that e.g. the 770 tiles x 4 waves of a 49k-pattern
// alignment fit the chip in one round (3 waves per SIMD hold only 768 tiles).  The
// theta variant keeps its full register budget (it would spill far more).
template <int N, int MODE>
constexpr int traverse_min_waves() { return (N == 20 && MODE != MODE_THETA) ? 4 : 1; }

template <int N, int MODE>
__global__ void __launch_bounds__(256, (traverse_min_waves<N, MODE>())) k_traverse_f64(KParams P) {
    traverse_f64_body<N, MODE>(P, blockIdx.x);
}

// 61 states with at most four categories: matrices staged in LDS (one workgroup per CU)
template <int MODE>
__global__ void __launch_bounds__(256, 1) k_traverse_f64_lds61(KParams P) {
    traverse_f64_body<61, MODE, false, true>(P, blockIdx.x);
}

// 61 states on the matrix cores.  The workgroups load the matrices
// once and take units in turn: SAFE a unit is (16 patterns, category), NORM four patterns with
// all categories.
template <bool SAFE>
__global__ void __launch_bounds__(SAFE ? 256 : 512, 2) k_traverse_f64_codon(KParams P) {
    __shared__ unsigned s_ok[2][PLK_GPU_MAX_CATS];
    __shared__ __attribute__((aligned(16))) double s_ui[64 * 64];
    const int lane = threadIdx.x & 63, w = wave_id(), ncat = P.ncat;
    double U[4][4][4];
#pragma unroll
    for (int i = 0; i < 64; i++) U[i / 16][i % 4][i / 4 % 4] = P.uinv_frag[(i / 2 * 64 + lane) * 2 + i % 2];
    for (int i = threadIdx.x; i < 64 * 64; i += blockDim.x) s_ui[i] = P.uinv_frag[64 * 64 + i];
    __syncthreads();
    const int units = P.ntiles * (SAFE ? 4 * ncat : 16), n = gridDim.x;
    int turn = 0;
    for (int u = blockIdx.x; u < units; u += n) {
        if (SAFE) traverse_f64_codon_body<true>(P, u / ncat, w, u % ncat, U, s_ui, s_ok, turn);
        else traverse_f64_codon_body<false>(P, u / 4, u % 4, w, U, s_ui, s_ok, turn);
    }
}

__global__ void __launch_bounds__(256) k_pmatrix_f64_codon(KParams P, const PJob *__restrict__ jobs) {
    pmatrix_f64_codon_body(P, jobs[blockIdx.x / P.ncat], blockIdx.x % P.ncat);
}

__global__ void __launch_bounds__(1024) k_branch_f64_codon(KParams P) { branch_f64_codon_body(P, blockIdx.x); }

// 20 states on the matrix cores; WIDE: 5-8 categories (two wavefronts per pattern unit).
// PG = 2 takes 160 registers (three wavefronts per SIMD), PG = 1 119 (four).
template <int MODE, int PG, bool WIDE>
__global__ void __launch_bounds__(WIDE ? 512 : 256, 2) k_traverse_f64_cat(KParams P) {
    traverse_f64_cat_body<MODE, PG>(P, blockIdx.x);
}

template <int MODE, int PG>
void launch_cat(const KParams &p, hipStream_t s) {
    const dim3 grid(p.nptn_pad / (4 * mc_unit(PG, p.ncat)));
    if (p.ncat <= 4) hipLaunchKernelGGL((k_traverse_f64_cat<MODE, PG, false>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((k_traverse_f64_cat<MODE, PG, true>), grid, dim3(512), 0, s, p);
}

// PG = 1 while its wavefronts do not outnumber the SIMDs (4 patterns each: up to 4,096 patterns
// with 3-4 categories on 256 compute units), where an op's latency is all that counts: 50
// taxa x 3,855 patterns, all directions, 196 us against 270; beyond that PG = 2 has more
// products in flight per wavefront and 64-byte pieces per row: 100 taxa x 6,000 patterns
// 197 against 226 us, 24,000 577 against 798, 49,994 1.31 ms against 1.80.  One category
// leaves no room for PG = 2 in a 64-pattern tile.
template <int MODE>
hipError_t traverse_cat(const KParams &p, hipStream_t s) {
    const int waves = p.nptn_pad / mc_unit(1, p.ncat) * ((p.ncat + 3) / 4);
    if (p.ncat > 1 && waves > 4 * p.ncu) launch_cat<MODE, 2>(p, s);
    else launch_cat<MODE, 1>(p, s);
    return hipGetLastError();
}

template <int N, int DERIV>
__global__ void __launch_bounds__(256) k_theta_eval_f64(KParams P) {
    theta_eval_f64_body<N, DERIV>(P, blockIdx.x, P.br_len);
}

// First Newton step, after the traversal that built theta left (d1, d2) in P.result.
__global__ void k_newton_first(NewtonState *st, const double *result) {
    if (threadIdx.x == 0) newton_after_eval(*st, result[0], result[1]);
}

// One Newton iteration: derivatives at the state's current iterate, then (in the
// workgroup that finishes the reduction) the step.  A finished solve makes every
// later launch of the queue return at once.
template <int N>
__global__ void __launch_bounds__(256) k_theta_newton_f64(KParams P, NewtonState *st) {
    if (st->done) return;
    const double len = st->rts;
    const bool last = theta_eval_f64_body<N, 1>(P, blockIdx.x, len);
    if (last && threadIdx.x == 0) newton_after_eval(*st, P.result[0], P.result[1]);
}

template <int N>
hipError_t traverse_n(const KParams &p0, int mode, hipStream_t s) {
    KParams p = p0;
    dim3 grid(p.ntiles), block(64 * p.ncw);
    if constexpr (N == 20) {
        if (p.f64_form == 1) {
            if (mode == MODE_LOGL) return traverse_cat<MODE_LOGL>(p, s);
            if (p.nops > 0) {
                const hipError_t e = traverse_cat<MODE_PARTIALS>(p, s);
                if (e != hipSuccess || mode == MODE_PARTIALS) return e;
            } else if (mode == MODE_PARTIALS) {
                return hipSuccess;
            }
            p.nops = 0;  // theta in the vector kernel, without ops
        }
    }
    if constexpr (N == 61) {
        if (p.f64_form == 1) {
            // the op list on the matrix cores, then the branch stage alone (theta: no ops, in
            // the vector kernel)
            if (p.nops > 0) {
                // One category: the checks over a pattern and over a category are the same, and
                // SAFE's workgroups have four wavefronts (NORM's one each left a compute unit two
                // of eight: 20 taxa x 20,000 sites 452 us, now 218).
                const bool safe = p.safe || p.ncat == 1;
                const int units = p.ntiles * (safe ? 4 * p.ncat : 16);
                // Workgroups that stay on a compute unit: eight wavefronts by registers, four
                // workgroups by LDS (two categories 466 -> 321 us).
                const int stay = safe ? 2 : std::min(4, 8 / p.ncat);
                const dim3 g(std::min(units, std::max(1, stay * p.ncu)));
                if (safe) hipLaunchKernelGGL(k_traverse_f64_codon<true>, g, dim3(256), 0, s, p);
                else hipLaunchKernelGGL(k_traverse_f64_codon<false>, g, dim3(64 * p.ncat), 0, s, p);
                if (mode == MODE_PARTIALS) return hipGetLastError();
                p.nops = 0;
            }
            if (mode == MODE_LOGL) hipLaunchKernelGGL(k_branch_f64_codon, grid, dim3(1024), 0, s, p);
            else if (mode == MODE_THETA) hipLaunchKernelGGL((k_traverse_f64<N, MODE_THETA>), grid, block, 0, s, p);
            return hipGetLastError();
        }
    }
    if (N == 61 && p.ncat <= 4) {
        if (mode == MODE_PARTIALS) hipLaunchKernelGGL((k_traverse_f64_lds61<MODE_PARTIALS>), grid, block, 0, s, p);
        else if (mode == MODE_LOGL) hipLaunchKernelGGL((k_traverse_f64_lds61<MODE_LOGL>), grid, block, 0, s, p);
        else hipLaunchKernelGGL((k_traverse_f64_lds61<MODE_THETA>), grid, block, 0, s, p);
        return hipGetLastError();
    }
    if (mode == MODE_PARTIALS) hipLaunchKernelGGL((k_traverse_f64<N, MODE_PARTIALS>), grid, block, 0, s, p);
    else if (mode == MODE_LOGL) hipLaunchKernelGGL((k_traverse_f64<N, MODE_LOGL>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((k_traverse_f64<N, MODE_THETA>), grid, block, 0, s, p);
    return hipGetLastError();
}

template <int N>
hipError_t theta_eval_n(const KParams &p, int deriv, hipStream_t s) {
    dim3 grid(p.ntiles), block(64 * p.ncw);
    if (deriv) hipLaunchKernelGGL((k_theta_eval_f64<N, 1>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((k_theta_eval_f64<N, 0>), grid, block, 0, s, p);
    return hipGetLastError();
}

template <int N>
hipError_t theta_newton_n(const KParams &p, NewtonState *st, hipStream_t s) {
    hipLaunchKernelGGL((k_theta_newton_f64<N>), dim3(p.ntiles), dim3(64 * p.ncw), 0, s, p, st);
    return hipGetLastError();
}

}  // namespace

hipError_t newton_first(NewtonState *st, const double *result, hipStream_t s) {
    hipLaunchKernelGGL(k_newton_first, dim3(1), dim3(64), 0, s, st, result);
    return hipGetLastError();
}

hipError_t f64_theta_newton(const KParams &p, NewtonState *st, hipStream_t s) {
    switch (p.n) {
        case 4: return theta_newton_n<4>(p, st, s);
        case 20: return theta_newton_n<20>(p, st, s);
        case 61: return theta_newton_n<61>(p, st, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t f64_pmatrix(const KParams &p, const PJob *jobs, int njobs, hipStream_t s) {
    if (p.n == 61 && p.f64_form == 1) hipLaunchKernelGGL(k_pmatrix_f64_codon, dim3(njobs * p.ncat), dim3(256), 0, s, p, jobs);
    else hipLaunchKernelGGL(k_pmatrix_f64, dim3(njobs * p.ncat), dim3(256), 0, s, p, jobs);
    return hipGetLastError();
}

hipError_t f64_traverse(const KParams &p, int mode, hipStream_t s) {
    switch (p.n) {
        case 4: return traverse_n<4>(p, mode, s);
        case 20: return traverse_n<20>(p, mode, s);
        case 61: return traverse_n<61>(p, mode, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t f64_theta_eval(const KParams &p, int deriv, hipStream_t s) {
    switch (p.n) {
        case 4: return theta_eval_n<4>(p, deriv, s);
        case 20: return theta_eval_n<20>(p, deriv, s);
        case 61: return theta_eval_n<61>(p, deriv, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace plk
