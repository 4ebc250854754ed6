// 4-state traversal kernels: thin __global__ wrappers over dev_dna.h.
#include "dev_dna.h"

namespace plk {
namespace {
using namespace dev;

// one thread per (job, category, state)
template <int FORM>
__global__ void __launch_bounds__(256) k_pmatrix_dna(KParams P, const PJob *__restrict__ jobs, int njobs) {
    const int idx = blockIdx.x * 256 + threadIdx.x, per = 4 * P.ncat;
    if (idx >= njobs * per) return;
    const PJob j = jobs[idx / per];
    const int c = (idx % per) >> 2, i = idx & 3, groups = (P.ncat + 3) / 4;
    dna_real<FORM> *M = (dna_real<FORM> *)P.mats + (int64_t)j.op * P.mat_stride + j.side * dna_side_len(FORM, groups);
    dna_pmat<FORM>(P, c, i, j.len, M, j.leaf ? M + groups * dna_p_len(FORM) : nullptr);
}

// blockIdx.y: range of the op list
template <int FORM, int CG, int MODE, bool STAGE, bool SAFE>
__device__ __forceinline__ void run_ranges(const KParams &P, char *smem) {
    int k0 = 0, k1 = P.nops;
    if (MODE == MODE_PARTIALS && P.nlevels > 1) {
        k0 = load_int(P.lvl, blockIdx.y);
        k1 = load_int(P.lvl, blockIdx.y + 1);
    }
    traverse_dna_body<FORM, CG, MODE, STAGE, SAFE>(P, blockIdx.x, k0, k1, smem);
}

template <int FORM, int CG, int MODE, bool STAGE, bool SAFE>
__global__ void __launch_bounds__(256, FORM == 1 && CG == 1 ? 8 : 1) k_traverse_dna(KParams P) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    run_ranges<FORM, CG, MODE, STAGE, SAFE>(P, smem);
}

// the same with the op list in the kernel arguments
template <int FORM, int CG, int MODE, bool SAFE>
__global__ void __launch_bounds__(256) k_traverse_dna_inl(KParams P, SmallInline in) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    KParams Q = P;
    Q.ops = (const DevOp *)in.data;
    Q.lvl = (const int32_t *)in.data + P.nops * (int)(sizeof(DevOp) / 4);
    run_ranges<FORM, CG, MODE, true, SAFE>(Q, smem);
}

template <int FORM, int CG, int MODE, bool SAFE>
hipError_t launch(const KParams &p, bool stage, const SmallInline *inl, hipStream_t s) {
    const int waves = p.ncat >= 3 ? 4 : p.ncat;
    const dim3 grid(p.ntiles, MODE == MODE_PARTIALS && p.nlevels > 1 ? p.nlevels : 1), block(64 * waves);
    const size_t lds = dna_lds_bytes(FORM, p.ncat, waves, p.nbuf, stage ? p.small_stage : 0, stage ? p.ntip : 0);
    if (lds > kDnaLdsMax) return hipErrorInvalidConfiguration;
    if (inl) hipLaunchKernelGGL((k_traverse_dna_inl<FORM, CG, MODE, SAFE>), grid, block, lds, s, p, *inl);
    else if (stage) hipLaunchKernelGGL((k_traverse_dna<FORM, CG, MODE, true, SAFE>), grid, block, lds, s, p);
    else hipLaunchKernelGGL((k_traverse_dna<FORM, CG, MODE, false, SAFE>), grid, block, lds, s, p);
    return hipGetLastError();
}

template <int FORM, int CG>
hipError_t launch_mode(const KParams &p, int mode, bool stage, const SmallInline *inl, hipStream_t s) {
    // (one category: SAFE's check and counts are NORM's, whose counts come in one load: 300 taxa x
    // 1,500 sites 220 -> 217 us)
    if (FORM == 0 && p.safe && p.ncat > 1)
        return mode == MODE_LOGL ? launch<FORM, CG, MODE_LOGL, FORM == 0>(p, stage, inl, s)
                                 : launch<FORM, CG, MODE_PARTIALS, FORM == 0>(p, stage, inl, s);
    return mode == MODE_LOGL ? launch<FORM, CG, MODE_LOGL, false>(p, stage, inl, s)
                             : launch<FORM, CG, MODE_PARTIALS, false>(p, stage, inl, s);
}

}  // namespace

size_t dna_lds_bytes(int form, int ncat, int waves, int nbuf, int nstage, int ntab) {
    const size_t rs = form == 0 ? 8 : 4, cg = (ncat + 3) / 4;
    size_t b = dna_window(nstage > 0) * 128;
    if (form == 0) b += (size_t)kDnaStates * 4 * rs;
    b += ((size_t)nstage * 2 * dna_p_len(form) + (form == 0 ? 0 : (size_t)ntab * dna_table_len())) * cg * rs;
    return b + (size_t)waves * nbuf * cg * (256 * rs + 64 * (form == 0 ? 8 : 4));
}

hipError_t dna_pmatrix(const KParams &p, int form, const PJob *jobs, int njobs, hipStream_t s) {
    if (njobs <= 0) return hipSuccess;
    const dim3 grid((njobs * 4 * p.ncat + 255) / 256);
    if (form == 0) hipLaunchKernelGGL(k_pmatrix_dna<0>, grid, dim3(256), 0, s, p, jobs, njobs);
    else hipLaunchKernelGGL(k_pmatrix_dna<1>, grid, dim3(256), 0, s, p, jobs, njobs);
    return hipGetLastError();
}

hipError_t dna_traverse(const KParams &p, int form, int mode, bool stage, const SmallInline *inl, hipStream_t s) {
    if (mode != MODE_PARTIALS && mode != MODE_LOGL) return hipErrorInvalidValue;
    if (form == 0) return p.ncat <= 4 ? launch_mode<0, 1>(p, mode, stage, inl, s) : launch_mode<0, 2>(p, mode, stage, inl, s);
    return p.ncat <= 4 ? launch_mode<1, 1>(p, mode, stage, inl, s) : launch_mode<1, 2>(p, mode, stage, inl, s);
}

}  // namespace plk
