// Newton branch solves in one launch: thin __global__ wrappers over dev_newton.h.
#include "dev_newton.h"

namespace plk {
namespace {
using namespace dev;

// wavefronts per SIMD that the registers of the products leave room for (newton_solve_fits)
constexpr int solve_waves(int n) { return n == 61 ? 2 : 4; }
// Tiles of a workgroup.  4 states: four, whose products take a wavefront 32 registers, for many
// branches (3,256 workgroups of one tile 173 us a solve, 814 of four 58) and for one long
// alignment; a short one, where only the latency counts, keeps one (64 taxa x 4,783 patterns: 36.5 -> 34.6 us a branch).
constexpr int solve_tiles(int n) { return n == 4 ? 4 : 1; }
int groups(int n, int ntiles) { return (ntiles + solve_tiles(n) - 1) / solve_tiles(n); }

template <int N, bool THETA, bool WIDE, int K>
__global__ void __launch_bounds__(WIDE ? 512 : 256, solve_waves(N)) k_newton_solve(KParams P, NewtonState start,
                                                                                 HandArea hand, NewtonState *out) {
    newton_solve_body<N, false, THETA, WIDE ? 8 : 4, K>(P, blockIdx.x, start, hand.use, hand.spare, hand.spare_len, out);
}

// many branches: the workgroups of a branch are neighbours; states is the host's mirror
template <int N, bool WIDE>
__global__ void __launch_bounds__(WIDE ? 512 : 256, solve_waves(N)) k_newton_solve_multi(
    const KParams *params, int nwg, int64_t hand_len, const NewtonState *start, HandArea hand, NewtonState *states) {
    const int br = blockIdx.x / nwg;
    const KParams P = load_uniform(params + br);
    newton_solve_body<N, true, false, WIDE ? 8 : 4, solve_tiles(N)>(P, blockIdx.x % nwg, load_uniform(start + br), hand.use + hand_len * br, hand.spare, hand.spare_len, states + br);
}

template <int N, bool THETA, int K>
void solve_k(const KParams &p, const NewtonState &start, HandArea hand, NewtonState *out, hipStream_t s) {
    const dim3 g((p.ntiles + K - 1) / K), b(64 * p.ncat);
    if (p.ncat <= 4) hipLaunchKernelGGL((k_newton_solve<N, THETA, false, K>), g, b, 0, s, p, start, hand, out);
    else hipLaunchKernelGGL((k_newton_solve<N, THETA, true, K>), g, b, 0, s, p, start, hand, out);
}

template <int N, bool THETA>
void solve_n(const KParams &p, const NewtonState &start, HandArea hand, NewtonState *out, hipStream_t s) {
    if (p.ntiles * p.ncat <= solve_waves(N) * p.ncu) solve_k<N, THETA, 1>(p, start, hand, out, s);
    else solve_k<N, THETA, solve_tiles(N)>(p, start, hand, out, s);
}

template <int N>
void solve_multi_n(int ncat, int ntiles, const KParams *params, const NewtonState *start, HandArea hand,
                   NewtonState *states, int nbr, hipStream_t s) {
    const int nwg = groups(N, ntiles);
    const dim3 g(nbr * nwg), b(64 * ncat);
    if (ncat <= 4) hipLaunchKernelGGL((k_newton_solve_multi<N, false>), g, b, 0, s, params, nwg, (int64_t)newton_hand_len(ntiles), start, hand, states);
    else hipLaunchKernelGGL((k_newton_solve_multi<N, true>), g, b, 0, s, params, nwg, (int64_t)newton_hand_len(ntiles), start, hand, states);
}

}  // namespace

bool newton_solve_fits(int n, int ncat, int ntiles, int ncu) { return groups(n, ntiles) * ncat <= solve_waves(n) * ncu; }

hipError_t newton_solve(const KParams &p, bool from_theta, const NewtonState &start, HandArea hand, NewtonState *out,
                        hipStream_t s) {
    switch (p.n) {
        case 4: from_theta ? solve_n<4, true>(p, start, hand, out, s) : solve_n<4, false>(p, start, hand, out, s); break;
        case 20: from_theta ? solve_n<20, true>(p, start, hand, out, s) : solve_n<20, false>(p, start, hand, out, s); break;
        case 61: from_theta ? solve_n<61, true>(p, start, hand, out, s) : solve_n<61, false>(p, start, hand, out, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t newton_solve_multi(int n, int ncat, int ntiles, const KParams *params, const NewtonState *start,
                              HandArea hand, NewtonState *states, int nbr, hipStream_t s) {
    switch (n) {
        case 4: solve_multi_n<4>(ncat, ntiles, params, start, hand, states, nbr, s); break;
        case 20: solve_multi_n<20>(ncat, ntiles, params, start, hand, states, nbr, s); break;
        case 61: solve_multi_n<61>(ncat, ntiles, params, start, hand, states, nbr, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace plk
