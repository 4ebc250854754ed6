// Newton branch solves in one launch: thin __global__ wrappers over dev_newton.h.
#include <algorithm>
#include <type_traits>

#include "dev_newton.h"

namespace plk {
namespace {
using namespace dev;

// wavefronts per SIMD that the registers of the products leave room for
constexpr int solve_waves(int n) { return n == 61 ? 2 : 4; }
// Tiles of a workgroup.  4 states: four, whose products take a wavefront 32 registers, for many
// branches (3,256 workgroups of one tile 173 us a solve, 814 of four 58) and for one long
// alignment; a short one, where only the latency counts, keeps one (64 taxa x 4,783 patterns: 36.5 -> 34.6 us a branch).
constexpr int solve_tiles(int n) { return n == 4 ? 4 : 1; }
// Categories that a workgroup's LDS has room for.  (Four tiles of 4 states with room for four
// categories are 33 KB, four workgroups a compute unit, which fewer wavefronts each do not fill: three
// categories x 300,000 sites, 12 taxa, an optimisation round 2.1 ms by launches, 1.3 in one.)
constexpr int solve_maxc(int n, int ncat) { return ncat > 4 ? 8 : n == 4 ? ncat : 4; }

// f(MAXC), with the category count as a compile-time bound
template <int N, typename F>
auto with_maxc(int ncat, F &&f) {
    const int m = solve_maxc(N, ncat);
    if constexpr (N == 4) {
        if (m == 1) return f(std::integral_constant<int, 1>{});
        if (m == 2) return f(std::integral_constant<int, 2>{});
        if (m == 3) return f(std::integral_constant<int, 3>{});
    }
    return m == 4 ? f(std::integral_constant<int, 4>{}) : f(std::integral_constant<int, 8>{});
}

// One branch's workgroups of K tiles against a quarter of the places.
template <int N, int K>
bool fits(int ncat, int ntiles, int ncu) {
    const int lds = with_maxc<N>(ncat, [](auto M) { return (int)sizeof(NewtonLds<N, decltype(M)::value, K>); });
    const int places = std::min(160 * 1024 / lds, 4 * solve_waves(N) / ncat);
    return 4 * ((ntiles + K - 1) / K) <= places * ncu;
}

template <int N, bool THETA, int MAXC, int K>
__global__ void __launch_bounds__(64 * MAXC, solve_waves(N)) k_newton_solve(KParams P, NewtonState start, HandArea hand,
                                                                          NewtonState *out) {
    newton_solve_body<N, false, THETA, MAXC, K>(P, blockIdx.x, start, hand.use, hand.spare, hand.spare_len, out);
}

// many branches: the workgroups of a branch are neighbours; states is the host's mirror
template <int N, int MAXC>
__global__ void __launch_bounds__(64 * MAXC, solve_waves(N)) k_newton_solve_multi(
    const KParams *params, int nwg, int64_t hand_len, const NewtonState *start, HandArea hand, NewtonState *states) {
    const int br = blockIdx.x / nwg;
    const KParams P = load_uniform(params + br);
    newton_solve_body<N, true, false, MAXC, solve_tiles(N)>(P, blockIdx.x % nwg, load_uniform(start + br), hand.use + hand_len * br, hand.spare, hand.spare_len, states + br);
}

template <int N, bool THETA, int K>
void solve_k(const KParams &p, const NewtonState &start, HandArea hand, NewtonState *out, hipStream_t s) {
    const dim3 g((p.ntiles + K - 1) / K), b(64 * p.ncat);
    with_maxc<N>(p.ncat, [&](auto M) {
        hipLaunchKernelGGL((k_newton_solve<N, THETA, decltype(M)::value, K>), g, b, 0, s, p, start, hand, out);
    });
}

template <int N, bool THETA>
void solve_n(const KParams &p, const NewtonState &start, HandArea hand, NewtonState *out, hipStream_t s) {
    if (fits<N, 1>(p.ncat, p.ntiles, p.ncu)) solve_k<N, THETA, 1>(p, start, hand, out, s);
    else solve_k<N, THETA, solve_tiles(N)>(p, start, hand, out, s);
}

template <int N>
void solve_multi_n(int ncat, int ntiles, const KParams *params, const NewtonState *start, HandArea hand,
                   NewtonState *states, int nbr, hipStream_t s) {
    const int nwg = (ntiles + solve_tiles(N) - 1) / solve_tiles(N);
    const dim3 g(nbr * nwg), b(64 * ncat);
    with_maxc<N>(ncat, [&](auto M) {
        hipLaunchKernelGGL((k_newton_solve_multi<N, decltype(M)::value>), g, b, 0, s, params, nwg, (int64_t)newton_hand_len(ntiles), start, hand, states);
    });
}

}  // namespace

bool newton_solve_fits(int n, int ncat, int ntiles, int ncu) {
    switch (n) {
        case 4: return fits<4, solve_tiles(4)>(ncat, ntiles, ncu);
        case 20: return fits<20, solve_tiles(20)>(ncat, ntiles, ncu);
        case 61: return fits<61, solve_tiles(61)>(ncat, ntiles, ncu);
        default: return false;
    }
}

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
