// A whole Newton branch solve (minimizeNewton, utils/optimization.cpp:422-499) in one launch.
//
// One derivative evaluation of an alignment of some thousand patterns is about a microsecond of
// arithmetic, so a solve of one launch per evaluation is its launches: on 64 DNA taxa x 4,783
// patterns a branch took seven of 4.1 us each (they are queued six at a time, and half of them
// came after the end of the solve), one more for the first step and two copies of the state:
// 68.6 us in all.  Now it is 34.2, the solve 17.8 of them; both moves of 37 internal branches
// on 40 taxa x 2,800 patterns took 90 launches, now five of 58 us (1,592 -> 652 us).
//
// Here a workgroup keeps the products theta of its 64-pattern tiles in registers (a wavefront per
// category), and the workgroups of a branch exchange their tiles' sums once per evaluation:
// each stores its own, reads all of them in tile order and takes the same step by itself.  A
// sum is its own signal: a place holds a NaN of all ones until the sum comes (a sum that is
// NaN is stored as the ordinary one), so an exchange is one store and one load through the
// device's coherence point.  With a counter raised after the stores it was two of each, and the
// many-branch counters, eight bytes apart, made a launch 700 us.
//
// Three sets of places take turns: a workgroup empties its places of evaluation r + 1 before it
// stores r; it has then read r - 1 from every workgroup, so all have read r - 2, the last to use
// those places.  They are all empty when a launch starts: two areas alternate between the
// launches of a context, and each launch empties the other one.  The workgroup of tile 0
// writes the state to the host.
//
// A wait needs the branch's other workgroups on the device.  The launch rule (newton_solve_fits)
// lets one branch take a quarter of the places (wavefront slots and LDS), and the workgroups of
// a branch are neighbours in dispatch order, so the oldest unfinished branch always gets its
// places once earlier work drains.  Should they still not come (kernels of more than four queues
// that hold each other's places), a wait ends after NewtonState::wait and the workgroup leaves;
// the state stays unfinished and the host solves with one launch per evaluation.
#pragma once

#include "dev_f64.h"

namespace plk {
namespace dev {

__device__ __forceinline__ double hand_empty() { return __longlong_as_double(-1ll); }
__device__ __forceinline__ bool is_empty(double v) { return __double_as_longlong(v) == -1ll; }

// A workgroup's LDS; MAXC: categories it has room for.
template <int N, int MAXC, int K>
struct alignas(16) NewtonLds {
    alignas(16) double val[3][MAXC * N];
    double cat[K][3][MAXC][64], inv[K][64], freq[K][64];
    NewtonState st;
    int sc[K][MAXC][64], go;
};

// L3: many-branch form (the logL of every evaluation, and one more evaluation at the answer where
// bisection ended on an older point).  THETA: the products are read from P.theta instead of
// formed from the partials at the branch.  hand: 3 NV ntiles empty places; spare: the places that
// the solve before this one used, emptied here for the next one.
template <int N, bool L3, bool THETA, int MAXC, int K>
__device__ inline void newton_solve_body(const KParams &P, const int wg, const NewtonState &start, double *hand,
                                         double *spare, int64_t spare_len, NewtonState *out) {
    constexpr int NV = L3 ? 3 : 2;
    const int lane = threadIdx.x & 63, c = wave_id(), ncat = P.ncat;
    __shared__ NewtonLds<N, MAXC, K> s;
    auto &s_val = s.val;
    auto &s_cat = s.cat;
    auto &s_sc = s.sc;
    auto &s_inv = s.inv, &s_freq = s.freq;
    auto &s_st = s.st;
    auto &s_go = s.go;
    if (threadIdx.x == 0) s_st = start;
    const uint64_t wait = (uint64_t)start.wait;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < spare_len; i += (int64_t)gridDim.x * blockDim.x)
        spare[i] = hand_empty();
    // a last workgroup with fewer tiles takes the alignment's last one again and drops its sums
    auto tile_of = [&](int k) { return min(wg * K + k, P.ntiles - 1); };
    double th[K][N];
    int sc[K];  // scale count of this lane's pattern (its minimum over the categories)
    double *__restrict__ theta = (double *)P.theta;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int tile = tile_of(k);
        const int64_t p = (int64_t)tile * 64 + lane;
        const int64_t toff = ((int64_t)tile * ncat + c) * N * 64 + lane;
        sc[k] = 0;
        if constexpr (THETA) {
#pragma unroll
            for (int i = 0; i < N; i++) th[k][i] = theta[toff + i * 64];
        } else {
            // theta = node * dad (2187-2193; tip 2104-2145)
            const int64_t off = ((int64_t)tile * ncat + c) * N * 64 + f64_loff(N, lane);
            const double *__restrict__ B = (const double *)P.part + (int64_t)P.br_b * P.slot_stride + off;
            const uint16_t *__restrict__ scB = (const uint16_t *)P.scale + (int64_t)P.br_b * P.scale_stride;
            const int64_t a = P.safe ? p * ncat + c : p;
            sc[k] = scB[a];
            if (P.br_a < 0) {
                const double *__restrict__ tip = P.tip_lh + P.states[(int64_t)(-P.br_a - 1) * P.nptn_pad + p] * N;
#pragma unroll
                for (int i = 0; i < N; i++) th[k][i] = tip[i] * B[f64_xoff(N, i)];
            } else {
                const double *__restrict__ A = (const double *)P.part + (int64_t)P.br_a * P.slot_stride + off;
                sc[k] += ((const uint16_t *)P.scale + (int64_t)P.br_a * P.scale_stride)[a];
#pragma unroll
                for (int i = 0; i < N; i++) th[k][i] = A[f64_xoff(N, i)] * B[f64_xoff(N, i)];
            }
            s_sc[k][c][lane] = sc[k];
        }
    }
    __syncthreads();
    if constexpr (!THETA) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int tile = tile_of(k);
            const int64_t p = (int64_t)tile * 64 + lane;
            // categories above the minimum count (2146-2171, 2194-2225)
            int mn = s_sc[k][0][lane];
            for (int q = 1; q < ncat; q++) mn = min(mn, s_sc[k][q][lane]);
            if (sc[k] != mn) {
                const double f = safe_factor(sc[k] - mn);
#pragma unroll
                for (int i = 0; i < N; i++) th[k][i] *= f;
            }
            sc[k] = mn;
            if (theta)
#pragma unroll
                for (int i = 0; i < N; i++) theta[((int64_t)tile * ncat + c) * N * 64 + lane + i * 64] = th[k][i];
            if (c == 0 && P.buf_scale) P.buf_scale[p] = mn * kLogST;
        }
    }
    for (int k = c; k < K; k += ncat) {
        const int64_t p = (int64_t)tile_of(k) * 64 + lane;
        s_inv[k][lane] = P.invar[p];
        s_freq[k][lane] = p < P.nptn ? P.freq[p] : 0.0;
    }
    // fill_val's factors: N values of a category for its wavefront
    const int vi = min(lane, N - 1);
    const double cof = P.eval[vi] * P.rates[c], prop = P.props[c];
    const int64_t hlen = (int64_t)NV * P.ntiles;
    for (int r = 0;; r++) {
        // this workgroup's places of the next evaluation are emptied; that is complete before
        // this evaluation's sums go out
        double *now = hand + (r % 3) * hlen, *next = hand + ((r + 1) % 3) * hlen;
        if (lane < NV && r > 0)
            for (int k = c; k < K && wg * K + k < P.ntiles; k += ncat) publish(&next[NV * (wg * K + k) + lane], hand_empty());
        if (lane < N) {
            const double val = exp(cof * s_st.rts) * prop, val1 = cof * val;
            s_val[0][c * N + lane] = val;
            s_val[1][c * N + lane] = val1;
            s_val[2][c * N + lane] = cof * val1;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const double *v0 = s_val[0] + c * N, *v1 = s_val[1] + c * N, *v2 = s_val[2] + c * N;
#pragma unroll
        for (int k = 0; k < K; k++) {
            double l0 = 0.0, l1 = 0.0, l2 = 0.0;
#pragma unroll
            for (int i = 0; i < N; i++) {
                l0 = fma(v0[i], th[k][i], l0);
                l1 = fma(v1[i], th[k][i], l1);
                l2 = fma(v2[i], th[k][i], l2);
            }
            s_cat[k][0][c][lane] = l0;
            s_cat[k][1][c][lane] = l1;
            s_cat[k][2][c][lane] = l2;
        }
        __syncthreads();
        for (int k = c; k < K && wg * K + k < P.ntiles; k += ncat) {
            const int tile = wg * K + k;
            const int64_t p = (int64_t)tile * 64 + lane;
            const bool mine = p < P.nptn;
            double lh = 0.0, d1 = 0.0, d2 = 0.0;
            for (int q = 0; q < ncat; q++) {
                lh += s_cat[k][0][q][lane];
                d1 += s_cat[k][1][q][lane];
                d2 += s_cat[k][2][q][lane];
            }
            lh = fabs(lh) + s_inv[k][lane];
            const double freq = s_freq[k][lane];
            const double inv = 1.0 / lh;
            const double dfr = d1 * inv, ddfr = d2 * inv;
            const double t1 = dfr * freq, t2 = ddfr * freq;
            if (P.g_frac && mine) P.g_frac[p] = dfr;  // G_matrix row (2518)
            double v[NV];
            v[0] = wave_sum(mine ? t1 : 0.0);
            v[1] = wave_sum(mine ? t2 - t1 * dfr : 0.0);
            if constexpr (L3) {
                int mn = s_sc[k][0][lane];
                for (int q = 1; q < ncat; q++) mn = min(mn, s_sc[k][q][lane]);
                v[2] = wave_sum(mine ? (log(lh) + mn * kLogST) * freq : 0.0);
            }
            if (r > 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (lane == 0) {
#pragma unroll
                for (int q = 0; q < NV; q++) publish(&now[NV * tile + q], v[q] == v[q] ? v[q] : (double)NAN);
            }
        }
        if (c == 0) {
            const uint64_t t0 = wall_clock64();
            bool ok = true;
            double v[NV];
#pragma unroll
            for (int q = 0; q < NV; q++) v[q] = 0.0;
            for (int i = lane; i < P.ntiles; i += 64) {
                double x[NV];
                for (;;) {
                    bool full = true;
#pragma unroll
                    for (int q = 0; q < NV; q++) {
                        x[q] = __hip_atomic_load(&now[NV * i + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        full = full && !is_empty(x[q]);
                    }
                    if (full) break;
                    if (wall_clock64() - t0 >= wait) {
                        ok = false;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
#pragma unroll
                for (int q = 0; q < NV; q++) v[q] += x[q];
            }
            ok = __all(ok);
#pragma unroll
            for (int q = 0; q < NV; q++) v[q] = wave_sum(v[q]);
            if (lane == 0) {
                NewtonState t = s_st;  // in registers: the step reads and writes its fields some 40 times
                if (ok) {
                    if constexpr (L3) {
                        const bool extra = t.eval_only != 0;
                        newton_record(t, v[0], v[1], v[2]);
                        if (t.done && !extra && t.status == NEWTON_OK && t.out != t.x_eval) {
                            t.rts = t.out;
                            t.eval_only = 1;
                            t.done = 0;
                        }
                    } else {
                        newton_after_eval(t, v[0], v[1]);
                    }
                    s_st = t;
                }
                s_go = ok && !t.done;
            }
        }
        __syncthreads();
        if (!s_go) break;
    }
    if (wg == 0 && threadIdx.x == 0 && s_st.done) *out = s_st;
}

}  // namespace dev
}  // namespace plk
