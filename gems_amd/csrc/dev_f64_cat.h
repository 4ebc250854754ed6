// FP64 traversal of 20-state models on the matrix cores: four categories side by side in one
// wavefront, and two constant matrices.
//
// Per op and category the eigen-space partial (tree/phylokernelnew.h:1911-2036) is
//   a = E_L L,  b = E_R R  (E = U diag(exp(Lambda r t))),  out = U^-1 (a o b)
// with tip children replaced by leaf-table rows (1729-1747, 1848-1890).  Written as
// a = U (exp(Lambda r t) o L), the matrices are U and U^-1 for every op, side and category, so
// they are in LDS for the whole launch (read anew in each product: in registers they would
// take 50 each) and an op reads from memory only its children's rows and 20 exponentials
// per side and category (reading E instead, 12.8 KB per side and
// wavefront, kept the vector L1 busy 70 % of the time: 1.60 ms for 100 taxa x 49,994
// patterns).
//
// The matrix instruction is v_mfma_f64_4x4x4_4b_f64, four independent 4 x 4 x 4 products:
// block b takes category b, its columns four patterns, so 20 states are 5 x 5 tiles without
// padding.  Lane layout (checked on the device): A[i][k] of block b in lane i + 4 b + 16 k,
// B[k][j] in lane j + 4 b + 16 k, D[i][j] in lane j + 4 b + 16 i.  D is laid out as the next
// product's B: a o b goes straight into the U^-1 product and an op's output straight into the
// next op, with nothing exchanged between lanes.  Measured on this card the 4 x 4 x 4
// instruction runs at 61 TFLOP/s, the 16 x 16 x 4 one at 47.
//
// A wavefront owns PG patterns per column (4 PG patterns) and all categories of them, so the
// scaling check over a pattern's categories (2019-2034, 1893-1907) is a ballot and the op
// loop has no barrier.  PG = 2 has twice the independent products; PG = 1 spreads a short
// alignment over more wavefronts.  One or two categories put pattern groups into
// the blocks that would be idle; 5-8 categories take two wavefronts, which then meet at
// the NORM check (SAFE checks each category alone).
#pragma once

#include "dev_common.h"

namespace plk {
namespace dev {

typedef double double2_t __attribute__((ext_vector_type(2)));

// d = M v for a 20 x 20 matrix in LDS (mc_frag order, read as 16-byte broadcasts); al = 4 k + i.
// The tiles of a k step are read while the previous step's products run: the barriers
// keep the compiler from holding the whole matrix in registers (25 tiles, 50 registers).
template <int PG>
__device__ __forceinline__ void mc_product(const double *F, int al, const double (&v)[5][PG], double (&d)[5][PG]) {
    double m[2][5];
    auto load = [&](int ks, double(&t)[5]) {
        const double2_t p = *(const double2_t *)(F + 80 * ks + 2 * al), q = *(const double2_t *)(F + 80 * ks + 32 + 2 * al);
        t[0] = p.x;
        t[1] = p.y;
        t[2] = q.x;
        t[3] = q.y;
        t[4] = F[80 * ks + 64 + al];
    };
#pragma unroll
    for (int xb = 0; xb < 5; xb++)
#pragma unroll
        for (int q = 0; q < PG; q++) d[xb][q] = 0.0;
    load(0, m[0]);
#pragma unroll
    for (int ks = 0; ks < 5; ks++) {
        if (ks < 4) load(ks + 1, m[(ks + 1) & 1]);
#pragma unroll
        for (int xb = 0; xb < 5; xb++)
#pragma unroll
            for (int q = 0; q < PG; q++)
                d[xb][q] = __builtin_amdgcn_mfma_f64_4x4x4f64(m[ks & 1][xb], v[ks][q], d[xb][q], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// PG consecutive values
template <int PG>
__device__ __forceinline__ void load_pg(const double *__restrict__ s, double (&v)[PG]) {
    if constexpr (PG == 1) {
        v[0] = s[0];
    } else {
#pragma unroll
        for (int q = 0; q < PG; q += 2) {
            const double2_t t = *(const double2_t *)(s + q);
            v[q] = t.x;
            v[q + 1] = t.y;
        }
    }
}
template <int PG>
__device__ __forceinline__ void store_pg(double *__restrict__ d, const double (&v)[PG]) {
    if constexpr (PG == 1) {
        d[0] = v[0];
    } else {
#pragma unroll
        for (int q = 0; q < PG; q += 2) *(double2_t *)(d + q) = double2_t{v[q], v[q + 1]};
    }
}

// fixed shuffle tree over each group of 16 lanes; valid in its first lane
__device__ __forceinline__ double sum16(double v) {
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// One workgroup: four pattern units of mc_unit(PG, ncat) patterns each (a wavefront per unit
// and group of four categories), 16, 32 or 64 patterns; wg counts them.
template <int MODE, int PG>
__device__ inline void traverse_f64_cat_body(const KParams &P, const int wg) {
    constexpr int N = 20, KS = 5;
    const int lane = threadIdx.x & 63, j = lane & 3, b = (lane >> 2) & 3, k4 = lane >> 4;
    const int ncat = P.ncat, ngrp = (ncat + 3) >> 2;
    const int ncb = ncat >= 3 ? 4 : ncat;  // categories side by side in a wavefront
    const int up_ = mc_unit(PG, ncat);     // patterns of a wavefront
    const int w = wave_id();
    const bool live = w < 4 * ngrp;  // batched launches: further wavefronts only join barriers
    const int unit = live ? w / ngrp : 0, grp = live ? w % ngrp : 0;
    const int cw = grp * 4 + b % ncb;
    const bool mine = live && cw < ncat;   // this lane's category exists
    const int c = min(cw, ncat - 1);
    const int nb = min(ncat - 4 * grp, 4);
    const int lt = k4 * nb + (c - 4 * grp);  // this lane's place in a row of mc_leaf order
    const int wp = unit * up_ + (b / ncb) * 4 * PG + j * PG;   // first pattern within the workgroup
    const int64_t p = (int64_t)wg * 4 * up_ + wp;
    const int tile = (int)(p >> 6), pl = (int)(p & 63);
    const bool safe = P.safe != 0, meet = !safe && ngrp > 1;
    double *__restrict__ part = (double *)P.part + ((int64_t)tile * ncat + c) * N * 64 + f64_loff(N, pl) + 8 * k4;
    uint16_t *__restrict__ scale = (uint16_t *)P.scale + (safe ? p * ncat + c : p);
    const int sstep = safe ? ncat : 1;  // pattern to pattern in the scale counts
    const uint8_t *__restrict__ states = P.states + p;
    const bool counts = mine && k4 == 0 && (safe || cw == 0);  // this lane keeps scale counts
    bool noinv[PG];
#pragma unroll
    for (int q = 0; q < PG; q++) noinv[q] = P.invar[p + q] == 0.0;
    __shared__ unsigned s_nb[2][4][2][PG];                // not-below masks of a unit's two groups
    __shared__ double s_cat[PLK_GPU_MAX_CATS][64];
    __shared__ int s_sc[PLK_GPU_MAX_CATS][64];

    // U^-1 and U in fragment order, read as 16-byte broadcasts
    __shared__ __attribute__((aligned(16))) double s_u[800];
    for (int i = threadIdx.x; i < 800; i += blockDim.x) s_u[i] = P.uinv_frag[i];
    __syncthreads();
    auto product = [&](const double *F, const double(&v)[KS][PG], double(&d)[KS][PG]) {
        mc_product<PG>(F, 4 * k4 + j, v, d);
    };

    auto load_rows = [&](int slot, double(&v)[KS][PG]) {
        const double *__restrict__ C = part + (int64_t)slot * P.slot_stride;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) load_pg<PG>(C + 32 * ks, v[ks]);
    };
    auto load_counts = [&](int slot, unsigned(&v)[PG]) {
        const uint16_t *__restrict__ s = scale + (int64_t)slot * P.scale_stride;
#pragma unroll
        for (int q = 0; q < PG; q++) v[q] = s[q * sstep];
    };
    auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // 20 values per category in mc_leaf order: this lane's five
    auto load_row = [&](const double *__restrict__ row, double(&v)[KS]) {
        row += grp * 80;
        const double2_t q0 = *(const double2_t *)(row + 2 * lt), q1 = *(const double2_t *)(row + 8 * nb + 2 * lt);
        v[0] = q0.x;
        v[1] = q0.y;
        v[2] = q1.x;
        v[3] = q1.y;
        v[4] = row[16 * nb + lt];
    };
    auto table = [&](const double *__restrict__ tab, unsigned st, double(&v)[KS][PG]) {
#pragma unroll
        for (int q = 0; q < PG; q++) {
            double t[KS];
            load_row(tab + (int64_t)((st >> (8 * q)) & 255) * ncat * N, t);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) v[ks][q] = t[ks];
        }
    };
    auto state = [&](bool tip, int taxon) -> unsigned {
        // (an internal child's slot is not a taxon: read taxon 0 and ignore it)
        const uint8_t *__restrict__ s = states + (int64_t)(tip ? taxon : 0) * P.nptn_pad;
        if constexpr (PG == 1) return *s;
        return *(const uint16_t *)s;
    };
    // In a post-order list nearly every op has the previous op's output as a child: it stays
    // in registers (cv, cc) and is not read back, and its stores are issued after the next
    // op's loads, so that no load waits behind them (a wavefront's vector memory operations
    // complete in issue order).
    double cv[KS][PG];
    unsigned cc[PG];
    int prev_out = -1;
#pragma unroll
    for (int q = 0; q < PG; q++) {
        cc[q] = 0;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) cv[ks][q] = 0.0;
    }
    // straight-line (a branch would make the waits for the next op's loads cover these
    // stores too): no real target -> the context's sink
    auto store_carried = [&]() {
        double *__restrict__ po = (prev_out >= 0 && mine) ? part + (int64_t)prev_out * P.slot_stride : (double *)P.sink;
        uint16_t *__restrict__ ps = (prev_out >= 0 && counts) ? scale + (int64_t)prev_out * P.scale_stride : (uint16_t *)P.sink;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) store_pg<PG>(po + 32 * ks, cv[ks]);
#pragma unroll
        for (int q = 0; q < PG; q++) ps[q * sstep] = (uint16_t)cc[q];
    };
    // op descriptors and tip states are fetched one op ahead
    const int last = P.nops - 1;
    DevOp nxt{};
    unsigned nl = 0, nr = 0;
    auto prefetch = [&](int k) {
        nxt = load_op(P.ops, k);
        nl = state(nxt.kind <= KIND_TI, nxt.left);
        nr = state(nxt.kind == KIND_TT, nxt.right);
    };
    if (last >= 0) prefetch(0);
    int par = 0;
    for (int k = 0; k <= last; k++) {
        const DevOp op = nxt;
        const unsigned stl = nl, str = nr;
        const double *__restrict__ M = (const double *)P.mats + (int64_t)k * P.mat_stride;
        const double *__restrict__ tabs = M + (int64_t)2 * ncat * N * N;
        with_kind(op.kind, [&](auto KC) {
            constexpr int KIND = decltype(KC)::value;
            const bool carry = KIND != KIND_TT && op.right == prev_out;
            if (KIND == KIND_II && op.left == prev_out) {
                store_carried();  // read from memory: written first
                fence();
            }
            double xr[KS], xl[KS], r[KS][PG], l[KS][PG], o[KS][PG];
            unsigned sc[PG];
            if constexpr (KIND != KIND_TT) {
                load_row(M + (int64_t)ncat * N * N, xr);
                if (carry) {
#pragma unroll
                    for (int q = 0; q < PG; q++) {
                        sc[q] = cc[q];
#pragma unroll
                        for (int ks = 0; ks < KS; ks++) r[ks][q] = cv[ks][q];
                    }
                } else {
                    load_rows(op.right, r);
                    load_counts(op.right, sc);
                }
            } else {
                table(tabs + (int64_t)(P.su + 1) * ncat * N, str, r);
#pragma unroll
                for (int q = 0; q < PG; q++) sc[q] = 0;
            }
            unsigned sl[PG];
            if constexpr (KIND == KIND_II) {
                load_row(M, xl);
                load_rows(op.left, l);
                load_counts(op.left, sl);
            } else {
                table(tabs, stl, l);
            }
            fence();
            store_carried();
            prefetch(min(k + 1, last));
            if constexpr (KIND != KIND_TT) {
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
#pragma unroll
                    for (int q = 0; q < PG; q++) r[ks][q] *= xr[ks];
                product(s_u + 400, r, o);
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
#pragma unroll
                    for (int q = 0; q < PG; q++) r[ks][q] = o[ks][q];
            }
            if constexpr (KIND == KIND_II) {
#pragma unroll
                for (int q = 0; q < PG; q++) sc[q] += sl[q];
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
#pragma unroll
                    for (int q = 0; q < PG; q++) l[ks][q] *= xl[ks];
                product(s_u + 400, l, o);
#pragma unroll
                for (int ks = 0; ks < KS; ks++)
#pragma unroll
                    for (int q = 0; q < PG; q++) l[ks][q] = o[ks][q];
            }
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int q = 0; q < PG; q++) l[ks][q] *= r[ks][q];
            product(s_u, l, o);
            if constexpr (KIND != KIND_TT) {
                // lanes with a value at or above 2^-256, folded onto the lanes of a pattern
                unsigned not_below[PG];
#pragma unroll
                for (int q = 0; q < PG; q++) {
                    double m = 0.0;
#pragma unroll
                    for (int ks = 0; ks < KS; ks++) m = fmax(m, fabs(o[ks][q]));
                    const unsigned long long x = __ballot(mine && !(m < kST));
                    unsigned y = (unsigned)(x | x >> 32);
                    y = (y | y >> 16) & 0xffffu;  // [block][column]
                    if (!safe) {
                        if (ncb > 1) y |= (y >> 4 & 0x0f0fu) | (y << 4 & 0xf0f0u);  // blocks 0, 1 and 2, 3
                        if (ncb > 2) y = (y | y >> 8 | y << 8) & 0xffffu;
                    }
                    not_below[q] = y;
                }
                if (meet) {
                    // the other four categories' wavefront
                    if (live && lane == 0)
#pragma unroll
                        for (int q = 0; q < PG; q++) s_nb[par][unit][grp][q] = not_below[q];
                    __syncthreads();
#pragma unroll
                    for (int q = 0; q < PG; q++) not_below[q] = s_nb[par][unit][0][q] | s_nb[par][unit][1][q];
                    par ^= 1;
                }
#pragma unroll
                for (int q = 0; q < PG; q++) {
                    const bool up = !(not_below[q] >> (lane & 15) & 1) && noinv[q];
                    if (__any(up)) {
                        const double f = up ? kTwo256 : 1.0;
                        sc[q] += up ? 1 : 0;
#pragma unroll
                        for (int ks = 0; ks < KS; ks++) o[ks][q] *= f;
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < PG; q++) {
                cc[q] = sc[q];
#pragma unroll
                for (int ks = 0; ks < KS; ks++) cv[ks][q] = o[ks][q];
            }
        });
        prev_out = op.out_slot;
        fence();
    }
    if (prev_out >= 0) {
        store_carried();
        fence();
    }
    if (MODE == MODE_PARTIALS) return;

    // -------- branch logL: lh_c = sum_i val_i a_i b_i (2903-2914, 3044-3057)
    const bool atip = P.br_a < 0;
    {
        double x[KS][PG], y[KS][PG];
        unsigned sb[PG], sa[PG];
        load_rows(P.br_b, y);
        load_counts(P.br_b, sb);
        if (atip) {
            const unsigned st = state(true, -P.br_a - 1);
#pragma unroll
            for (int q = 0; q < PG; q++) {
                sa[q] = 0;
#pragma unroll
                for (int ks = 0; ks < KS; ks++) x[ks][q] = P.tip_lh[(st >> (8 * q) & 255) * N + 5 * k4 + ks];
            }
        } else {
            load_rows(P.br_a, x);
            load_counts(P.br_a, sa);
        }
        double acc[PG];
#pragma unroll
        for (int q = 0; q < PG; q++) acc[q] = 0.0;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const double cof = P.eval[5 * k4 + ks] * P.rates[c];
            const double val = exp(cof * P.br_len) * P.props[c];
#pragma unroll
            for (int q = 0; q < PG; q++) acc[q] = fma(val * x[ks][q], y[ks][q], acc[q]);
        }
#pragma unroll
        for (int q = 0; q < PG; q++) {
            acc[q] += __shfl_xor(acc[q], 16, 64);
            acc[q] += __shfl_xor(acc[q], 32, 64);
            if (mine && k4 == 0) {
                s_cat[c][wp + q] = acc[q];
                s_sc[c][wp + q] = (int)(sb[q] + sa[q]);
            }
        }
    }
    __syncthreads();
    const int wpat = 4 * up_;  // patterns of the workgroup: wavefront 0 finishes them
    double sum = 0.0;
    if (w == 0) {
        const int64_t pp = (int64_t)wg * wpat + lane;
        if (lane < wpat && pp < P.nptn) {
            int mn = s_sc[0][lane];
            if (safe)
                for (int cc = 1; cc < ncat; cc++) mn = min(mn, s_sc[cc][lane]);
            // categories above the minimum count are scaled by 2^-256 or dropped (2918-2944)
            auto value = [&](int cc) {
                const int d = safe ? s_sc[cc][lane] - mn : 0;
                return s_cat[cc][lane] * (d == 0 ? 1.0 : (d == 1 ? kST : 0.0));
            };
            double lh = 0.0;
            for (int cc = 0; cc < ncat; cc++) lh += value(cc);
            const double lg = log(fabs(lh) + P.invar[pp]) + mn * kLogST;
            P.ptn_lh[pp] = lg;
            if (P.ptn_lh_cat) {
                for (int cc = 0; cc < ncat; cc++) P.ptn_lh_cat[pp * ncat + cc] = value(cc);
                P.ptn_scaling[pp] = mn * kLogST;
            }
            sum = lg * P.freq[pp];
        }
        sum = sum16(sum);
    }
    finish_blocks(P, sum, wg, wpat >> 4);
}

}  // namespace dev
}  // namespace plk
