// FP64 traversal of 61-state models on the matrix cores: a wavefront takes four patterns of
// one category through the op list, with U in its registers and U^-1 in LDS.
//
// Per op and category the eigen-space partial (tree/phylokernelnew.h:1911-2036) is
//   a = U (exp(Lambda r t_L) o L),  b alike,  out = U^-1 (a o b)
// with tip children replaced by leaf-table rows (1729-1747, 1848-1890), so an op reads 61
// exponentials a side where E = U diag(exp) would be 30 KB.
//
// The instruction is v_mfma_f64_4x4x4_4b_f64 (61 TFLOP/s on this card; 16 x 16 x 4: 47), four
// independent 4 x 4 x 4 products.  Block b takes the states 16 R + 4 b + k as its share of the
// sum, its columns are the wavefront's four patterns.  Lane j + 4 b + 16 k then holds the
// states 16 R + 4 b + k (R = 0..3) of pattern j: a child, 61 x 4 values, is four registers
// a lane and nothing is held twice.  A product is 64 instructions; accumulator (R, s) of
// block b collects its share of the rows 16 R + 4 ((b + s) mod 4) + i, so that adding the
// four accumulators of an R rotated by s blocks within each row of 16 lanes puts row
// 16 R + 4 b + i where the next product reads it.  U in this order is 64 registers of doubles,
// loaded once per workgroup, U^-1 is read from LDS (both in registers leave one wavefront a
// SIMD, which issues these instructions every 31 cycles; two reach 20).
//
// Scaling as the reference: SAFE checks each category alone, and a workgroup is four
// wavefronts of one category (16 patterns); NORM checks max |out| over the categories of a
// pattern, and a workgroup is the categories of four patterns, which meet at a barrier.
// A lane reads back only what it stored itself, so the op loop needs no other exchange.
// The sums run in another order than the vector kernels', so values differ at the rounding
// level (checked against the oracle's 1e-10).
//
// The sums differ from the former E L on 16 x 16 x 4 tiles in the last places; against long
// double the logL of simulated codon patterns is 0.6-1.0 times as far off (rms, 20-100 taxa).
//
// 48 taxa x 4,700 patterns x 4 categories, SAFE: 700 us with E from memory, a wavefront per
// 16 rows and three barriers an op; 390 us now.  The matrix instructions alone take 180 us;
// the units are 2.3 for each workgroup that fits (three rounds), and 29 % of the wavefronts'
// cycles wait.  Measured on the way: partials as rows of 64 patterns (16 pieces of 32 bytes a
// load) 530 us; U^-1 in registers too, one wavefront a SIMD, 540.
#pragma once

#include "dev_common.h"

namespace plk {
namespace dev {

typedef double codon_d2 __attribute__((ext_vector_type(2)));

// y = sum over s of d[s] from s blocks (of four lanes) below, in each row of 16 lanes
template <int S>
__device__ __forceinline__ double codon_rotate(double v) {
    constexpr int ctrl = 0x120 + 4 * S;  // row_ror
    int2 w = __builtin_bit_cast(int2, v);
    w.x = __builtin_amdgcn_update_dpp(0, w.x, ctrl, 0xf, 0xf, true);
    w.y = __builtin_amdgcn_update_dpp(0, w.y, ctrl, 0xf, 0xf, true);
    return __builtin_bit_cast(double, w);
}

// y = M x, the tiles of M from get(R, q, t): the four of row group R and states q.  A row group at
// a time: four products in flight and 8 registers of sums.
template <typename F>
__device__ __forceinline__ void codon_product(F &&get, const double (&x)[4], double (&y)[4]) {
    double v[4];
#pragma unroll
    for (int R = 0; R < 4; R++) {
        double d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            double t[4];
            get(R, q, t);
#pragma unroll
            for (int s = 0; s < 4; s++) d[s] = __builtin_amdgcn_mfma_f64_4x4x4f64(t[s], x[q], d[s], 0, 0, 0);
        }
        v[R] = (d[0] + codon_rotate<1>(d[1])) + (codon_rotate<2>(d[2]) + codon_rotate<3>(d[3]));
    }
#pragma unroll
    for (int R = 0; R < 4; R++) y[R] = v[R];
}

// The op list for the patterns 16 blk + 4 quad .. + 3 of category c.  s_ok: NORM's exchange, two
// buffers used in turn (turn goes on over the units: not every op has an exchange).
template <bool SAFE>
__device__ inline void traverse_f64_codon_body(const KParams &P, const int blk, const int quad, const int c,
                                               const double (&U)[4][4][4], const double *s_ui, unsigned (*s_ok)[PLK_GPU_MAX_CATS],
                                               int &turn) {
    constexpr int N = 61;
    const int lane = threadIdx.x & 63, j = lane & 3, s4 = ((lane >> 2) & 3) * 4 + (lane >> 4);
    const int ncat = P.ncat, tile = blk >> 2, pl = (blk & 3) * 16 + quad * 4 + j;
    const int64_t p = (int64_t)tile * 64 + pl;
    const int64_t cbase = ((int64_t)tile * ncat + c) * N * 64 + ((blk & 3) * 4 + quad) * 4 * N;  // (f64_loff)
    const int64_t at = SAFE ? p * ncat + c : p;  // the pattern's scale count
    double *__restrict__ part = (double *)P.part;
    uint16_t *__restrict__ scale = (uint16_t *)P.scale;
    const bool noinv = P.invar[p] == 0.0;
    // the lane's rows 16 R + s4; past the last one it repeats row 60 and stores to the sink
    // (U's columns and the exponentials are zero there); bytes from the quad's block
    unsigned row[4], at_row[4];
#pragma unroll
    for (int R = 0; R < 4; R++) {
        row[R] = min(16 * R + s4, N - 1) * 8;
        at_row[R] = row[R] * 4 + j * 8;
    }
    const bool last = 48 + s4 < N;
    const unsigned at_e = s4 * 8, at_n = (unsigned)at * 2, st_step = ncat * N * 8;

    // the operands of one side of the op at hand
    struct Side {
        double v[4], e[4];
        unsigned n, st;
    };
    Side lft{}, rgt{};
    double cv[4] = {0.0, 0.0, 0.0, 0.0};  // the last op's output, with its count
    unsigned cn = 0;
    // Straight-line loads: behind a branch the wait for them would cover the last op's
    // stores too, so a tip reads some count and exponentials that it leaves alone, and a
    // child that is still in registers is read from memory in vain.
    auto fetch_side = [&](int k, const DevOp &op, int side, bool tip, int ref, Side &d) {
        const char *M = (const char *)((const double *)P.mats + (int64_t)k * P.mat_stride);
        const char *src = tip ? M + (2 * ncat * N * N + side * (P.su + 1) * ncat * N + c * N) * 8
                              : (const char *)(part + (int64_t)ref * P.slot_stride + cbase);
        const unsigned tab = d.st * st_step;
#pragma unroll
        for (int R = 0; R < 4; R++) d.v[R] = *(const double *)(src + (tip ? tab + row[R] : at_row[R]));
        const char *e = M + (side * ncat * N * N + c * 64) * 8;
#pragma unroll
        for (int R = 0; R < 4; R++) d.e[R] = *(const double *)(e + at_e + 128 * R);
        d.n = *(const uint16_t *)((const char *)(scale + (int64_t)(tip ? op.out_slot : ref) * P.scale_stride) + at_n);
    };
    auto fetch = [&](int k, const DevOp &op) {
        fetch_side(k, op, 0, op.kind <= KIND_TI, op.left, lft);
        fetch_side(k, op, 1, op.kind == KIND_TT, op.right, rgt);
    };
    auto states = [&](const DevOp &op) {
        lft.st = P.states[(int64_t)(op.kind <= KIND_TI ? op.left : 0) * P.nptn_pad + p];
        rgt.st = P.states[(int64_t)(op.kind == KIND_TT ? op.right : 0) * P.nptn_pad + p];
    };
    const int last_op = P.nops - 1;
    DevOp op = load_op(P.ops, 0), nxt = load_op(P.ops, min(1, last_op)), ahead = load_op(P.ops, min(2, last_op));
    states(op);
    fetch(0, op);
    states(nxt);
    int before = -1;
    for (int k = 0; k <= last_op; k++) {
        const bool ltip = op.kind <= KIND_TI, rtip = op.kind == KIND_TT;
        const bool lcarry = !ltip && op.left == before, rcarry = !rtip && op.right == before;
        double a[4], b[4], y[4];
        auto take = [&](const Side &d, bool tip, bool carry, double(&x)[4]) {
            if (tip) {
#pragma unroll
                for (int R = 0; R < 4; R++) x[R] = d.v[R];
            } else if (carry) {
#pragma unroll
                for (int R = 0; R < 4; R++) x[R] = cv[R] * d.e[R];
            } else {
#pragma unroll
                for (int R = 0; R < 4; R++) x[R] = d.v[R] * d.e[R];
            }
            return tip ? 0u : carry ? cn : d.n;
        };
        unsigned n = take(rgt, rtip, rcarry, a) + take(lft, ltip, lcarry, b);
        fetch(min(k + 1, last_op), nxt);
        states(ahead);
        const DevOp ahead2 = load_op(P.ops, min(k + 3, last_op));
        auto tiles_u = [&](int R, int q, double(&t)[4]) {
#pragma unroll
            for (int s = 0; s < 4; s++) t[s] = U[R][s][q];
        };
        if (!rtip) codon_product(tiles_u, a, a);
        if (!ltip) codon_product(tiles_u, b, b);
#pragma unroll
        for (int R = 0; R < 4; R++) a[R] *= b[R];
        int f = 2 * lane;
        asm volatile("" : "+v"(f));  // read per op, not held in registers
        codon_product([&](int R, int q, double(&t)[4]) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const codon_d2 v = *(const codon_d2 *)(s_ui + f + ((R * 4 + q) * 2 + h) * 128);
                t[2 * h] = v.x;
                t[2 * h + 1] = v.y;
            }
        }, a, y);

        if (op.kind != KIND_TT) {
            // bit j: pattern j has a value at or above 2^-256 (2019-2034, 1997-2013)
            bool big = false;
#pragma unroll
            for (int R = 0; R < 4; R++) big = big || (fabs(y[R]) >= kST && (R < 3 || last));
            unsigned long long m = __ballot(big);
            unsigned ok = (unsigned)(m | m >> 32);
            ok |= ok >> 16;
            ok |= ok >> 8;
            ok = (ok | ok >> 4) & 0xf;
            if (!SAFE) {
                unsigned *s = s_ok[turn ^= 1];
                if (lane == 0) s[c] = ok;
                // (LDS only: the stores in flight are this wavefront's own business)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                for (int q = 0; q < ncat; q++) ok |= s[q];
            }
            const bool up = !(ok >> j & 1) && noinv;
#pragma unroll
            for (int R = 0; R < 4; R++) y[R] = up ? y[R] * kTwo256 : y[R];
            n += up ? 1u : 0u;
        }
        char *out = (char *)(part + (int64_t)op.out_slot * P.slot_stride + cbase);
#pragma unroll
        for (int R = 0; R < 3; R++) *(double *)(out + at_row[R]) = y[R];
        *(double *)(last ? out + at_row[3] : (char *)P.sink) = y[3];
        *(uint16_t *)((char *)(scale + (int64_t)op.out_slot * P.scale_stride) + at_n) = (uint16_t)n;
#pragma unroll
        for (int R = 0; R < 4; R++) cv[R] = y[R];
        cn = n & 0xffffu;
        before = op.out_slot;
        op = nxt;
        nxt = ahead;
        ahead = ahead2;
    }
}

// P(t) data of a (job, category) for it: the 64 exponentials (zero past the last state) and
// for a tip the leaf table [state][category][row], 16 rows a wavefront: block b of the
// 4 x 4 x 4 tiles takes the rows 4 b + j, the states are the tile's rows, so a table row is
// written in pieces of 128 bytes.  The instruction adds its four terms in order, so an entry
// is the sum over the states in order that the oracle and the vector kernels form: entries
// that are small because their terms cancel (two or three substitutions in a codon) carry the
// same rounding.  All sides of 48 taxa: 92 us one dot product a thread, 27 now.
__device__ inline void pmatrix_f64_codon_body(const KParams &P, const PJob &job, const int c) {
    constexpr int N = 61, S = 4;  // S: groups of four states at once
    const int lane = threadIdx.x & 63, k = lane >> 4, ncat = P.ncat;
    double *M = (double *)P.mats + (int64_t)job.op * P.mat_stride;
    __shared__ double ex[64];
    if (threadIdx.x < 64) {
        const double v = lane < N ? exp(P.eval[min(lane, N - 1)] * (P.rates[c] * job.len)) : 0.0;
        ex[lane] = v;
        M[(int64_t)job.side * ncat * N * N + c * 64 + lane] = v;
    }
    if (!job.leaf) return;
    __syncthreads();
    double *T = M + (int64_t)2 * ncat * N * N + (int64_t)job.side * (P.su + 1) * ncat * N + c * N;
    const int x = wave_id() * 16 + (lane & 15);  // (as a column; D's columns are the same lanes)
    double e[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int i = 4 * q + k;
        const double u = P.evec[min(x, N - 1) * N + min(i, N - 1)];
        e[q] = i < N ? u * ex[i] : 0.0;
    }
    for (int s0 = 0; s0 < P.su; s0 += 4 * S) {
        double t[S][16], d[S];
#pragma unroll
        for (int g = 0; g < S; g++) {
            d[g] = 0.0;
#pragma unroll
            for (int q = 0; q < 16; q++)
                t[g][q] = P.tip_lh[min(s0 + 4 * g + (lane & 3), P.su - 1) * N + min(4 * q + k, N - 1)];
        }
#pragma unroll
        for (int q = 0; q < 16; q++)
#pragma unroll
            for (int g = 0; g < S; g++) d[g] = __builtin_amdgcn_mfma_f64_4x4x4f64(t[g][q], e[q], d[g], 0, 0, 0);
#pragma unroll
        for (int g = 0; g < S; g++) {
            const int s = s0 + 4 * g + k;
            if (s < P.su && x < N) T[(int64_t)s * ncat * N + x] = d[g];
        }
    }
    if (threadIdx.x < N) T[(int64_t)P.su * ncat * N + threadIdx.x] = 1.0;
}

// Branch logL of a tile (no ops): 16 wavefronts, four patterns each, the lanes' states as in
// the traversal, four categories' rows in flight at once (with one wavefront a category,
// a pattern a lane, walking the 61 rows took 41 us of latency).
__device__ inline void branch_f64_codon_body(const KParams &P, const int tile) {
    constexpr int N = 61, C = 4;
    const int lane = threadIdx.x & 63, w = wave_id(), ncat = P.ncat;
    const int j = lane & 3, s4 = ((lane >> 2) & 3) * 4 + (lane >> 4), pl = w * 4 + j;
    const int64_t p = (int64_t)tile * 64 + pl;
    const bool atip = P.br_a < 0;
    const int64_t off = (int64_t)tile * ncat * N * 64 + f64_loff(N, pl);
    const double *__restrict__ B = (const double *)P.part + (int64_t)P.br_b * P.slot_stride + off;
    const double *__restrict__ A = (const double *)P.part + (int64_t)(atip ? P.br_b : P.br_a) * P.slot_stride + off;
    const double *__restrict__ T = P.tip_lh + (atip ? P.states[(int64_t)(-P.br_a - 1) * P.nptn_pad + p] : 0) * N;
    const uint16_t *scB = (const uint16_t *)P.scale + (int64_t)P.br_b * P.scale_stride;
    const uint16_t *scA = (const uint16_t *)P.scale + (int64_t)(atip ? P.br_b : P.br_a) * P.scale_stride;
    __shared__ double s_val[PLK_GPU_MAX_CATS][64], s_lh[64];
    for (int i = threadIdx.x; i < ncat * 64; i += blockDim.x) {
        const int c = i >> 6, x = i & 63;
        s_val[c][x] = x < N ? exp(P.eval[min(x, N - 1)] * P.rates[c] * P.br_len) * P.props[c] : 0.0;
    }
    __syncthreads();
    double lh = 0.0;
    int sc = 0x7fffffff;
    double v[PLK_GPU_MAX_CATS];
    int n[PLK_GPU_MAX_CATS];
#pragma unroll
    for (int c0 = 0; c0 < PLK_GPU_MAX_CATS; c0 += C) {
        if (c0 >= ncat) break;
        double va[C][4], vb[C][4];
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int cc = min(c0 + c, ncat - 1);
#pragma unroll
            for (int R = 0; R < 4; R++) {
                const int i = min(16 * R + s4, N - 1);
                vb[c][R] = B[cc * N * 64 + f64_xoff(N, i)];
                va[c][R] = atip ? T[i] : A[cc * N * 64 + f64_xoff(N, i)];
            }
            const int64_t at = P.safe ? p * ncat + cc : p;
            n[c0 + c] = (int)scB[at] + (atip ? 0 : (int)scA[at]);
        }
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int cc = min(c0 + c, ncat - 1);
            double t = 0.0;
#pragma unroll
            for (int R = 0; R < 4; R++) t = 16 * R + s4 < N ? fma(s_val[cc][16 * R + s4] * va[c][R], vb[c][R], t) : t;
            t += codon_rotate<2>(t);
            t += codon_rotate<1>(t);
            t += __shfl_xor(t, 16, 64);
            v[c0 + c] = t + __shfl_xor(t, 32, 64);
            if (c0 + c < ncat) sc = min(sc, n[c0 + c]);
        }
    }
    // SAFE: categories above the minimum count are scaled by 2^-256 or dropped (3063-3088)
#pragma unroll
    for (int c = 0; c < PLK_GPU_MAX_CATS; c++) {
        if (c >= ncat) break;
        if (n[c] != sc) v[c] *= n[c] == sc + 1 ? kST : 0.0;
        lh += v[c];
        if (P.ptn_lh_cat && s4 == 0 && p < P.nptn) P.ptn_lh_cat[p * ncat + c] = v[c];  // 3023, 3076-3083
    }
    const double l = log(fabs(lh) + P.invar[p]) + sc * kLogST;  // 3096-3108
    if (s4 == 0) {
        if (p < P.nptn) {
            P.ptn_lh[p] = l;
            if (P.ptn_lh_cat) P.ptn_scaling[p] = sc * kLogST;
        }
        s_lh[pl] = p < P.nptn ? l * P.freq[p] : 0.0;
    }
    __syncthreads();
    double r0 = 0.0;
    if (w == 0) r0 = wave_sum(s_lh[lane]);
    finish_tiles(P, r0, 0.0, tile, P.ntiles);
}

}  // namespace dev
}  // namespace plk
