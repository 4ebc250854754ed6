// Traversal of 4-state (DNA) models: a wavefront walks the op list alone.
//
// A wavefront owns 16 patterns and all categories of them, so neither the products nor the
// check over a pattern's categories needs another wavefront: the op loop has no barrier.
// The transition products are 4 x 4 matrix instructions whose output lanes are the input
// lanes of the next product, so an op's output is the next op's child as it stands.
//
//   FORM 0 (FP64, eigen space, tree/phylokernelnew.h:1636-2036):
//     a = U (exp(Lambda r t_L) o L), b alike, out = U^-1 (a o b); U and U^-1 are one register
//     each.  v_mfma_f64_4x4x4_4b_f64: block b = category, columns = four patterns.  Lane
//     j + 4 b + 16 k holds state k of category b of patterns 4 j .. 4 j + 3 (four products).
//   FORM 1 (FP32, real space): out = (P_L L) o (P_R R), renormalised per pattern.
//     v_mfma_f32_4x4x1_16b_f32 four times (k = 0..3): block = (category, four patterns).  Lane
//     16 b + p holds the four states of category b of pattern p.
//
// Either way a lane's four values are contiguous in memory.  A tip's product comes from its
// row of a table of P(t) times the tip vectors, formed in FP64 (FORM 1), or the tip is a child
// whose vectors are read from LDS (FORM 0); it is 1 for the unknown state.
//
// A small alignment is bound by the op's own chain of instructions (one wavefront per SIMD or
// fewer), a large one by the partials it writes.  For the first, an op issues as little as it
// can, and waits for no store:
//   - the previous op's output stays in registers,
//   - outputs read again soon are also kept in LDS, in buffers private to the wavefront
//     (assigned on the host by liveness; a post-order list needs about log2 of the taxa),
//   - the list's fields, the outputs' addresses and the tip states come from lanes and LDS,
//     filled a window of ops at a time; operands are read an op ahead, before the op's stores
//     are issued (a wavefront's vector memory operations complete in order),
//   - a short list's exponentials (FP64) or P(t) rows (FP32) are formed in LDS by the
//     workgroup (STAGE), which saves the P(t) launch.
// Every partial is stored to memory.  One or two categories put pattern groups into the
// blocks that would be idle; with 5-8 a lane holds two categories (CG = 2).
//
// Measured (logL, against the level-parallel kernel below 320 tiles and the category-split
// kernels above): 12 taxa x 400 sites FP64 34 -> 26 us a call, 32 taxa x 10,000 sites 56 -> 40 us
// (0.5 us an op, 0.7 before the waits and address arithmetic left the loop), 512 taxa x
// 100,000 sites FP32 2700 -> 1050 us (3.5 GB of partials and counts: 3.4 TB/s).
#pragma once

#include "dev_common.h"

namespace plk {
namespace dev {

typedef double dna_d2 __attribute__((ext_vector_type(2)));

template <int FORM>
using dna_real = std::conditional_t<FORM == 0, double, float>;

// Place of (category c, state / row i) in one side's P(t) data: FORM 0 [group][state][category],
// FORM 1 [group][category][row][4].
template <int FORM>
__device__ __forceinline__ int dna_place(int c, int i) {
    const int g = c >> 2, b = c & 3;
    return FORM == 0 ? g * 16 + i * 4 + b : g * 64 + (b * 4 + i) * 4;
}

// One thread's share of P(t) for category c of length t: FORM 0 the exponential of state i,
// FORM 1 row i of P and, for a tip, row i of its table ([group][state][category][row]); FP64
// sums rounded once (the P(t) kernel's arithmetic).
template <int FORM>
__device__ __forceinline__ void dna_pmat(const KParams &P, int c, int i, double t, dna_real<FORM> *dst, dna_real<FORM> *tab) {
    const double rt = P.rates[c] * t;
    dst += dna_place<FORM>(c, i);
    if constexpr (FORM == 0) {
        *dst = exp(P.eval[i] * rt);
    } else {
        double pr[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const double ue = P.evec[i * 4 + k] * exp(P.eval[k] * rt);
#pragma unroll
            for (int y = 0; y < 4; y++) pr[y] = fma(ue, P.inv_evec[k * 4 + y], pr[y]);
        }
#pragma unroll
        for (int y = 0; y < 4; y++) dst[y] = (float)pr[y];
        if (!tab) return;
        tab += (c >> 2) * dna_table_len() + (c & 3) * 4 + i;
        for (int s = 0; s < P.su; s++) {
            double v = 0.0;
#pragma unroll
            for (int y = 0; y < 4; y++) v = fma(pr[y], P.tipvec[s * 4 + y], v);
            tab[s * 16] = (float)v;
        }
        tab[P.su * 16] = 1.0f;
    }
}

// The value, read where it is written down and not earlier: copied ahead of a branch, a
// register that a load may still fill would have the wavefront wait for everything in flight,
// the last op's stores included, on the path that does not need it.
template <typename T>
__device__ __forceinline__ T stay(T v) {
    asm volatile("" : "+v"(v));
    return v;
}

// max over the lanes of a pattern (FORM 1: lane bits 4 and 5 are the category)
__device__ __forceinline__ float dna_max(float m, int ncb) {
    if (ncb > 1) {
        const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
        m = fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
    }
    if (ncb > 2) {
        const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
        m = fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
    }
    return m;
}

// An address of device memory, from the two words a lane holds.
typedef __attribute__((address_space(1))) char dna_mem;
__device__ __forceinline__ dna_mem *dna_addr(int lo, int hi) {
    return (dna_mem *)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// Dynamic LDS of a workgroup, in this order: tip states, tip vectors (FORM 0), staged P(t)
// data and tip tables, then per wavefront nbuf buffers of values and counts.
template <int FORM, int CG>
struct DnaLds {
    using REAL = dna_real<FORM>;
    uint8_t *tip;  // this wavefront's tip states: [op of the window][side][pattern]
    REAL *tipv;   // FORM 0: 19 x 4
    REAL *pm;     // staged P(t) data, [op][side][CG * dna_p_len]
    REAL *tab;    // FORM 1: staged tip tables, [index][CG * dna_table_len]
    REAL *val;    // this wavefront's buffers: [buffer][group][half][lane][2]
    int32_t *cnt; // [buffer][group][lane][FORM 0: two words of 16-bit counts, FORM 1: exponent]
    __device__ __forceinline__ DnaLds(const KParams &P, char *base, int wave, int ncb, int nstage, int ntab) {
        tip = (uint8_t *)base + wave * (dna_window(nstage > 0) * 128 / ncb);
        base += dna_window(nstage > 0) * 128;
        tipv = (REAL *)base;
        if (FORM == 0) base += (size_t)kDnaStates * 4 * sizeof(REAL);
        pm = (REAL *)base;
        base += (size_t)nstage * 2 * CG * dna_p_len(FORM) * sizeof(REAL);
        tab = (REAL *)base;
        base += (size_t)ntab * CG * dna_table_len() * sizeof(REAL);
        const size_t vb = (size_t)CG * 256 * sizeof(REAL), cb = (size_t)CG * 64 * (FORM == 0 ? 8 : 4);
        base += (size_t)wave * P.nbuf * (vb + cb);
        val = (REAL *)base;
        cnt = (int32_t *)(base + P.nbuf * vb);
    }
};

// Fields of an op as the loop reads them: bits, then the LDS buffers (or tip tables)
enum : unsigned {
    DNA_LTIP = 1,        // the child is a tip
    DNA_RTIP = 2,
    DNA_LCARRY = 4,      // the child is the previous op's output
    DNA_RCARRY = 8,
    DNA_LFAR = 16,       // the child is in memory only
    DNA_RFAR = 32,
    DNA_LGAP = 64,       // FORM 0: one of the wavefront's patterns has the unknown state
    DNA_RGAP = 128,
};

// One 64-pattern tile: the ops [k0, k1) of the list, and in MODE_LOGL the branch stage.
// SAFE: FORM 0 scaling mode (FORM 1 keeps one exponent per pattern in either).
template <int FORM, int CG, int MODE, bool STAGE, bool SAFE>
__device__ inline void traverse_dna_body(const KParams &P, const int tile, const int k0, const int k1, char *smem) {
    using REAL = dna_real<FORM>;
    constexpr int QP = FORM == 0 ? 4 : 1;  // patterns of a lane
    static_assert(FORM == 0 || !SAFE, "SAFE / NORM does not apply to FORM 1");
    // counts of a lane: FORM 1 the exponent; FORM 0 four 16-bit counts in one word per category
    // group (NORM: group 0 only).  As loaded from memory (RW words): SAFE counts of one
    // category lie ncat apart, so they arrive one by one.  (Scalars, not small arrays: the
    // compiler turned copies of two-word arrays into copies through scratch memory.)
    constexpr int CC = SAFE ? CG : 1, RW = SAFE ? 4 : 1;
    using CNT = std::conditional_t<FORM == 0, unsigned long long, unsigned>;
    using RAW = std::conditional_t<SAFE, unsigned, CNT>;
    using CMEM = std::conditional_t<FORM == 0, uint16_t, uint32_t>;
    constexpr int SL = dna_side_len(FORM, CG), PL = CG * dna_p_len(FORM), TL = CG * dna_table_len();
    constexpr int XN = FORM == 0 ? 1 : 4;  // P(t) data of a lane, side and category group
    const int lane = threadIdx.x & 63;
    const int ncat = P.ncat, ncb = ncat >= 3 ? 4 : ncat;
    const int b = FORM == 0 ? (lane >> 2) & 3 : lane >> 4;  // block: category, or further patterns
    const int s4 = lane >> 4;                               // FORM 0: state of the lane
    const int row = lane & 3;                               // matrix row of the lane (A operand)
    const int w = wave_id();
    const bool live = w < ncb;       // 4 / (4 / ncb) wavefronts cover the tile; batched launches may hold more
    const int np = 16 * (4 / ncb);   // patterns of a wavefront
    const int pl = (live ? w : 0) * np + (b / ncb) * 16 + (FORM == 0 ? 4 * (lane & 3) : lane & 15);
    const int64_t p = (int64_t)tile * 64 + pl;  // first pattern of the lane
    // Lanes without a category of their own (three, or five to seven of them) repeat the last
    // one: they form and store the same values, so no access needs a test.
    int cat[CG];
    bool mine[CG];
    unsigned off[CG], coff[CG];  // bytes from a slot's tile: the lane's values, its counts
#pragma unroll
    for (int g = 0; g < CG; g++) {
        const int c = 4 * g + b % ncb;
        mine[g] = live && c < ncat;
        cat[g] = min(c, ncat - 1);
        off[g] = (FORM == 0 ? (cat[g] * 4 + s4) * 64 + pl : cat[g] * 256 + pl * 4) * (int)sizeof(REAL);
        coff[g] = (SAFE ? pl * ncat + cat[g] : pl) * (int)sizeof(CMEM);
    }
    const int64_t tile_part = (int64_t)tile * ncat * 256, tile_cnt = (int64_t)tile * 64 * (SAFE ? ncat : 1);
    auto part_of = [&](int slot) { return (unsigned long long)((REAL *)P.part + (int64_t)slot * P.slot_stride + tile_part); };
    auto cnt_of = [&](int slot) { return (unsigned long long)((CMEM *)P.scale + (int64_t)slot * P.scale_stride + tile_cnt); };
    // FORM 0 needs the patterns' invariant terms in the loop; a staged list is short and also
    // brings what the branch stage needs ahead of it, a long one spares the registers.
    double inv[QP], frq[QP];
    auto load_inv = [&] {
#pragma unroll
        for (int q = 0; q < QP; q++) inv[q] = P.invar[p + q];
    };
    auto load_freq = [&] {
#pragma unroll
        for (int q = 0; q < QP; q++) frq[q] = P.freq[min(p + q, (int64_t)P.nptn - 1)];
    };
    if (FORM == 0 || (STAGE && MODE == MODE_LOGL)) load_inv();
    if (STAGE && MODE == MODE_LOGL) load_freq();

    const int nstage = STAGE ? k1 - k0 + 1 : 0;
    const DnaLds<FORM, CG> L(P, smem, live ? w : 0, ncb, nstage, STAGE && FORM == 1 ? P.ntip : 0);
    if (FORM == 0)
        for (int i = threadIdx.x; i < (P.su + 1) * 4; i += blockDim.x) L.tipv[(i & 3) * kDnaStates + (i >> 2)] = (REAL)P.tip_lh[i];
    if constexpr (STAGE) {
        for (int idx = threadIdx.x; idx < (k1 - k0) * 8 * ncat; idx += blockDim.x) {
            const int i = idx & 3, c = (idx >> 2) % ncat, side = (idx / (4 * ncat)) & 1, k = idx / (8 * ncat);
            const DevOp *o = P.ops + k0 + k;
            const int at = side ? o->lds_right : o->lds_left;
            const bool tip = side ? o->kind == KIND_TT : o->kind <= KIND_TI;
            dna_pmat<FORM>(P, c, i, side ? o->len_right : o->len_left, L.pm + (k * 2 + side) * PL, tip ? L.tab + at * TL : nullptr);
        }
        if (FORM == 1 && MODE == MODE_LOGL)
            for (int idx = threadIdx.x; idx < 4 * ncat; idx += blockDim.x)
                dna_pmat<FORM>(P, idx >> 2, idx & 3, P.br_len, L.pm + (k1 - k0) * 2 * PL, nullptr);
    }
    __syncthreads();

    // A operands: FORM 0 the constant U and U^-1 (U[row][state])
    double aU = 0.0, aUi = 0.0;
    if constexpr (FORM == 0) {
        aU = P.evec[row * 4 + s4];
        aUi = P.inv_evec[row * 4 + s4];
    }
    auto load4 = [&](const REAL *src, REAL(&v)[4]) {
        if constexpr (FORM == 0) {
            const dna_d2 x = *(const dna_d2 *)src, y = *(const dna_d2 *)(src + 2);
            v[0] = x.x;
            v[1] = x.y;
            v[2] = y.x;
            v[3] = y.y;
        } else {
            const floatx4 x = *(const floatx4 *)src;
#pragma unroll
            for (int y = 0; y < 4; y++) v[y] = x[y];
        }
    };
    auto store4 = [&](dna_mem *dst, const REAL(&v)[4]) {
        if constexpr (FORM == 0) {
            *(__attribute__((address_space(1))) dna_d2 *)dst = dna_d2{v[0], v[1]};
            *(__attribute__((address_space(1))) dna_d2 *)(dst + 16) = dna_d2{v[2], v[3]};
        } else {
            *(__attribute__((address_space(1))) floatx4 *)dst = floatx4{v[0], v[1], v[2], v[3]};
        }
    };
    auto load_mem = [&](int slot, REAL(&v)[CG][4]) {
        const char *src = (const char *)((const REAL *)P.part + (int64_t)slot * P.slot_stride + tile_part);
#pragma unroll
        for (int g = 0; g < CG; g++) load4((const REAL *)(src + off[g]), v[g]);
    };
    auto load_counts = [&](int slot, RAW(&v)[CC][RW]) {
        const char *src = (const char *)((const CMEM *)P.scale + (int64_t)slot * P.scale_stride + tile_cnt);
#pragma unroll
        for (int g = 0; g < CC; g++)
#pragma unroll
            for (int q = 0; q < RW; q++) {
                if constexpr (SAFE) v[g][q] = *((const CMEM *)(src + coff[g]) + q * ncat);
                else v[g][q] = *(const RAW *)(src + coff[g]);
            }
    };
    auto pack = [&](const RAW(&v)[CC][RW], CNT(&n)[CC]) {
#pragma unroll
        for (int g = 0; g < CC; g++) {
            if constexpr (SAFE)
                n[g] = (CNT)(v[g][0] | v[g][1 % RW] << 16) | (CNT)(v[g][2 % RW] | v[g][3 % RW] << 16) << 32;
            else n[g] = v[g][0];
        }
    };
    auto store_counts = [&](dna_mem *dst, const CNT(&n)[CC]) {
#pragma unroll
        for (int g = 0; g < CC; g++) {
            if constexpr (SAFE) {
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *((__attribute__((address_space(1))) uint16_t *)(dst + coff[g]) + q * ncat) = (uint16_t)(n[g] >> (16 * q));
            } else {
                *(__attribute__((address_space(1))) CNT *)(dst + coff[g]) = n[g];
            }
        }
    };
    auto lds_val = [&](int buf, int g, int half) { return L.val + (((size_t)buf * CG + g) * 2 + half) * 128 + lane * 2; };
    auto lds_cnt = [&](int buf, int g) { return (CNT *)L.cnt + ((size_t)buf * CG + g) * 64 + lane; };
    auto load_lds = [&](int buf, REAL(&v)[CG][4], CNT(&n)[CC]) {
#pragma unroll
        for (int g = 0; g < CG; g++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                v[g][2 * h] = lds_val(buf, g, h)[0];
                v[g][2 * h + 1] = lds_val(buf, g, h)[1];
            }
#pragma unroll
        for (int g = 0; g < CC; g++) n[g] = *lds_cnt(buf, g);
    };
    auto store_lds = [&](int buf, const REAL(&v)[CG][4], const CNT(&n)[CC]) {
#pragma unroll
        for (int g = 0; g < CG; g++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                lds_val(buf, g, h)[0] = v[g][2 * h];
                lds_val(buf, g, h)[1] = v[g][2 * h + 1];
            }
#pragma unroll
        for (int g = 0; g < CC; g++) *lds_cnt(buf, g) = n[g];
    };
    // FORM 0: the tip vectors of the lane's patterns (st: four states, times eight)
    auto tip_rows = [&](unsigned st, REAL(&v)[CG][4]) {
        const char *t = (const char *)(L.tipv + s4 * kDnaStates);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const REAL x = *(const REAL *)(t + ((st >> (8 * q)) & 255));
#pragma unroll
            for (int g = 0; g < CG; g++) v[g][q] = x;
        }
    };
    // P(t) data of an op's side: FORM 0 the lane's exponential, FORM 1 its row of P or, for a
    // tip, of the op's table
    auto load_pm = [&](int k, int side, bool tip, int at, unsigned st, REAL(&x)[CG][XN]) {
        const REAL *src = STAGE ? L.pm + ((k - k0) * 2 + side) * PL : (const REAL *)P.mats + (int64_t)k * P.mat_stride + side * SL;
        if constexpr (FORM == 0) {
#pragma unroll
            for (int g = 0; g < CG; g++) x[g][0] = src[dna_place<0>(cat[g], s4)];
        } else {
            const REAL *t = STAGE ? L.tab + at * TL : src + PL;
            src = tip ? t : src;
#pragma unroll
            for (int g = 0; g < CG; g++) {
                const int i = (cat[g] >> 2) * dna_table_len() + (int)st * 16 + (cat[g] & 3) * 4;
                load4(src + (tip ? i : dna_place<1>(cat[g], row)), x[g]);
            }
        }
    };
    // one side of the product
    auto side = [&](const REAL(&x)[CG][XN], const REAL(&v)[CG][4], bool tip, bool gap, unsigned st, REAL(&d)[CG][4]) {
#pragma unroll
        for (int g = 0; g < CG; g++) {
            if constexpr (FORM == 0) {
#pragma unroll
                for (int q = 0; q < 4; q++) d[g][q] = __builtin_amdgcn_mfma_f64_4x4x4f64(aU, x[g][0] * v[g][q], 0.0, 0, 0, 0);
                if (gap)
#pragma unroll
                    for (int q = 0; q < 4; q++) d[g][q] = (int)((st >> (8 * q)) & 255) == P.su * 8 ? 1.0 : d[g][q];
            } else if (tip) {
#pragma unroll
                for (int q = 0; q < 4; q++) d[g][q] = x[g][q % XN];
            } else {
                floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int y = 0; y < 4; y++) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(x[g][y % XN], v[g][y], acc, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 4; q++) d[g][q] = acc[q];
            }
        }
    };
    auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    // -------- the op list
    // Lane i of a wavefront holds op w0 + i as the loop needs it: its output's addresses, its
    // children's slots and its fields, read across lanes with no memory access in the loop.
    // It also brings the op's tip states of the wavefront's patterns to LDS.
    typedef int int4v __attribute__((ext_vector_type(4)));
    int f_plo = 0, f_phi = 0, f_clo = 0, f_chi = 0, f_left = 0, f_right = 0, f_bits = 0;
    int w0 = k0;
    constexpr int kWindow = dna_window(STAGE);
    auto window = [&](int from) {
        const int at = min(from + lane, k1 - 1);
        const int4v *o = (const int4v *)(P.ops + at);
        const int4v wa = o[0], wb = o[1];
        const int before = at > k0 ? P.ops[at - 1].out_slot : -1;
        const bool ltip = wa.y <= KIND_TI, rtip = wa.y == KIND_TT;
        const int64_t base = (int64_t)tile * 64 + (live ? w : 0) * np;
        uint8_t *dst = L.tip + (lane & (kWindow - 1)) * 2 * np;  // (ops past the window are not read)
        unsigned bits = (ltip ? DNA_LTIP : wa.z == before ? DNA_LCARRY : wb.y < 0 ? DNA_LFAR : 0) |
                        (rtip ? DNA_RTIP : wa.w == before ? DNA_RCARRY : wb.z < 0 ? DNA_RFAR : 0);
        for (int i = 0; i < np; i += 16) {
            int4v l = {0, 0, 0, 0}, r = {0, 0, 0, 0};
            if (ltip && lane < kWindow) l = *(const int4v *)(P.states + (int64_t)wa.z * P.nptn_pad + base + i);
            if (rtip && lane < kWindow) r = *(const int4v *)(P.states + (int64_t)wa.w * P.nptn_pad + base + i);
            if constexpr (FORM == 0) {
                // any byte equal to the unknown state; then the states times the size of a value
                const unsigned u = 0x01010101u * (unsigned)P.su;
                unsigned lz = 0, rz = 0;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const unsigned x = (unsigned)l[j] ^ u, y = (unsigned)r[j] ^ u;
                    lz |= (x - 0x01010101u) & ~x & 0x80808080u;
                    rz |= (y - 0x01010101u) & ~y & 0x80808080u;
                    l[j] <<= 3;
                    r[j] <<= 3;
                }
                bits |= (ltip && lz ? DNA_LGAP : 0) | (rtip && rz ? DNA_RGAP : 0);
            }
            if (lane < kWindow) {
                *(int4v *)(dst + i) = l;
                *(int4v *)(dst + np + i) = r;
            }
        }
        bits |= (unsigned)(wb.x & 255) << 8 | (unsigned)(wb.y & 255) << 16 | (unsigned)(wb.z & 255) << 24;
        const unsigned long long pa = part_of(wa.x), ca = cnt_of(wa.x);
        // (stay: wait for the loads here, not at every use in the loop)
        f_plo = stay((int)pa);
        f_phi = stay((int)(pa >> 32));
        f_clo = stay((int)ca);
        f_chi = stay((int)(ca >> 32));
        f_left = stay(wa.z);
        f_right = stay(wa.w);
        f_bits = stay((int)bits);
        w0 = from;
        fence();
    };
    auto field = [&](int f, int k) { return __builtin_amdgcn_readlane(f, k - w0); };
    // states of the lane's patterns (whatever is there for a side that is no tip)
    auto states_of = [&](int k, unsigned &ls, unsigned &rs) {
        const uint8_t *s = L.tip + (k - w0) * 2 * np + (pl & (np - 1));
        if constexpr (FORM == 0) {
            ls = *(const unsigned *)s;
            rs = *(const unsigned *)(s + np);
        } else {
            ls = *s;
            rs = s[np];
        }
    };
    // One side of the op at hand: the tip's states (ahead: an op ahead); P(t) data; the child,
    // or a FORM 0 tip's vectors, with its counts.
    struct Side {
        unsigned st, ahead;
        REAL x[CG][XN], m[CG][4];
        CNT n[CC];
    };
    Side lft{}, rgt{};
    REAL cv[CG][4] = {};  // the last op's output
    CNT cn[CC] = {};
    // A side's operands.  The previous op's output is handed over in registers.  A child that is
    // neither that nor in LDS is waited for on the spot: a wait after the branches would
    // cover the stores in flight of every op.
    auto fetch_side = [&](int k, int which, bool tip, bool carry, bool far, int lds, Side &d) {
        d.st = d.ahead;
#pragma unroll
        for (int g = 0; g < CC; g++) d.n[g] = 0;
        if (tip) {
            if constexpr (FORM == 0) tip_rows(d.st, d.m);
        } else if (!carry) {
            if (!far) {
                load_lds(lds, d.m, d.n);
            } else {
                const int slot = field(which ? f_right : f_left, k);
                RAW t[CC][RW];
                load_mem(slot, d.m);
                load_counts(slot, t);
#pragma unroll
                for (int g = 0; g < CG; g++)
#pragma unroll
                    for (int q = 0; q < 4; q++) d.m[g][q] = stay(d.m[g][q]);
#pragma unroll
                for (int g = 0; g < CC; g++)
#pragma unroll
                    for (int q = 0; q < RW; q++) t[g][q] = stay(t[g][q]);
                pack(t, d.n);
            }
        }
        load_pm(min(k, k1 - 1), which, tip, lds, d.st, d.x);
    };
    auto fetch = [&](int k, unsigned bits) {
        fetch_side(k, 0, bits & DNA_LTIP, bits & DNA_LCARRY, bits & DNA_LFAR, bits >> 16 & 255, lft);
        fetch_side(k, 1, bits & DNA_RTIP, bits & DNA_RCARRY, bits & DNA_RFAR, bits >> 24, rgt);
    };
    const int kend = live ? k1 : k0;
    unsigned nxt = 0;
    if (k0 < kend) {
        window(k0);
        nxt = (unsigned)field(f_bits, k0);
        states_of(k0, lft.ahead, rgt.ahead);
        fetch(k0, nxt);
        states_of(k0 + 1, lft.ahead, rgt.ahead);
    }
    // (a load still in flight here would be waited for in every turn of the loop)
    aU = stay(aU);
    aUi = stay(aUi);
    __builtin_amdgcn_s_waitcnt(0);
    for (int k = k0; k < kend; k++) {
        const unsigned bits = nxt;
        REAL a[CG][4], o[CG][4];
        CNT n[CC];
        side(rgt.x, rgt.m, bits & DNA_RTIP, bits & DNA_RGAP, rgt.st, a);
        side(lft.x, lft.m, bits & DNA_LTIP, bits & DNA_LGAP, lft.st, o);
#pragma unroll
        for (int g = 0; g < CC; g++) n[g] = rgt.n[g] + lft.n[g];  // (16-bit counts: no carry, counts < ops)
        dna_mem *const pout = dna_addr(field(f_plo, k), field(f_phi, k));
        dna_mem *const cout = dna_addr(field(f_clo, k), field(f_chi, k));
        if (!STAGE && k + 2 >= w0 + kWindow) window(k);
        nxt = (unsigned)field(f_bits, k + 1);
        fetch(k + 1, nxt);
        states_of(k + 2, lft.ahead, rgt.ahead);
#pragma unroll
        for (int g = 0; g < CG; g++) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                o[g][q] *= a[g][q];
                if constexpr (FORM == 0) o[g][q] = __builtin_amdgcn_mfma_f64_4x4x4f64(aUi, o[g][q], 0.0, 0, 0, 0);
            }
        }
        if constexpr (FORM == 1) {
            float m = 0.0f;
#pragma unroll
            for (int g = 0; g < CG; g++)
#pragma unroll
                for (int q = 0; q < 4; q++) m = fmaxf(m, fabsf(o[g][q]));
            const int e = norm_exponent(dna_max(m, ncb));
#pragma unroll
            for (int g = 0; g < CG; g++)
#pragma unroll
                for (int q = 0; q < 4; q++) o[g][q] = ldexpf(o[g][q], -e);
            n[0] += e;
        } else if (!(bits & DNA_RTIP)) {
            // some value of the wavefront is below 2^-256 (or no number): see which pattern
            // (NORM) or pattern and category (SAFE) has none above it (2019-2034, 1997-2013)
            unsigned long long ok[CG][4], every = ~0ull;
#pragma unroll
            for (int g = 0; g < CG; g++)
#pragma unroll
                for (int q = 0; q < 4; q++) every &= ok[g][q] = __ballot(fabs(o[g][q]) >= kST);
            if (~every) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    unsigned y[CG], all = 0;
#pragma unroll
                    for (int g = 0; g < CG; g++) {
                        y[g] = (unsigned)(ok[g][q] | ok[g][q] >> 32);
                        y[g] = (y[g] | y[g] >> 16) & 0xffffu;  // [block][column]
                        all |= y[g];
                    }
                    if (ncb > 1) all |= (all >> 4 & 0x0f0fu) | (all << 4 & 0xf0f0u);
                    if (ncb > 2) all = (all | all >> 8 | all << 8) & 0xffffu;
                    if ((SAFE ? y[0] & y[CG - 1] : all) == 0xffffu) continue;
#pragma unroll
                    for (int g = 0; g < CG; g++) {
                        const bool up = !((SAFE ? y[g] : all) >> (lane & 15) & 1) && inv[q] == 0.0;
                        o[g][q] *= up ? kTwo256 : 1.0;
                        if (SAFE || g == 0) n[SAFE ? g : 0] += up ? (CNT)1 << (16 * q) : 0;
                    }
                }
            }
        }
        // the next op's child, handed over
        auto hand = [&](REAL(&m)[CG][4], CNT(&nm)[CC]) {
#pragma unroll
            for (int g = 0; g < CG; g++)
#pragma unroll
                for (int q = 0; q < 4; q++) m[g][q] = o[g][q];
#pragma unroll
            for (int g = 0; g < CC; g++) nm[g] = n[g];
        };
        if (nxt & DNA_RCARRY) hand(rgt.m, rgt.n);
        if (nxt & DNA_LCARRY) hand(lft.m, lft.n);
        if ((bits >> 8 & 255) != 255) store_lds(bits >> 8 & 255, o, n);
#pragma unroll
        for (int g = 0; g < CG; g++) store4(pout + off[g], o[g]);
        store_counts(cout, n);
        if (MODE == MODE_LOGL && k + 1 == kend) hand(cv, cn);
        fence();  // other lanes of this wavefront read these values later
    }
    if (MODE == MODE_PARTIALS) return;

    // -------- branch logL
    __shared__ double s_lh[64];
    if (FORM == 1 && !STAGE) load_inv();
    if (!STAGE) load_freq();
    {
        const bool atip = P.br_a < 0;
        REAL vb[CG][4], va[CG][4];
        CNT nb[CC], na[CC];
        RAW raw[CC][RW];
#pragma unroll
        for (int g = 0; g < CC; g++) na[g] = 0;
        if (k0 < kend && P.br_b == P.ops[k1 - 1].out_slot) {
#pragma unroll
            for (int g = 0; g < CG; g++)
#pragma unroll
                for (int q = 0; q < 4; q++) vb[g][q] = cv[g][q];
#pragma unroll
            for (int g = 0; g < CC; g++) nb[g] = cn[g];
        } else {
            load_mem(P.br_b, vb);
            load_counts(P.br_b, raw);
            pack(raw, nb);
        }
        if (atip) {
            const uint8_t *m = P.states + (int64_t)(-P.br_a - 1) * P.nptn_pad + p;
            const unsigned st = FORM == 0 ? *(const unsigned *)m : *m;
            if constexpr (FORM == 0) {
                tip_rows(st << 3, va);
            } else {
#pragma unroll
                for (int g = 0; g < CG; g++)
#pragma unroll
                    for (int q = 0; q < 4; q++) va[g][q] = (REAL)P.tipvec[st * 4 + q];
            }
        } else {
            load_mem(P.br_a, va);
            load_counts(P.br_a, raw);
            pack(raw, na);
        }
        // per lane: the category's likelihood of each of its patterns
        double lh[CG][QP];
        if constexpr (FORM == 0) {
            // lh_c = sum_i val_i a_i b_i (2903-2914, 3044-3057)
#pragma unroll
            for (int g = 0; g < CG; g++) {
                const double cof = P.eval[s4] * P.rates[cat[g]];
                const double val = exp(cof * P.br_len) * P.props[cat[g]];
#pragma unroll
                for (int q = 0; q < QP; q++) {
                    double v = val * va[g][q] * vb[g][q];
                    v += __shfl_xor(v, 16, 64);
                    v += __shfl_xor(v, 32, 64);
                    lh[g][q] = v;
                }
            }
        } else {
            // lh_c = sum_x pi_x a_x (P_c(t) b)_x
            REAL x[CG][XN], d[CG][4];
            load_pm(P.nops, 0, false, 0, 0, x);
            side(x, vb, false, false, 0, d);
#pragma unroll
            for (int g = 0; g < CG; g++) {
                float acc = 0.0f;
#pragma unroll
                for (int q = 0; q < 4; q++) acc = fmaf((float)P.pi[q] * va[g][q], d[g][q], acc);
                lh[g][0] = (double)acc;
            }
        }
        // the pattern's value, formed in the lanes of its first category (FORM 0: state 0)
#pragma unroll
        for (int q = 0; q < QP; q++) {
            int sc[CG], mn = 0;
#pragma unroll
            for (int g = 0; g < CG; g++) {
                const CNT t = nb[SAFE ? g : 0] + na[SAFE ? g : 0];
                sc[g] = FORM == 0 ? (int)(t >> (FORM == 0 ? 16 * q : 0) & 0xffff) : (int)t;
            }
            auto from = [&](int cc) { return FORM == 0 ? (lane & 3) | ((b / ncb) * ncb + cc) << 2 : (lane & 15) | ((b / ncb) * ncb + cc) << 4; };
            mn = sc[0];
            if (SAFE) {
                mn = __shfl(sc[0], from(0), 64);
                for (int c = 1; c < ncat; c++) mn = min(mn, __shfl(c < 4 ? sc[0] : sc[CG - 1], from(c & 3), 64));
            }
            // SAFE: categories above the minimum count are scaled by 2^-256 or dropped (3063-3088)
#pragma unroll
            for (int g = 0; g < CG; g++)
                if (SAFE) lh[g][q] *= sc[g] == mn ? 1.0 : sc[g] == mn + 1 ? kST : 0.0;
            double sum = 0.0;
            for (int c = 0; c < ncat; c++) {
                const double v = __shfl(c < 4 ? lh[0][q] : lh[CG - 1][q], from(c & 3), 64);
                sum += FORM == 0 ? v : P.props[c] * v;
            }
            const int64_t pp = p + q;
            double l;
            if constexpr (FORM == 0) l = log(fabs(sum) + inv[q]) + mn * kLogST;
            else l = log_lh_expo(sum, mn, inv[q]);
            const bool first = live && b % ncb == 0 && (FORM == 1 || s4 == 0);
            if (first) {
                if (pp < P.nptn) P.ptn_lh[pp] = l;
                s_lh[pl + q] = pp < P.nptn ? l * frq[q] : 0.0;
                if (FORM == 0 && P.ptn_scaling && pp < P.nptn) P.ptn_scaling[pp] = mn * kLogST;
            }
            // side output _pattern_lh_cat (3023, SAFE-adjusted 3076-3083)
            if (FORM == 0 && P.ptn_lh_cat && s4 == 0 && pp < P.nptn)
#pragma unroll
                for (int g = 0; g < CG; g++)
                    if (mine[g]) P.ptn_lh_cat[pp * ncat + cat[g]] = lh[g][q];
        }
    }
    __syncthreads();
    double r0 = 0.0;
    if (w == 0) r0 = wave_sum(s_lh[lane]);
    finish_tiles(P, r0, 0.0, tile, P.ntiles);
}

}  // namespace dev
}  // namespace plk
