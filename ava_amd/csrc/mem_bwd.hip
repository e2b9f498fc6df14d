// The backward of the fast-weight (delta-rule) memory recurrence for gfx950, one workgroup per head
// (delta_rec's gradient, gpu/arch.rs:1091-1136; the CUDA forms memg_bwd / memg_bwd4,
// gpu/lif.cu:3411-3888).
//
// Forward, per head and step: r = F^T e;  u_ij = b_i k_i v_j - a_i b_i e_i r_j;  S' = M S + u;
// P = a_i F_ij + S'_ij (M = 0: + u_ij);  F' = clamp(P, +-cap);  y = F'^T q.
// Backward, from the last step (dF, dS carried): gP = (dF + q dy^T) where |F'| < cap, else 0;
//   dq_i = sum_j dy_j F'_ij;  dalpha_i += sum_j gP_ij F_ij;  du = gP + dS;  dS <- M du;
//   dv_j = sum_i du_ij b_i k_i;  dr_j = -sum_i du_ij a_i b_i e_i;
//   with sv_i = sum_j du_ij v_j and sr_i = sum_j du_ij r_j:  dk_i = b_i sv_i;
//   db_i = k_i sv_i - a_i e_i sr_i;  dalpha_i -= b_i e_i sr_i;  de_i = -a_i b_i sr_i + sum_j dr_j F_ij;
//   dF <- a_i gP_ij + e_i dr_j;  dla = dalpha a (summed over the head's rows for per-head gates).
//
// Columns of F never mix in the forward, nor in the carried gradients; only the row sums above (over all 64
// columns) couple them, and nothing carried depends on those. So the serial part is two walks of the T
// steps, each its own recurrence and no more, and everything else is parallel over the chunks of CK steps:
//   1. mem_bwd_walk_kernel: the forward from (F0, S0), parking (F, S) at every chunk's start and r_j of
//      every step; and, in other workgroups of the same launch, the reverse walk of (dF, dS) as if no
//      element reached the bound, parking (dF, dS) at every chunk's end and dr_j of every step, and writing dv.
//      The forward marks the workgroups in which an element did reach it.
//   2. mem_bwd_bound_kernel: the reverse walk again from the parked end, with the bound's mask, in the marked
//      workgroups' columns (the others return at once).
//   3. mem_bwd_rows_kernel: per (head, chunk) the steps replayed from the parked states and walked back from
//      the parked gradients. r_j and dr_j are known, so no column sum is left: lane = row, each wave 8
//      columns, the row sums in the lane, the per-column values in scalar registers. The first chunk's workgroups end
//      with dF0 and dS0. Every output but dv is written here, after the last read of the inputs it may lie on.
// Measured, per-channel gates and momentum: 64 heads x 2048 steps 783 us (under the profiler walks 426, rows 438), 16 heads 343
// us, 256 heads 2.64 ms, 1024 heads x 512 steps 2.59 ms; one kernel that parked every 4th state and walked three times
// in series, the last walk forming the row sums too: 2.41, 1.87, 5.14 and 3.49 ms. With elements at the bound in every head
// 64 heads x 2048 1.33 ms, 16 heads 0.84, 256 4.2, 512 x 1024 3.6, 1024 x 1024 7.2 (that kernel, bound or not: 2.40, 1.91, 5.1, 3.6,
// 7.0); with the bound's walk waiting for each chunk's loads in turn, and every head's unmasked reverse walk before it, 2.41, 1.61,
// 5.0, 4.9 and 9.8.
// Workspace per (head, chunk): (F, S, dF, dS) of 16 KB (F and dF without momentum), and r, dr and room for dv per step.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {

constexpr int HS = 64, CK = 16;

typedef float f32x4 __attribute__((ext_vector_type(4)));
// the caller's tensors, which need not lie on 16 bytes (the hardware takes any multiple of 4)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
// The sum over the 16 lanes of v's DPP row (quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror,
// row_mirror), in every one of them.
__device__ __forceinline__ float sum16(float v) {
    v += dppf<0xB1>(v);
    v += dppf<0x4E>(v);
    v += dppf<0x141>(v);
    return v + dppf<0x140>(v);
}

// A column's 64 rows over 64 / R lanes (R = 4: a DPP row, R = 2: two), lane l its rows R l .. R l + R - 1: the sum
// over those lanes, in every one of them.
template <int R>
__device__ __forceinline__ float col_sum(float v) {
    v = sum16(v);
    if (R == 2) {
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    }
    return v;
}

struct MemBwdArgs {
    const float *q, *k, *e, *v, *la, *b, *F0, *S0, *dy, *dFT, *dST;
    float *dq, *dk, *de, *dv, *dla, *db, *dF0, *dS0;
    float *ck;       // [BH][chunk][state][64 columns][64 rows]: F, dF (and S, dS with momentum)
    float *r, *dr;   // [BH][T][64]
    int *hit;        // [BH][groups]: an element of the forward workgroup's columns reached the bound
    int groups, part, BH, T;  // part: which walks a launch holds (0 both, 1 the forward, 2 the reverse)
    float m, cap;
};

// Whether an element of the head reached the bound, by the forward walk's workgroups.
__device__ __forceinline__ bool head_hit(const MemBwdArgs &p, int bh) {
    int any = 0;
    for (int g = 0; g < p.groups; g++) any |= p.hit[bh * p.groups + g];
    return any != 0;
}

// Whether one did in the 16 columns from 16 cg, by the forward workgroups that hold some of them. (Columns mix in
// neither walk: the first one's results stand where none did.)
__device__ __forceinline__ bool cols_hit(const MemBwdArgs &p, int bh, int cg) {
    int any = 0;
    for (int g = cg * p.groups / 4; 4 * g < (cg + 1) * p.groups; g++) any |= p.hit[bh * p.groups + g];
    return any != 0;
}

// The parked state `which` of (head, chunk): 0 F, 1 dF, 2 S, 3 dS
template <bool MOM>
__device__ __forceinline__ float *parked(const MemBwdArgs &p, int bh, int c, int which) {
    const int nck = (p.T + CK - 1) / CK;
    return p.ck + (((size_t)bh * nck + c) * (MOM ? 4 : 2) + which) * (HS * HS);
}

// One chunk's inputs of a head in LDS: [step][row] each. The walks stage the next chunk while they scan this one.
struct Stage {
    float q[CK][HS], e[CK][HS], a[CK][HS], bk[CK][HS], abe[CK][HS], c[CK][HS];  // c: v (forward), dy (reverse)
};

// A thread's share of a chunk's inputs (step st, rows si .. si + 3), loaded one chunk ahead of its staging.
template <bool G1, bool FWD>
struct Loader {
    f32x4 q, k, e, c, la, b;
    __device__ __forceinline__ void load(const MemBwdArgs &p, int bh, int t0, int tid) {
        const int t = t0 + (tid >> 4), si = (tid & 15) * 4;
        const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
        q = k = e = c = la = b = z;
        if (t0 < 0 || t >= p.T) return;
        const size_t o = ((size_t)bh * p.T + t) * HS + si;
        auto at = [&](const float *x) -> f32x4 { return *reinterpret_cast<const f32x4u *>(x + o); };
        k = at(p.k);
        e = at(p.e);
        c = at(FWD ? p.v : p.dy);
        if (!FWD) q = at(p.q);
        if (G1) {
            const float l = p.la[(size_t)bh * p.T + t], g = p.b[(size_t)bh * p.T + t];
            la = f32x4{l, l, l, l};
            b = f32x4{g, g, g, g};
        } else {
            la = at(p.la);
            b = at(p.b);
        }
    }
    __device__ __forceinline__ void stage(Stage &s, int tid) const {
        const int st = tid >> 4, si = (tid & 15) * 4;
        f32x4 a, bk, abe;
#pragma unroll
        for (int z = 0; z < 4; z++) {
            a[z] = expf(la[z]);
            bk[z] = b[z] * k[z];
            abe[z] = (a[z] * b[z]) * e[z];
        }
        auto put = [&](float (&d)[CK][HS], const f32x4 &x) { *reinterpret_cast<f32x4 *>(&d[st][si]) = x; };
        if (!FWD) put(s.q, q);
        put(s.e, e);
        put(s.a, a);
        put(s.bk, bk);
        put(s.abe, abe);
        put(s.c, c);
    }
};

// The lane's operands of one step: its R rows' and its CPL columns'.
template <int R, int CPL, bool FWD>
struct StepIn {
    typedef float vec __attribute__((ext_vector_type(R)));
    vec q, e, a, k, x;
    float c[CPL];
    __device__ __forceinline__ void read(const Stage &s, int t, int i0, int j0) {
        auto at = [&](const float (&d)[CK][HS]) { return *reinterpret_cast<const vec *>(&d[t][i0]); };
        e = at(s.e);
        x = at(s.abe);
        k = at(s.bk);
        a = at(s.a);
        if (!FWD) q = at(s.q);
#pragma unroll
        for (int z = 0; z < CPL; z++) c[z] = s.c[t][j0 + z];
    }
};

// One forward step on the lane's R x CPL block (element CPL ri + c): r gets the columns' e^T F.
template <bool MOM, int R, int CPL>
__device__ __forceinline__ void fwd_step(float (&F)[R * CPL], float (&S)[R * CPL], const StepIn<R, CPL, true> &in,
                                         float M, float cap, float (&r)[CPL]) {
#pragma unroll
    for (int c = 0; c < CPL; c++) {
        r[c] = in.e[0] * F[c];
#pragma unroll
        for (int ri = 1; ri < R; ri++) r[c] = fmaf(in.e[ri], F[CPL * ri + c], r[c]);
    }
#pragma unroll
    for (int c = 0; c < CPL; c++) r[c] = col_sum<R>(r[c]);
#pragma unroll
    for (int ri = 0; ri < R; ri++)
#pragma unroll
        for (int c = 0; c < CPL; c++) {
            const int m = CPL * ri + c;
            const float u = fmaf(-in.x[ri], r[c], in.k[ri] * in.c[c]);
            float f;
            if (MOM) {
                S[m] = fmaf(M, S[m], u);
                f = fmaf(in.a[ri], F[m], S[m]);
            } else {
                f = fmaf(in.a[ri], F[m], u);
            }
            F[m] = __builtin_amdgcn_fmed3f(f, -cap, cap);
        }
}

// One reverse step: (dF, dS) before it from those after it. Fb: F after the step, where the bound's mask is wanted
// (NULL: it passes every gradient). dr, dv: the columns' sums.
template <bool MOM, int R, int CPL>
__device__ __forceinline__ void rev_step(float (&dF)[R * CPL], float (&dS)[R * CPL], const StepIn<R, CPL, false> &in,
                                         float M, const float *Fb, float cap, float (&dr)[CPL], float (&dv)[CPL]) {
#pragma unroll
    for (int c = 0; c < CPL; c++) dr[c] = dv[c] = 0.0f;
#pragma unroll
    for (int ri = 0; ri < R; ri++)
#pragma unroll
        for (int c = 0; c < CPL; c++) {
            const int m = CPL * ri + c;
            float gP = fmaf(in.q[ri], in.c[c], dF[m]);
            if (Fb) gP = fabsf(Fb[m]) < cap ? gP : 0.0f;
            float du = gP;
            if (MOM) {
                du = gP + dS[m];
                dS[m] = M * du;
            }
            dr[c] = fmaf(-du, in.x[ri], dr[c]);
            dv[c] = fmaf(du, in.k[ri], dv[c]);
            dF[m] = in.a[ri] * gP;
        }
#pragma unroll
    for (int c = 0; c < CPL; c++) {
        dr[c] = col_sum<R>(dr[c]);
        dv[c] = col_sum<R>(dv[c]);
    }
#pragma unroll
    for (int ri = 0; ri < R; ri++)
#pragma unroll
        for (int c = 0; c < CPL; c++) dF[CPL * ri + c] = fmaf(in.e[ri], dr[c], dF[CPL * ri + c]);
}

template <int R, int CPL>
__device__ __forceinline__ void park(float *dst, const float (&X)[R * CPL], int i0, int j0) {
    typedef float vec __attribute__((ext_vector_type(R)));
#pragma unroll
    for (int c = 0; c < CPL; c++) {
        vec v;
#pragma unroll
        for (int ri = 0; ri < R; ri++) v[ri] = X[CPL * ri + c];
        *reinterpret_cast<vec *>(dst + (j0 + c) * HS + i0) = v;
    }
}

// 1. The walks. Lane l of the 64 / R lanes of a column holds its rows R l .. R l + R - 1, a wave R CPL columns, so a head and
// direction has 16 / (R CPL) workgroups: 8 (R = 2), or 4, 2 and 1 (R = 4; CPL = 1, 2, 4). A column sum is R FMAs and 4 DPP adds
// over the 16 lanes of a DPP row (R = 2: and a lane swap between two rows). A step's time is the dependent
// chain through that sum and back (about 15 operations) against its issue and its LDS reads (5 vectors of R floats a
// lane): step t + 1's operands are read during step t, and one barrier per chunk
// covers the staging of the next. A wave alone on its SIMD issues one VALU operation per 8 cycles, two waves share
// them: so few heads are split into more, smaller workgroups, and the operations per element fall with more columns a lane (9, 8
// and 7 forward). The columns' r (dr, dv) of step s stay in lane s, so a chunk's go out in
// one store. Workgroups: the forward walks first, then the reverse (see ava_mem_scan_bwd for many heads).
template <bool G1, bool MOM, int R, int CPL>
__global__ __launch_bounds__(256) void mem_bwd_walk_kernel(MemBwdArgs p) {
    constexpr int LPC = HS / R, WC = CPL * R, NG = HS / (4 * WC), NE = R * CPL;  // lanes a column, columns a wave
    __shared__ __attribute__((aligned(16))) Stage sg[2];
    const bool rev = p.part ? p.part == 2 : (int)blockIdx.x >= p.BH * NG;
    const int wg = blockIdx.x - (rev && !p.part ? p.BH * NG : 0), bh = wg / NG, cg = wg - bh * NG;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lc = lane & (LPC - 1);
    const int i0 = R * lc, j0 = 4 * WC * cg + WC * wave + CPL * (lane / LPC);
    const int T = p.T, nck = (T + CK - 1) / CK;
    const size_t hb = (size_t)bh * T * HS, fb = (size_t)bh * HS * HS;
    const float M = p.m, cap = p.cap;

    if (!rev) {
        float F[NE], S[NE], top = 0.0f;
#pragma unroll
        for (int m = 0; m < NE; m++) {
            const size_t o = fb + (size_t)(i0 + m / CPL) * HS + j0 + m % CPL;
            F[m] = p.F0 ? p.F0[o] : 0.0f;
            S[m] = (MOM && p.S0) ? p.S0[o] : 0.0f;
        }
        Loader<G1, true> in;
        in.load(p, bh, 0, tid);
        in.stage(sg[0], tid);
        in.load(p, bh, CK, tid);
        for (int c = 0; c < nck; c++) {
            __syncthreads();  // chunk c is staged; everyone is done with the other buffer
            if (c + 1 < nck) in.stage(sg[(c + 1) & 1], tid);
            in.load(p, bh, (c + 2) * CK, tid);
            const Stage &st = sg[c & 1];
            park<R, CPL>(parked<MOM>(p, bh, c, 0), F, i0, j0);
            if (MOM) park<R, CPL>(parked<MOM>(p, bh, c, 2), S, i0, j0);
            const int n = min(CK, T - c * CK);
            float kept[CPL];
            auto step = [&](const StepIn<R, CPL, true> &x, int s) {
                float r[CPL];
                fwd_step<MOM, R, CPL>(F, S, x, M, cap, r);
#pragma unroll
                for (int z = 0; z < CPL; z++) kept[z] = lc == s ? r[z] : kept[z];
#pragma unroll
                for (int m = 0; m < NE; m++) top = fmaxf(top, fabsf(F[m]));
            };
#pragma unroll
            for (int z = 0; z < CPL; z++) kept[z] = 0.0f;
            StepIn<R, CPL, true> cur, nxt;
            cur.read(st, 0, i0, j0);
            if (n == CK) {
#pragma unroll
                for (int s = 0; s < CK; s++) {
                    if (s + 1 < CK) nxt.read(st, s + 1, i0, j0);
                    step(cur, s);
                    cur = nxt;
                }
            } else {
                for (int s = 0; s < n; s++) {
                    nxt.read(st, min(s + 1, CK - 1), i0, j0);
                    step(cur, s);
                    cur = nxt;
                }
            }
            if (lc < n)
#pragma unroll
                for (int z = 0; z < CPL; z++) p.r[hb + (size_t)(c * CK + lc) * HS + j0 + z] = kept[z];
        }
        // (a bounded element holds +-cap, a NaN became -cap)
        const int any = __syncthreads_or(!(top < cap));
        if (tid == 0) p.hit[bh * NG + cg] = any;
        return;
    }

    float dF[NE], dS[NE];
#pragma unroll
    for (int m = 0; m < NE; m++) {
        const size_t o = fb + (size_t)(i0 + m / CPL) * HS + j0 + m % CPL;
        dF[m] = p.dFT ? p.dFT[o] : 0.0f;
        dS[m] = (MOM && p.dST) ? p.dST[o] : 0.0f;
    }
    if (p.part && p.hit[bh * NG + cg]) {  // these columns are walked with the bound's mask
        park<R, CPL>(parked<MOM>(p, bh, nck - 1, 1), dF, i0, j0);
        if (MOM) park<R, CPL>(parked<MOM>(p, bh, nck - 1, 3), dS, i0, j0);
        return;
    }
    Loader<G1, false> in;
    in.load(p, bh, (nck - 1) * CK, tid);
    in.stage(sg[(nck - 1) & 1], tid);
    in.load(p, bh, (nck - 2) * CK, tid);
    for (int c = nck - 1; c >= 0; c--) {
        __syncthreads();
        if (c > 0) in.stage(sg[(c - 1) & 1], tid);
        in.load(p, bh, (c - 2) * CK, tid);
        const Stage &st = sg[c & 1];
        park<R, CPL>(parked<MOM>(p, bh, c, 1), dF, i0, j0);
        if (MOM) park<R, CPL>(parked<MOM>(p, bh, c, 3), dS, i0, j0);
        const int n = min(CK, T - c * CK);
        float keptr[CPL], keptv[CPL];
        auto step = [&](const StepIn<R, CPL, false> &x, int s) {
            float dr[CPL], dv[CPL];
            rev_step<MOM, R, CPL>(dF, dS, x, M, nullptr, cap, dr, dv);
#pragma unroll
            for (int z = 0; z < CPL; z++) {
                keptr[z] = lc == s ? dr[z] : keptr[z];
                keptv[z] = lc == s ? dv[z] : keptv[z];
            }
        };
#pragma unroll
        for (int z = 0; z < CPL; z++) keptr[z] = keptv[z] = 0.0f;
        StepIn<R, CPL, false> cur, nxt;
        cur.read(st, n - 1, i0, j0);
        if (n == CK) {
#pragma unroll
            for (int s = CK - 1; s >= 0; s--) {
                if (s > 0) nxt.read(st, s - 1, i0, j0);
                step(cur, s);
                cur = nxt;
            }
        } else {
            for (int s = n - 1; s >= 0; s--) {
                nxt.read(st, max(s - 1, 0), i0, j0);
                step(cur, s);
                cur = nxt;
            }
        }
        if (lc < n) {
#pragma unroll
            for (int z = 0; z < CPL; z++) {
                const size_t o = hb + (size_t)(c * CK + lc) * HS + j0 + z;
                p.dr[o] = keptr[z];
                p.dv[o] = keptv[z];
            }
        }
    }
}

// 2. The reverse walk with the bound's mask, in the marked columns: every chunk's states are replayed from its parked
// ones (r is known) and kept, then the chunk is walked back. As in the walks above, a chunk's inputs are loaded two chunks
// ahead into registers and staged one ahead (double-buffered, one barrier a chunk), and the parked states come one ahead.
template <bool G1, bool MOM>
__global__ __launch_bounds__(256) void mem_bwd_bound_kernel(MemBwdArgs p) {
    const int bh = blockIdx.x >> 2, cg = blockIdx.x & 3;
    if (!cols_hit(p, bh, cg)) return;
    __shared__ __attribute__((aligned(16))) Stage sg[2];
    __shared__ float sv[2][CK][16], sr[2][CK][16];  // v and r of the workgroup's 16 columns
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15;
    const int i0 = 4 * l16, jl = 4 * wave + (lane >> 4), j = 16 * cg + jl;
    const int T = p.T, nck = (T + CK - 1) / CK;
    const size_t hb = (size_t)bh * T * HS;
    const float M = p.m, cap = p.cap;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto state = [&](int c, int which) {
        return *reinterpret_cast<const f32x4 *>(parked<MOM>(p, bh, c, which) + j * HS + i0);
    };
    // the gradients after the last step, as the first walk parked them
    float dF[4], dS[4];
    {
        const f32x4 f = state(nck - 1, 1), s = MOM ? state(nck - 1, 3) : zero;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            dF[m] = f[m];
            dS[m] = s[m];
        }
    }
    Loader<G1, false> in;
    float lv, lr;  // v and r of step tid / 16, column tid % 16
    auto load = [&](int c) {
        in.load(p, bh, c * CK, tid);
        const int t = c * CK + (tid >> 4);
        lv = lr = 0.0f;
        if (c < 0 || t >= T) return;
        const size_t o = hb + (size_t)t * HS + 16 * cg + (tid & 15);
        lv = p.v[o];
        lr = p.r[o];
    };
    auto stage = [&](int b) {
        in.stage(sg[b], tid);
        sv[b][tid >> 4][tid & 15] = lv;
        sr[b][tid >> 4][tid & 15] = lr;
    };
    load(nck - 1);
    stage((nck - 1) & 1);
    load(nck - 2);
    f32x4 f0 = state(nck - 1, 0), s0 = MOM ? state(nck - 1, 2) : zero;
    for (int c = nck - 1; c >= 0; c--) {
        __syncthreads();  // chunk c is staged; everyone is done with the other buffer
        if (c > 0) stage((c - 1) & 1);
        load(c - 2);
        float Ft[CK + 1][4], S[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            Ft[0][m] = f0[m];
            S[m] = s0[m];
        }
        if (c > 0) {
            f0 = state(c - 1, 0);
            if (MOM) s0 = state(c - 1, 2);
        }
        park<4, 1>(parked<MOM>(p, bh, c, 1), dF, i0, j);
        if (MOM) park<4, 1>(parked<MOM>(p, bh, c, 3), dS, i0, j);
        const int n = min(CK, T - c * CK), b = c & 1;
        const Stage &st = sg[b];
        float keptr = 0.0f, keptv = 0.0f;
        auto chunk = [&](auto full) {
            constexpr bool FULL = decltype(full)::value;
            // a step's operands are read during the step before it, and not earlier (registers: see sched_barrier)
            struct {
                f32x4 x, k, a;
                float r, v;
            } in[2];
            auto read = [&](int s) {
                auto at = [&](const float (&d)[CK][HS]) { return *reinterpret_cast<const f32x4 *>(&d[s][i0]); };
                in[s & 1] = {at(st.abe), at(st.bk), at(st.a), sr[b][s][jl], sv[b][s][jl]};
            };
            read(0);
#pragma unroll
            for (int s = 0; s < CK; s++)
                if (FULL || s < n) {
                    if (s + 1 < CK) read(s + 1);
                    const auto &z = in[s & 1];
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const float u = fmaf(-z.x[m], z.r, z.k[m] * z.v);
                        if (MOM) S[m] = fmaf(M, S[m], u);
                        const float f = fmaf(z.a[m], Ft[s][m], MOM ? S[m] : u);
                        Ft[s + 1][m] = __builtin_amdgcn_fmed3f(f, -cap, cap);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            StepIn<4, 1, false> x[2];
            x[1].read(st, n - 1, i0, j);
            if (!FULL) x[0] = x[1];
#pragma unroll
            for (int s = CK - 1; s >= 0; s--)
                if (FULL || s < n) {
                    if (s > 0) x[(s - 1) & 1].read(st, s - 1, i0, j);
                    float dr[1], dv[1];
                    rev_step<MOM, 4, 1>(dF, dS, x[s & 1], M, Ft[s + 1], cap, dr, dv);
                    keptr = l16 == s ? dr[0] : keptr;
                    keptv = l16 == s ? dv[0] : keptv;
                    __builtin_amdgcn_sched_barrier(0);
                }
        };
        if (n == CK) chunk(std::integral_constant<bool, true>{});
        else chunk(std::integral_constant<bool, false>{});
        if (l16 < n) {
            const size_t o = hb + (size_t)(c * CK + l16) * HS + j;
            p.dr[o] = keptr;
            p.dv[o] = keptv;
        }
    }
}

// 3. The rows' gradients of one (head, chunk): lane = row, wave w columns 8w .. 8w + 7. The steps are replayed from
// the parked (F, S), every F of half a chunk kept (the first half is replayed twice: 72 registers instead of 136
// leave room for two workgroups on a CU, whose loads and barriers then hide behind each other), and walked back
// from the parked (dF, dS); a step's five row sums over the wave's columns go to LDS, and once per two steps (two
// buffers, one barrier) the eight waves' are added in order. 17 VALU operations per element and step (21 with the
// bound's mask) and no exchange between lanes. 64 heads x 2048 steps: 445 us, of which the VALU 170 and the 1.05 GB
// 210; keeping all 16 F (one workgroup per CU) 580, without the operands' read-ahead 487.
constexpr int RW = 8, RG = 2, HC = CK / 2;  // waves (8 columns each), steps per combine, steps whose F are kept

typedef const __attribute__((address_space(4))) float *ScalarPtr;  // uniform, written (by an output on an input) after the last read only

struct RowsLds {
    float q[CK][HS], k[CK][HS], e[CK][HS], a[CK][HS], b[CK][HS], abe[CK][HS];
    float red[2][RW][RG][5][HS];  // per buffer, wave and step: dq, sum gP F, sv, sr, sum dr F
};

template <bool G1, bool MOM, bool FULL, bool BOUND>
__device__ __forceinline__ void rows_chunk(const MemBwdArgs &p, RowsLds &L, int bh, int c, int n, int lane, int wave) {
    constexpr int NC = HS / RW;
    const float M = p.m, cap = p.cap;
    const size_t hb = (size_t)bh * p.T * HS, o0 = hb + (size_t)c * CK * HS;
    ScalarPtr v = (ScalarPtr)(p.v + o0 + NC * wave), rr = (ScalarPtr)(p.r + o0 + NC * wave);
    const ScalarPtr dy = (ScalarPtr)(p.dy + o0 + NC * wave), drr = (ScalarPtr)(p.dr + o0 + NC * wave);
    // the two pointers made new to the compiler: each pass over the steps loads its v and r again, where keeping a
    // pass's for the next would spill the scalar registers
    auto renew = [&]() {
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+s"(v), "+s"(rr));
#endif
    };
    float Ft[HC + 1][NC], S[NC], dF[NC], dS[NC];
    auto get = [&](float (&X)[NC], int which) {
        const float *src = parked<MOM>(p, bh, c, which) + NC * wave * HS + lane;
#pragma unroll
        for (int z = 0; z < NC; z++) X[z] = src[z * HS];
    };
    // A step's operands are read while the step before it is computed, and not earlier (sched_barrier ends each
    // step: the scalar registers hold two steps').
    struct FwdIn {
        float v[NC], r[NC], a, b, k, x;
    };
    struct RevIn {
        float v[NC], r[NC], y[NC], d[NC], q, e, a;
    };
    auto read_fwd = [&](FwdIn &in, int s) {
#pragma unroll
        for (int z = 0; z < NC; z++) {
            in.v[z] = v[s * HS + z];
            in.r[z] = rr[s * HS + z];
        }
        in.a = L.a[s][lane];
        in.b = L.b[s][lane];
        in.k = L.k[s][lane];
        in.x = L.abe[s][lane];
    };
    auto read_rev = [&](RevIn &in, int s) {
#pragma unroll
        for (int z = 0; z < NC; z++) {
            in.v[z] = v[s * HS + z];
            in.r[z] = rr[s * HS + z];
            in.y[z] = dy[s * HS + z];
            in.d[z] = drr[s * HS + z];
        }
        in.q = L.q[s][lane];
        in.e = L.e[s][lane];
        in.a = L.a[s][lane];
    };
    // F after a step from F before it (S in place)
    auto replay = [&](const FwdIn &in, const float (&Fa)[NC], float (&Fb)[NC]) {
        const float bk = in.b * in.k;
#pragma unroll
        for (int z = 0; z < NC; z++) {
            const float u = fmaf(-in.x, in.r[z], bk * in.v[z]);
            if (MOM) S[z] = fmaf(M, S[z], u);
            const float f = fmaf(in.a, Fa[z], MOM ? S[z] : u);
            Fb[z] = BOUND ? __builtin_amdgcn_fmed3f(f, -cap, cap) : f;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    get(dF, 1);
    if (MOM) get(dS, 3);
#pragma unroll
    for (int h = 1; h >= 0; h--) {
        const int s0 = h * HC;
        if (!FULL && s0 >= n) continue;
        get(Ft[0], 0);
        if (MOM) get(S, 2);
        // (an operand past the chunk's last step, read ahead, is the last step's again: in bounds, unused)
        auto at = [&](int s) { return FULL ? s : min(s, n - 1); };
        FwdIn fin[2];
        read_fwd(fin[0], 0);
        if (h) {
#pragma unroll
            for (int s = 0; s < HC; s++) {
                read_fwd(fin[(s + 1) & 1], at(s + 1));
                replay(fin[s & 1], Ft[0], Ft[0]);
            }
        }
        renew();
#pragma unroll
        for (int s = 0; s < HC; s++)
            if (FULL || s0 + s < n) {
                if (s + 1 < HC) read_fwd(fin[(s + 1) & 1], at(s0 + s + 1));
                replay(fin[s & 1], Ft[s], Ft[s + 1]);
            }
        renew();
        RevIn rin[2];
        const int top = FULL ? s0 + HC - 1 : min(s0 + HC, n) - 1;  // the half's last step
        read_rev(rin[(HC - 1) & 1], top);
        if (!FULL) rin[0] = rin[1];
#pragma unroll
        for (int g = HC / RG - 1; g >= 0; g--) {
            const int g0 = s0 + g * RG;
            if (!FULL && g0 >= n) continue;
#pragma unroll
            for (int w = RG - 1; w >= 0; w--) {
                const int s = g0 + w;
                if (FULL || s < n) {
                    const float(&Fa)[NC] = Ft[g * RG + w];
                    const float(&Fb)[NC] = Ft[g * RG + w + 1];
                    const RevIn &in = rin[s & 1];
                    if (g * RG + w > 0) read_rev(rin[(s - 1) & 1], s - 1);
                    float sq = 0.0f, sa = 0.0f, sv = 0.0f, sr = 0.0f, sd = 0.0f;
#pragma unroll
                    for (int z = 0; z < NC; z++) {
                        const float yz = in.y[z], dz = in.d[z];
                        sq = fmaf(yz, Fb[z], sq);
                        float gP = fmaf(in.q, yz, dF[z]);
                        if (BOUND) gP = fabsf(Fb[z]) < cap ? gP : 0.0f;
                        sa = fmaf(gP, Fa[z], sa);
                        float du = gP;
                        if (MOM) {
                            du = gP + dS[z];
                            dS[z] = M * du;
                        }
                        sv = fmaf(du, in.v[z], sv);
                        sr = fmaf(du, in.r[z], sr);
                        sd = fmaf(dz, Fa[z], sd);
                        dF[z] = fmaf(in.e, dz, in.a * gP);
                    }
                    float(&o)[5][HS] = L.red[g & 1][wave][w];
                    o[0][lane] = sq;
                    o[1][lane] = sa;
                    o[2][lane] = sv;
                    o[3][lane] = sr;
                    o[4][lane] = sd;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __syncthreads();  // the group's sums are in; this buffer's last ones were combined before this barrier
            // wave 2 i (waves 0 and 2) finishes dq and dla of step i of the group, wave 2 i + 1 its dk, de and db
            const int i = wave >> 1, s = g0 + i, t = c * CK + s;
            if (i < RG && (FULL || s < n)) {
                auto sum = [&](int z) {
                    float x = L.red[g & 1][0][i][z][lane];
#pragma unroll
                    for (int w = 1; w < RW; w++) x += L.red[g & 1][w][i][z][lane];
                    return x;
                };
                const size_t o = hb + (size_t)t * HS + lane, og = G1 ? (size_t)bh * p.T + t : o;
                const float a = L.a[s][lane], b = L.b[s][lane], e = L.e[s][lane], sr = sum(3);
                if ((wave & 1) == 0) {
                    p.dq[o] = sum(0);
                    const float da = fmaf(-(b * e), sr, sum(1)) * a;
                    if (G1) {
                        const float x = ava::wave_sum(da);
                        if (lane == 0) p.dla[og] = x;
                    } else {
                        p.dla[o] = da;
                    }
                } else {
                    const float sv = sum(2);
                    p.dk[o] = b * sv;
                    p.de[o] = fmaf(-(a * b), sr, sum(4));
                    const float db = fmaf(-(a * e), sr, L.k[s][lane] * sv);
                    if (G1) {
                        const float x = ava::wave_sum(db);
                        if (lane == 0) p.db[og] = x;
                    } else {
                        p.db[o] = db;
                    }
                }
            }
        }
    }
    if (c == 0) {
        const size_t o = (size_t)bh * HS * HS + (size_t)lane * HS + NC * wave;
        auto put = [&](float *dst, const float (&X)[NC]) {
            if (!dst) return;
#pragma unroll
            for (int z = 0; z < NC; z++) dst[o + z] = X[z];
        };
        put(p.dF0, dF);
        if (MOM) put(p.dS0, dS);
    }
}

template <bool G1, bool MOM>
__global__ __launch_bounds__(64 * RW, 4) void mem_bwd_rows_kernel(MemBwdArgs p) {
    __shared__ __attribute__((aligned(16))) RowsLds L;
    const int nck = (p.T + CK - 1) / CK, bh = blockIdx.x / nck, c = blockIdx.x - bh * nck, n = min(CK, p.T - c * CK);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
    for (int h = 0; h < CK / RW; h++) {
        const int s = wave + RW * h;
        if (s < n) {
            const size_t o = ((size_t)bh * p.T + c * CK + s) * HS + lane, og = G1 ? (size_t)bh * p.T + c * CK + s : o;
            const float a = expf(p.la[og]), b = p.b[og], e = p.e[o];
            L.q[s][lane] = p.q[o];
            L.k[s][lane] = p.k[o];
            L.e[s][lane] = e;
            L.a[s][lane] = a;
            L.b[s][lane] = b;
            L.abe[s][lane] = (a * b) * e;
        }
    }
    // the chunk's v, dy, r and dr rows come into L2 together here; the scalar loads of a step then miss no further
    float warm = 0.0f;
    {
        const size_t o = ((size_t)bh * p.T + c * CK) * HS + min(2 * tid, n * HS - 2);
        for (const float *x : {p.v, p.dy, (const float *)p.r, (const float *)p.dr}) {
            const f32x2u w = *reinterpret_cast<const f32x2u *>(x + o);
            warm += w[0] + w[1];
        }
    }
    const bool bound = head_hit(p, bh);
    asm volatile("" ::"v"(warm));
    __syncthreads();
    if (bound)
        rows_chunk<G1, MOM, false, true>(p, L, bh, c, n, lane, wave);
    else if (n == CK)
        rows_chunk<G1, MOM, true, false>(p, L, bh, c, n, lane, wave);
    else
        rows_chunk<G1, MOM, false, false>(p, L, bh, c, n, lane, wave);
}

// dv, formed in the workspace (see ava_mem_scan_bwd)
__global__ __launch_bounds__(256) void mem_bwd_copy_kernel(const float *__restrict__ x, float *__restrict__ y, size_t n) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) y[i] = x[i];
}

struct Layout {
    size_t ck, r, hit;  // floats: the parked states; r, dr, and dv where it cannot go out at once; the marks
    size_t bytes() const { return (ck + 3 * r + hit) * sizeof(float); }
};
Layout layout(int BH, int T, bool mom) {
    return {(size_t)BH * ((T + CK - 1) / CK) * (mom ? 4 : 2) * HS * HS, (size_t)BH * T * HS, (size_t)BH * 8};
}

}  // namespace

extern "C" size_t ava_mem_scan_bwd_workspace(int BH, int T, int momentum) {
    if (BH <= 0 || T <= 0) return 0;
    return layout(BH, T, momentum != 0).bytes();
}

// The backward of ava_mem_scan (same layout and gates), from the initial state F0, S0 (nullable:
// zeros) and the gradients dy of y and dF_T, dS_T of the final state (nullable: zeros): dq, dk, de,
// dv [BH][T][hs]; dla, db [BH][T][g]; dF0, dS0 (nullable) the gradients of the initial state.
extern "C" int ava_mem_scan_bwd(const float *q, const float *k, const float *e, const float *v, const float *la,
                                const float *b, int BH, int T, int hs, int g, float m, float cap, const float *F0,
                                const float *S0, const float *dy, const float *dF_T, const float *dS_T, float *dq,
                                float *dk, float *de, float *dv, float *dla, float *db, float *dF0, float *dS0,
                                void *work, size_t work_bytes, ava_stream stream) {
    AVA_REQUIRE(hs == HS, AVA_ERR_UNSUPPORTED, "mem_scan_bwd: head size %d (this build runs 64)", hs);
    AVA_REQUIRE(g == 1 || g == HS, AVA_ERR_SHAPE, "mem_scan_bwd: g=%d (1 or hs)", g);
    AVA_REQUIRE(BH > 0 && T > 0, AVA_ERR_SHAPE, "mem_scan_bwd: BH=%d T=%d", BH, T);
    AVA_REQUIRE(q && k && e && v && la && b && dy && dq && dk && de && dv && dla && db && work, AVA_ERR_ARG,
                "mem_scan_bwd: NULL buffer");
    const bool mom = m != 0.0f;
    const size_t need = ava_mem_scan_bwd_workspace(BH, T, mom);
    AVA_REQUIRE(work_bytes >= need, AVA_ERR_SHAPE, "mem_scan_bwd: workspace %zu < %zu bytes", work_bytes, need);
    const Layout lo = layout(BH, T, mom);
    float *w = (float *)work;
    MemBwdArgs p{q, k, e, v, la, b, F0, mom ? S0 : nullptr, dy, dF_T, mom ? dS_T : nullptr, dq, dk, de, dv, dla, db,
                 dF0, mom ? dS0 : nullptr, w, w + lo.ck, w + lo.ck + lo.r, (int *)(w + lo.ck + 3 * lo.r), 0, 0, BH, T, m, cap};
    const hipStream_t st = (hipStream_t)stream;
    int cus = 0;
    if (int r = ava::device_cus(&cus)) return r;
    // An output may be an input's buffer. The rows kernel writes the others, each element after its last read; the
    // walks write dv while the inputs are still wanted, so on one of them it goes through the workspace.
    const size_t nv = lo.r, ng = (size_t)BH * T * g;
    auto on = [&](const float *x, size_t n) { return (uintptr_t)dv < (uintptr_t)(x + n) && (uintptr_t)x < (uintptr_t)(dv + nv); };
    const bool late = on(q, nv) || on(k, nv) || on(e, nv) || on(v, nv) || on(dy, nv) || on(la, ng) || on(b, ng);
    if (late) p.dv = w + lo.ck + 2 * lo.r;
    const int rows = BH * ava::ceil_div(T, CK);
    auto walk = [&](auto kern, int groups) {
        p.groups = groups;
        // From two heads a CU the forward walks alone fill the chip: they go first, and the reverse walks of columns that
        // reached the bound are left to the bound kernel. (Up to two chunks the launch more costs what they take.)
        if (BH >= 2 * cus && T > 2 * CK) {
            p.part = 1;
            kern<<<BH * groups, 256, 0, st>>>(p);
            p.part = 2;
            kern<<<BH * groups, 256, 0, st>>>(p);
        } else {
            kern<<<BH * groups * 2, 256, 0, st>>>(p);
        }
    };
    auto run = [&](auto w8, auto w4, auto w2, auto w1, auto bound, auto rows_k) {
        // A head's columns over 4 or 2 workgroups a direction while the CUs hold them all at once (three each, by LDS), over 8
        // only while each has a CU to itself. All three launches, T = 1024, momentum, 8 / 4 / 2 / 1 workgroups: 16 heads
        // 198 / 200 / 271 / 424 us, 32 277 / 241 / 311 / 462, 64 559 / 400 / 421 / 583, 96 747 / 569 / 589 / 671, 128 980 / 797 / 702
        // / 769, 192 1427 / 1101 / 1004 / 1123, 256 - / 1446 / 1301 / 1296.
        if (16L * BH <= cus) walk(w8, 8);
        else if (8L * BH <= 3L * cus) walk(w4, 4);
        else if (4L * BH <= 3L * cus) walk(w2, 2);
        else walk(w1, 1);
        bound<<<BH * 4, 256, 0, st>>>(p);
        rows_k<<<rows, 64 * RW, 0, st>>>(p);
        if (late) mem_bwd_copy_kernel<<<(unsigned)std::min<size_t>(2048, (nv + 255) / 256), 256, 0, st>>>(p.dv, dv, nv);
    };
#define AVA_MB(G1_, MOM_)                                                                                            \
    run(mem_bwd_walk_kernel<G1_, MOM_, 2, 1>, mem_bwd_walk_kernel<G1_, MOM_, 4, 1>,                                 \
        mem_bwd_walk_kernel<G1_, MOM_, 4, 2>, mem_bwd_walk_kernel<G1_, MOM_, 4, 4>, mem_bwd_bound_kernel<G1_, MOM_>, \
        mem_bwd_rows_kernel<G1_, MOM_>)
    if (g == 1) {
        if (mom) AVA_MB(true, true);
        else AVA_MB(true, false);
    } else {
        if (mom) AVA_MB(false, true);
        else AVA_MB(false, false);
    }
#undef AVA_MB
    AVA_LAUNCHED("mem_scan_bwd");
    return AVA_OK;
}
