// The backward of the general LIF scan for gfx950 (the surrogate gradient of the straight-through
// spikes: gpu/arch.rs:964-1071 lif_ref's autograd; the CUDA form lifg_bwd, gpu/lif.cu:3228-3290).
//
// One lane per (b, c), channel-contiguous as the forward, walking T twice:
//   1. the forward replayed from (v0, s0, a0), nothing kept but the state at the start of every
//      segment of K steps (segments are cut from the end, so only the first may be short). That
//      state (v, s, a) is parked in the segment's own first three rows of dI, which the reverse
//      pass overwrites last: no workspace and 12 bytes per segment of traffic.
//   2. segment by segment from the last: the K steps replayed from the parked state with v_t and
//      a_t in registers, then walked back. The next (earlier) segment's currents, incoming
//      gradients and parked state are loaded while this one is processed.
// HBM per element: the currents twice, the incoming gradient once and dI once, 16 bytes (a
// backward that stores the membrane and trace instead moves 28).
//
// Per step, backwards (G = dL/dv_t, carried: cv = beta G_{t+1}, ca = dL/da_{t+1} rho):
//   ds/dv, ds/dth from the surrogate 1 / (1 + S |x|)^2 of each spike edge x = v - k th, -v - k th;
//   gs = dL/ds_t (minus te G_{t+1} when the reset carries gradient, te = th_t or 2 beta / (ds/dv)
//   where th_t ds/dv > 2 beta);  G = gs ds/dv + cv;  dbeta += G v_{t-1};
//   ALIF: gth = gs ds/dth (- s_t G_{t+1}), ga = gth gain + ca, dgain += gth a_t,
//   drho += ga (a_{t-1} - |s_{t-1}|), ca = rho ga.
// Every operation is rounded on its own (-ffp-contract=off), in the order of the CPU statement.
// Measured, 64 x 2048 x 2048: 960 us, 4.3 GB at 4.5 TB/s (a device copy: 5.0); 1244 us, VALU-bound, with IEEE divides
// in the surrogates and the spikes by differences and formed again on the way back.
#include <type_traits>

#include "common.h"

namespace {

template <int LEVELS, bool SIGNED>
__device__ __forceinline__ float spike_of(float v, float th) {
    if (!SIGNED) return (v - th >= 0.0f) ? 1.0f : 0.0f;
    float h = 0.0f;
#pragma unroll
    for (int k = 1; k <= LEVELS; k++) {
        const float kth = th * (float)k;
        h += ((v - kth >= 0.0f) ? 1.0f : 0.0f) - ((-v - kth >= 0.0f) ? 1.0f : 0.0f);
    }
    return h;
}

// 1 / d for d in [1, 2^125) as the IEEE divide rounds it: the hardware's reciprocal (within an ulp) and one Newton
// step with a fused residual; compared with the divide on every float of the range. 3 operations instead of about 10.
__device__ __forceinline__ float recip(float d) {
    const float r = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, r, 1.0f), r, r);
}

template <int LEVELS, bool SIGNED, bool FIN>
__device__ __forceinline__ float spike(float v, float th) {
    return FIN ? (float)ava::lif_count<LEVELS, SIGNED>(v, th) : spike_of<LEVELS, SIGNED>(v, th);
}

// NEAR: slope |x| is below 2^60 (or NaN), so a^2 is in recip's range.
template <bool NEAR>
__device__ __forceinline__ float surrogate(float x, float slope) {
    const float a = 1.0f + slope * fabsf(x);
    return NEAR ? recip(a * a) : 1.0f / (a * a);
}

// d s / d v and d s / d th of one step's surrogate spike.
template <int LEVELS, bool SIGNED, bool NEAR>
__device__ __forceinline__ void dspike(float v, float th, float slope, float &dv, float &dth) {
    if (!SIGNED) {
        const float g = surrogate<NEAR>(v - th, slope);
        dv = g;
        dth = -g;
        return;
    }
    float a = 0.0f, b = 0.0f;
#pragma unroll
    for (int k = 1; k <= LEVELS; k++) {
        const float kth = th * (float)k;
        const float gu = surrogate<NEAR>(v - kth, slope), gd = surrogate<NEAR>(-v - kth, slope);
        a += gu + gd;
        b += (float)k * (gd - gu);
    }
    dv = a;
    dth = b;
}

// Whether a chain's thresholds stay below 3e8 (rho in [0, 1] keeps the trace within its start, the carried spike and
// 2) and the slope is in [0, 1e6): then spikes count by ava::lif_count, and membranes below NEAR_V give NEAR surrogates. (A
// trainer's slope may be negative, and 1 + slope |x| then anything down to 0.)
constexpr float NEAR_V = 1e9f;
__device__ __forceinline__ bool tame(float th0, float rho, float gain, float a0, float s0, float slope) {
    return fabsf(th0) < 1e8f && rho >= 0.0f && rho <= 1.0f && fabsf(gain) < 1e4f && fabsf(a0) < 1e4f &&
           fabsf(s0) < 1e4f && slope >= 0.0f && slope < 1e6f;
}

struct LifBwdArgs {
    const float *cur, *ps, *v0, *s0, *a0, *gs, *gv, *ga;
    float *dI, *dv0, *da0, *dbeta, *drho, *dgain;
    int B, T, D;
    float slope;
    int rg;
};

// Whether the wave's chains (this lane's: channel c, state index i) are tame.
template <bool ALIF>
__device__ __forceinline__ bool wave_tame(const LifBwdArgs &p, int c, int i) {
    return __all(tame(p.ps[p.D + c], ALIF ? p.ps[2 * p.D + c] : 0.0f, ALIF ? p.ps[3 * p.D + c] : 0.0f,
                      ALIF ? p.a0[i] : 0.0f, p.s0[i], p.slope));
}

// FIN: the wave's chains are tame. KEEP: the spikes are kept for the way back, not formed again (see ava_lif_scan_bwd).
template <int K, int LEVELS, bool SIGNED, bool ALIF, bool FIN, bool KEEP>
__device__ __forceinline__ void lif_bwd_chain(const LifBwdArgs &p, int gid) {
    const int D = p.D, T = p.T;
    const int b = gid / D, c = gid - b * D;
    const float bt = p.ps[c], th0 = p.ps[D + c], rho = p.ps[2 * D + c], gain = p.ps[3 * D + c];
    const float omr = 1.0f - rho;
    const size_t col = (size_t)b * T * D + c;
    const float *x = p.cur + col, *g = p.gs + col;
    float *o = p.dI + col;
    const float v0 = p.v0[gid], s0 = p.s0[gid], a0 = ALIF ? p.a0[gid] : 0.0f;
    const int nseg = (T + K - 1) / K;
    // segment q (0 = the last) covers [max(0, T - (q + 1) K), T - q K)
    auto seg0 = [&](int q) { return max(0, T - (q + 1) * K); };

    float buf[K] = {}, nxt[K] = {};  // (entries past a short segment are never read)
    auto load_cur = [&](int q, float (&dst)[K]) {
        const int t0 = seg0(q), n = T - q * K - t0;
#pragma unroll
        for (int i = 0; i < K; i++)
            if (i < n) dst[i] = __builtin_nontemporal_load(x + (size_t)(t0 + i) * D);
    };

    // 1. the forward, parking the state at each segment's start (segments after the first)
    {
        float v = v0, sp = s0, a = a0, thp = ALIF ? th0 + a0 * gain : th0;
        load_cur(nseg - 1, buf);
        for (int q = nseg - 1; q >= 0; q--) {
            if (q > 0) load_cur(q - 1, nxt);
            const int t0 = seg0(q), n = T - q * K - t0;
            if (t0 > 0) {
                o[(size_t)t0 * D] = v;
                o[(size_t)(t0 + 1) * D] = sp;
                if (ALIF) o[(size_t)(t0 + 2) * D] = a;
            }
#pragma unroll
            for (int i = 0; i < K; i++) {
                if (i < n) {
                    float tht = th0;
                    if (ALIF) {
                        a = a * rho + fabsf(sp) * omr;
                        tht = th0 + a * gain;
                    }
                    v = (v * bt + buf[i]) - sp * thp;
                    sp = spike<LEVELS, SIGNED, FIN>(v, tht);
                    thp = tht;
                }
            }
#pragma unroll
            for (int i = 0; i < K; i++) buf[i] = nxt[i];
        }
    }

    // 2. backwards, segment by segment
    float cv = p.gv ? p.gv[gid] : 0.0f, ca = (ALIF && p.ga) ? p.ga[gid] : 0.0f;
    float gb = 0.0f, gr = 0.0f, gg = 0.0f, Gn = 0.0f;  // Gn = dL/dv_{t+1}
    float gbuf[K] = {}, gnxt[K] = {};
    auto load_g = [&](int q, float (&dst)[K]) {
        const int t0 = seg0(q), n = T - q * K - t0;
#pragma unroll
        for (int i = 0; i < K; i++)
            if (i < n) dst[i] = g[(size_t)(t0 + i) * D];
    };
    float ckv, cks, cka, nkv = 0.0f, nks = 0.0f, nka = 0.0f;
    auto load_ck = [&](int q, float &kv, float &ks, float &ka) {
        const int t0 = seg0(q);
        kv = v0;
        ks = s0;
        ka = a0;
        if (t0 > 0) {
            kv = o[(size_t)t0 * D];
            ks = o[(size_t)(t0 + 1) * D];
            ka = ALIF ? o[(size_t)(t0 + 2) * D] : 0.0f;
        }
    };
    load_cur(0, buf);
    load_g(0, gbuf);
    load_ck(0, ckv, cks, cka);
    for (int q = 0; q < nseg; q++) {
        if (q + 1 < nseg) {
            load_cur(q + 1, nxt);
            load_g(q + 1, gnxt);
            load_ck(q + 1, nkv, nks, nka);
        }
        const int t0 = seg0(q), n = T - q * K - t0;
        float vs[K] = {}, as[K] = {}, ss[KEEP ? K : 1] = {}, top = 0.0f;
        auto spk = [&](int i) {
            if constexpr (KEEP) return ss[i];
            else return spike<LEVELS, SIGNED, FIN>(vs[i], ALIF ? th0 + as[i] * gain : th0);
        };
        {
            float v = ckv, sp = cks, a = cka, thp = ALIF ? th0 + cka * gain : th0;
#pragma unroll
            for (int i = 0; i < K; i++) {
                if (i < n) {
                    float tht = th0;
                    if (ALIF) {
                        a = a * rho + fabsf(sp) * omr;
                        tht = th0 + a * gain;
                    }
                    v = (v * bt + buf[i]) - sp * thp;
                    sp = spike<LEVELS, SIGNED, FIN>(v, tht);
                    thp = tht;
                    vs[i] = v;
                    as[i] = a;
                    if constexpr (KEEP) ss[i] = sp;
                    if (FIN) top = fmaxf(top, fabsf(v));
                }
            }
        }
        auto back = [&](auto near) {
            constexpr bool NEAR = decltype(near)::value;
#pragma unroll
            for (int i = K - 1; i >= 0; i--) {
                if (i < n) {
                    const float vt = vs[i], at = ALIF ? as[i] : 0.0f;
                    const float tht = ALIF ? th0 + at * gain : th0;
                    float dv, dth;
                    dspike<LEVELS, SIGNED, NEAR>(vt, tht, p.slope, dv, dth);
                    float gst = gbuf[i];
                    if (p.rg) {
                        const float qq = tht * dv, cap = 2.0f * bt;
                        gst -= (qq > cap ? cap / dv : tht) * Gn;
                    }
                    const float G = gst * dv + cv;
                    gb += G * (i > 0 ? vs[i - 1] : ckv);
                    if (ALIF) {
                        float gth = gst * dth;
                        if (p.rg) gth -= spk(i) * Gn;
                        const float gaa = gth * gain + ca;
                        gg += gth * at;
                        const float ap = i > 0 ? as[i - 1] : cka;
                        const float sprev = i > 0 ? spk(i - 1) : cks;
                        gr += gaa * (ap - fabsf(sprev));
                        ca = rho * gaa;
                    }
                    o[(size_t)(t0 + i) * D] = G;
                    Gn = G;
                    cv = bt * G;
                }
            }
        };
        if (FIN && __all(top < NEAR_V)) back(std::integral_constant<bool, true>{});
        else back(std::integral_constant<bool, false>{});
#pragma unroll
        for (int i = 0; i < K; i++) {
            buf[i] = nxt[i];
            gbuf[i] = gnxt[i];
        }
        ckv = nkv;
        cks = nks;
        cka = nka;
    }
    if (ALIF && p.rg) {  // the first step's reset used the initial threshold theta + a0 gain
        const float g0 = -s0 * Gn;
        gg += g0 * a0;
        ca += g0 * gain;
    }
    p.dv0[gid] = cv;
    if (p.da0) p.da0[gid] = ALIF ? ca : 0.0f;
    p.dbeta[gid] = gb;
    if (p.drho) p.drho[gid] = ALIF ? gr : 0.0f;
    if (p.dgain) p.dgain[gid] = ALIF ? gg : 0.0f;
}

template <int K, int LEVELS, bool SIGNED, bool ALIF, bool KEEP>
__global__ __launch_bounds__(256, 2) void lif_bwd_kernel(LifBwdArgs p) {
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = gid < p.B * p.D;
    const bool fin = wave_tame<ALIF>(p, in ? gid % p.D : 0, in ? gid : 0);
    if (!in) return;
    if (fin) lif_bwd_chain<K, LEVELS, SIGNED, ALIF, true, KEEP>(p, gid);
    else lif_bwd_chain<K, LEVELS, SIGNED, ALIF, false, KEEP>(p, gid);
}

// Steps per segment: 5 x 16 registers of currents, gradients and replayed state. 32-step segments
// (226 VGPRs, the same two waves per SIMD) measured 7% slower at config[1]'s shape.
constexpr int SEG = 16;

// ------------------------------------------------------------------ the backward in parallel segments
//
// With few (stream, channel) chains (the training step's B = 4: 4,096 lanes, a sixteenth of the SIMDs)
// the walk above is a long dependent chain per lane. Given the forward trajectory, though, the walk
// is linear in what it carries between steps, X = (Gn, cv, ca): per step
//   gst = g - te Gn;  G = gst dv + cv;  ALIF: gth = gst dth - s Gn (reset gradient), gaa = gth gain + ca;
//   then (Gn, cv, ca) <- (G, beta G, rho gaa), and dbeta, dgain, drho gather G v_prev, gth a, gaa (a_prev -
//   |s_prev|),
// so a segment of SK steps maps the X entering it (from the later steps) to the X leaving it, and its
// parameter gradients, by affine functions of X. Four passes:
//   A (one lane per chain): the forward replayed, the state (v, s, a) parked at every segment start
//      (skipped when the caller's forward parked them: ava::lif_scan's park);
//   B (one lane per (chain, segment)): the segment's forward replayed from its parked state, then walked
//      back with every carried and gathered quantity held as its 4 coefficients (1, X) — the affine
//      functions, written to the workspace;
//   C (one lane per chain): the segments' functions applied from the last to the first, from X = (0, dL/dv_T,
//      dL/da_T): each segment's entering X is kept, and the parameter gradients are summed;
//   D (one lane per (chain, segment)): the segment replayed and walked back with its entering X, as the
//      walk above, writing dI.
// The forward arithmetic is the scan's own (the same spikes and states); the backward sums associate
// differently from the one-lane walk (rounding only). Per (chain, segment): 3 parked state floats and
// 27 workspace floats (24 coefficients, the entering X).
constexpr int SK = ava::LIF_SEG_STEPS;
constexpr int SW = 27;  // workspace floats per (chain, segment): 24 coefficients, the entering X

struct LifSegArgs {
    LifBwdArgs p;
    float *ws;    // [nseg][SW][chains]
    float *park;  // [nseg][3][chains]: the state at each segment's start
    int nseg;
};

// field f of (segment sg, chain ch): 0..23 the coefficients, 24..26 the entering X
__device__ __forceinline__ float *ws_at(const LifSegArgs &a, int sg, int f, int ch) {
    return a.ws + ((size_t)sg * SW + f) * (size_t)(a.p.B * a.p.D) + ch;
}
__device__ __forceinline__ float *park_at(const LifSegArgs &a, int sg, int f, int ch) {
    return a.park + ((size_t)sg * 3 + f) * (size_t)(a.p.B * a.p.D) + ch;
}

// one forward step of the scan (lif_scan_kernel's loop body)
template <int LEVELS, bool SIGNED, bool ALIF, bool FIN>
__device__ __forceinline__ void fwd1(float x, float bt, float th0, float rho, float omr, float gain, float &v,
                                     float &sp, float &a, float &thp) {
    float tht = th0;
    if (ALIF) {
        a = a * rho + fabsf(sp) * omr;
        tht = th0 + a * gain;
    }
    v = (v * bt + x) - sp * thp;
    sp = spike<LEVELS, SIGNED, FIN>(v, tht);
    thp = tht;
}

template <int LEVELS, bool SIGNED, bool ALIF>
__global__ __launch_bounds__(256) void lif_seg_park_kernel(LifSegArgs A) {
    const LifBwdArgs &p = A.p;
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int D = p.D, T = p.T;
    if (gid >= p.B * D) return;
    const int b = gid / D, c = gid - b * D;
    const float bt = p.ps[c], th0 = p.ps[D + c], rho = p.ps[2 * D + c], gain = p.ps[3 * D + c], omr = 1.0f - rho;
    const float *x = p.cur + (size_t)b * T * D + c;
    float v = p.v0[gid], sp = p.s0[gid], a = ALIF ? p.a0[gid] : 0.0f;
    float thp = ALIF ? th0 + a * gain : th0;
    *park_at(A, 0, 0, gid) = v;
    *park_at(A, 0, 1, gid) = sp;
    *park_at(A, 0, 2, gid) = a;
    // two segments' currents in flight, as the scan's
    auto scan = [&](auto fin) {
        constexpr bool FIN = decltype(fin)::value;
        float buf[SK];
#pragma unroll
        for (int i = 0; i < SK; i++) buf[i] = __builtin_nontemporal_load(x + (size_t)min(i, T - 1) * D);
        for (int t0 = 0; t0 < T; t0 += SK) {
            float nxt[SK];
#pragma unroll
            for (int i = 0; i < SK; i++) nxt[i] = __builtin_nontemporal_load(x + (size_t)min(t0 + SK + i, T - 1) * D);
            if (t0 + SK < T) {
#pragma unroll
                for (int i = 0; i < SK; i++) fwd1<LEVELS, SIGNED, ALIF, FIN>(buf[i], bt, th0, rho, omr, gain, v, sp, a, thp);
                const int sg = t0 / SK + 1;
                *park_at(A, sg, 0, gid) = v;
                *park_at(A, sg, 1, gid) = sp;
                *park_at(A, sg, 2, gid) = a;
            }
#pragma unroll
            for (int i = 0; i < SK; i++) buf[i] = nxt[i];
        }
    };
    if (wave_tame<ALIF>(p, c, gid)) scan(std::integral_constant<bool, true>{});
    else scan(std::integral_constant<bool, false>{});
}

// The segment's forward from its parked state: vs, as after each of its n steps (and the state before)
// (FIN: as fwd1's; returns the largest |v|)
template <int LEVELS, bool SIGNED, bool ALIF, bool FIN>
__device__ __forceinline__ float seg_replay(const float *x, int D, int t0, int n, float bt, float th0, float rho,
                                           float omr, float gain, float v, float sp, float a, float (&vs)[SK],
                                           float (&as)[SK]) {
    float thp = ALIF ? th0 + a * gain : th0, top = 0.0f;
#pragma unroll
    for (int i = 0; i < SK; i++) {
        if (i < n) {
            fwd1<LEVELS, SIGNED, ALIF, FIN>(x[(size_t)(t0 + i) * D], bt, th0, rho, omr, gain, v, sp, a, thp);
            vs[i] = v;
            as[i] = a;
            top = fmaxf(top, fabsf(v));
        }
    }
    return top;
}

// an affine function of X = (Gn, cv, ca): c[0] + c[1] Gn + c[2] cv + c[3] ca
struct Aff {
    float c[4];
};
__device__ __forceinline__ Aff aff(float k) { return Aff{{k, 0.0f, 0.0f, 0.0f}}; }
__device__ __forceinline__ Aff axpy(float s, const Aff &x, const Aff &y) {  // s x + y
    Aff r;
#pragma unroll
    for (int i = 0; i < 4; i++) r.c[i] = fmaf(s, x.c[i], y.c[i]);
    return r;
}
__device__ __forceinline__ Aff scal(float s, const Aff &x) {
    Aff r;
#pragma unroll
    for (int i = 0; i < 4; i++) r.c[i] = s * x.c[i];
    return r;
}

template <int LEVELS, bool SIGNED, bool ALIF, bool FIN>
__device__ __forceinline__ void seg_affine(const LifSegArgs &A, int gid) {
    const LifBwdArgs &p = A.p;
    const int chains = p.B * p.D;
    const int sg = gid / chains, ch = gid - sg * chains;
    const int D = p.D, T = p.T, b = ch / D, c = ch - b * D;
    const float bt = p.ps[c], th0 = p.ps[D + c], rho = p.ps[2 * D + c], gain = p.ps[3 * D + c], omr = 1.0f - rho;
    const int t0 = sg * SK, n = min(SK, T - t0);
    const float *x = p.cur + (size_t)b * T * D + c, *g = p.gs + (size_t)b * T * D + c;
    const float pv = *park_at(A, sg, 0, ch), ps_ = *park_at(A, sg, 1, ch), pa = *park_at(A, sg, 2, ch);
    float vs[SK] = {}, as[SK] = {};
    const float top = seg_replay<LEVELS, SIGNED, ALIF, FIN>(x, D, t0, n, bt, th0, rho, omr, gain, pv, ps_, pa, vs, as);
    Aff Gn{{0.0f, 1.0f, 0.0f, 0.0f}}, cv{{0.0f, 0.0f, 1.0f, 0.0f}}, ca{{0.0f, 0.0f, 0.0f, 1.0f}};
    Aff gb = aff(0.0f), gg = aff(0.0f), gr = aff(0.0f);
    auto back = [&](auto near) {
        constexpr bool NEAR = decltype(near)::value;
#pragma unroll
        for (int i = SK - 1; i >= 0; i--) {
            if (i < n) {
                const float vt = vs[i], at = ALIF ? as[i] : 0.0f;
                const float tht = ALIF ? th0 + at * gain : th0;
                float dv, dth;
                dspike<LEVELS, SIGNED, NEAR>(vt, tht, p.slope, dv, dth);
                const float gt = g[(size_t)(t0 + i) * D];
                float te = 0.0f;
                if (p.rg) {
                    const float qq = tht * dv, cap = 2.0f * bt;
                    te = qq > cap ? cap / dv : tht;
                }
                const Aff gst = axpy(-te, Gn, aff(gt));   // g - te Gn
                const Aff G = axpy(dv, gst, cv);          // gst dv + cv
                gb = axpy(i > 0 ? vs[i - 1] : pv, G, gb);
                if (ALIF) {
                    Aff gth = scal(dth, gst);
                    if (p.rg) gth = axpy(-spike<LEVELS, SIGNED, FIN>(vt, tht), Gn, gth);
                    const Aff gaa = axpy(gain, gth, ca);
                    gg = axpy(at, gth, gg);
                    const float ap = i > 0 ? as[i - 1] : pa;
                    const float sprev = i > 0 ? spike<LEVELS, SIGNED, FIN>(vs[i - 1], th0 + as[i - 1] * gain) : ps_;
                    gr = axpy(ap - fabsf(sprev), gaa, gr);
                    ca = scal(rho, gaa);
                }
                Gn = G;
                cv = scal(bt, G);
            }
        }
    };
    if (FIN && __all(top < NEAR_V)) back(std::integral_constant<bool, true>{});
    else back(std::integral_constant<bool, false>{});
    const Aff *out[6] = {&Gn, &cv, &ca, &gb, &gg, &gr};
#pragma unroll
    for (int f = 0; f < 6; f++)
#pragma unroll
        for (int i = 0; i < 4; i++) *ws_at(A, sg, 4 * f + i, ch) = out[f]->c[i];
}

template <int LEVELS, bool SIGNED, bool ALIF>
__global__ __launch_bounds__(256) void lif_seg_affine_kernel(LifSegArgs A) {
    const LifBwdArgs &p = A.p;
    const int chains = p.B * p.D, gid = blockIdx.x * blockDim.x + threadIdx.x;  // chain fastest
    const bool in = gid < chains * A.nseg;
    const int ch = in ? gid % chains : 0;
    const bool fin = wave_tame<ALIF>(p, ch % p.D, ch);
    if (!in) return;
    if (fin) seg_affine<LEVELS, SIGNED, ALIF, true>(A, gid);
    else seg_affine<LEVELS, SIGNED, ALIF, false>(A, gid);
}

__device__ __forceinline__ float apply_aff(const LifSegArgs &A, int sg, int f, int ch, float Gn, float cv, float ca) {
    const float *w = ws_at(A, sg, 4 * f, ch);
    const size_t st = (size_t)A.p.B * A.p.D;
    return fmaf(w[3 * st], ca, fmaf(w[2 * st], cv, fmaf(w[st], Gn, w[0])));
}

template <bool ALIF>
__global__ __launch_bounds__(256) void lif_seg_carry_kernel(LifSegArgs A) {
    const LifBwdArgs &p = A.p;
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= p.B * p.D) return;
    const int c = gid % p.D;
    const float gain = p.ps[3 * p.D + c];
    float Gn = 0.0f, cv = p.gv ? p.gv[gid] : 0.0f, ca = (ALIF && p.ga) ? p.ga[gid] : 0.0f;
    float gb = 0.0f, gg = 0.0f, gr = 0.0f;
    for (int sg = A.nseg - 1; sg >= 0; sg--) {
        *ws_at(A, sg, 24, gid) = Gn;
        *ws_at(A, sg, 25, gid) = cv;
        *ws_at(A, sg, 26, gid) = ca;
        gb += apply_aff(A, sg, 3, gid, Gn, cv, ca);
        if (ALIF) {
            gg += apply_aff(A, sg, 4, gid, Gn, cv, ca);
            gr += apply_aff(A, sg, 5, gid, Gn, cv, ca);
        }
        const float nG = apply_aff(A, sg, 0, gid, Gn, cv, ca), ncv = apply_aff(A, sg, 1, gid, Gn, cv, ca);
        const float nca = ALIF ? apply_aff(A, sg, 2, gid, Gn, cv, ca) : 0.0f;
        Gn = nG;
        cv = ncv;
        ca = nca;
    }
    if (ALIF && p.rg) {  // the first step's reset used the initial threshold theta + a0 gain
        const float g0 = -p.s0[gid] * Gn;
        gg += g0 * p.a0[gid];
        ca += g0 * gain;
    }
    p.dv0[gid] = cv;
    if (p.da0) p.da0[gid] = ALIF ? ca : 0.0f;
    p.dbeta[gid] = gb;
    if (p.drho) p.drho[gid] = ALIF ? gr : 0.0f;
    if (p.dgain) p.dgain[gid] = ALIF ? gg : 0.0f;
}

template <int LEVELS, bool SIGNED, bool ALIF, bool FIN>
__device__ __forceinline__ void seg_walk(const LifSegArgs &A, int gid) {
    const LifBwdArgs &p = A.p;
    const int chains = p.B * p.D;
    const int sg = gid / chains, ch = gid - sg * chains;
    const int D = p.D, T = p.T, b = ch / D, c = ch - b * D;
    const float bt = p.ps[c], th0 = p.ps[D + c], rho = p.ps[2 * D + c], gain = p.ps[3 * D + c], omr = 1.0f - rho;
    const int t0 = sg * SK, n = min(SK, T - t0);
    const float *x = p.cur + (size_t)b * T * D + c, *g = p.gs + (size_t)b * T * D + c;
    float *o = p.dI + (size_t)b * T * D + c;
    const float pv = *park_at(A, sg, 0, ch), ps_ = *park_at(A, sg, 1, ch), pa = *park_at(A, sg, 2, ch);
    float Gn = *ws_at(A, sg, 24, ch), cv = *ws_at(A, sg, 25, ch), ca = *ws_at(A, sg, 26, ch);
    float vs[SK] = {}, as[SK] = {};
    const float top = seg_replay<LEVELS, SIGNED, ALIF, FIN>(x, D, t0, n, bt, th0, rho, omr, gain, pv, ps_, pa, vs, as);
    auto back = [&](auto near) {
        constexpr bool NEAR = decltype(near)::value;
#pragma unroll
        for (int i = SK - 1; i >= 0; i--) {
            if (i < n) {
                const float vt = vs[i], at = ALIF ? as[i] : 0.0f;
                const float tht = ALIF ? th0 + at * gain : th0;
                float dv, dth;
                dspike<LEVELS, SIGNED, NEAR>(vt, tht, p.slope, dv, dth);
                float gst = g[(size_t)(t0 + i) * D];
                if (p.rg) {
                    const float qq = tht * dv, cap = 2.0f * bt;
                    gst -= (qq > cap ? cap / dv : tht) * Gn;
                }
                const float G = gst * dv + cv;
                if (ALIF) {
                    float gth = gst * dth;
                    if (p.rg) gth -= spike<LEVELS, SIGNED, FIN>(vt, tht) * Gn;
                    ca = rho * (gth * gain + ca);
                }
                o[(size_t)(t0 + i) * D] = G;
                Gn = G;
                cv = bt * G;
            }
        }
    };
    if (FIN && __all(top < NEAR_V)) back(std::integral_constant<bool, true>{});
    else back(std::integral_constant<bool, false>{});
}

template <int LEVELS, bool SIGNED, bool ALIF>
__global__ __launch_bounds__(256) void lif_seg_walk_kernel(LifSegArgs A) {
    const LifBwdArgs &p = A.p;
    const int chains = p.B * p.D, gid = blockIdx.x * blockDim.x + threadIdx.x;  // chain fastest
    const bool in = gid < chains * A.nseg;
    const int ch = in ? gid % chains : 0;
    const bool fin = wave_tame<ALIF>(p, ch % p.D, ch);
    if (!in) return;
    if (fin) seg_walk<LEVELS, SIGNED, ALIF, true>(A, gid);
    else seg_walk<LEVELS, SIGNED, ALIF, false>(A, gid);
}

template <int LEVELS, bool SIGNED, bool ALIF>
int launch_seg(const LifSegArgs &A, bool parked, hipStream_t st) {
    const long chains = (long)A.p.B * A.p.D, lanes = chains * A.nseg;
    if (!parked) lif_seg_park_kernel<LEVELS, SIGNED, ALIF><<<ava::ceil_div(chains, 256), 256, 0, st>>>(A);
    lif_seg_affine_kernel<LEVELS, SIGNED, ALIF><<<ava::ceil_div(lanes, 256), 256, 0, st>>>(A);
    lif_seg_carry_kernel<ALIF><<<ava::ceil_div(chains, 256), 256, 0, st>>>(A);
    lif_seg_walk_kernel<LEVELS, SIGNED, ALIF><<<ava::ceil_div(lanes, 256), 256, 0, st>>>(A);
    AVA_LAUNCHED("lif_scan_bwd segments");
    return AVA_OK;
}

}  // namespace

// The LIF scan's backward. Outputs per (b, c): dI [B][T][D], dv0, da0 and this stream's shares of
// dbeta, drho, dgain ([B][D] each; the parameter gradients are their sums over b).
extern "C" int ava_lif_scan_bwd(const float *cur, int B, int T, int D, const float *ps, const float *v0,
                                const float *s0, const float *a0, int levels, int is_signed, int alif, float slope,
                                int reset_grad, const float *g_spk, const float *g_vT, const float *g_aT, float *dI,
                                float *dv0, float *da0, float *dbeta, float *drho, float *dgain, ava_stream stream) {
    AVA_REQUIRE(cur && ps && v0 && s0 && g_spk && dI && dv0 && dbeta, AVA_ERR_ARG, "lif_scan_bwd: NULL buffer");
    AVA_REQUIRE(!alif || (a0 && da0 && drho && dgain), AVA_ERR_ARG, "lif_scan_bwd: ALIF needs a0, da0, drho, dgain");
    AVA_REQUIRE(B > 0 && T > 0 && D > 0 && (long)B * D <= (1L << 30), AVA_ERR_SHAPE, "lif_scan_bwd: B=%d T=%d D=%d",
                B, T, D);
    AVA_REQUIRE(levels == 1 || levels == 2, AVA_ERR_ARG, "lif_scan_bwd: levels %d (1 or 2)", levels);
    AVA_REQUIRE(slope >= 0.0f, AVA_ERR_ARG, "lif_scan_bwd: slope %g (the reset gradient is reset_grad)", slope);
    LifBwdArgs p{cur, ps, v0, s0, a0, g_spk, g_vT, alif ? g_aT : nullptr, dI, dv0, da0, dbeta, drho, dgain,
                 B, T, D, slope, reset_grad ? 1 : 0};
    const hipStream_t st = (hipStream_t)stream;
    dim3 grid(ava::ceil_div((long)B * D, 256)), block(256);
    // One level's spikes cost little to form again, and keeping them takes 140 registers where 123 let a fourth wave share
    // a SIMD: kept while three waves a SIMD hold all chains (unsigned, us kept / not: 32 x 1024 x 2048 308 / 325, 64 x 512 x 2048
    // 216 / 219, 256 x 128 x 1024 114 / 101, 256 x 256 x 1024 225 / 211). Two levels' are always kept.
    int cus = 0;
    if (int r = ava::device_cus(&cus)) return r;
    const bool keep = (long)B * D <= 3L * 256 * cus;
#define AVA_LB(L, S, A, K) lif_bwd_kernel<SEG, L, S, A, K><<<grid, block, 0, st>>>(p)
    if (!is_signed) {
        if (!alif) AVA_LB(1, false, false, false);
        else if (keep) AVA_LB(1, false, true, true);
        else AVA_LB(1, false, true, false);
    } else if (levels == 1) {
        if (!alif) AVA_LB(1, true, false, false);
        else if (keep) AVA_LB(1, true, true, true);
        else AVA_LB(1, true, true, false);
    } else {
        if (alif) AVA_LB(2, true, true, true);
        else AVA_LB(2, true, false, true);
    }
#undef AVA_LB
    AVA_LAUNCHED("lif_scan_bwd");
    return AVA_OK;
}

namespace ava {

size_t lif_bwd_seg_floats(int B, int T, int D) {
    return (size_t)((T + SK - 1) / SK) * (SW + 3) * (size_t)B * D;
}

// ava_lif_scan_bwd in parallel segments (the training step's form for few chains): the same outputs
// up to the association of the backward sums; ws holds lif_bwd_seg_floats(B, T, D) floats (the parked
// states at its end unless park, the forward's, is given).
int lif_scan_bwd_seg(const float *cur, int B, int T, int D, const float *ps, const float *v0, const float *s0,
                     const float *a0, int levels, int is_signed, int alif, float slope, int reset_grad,
                     const float *g_spk, const float *g_vT, const float *g_aT, float *dI, float *dv0, float *da0,
                     float *dbeta, float *drho, float *dgain, float *ws, size_t ws_floats, const float *park,
                     hipStream_t st) {
    AVA_REQUIRE(cur && ps && v0 && s0 && g_spk && dI && dv0 && dbeta && ws, AVA_ERR_ARG,
                "lif_scan_bwd_seg: NULL buffer");
    AVA_REQUIRE(!alif || (a0 && da0 && drho && dgain), AVA_ERR_ARG, "lif_scan_bwd_seg: ALIF needs a0, da0, drho, dgain");
    AVA_REQUIRE(B > 0 && T > 0 && D > 0 && (long)B * D * ((T + SK - 1) / SK) <= (1L << 30), AVA_ERR_SHAPE,
                "lif_scan_bwd_seg: B=%d T=%d D=%d", B, T, D);
    AVA_REQUIRE(ws_floats >= lif_bwd_seg_floats(B, T, D), AVA_ERR_SHAPE, "lif_scan_bwd_seg: workspace of %zu floats",
                ws_floats);
    AVA_REQUIRE(levels == 1 || levels == 2, AVA_ERR_ARG, "lif_scan_bwd_seg: levels %d (1 or 2)", levels);
    const int nseg = (T + SK - 1) / SK;
    float *own_park = ws + (size_t)nseg * SW * B * D;
    LifSegArgs A{LifBwdArgs{cur, ps, v0, s0, a0, g_spk, g_vT, alif ? g_aT : nullptr, dI, dv0, da0, dbeta, drho,
                            dgain, B, T, D, slope, reset_grad ? 1 : 0},
                 ws, park ? const_cast<float *>(park) : own_park, nseg};
    const bool parked = park != nullptr;
    if (!is_signed) return alif ? launch_seg<1, false, true>(A, parked, st) : launch_seg<1, false, false>(A, parked, st);
    if (levels == 1) return alif ? launch_seg<1, true, true>(A, parked, st) : launch_seg<1, true, false>(A, parked, st);
    return alif ? launch_seg<2, true, true>(A, parked, st) : launch_seg<2, true, false>(A, parked, st);
}

}  // namespace ava

extern "C" size_t ava_lif_scan_bwd_segments_workspace(int B, int T, int D) {
    return B > 0 && T > 0 && D > 0 ? ava::lif_bwd_seg_floats(B, T, D) * sizeof(float) : 0;
}

extern "C" int ava_lif_scan_bwd_segments(const float *cur, int B, int T, int D, const float *ps, const float *v0,
                                         const float *s0, const float *a0, int levels, int is_signed, int alif,
                                         float slope, int reset_grad, const float *g_spk, const float *g_vT,
                                         const float *g_aT, float *dI, float *dv0, float *da0, float *dbeta,
                                         float *drho, float *dgain, void *ws, size_t ws_bytes, ava_stream stream) {
    AVA_REQUIRE(slope >= 0.0f, AVA_ERR_ARG, "lif_scan_bwd_segments: slope %g (the reset gradient is reset_grad)",
                slope);
    return ava::lif_scan_bwd_seg(cur, B, T, D, ps, v0, s0, a0, levels, is_signed, alif, slope, reset_grad, g_spk, g_vT,
                                 g_aT, dI, dv0, da0, dbeta, drho, dgain, static_cast<float *>(ws),
                                 ws_bytes / sizeof(float), nullptr, (hipStream_t)stream);
}
