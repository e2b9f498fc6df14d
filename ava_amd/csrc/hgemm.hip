// The training step's f32 products on the f16 matrix cores of gfx950.
//
// C [m][n] = A . B (+ C) for f32 operands, with each operand split into two f16 terms under a power of
// two per row of A and per column of B: x = 2^e (hi + 2^-12 lo + r), hi the f16 nearest x 2^-e and lo the f16
// nearest 2^12 times the rest. The row's largest value is scaled to [2^14, 2^15), lo's factor gives the rest hi's
// range: |r| <= 2^-23 |x 2^-e|, and at most 2^-51 of the row's largest for values some 2^28 below it. Three of the four term
// products are kept, hi hi in one accumulator, hi lo and lo hi in another (lo lo is at most 2^-22 of the product), f32
// accumulation, and the powers of two go back exactly in the epilogue. The sum is rounded once per matrix instruction
// of 16 products, K/16 times instead of K/4. Relative 2-norm against float64, this form / a library f32 product: normal
// operands K = 64 9.8e-8 / 1.4e-7, 1024 1.4e-7 / 5.7e-7, 4096 2.2e-7 / 1.2e-6; rows spread over 40 binades the same;
// log-normal (sigma 1, 2) at K = 1024 1.4e-7 / 5.7e-7, 1.5e-7 / 5.3e-7; a training step's operands (spikes, normed rows, relu^2
// rows, the logits' gradient, token gradients of log-normal size) 0.7-2.9e-7 / 1.3-9.0e-7; one element of a row 1e8 times the others, meeting
// zeros 1.4e-7 / 5.7e-7 (1e9 2.8e-7, 1e10 2.6e-6). Where one product is nearly all of a sum, an f32 product rounds it
// once and this one's operands count: one-hot rows 4.4e-8 / 0, log-normal of sigma 3 8.1e-8 / 1.3e-8.
// Infinities and NaN give what they give in an f32 product (a value more than 2^39 below its row's largest counts as zero to
// an infinity it meets).
// Measured: 8192 x 1024 x 1024 49 us (352 TFLOP/s of f32 products, 1.05 PFLOP/s of f16) against 148 us in
// rocBLAS, 8192 x 8192 x 1024 361 / 1000, 1024 x 4096 x 8192 171 / 460; a large bf16 library product runs at
// 1.2 PFLOP/s on the same card, so the matrix cores bound it. The splits move 12 bytes an element.
//
// The operands are laid out K-contiguous by the split passes (split_rows for an operand whose K runs along
// its rows, split_cols for one whose K runs down its columns): per row of A (column of B), blocks of 32 k
// values, 64 bytes of hi then 64 bytes of lo, so a stage row is one 128-byte line.
#include <algorithm>

#include "common.h"
#include "hgemm.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ the operands' split

// |x|, or 0 where x is not finite: an infinity or NaN passes through the split under any scale, and the row's finite
// values keep theirs.
__device__ __forceinline__ float finite_abs(float x) { return fabsf(x) < INFINITY ? fabsf(x) : 0.0f; }

// The exponent of a row whose largest finite magnitude is amax: x 2^-e < 2^15 (0 for a row of zeros).
__device__ __forceinline__ int split_exp(float amax) {
    if (!(amax > 0.0f)) return 0;
    int ex;
    (void)frexpf(amax, &ex);
    return ex - 15;
}

constexpr float LO_SCALE = 4096.0f;  // |x 2^-e - hi| <= 2^-11 of a value below 2^15: lo stays below 2^15 too
__device__ __forceinline__ void split1(float x, int e, _Float16 &hi, _Float16 &lo) {
    const float t = ldexpf(x, -e);
    hi = (_Float16)t;
    lo = (_Float16)((t - (float)hi) * LO_SCALE);
}

// W waves per row of x [rows][cols] (cols <= 256 W NV): its exponent, then its blocks of 32. A lane holds
// NV groups of 4 consecutive values (16-byte loads when V4), so the row is read once (8192 x 8192: 96 us; one
// wave a row, reading it twice: 151 us); longer rows (NV = 0) are read again from the caches.
template <bool V4, int W, int NV>
__global__ __launch_bounds__(256) void split_rows_kernel(const float *__restrict__ x, int rows, int cols, int ld,
                                                         int ldk, _Float16 *__restrict__ out, int *__restrict__ exps) {
    __shared__ float smax[4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & (64 * W - 1);
    const int row = W == 1 ? blockIdx.x * 4 + wave : blockIdx.x;
    if (W == 1 && row >= rows) return;
    const float *xr = x + (size_t)row * ld;
    auto at = [&](int j) {
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        if (V4) {
            if (j < cols) v = *reinterpret_cast<const f32x4 *>(xr + j);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (j + i < cols) v[i] = xr[j + i];
        }
        return v;
    };
    float amax = 0.0f;
    f32x4 held[NV ? NV : 1];
    auto top = [&](const f32x4 &v) {
#pragma unroll
        for (int i = 0; i < 4; i++) amax = fmaxf(amax, finite_abs(v[i]));
    };
    if (NV) {
#pragma unroll
        for (int k = 0; k < NV; k++) held[k] = at(lane * 4 + k * 256 * W);
#pragma unroll
        for (int k = 0; k < NV; k++) top(held[k]);
    } else {
        for (int j = lane * 4; j < cols; j += 256 * W) top(at(j));
    }
    amax = ava::wave_max(amax);
    if (W > 1) {
        if ((threadIdx.x & 63) == 0) smax[wave] = amax;
        __syncthreads();
        amax = fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3]));
    }
    const int e = split_exp(amax);
    if (lane == 0) exps[row] = e;
    _Float16 *o = out + (size_t)row * ldk * 2;
    auto put = [&](int j, const f32x4 &v) {
        f16x4 hi, lo;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            _Float16 h, l;
            split1(v[i], e, h, l);
            hi[i] = h;
            lo[i] = l;
        }
        _Float16 *p = o + (j >> 5) * 64 + (j & 31);
        *reinterpret_cast<f16x4 *>(p) = hi;
        *reinterpret_cast<f16x4 *>(p + 32) = lo;
    };
    if (NV) {
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (lane * 4 + k * 256 * W < ldk) put(lane * 4 + k * 256 * W, held[k]);
    } else {
        for (int j = lane * 4; j < ldk; j += 256 * W) put(j, at(j));
    }
}

// The columns' largest magnitudes over SPLIT_ROWS rows at a time: part [row block][cols].
constexpr int SPLIT_ROWS = 128;
__global__ __launch_bounds__(256) void col_max_kernel(const float *__restrict__ x, int rows, int cols, int ld,
                                                      float *__restrict__ part) {
    __shared__ float s[4][64];
    const int c = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6, r0 = blockIdx.y * SPLIT_ROWS;
    float m = 0.0f;
    if (c < cols) {
        const int r1 = min(rows, r0 + SPLIT_ROWS);
#pragma unroll 8
        for (int r = r0 + w; r < r1; r += 4) m = fmaxf(m, finite_abs(x[(size_t)r * ld + c]));
    }
    s[w][threadIdx.x & 63] = m;
    __syncthreads();
    if (w == 0 && c < cols)
        part[(size_t)blockIdx.y * cols + c] = fmaxf(fmaxf(s[0][threadIdx.x], s[1][threadIdx.x]),
                                                    fmaxf(s[2][threadIdx.x], s[3][threadIdx.x]));
}

// A 64 x 64 tile of x transposed through LDS: row c of the output holds column c of x.
// Bound by HBM (12 bytes an element with the maxima's pass) once its loads overlap: the partial maxima, up to 64 a column,
// were a chain of L2 latencies ahead of the tile's loads (a training step's splits 15.8 us on average, 10.3 now; one d = 1024
// block at B = 4, T = 2048 9.67 -> 9.35 ms a step).
__global__ __launch_bounds__(256) void split_cols_kernel(const float *__restrict__ x, int rows, int cols, int ld,
                                                         int ldk, const float *__restrict__ part, int nparts,
                                                         _Float16 *__restrict__ out, int *__restrict__ exps) {
    __shared__ float tile[64][65];
    __shared__ float smax[4][64];
    __shared__ int se[64];
    const int c0 = blockIdx.x * 64, r0 = blockIdx.y * 64, tx = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c = c0 + tx;
    // the tile's values are in flight while the partial maxima come, eight at a time
    float t[16], m = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) t[i] = (c < cols && r0 + w + 4 * i < rows) ? x[(size_t)(r0 + w + 4 * i) * ld + c] : 0.0f;
    AVA_ISSUE_FENCE();
    if (c < cols) {
#pragma unroll 8
        for (int k = w; k < nparts; k += 4) m = fmaxf(m, part[(size_t)k * cols + c]);
    }
    smax[w][tx] = m;
#pragma unroll
    for (int i = 0; i < 16; i++) tile[w + 4 * i][tx] = t[i];
    __syncthreads();
    if (w == 0) {
        const int e = split_exp(fmaxf(fmaxf(smax[0][tx], smax[1][tx]), fmaxf(smax[2][tx], smax[3][tx])));
        se[tx] = e;
        if (blockIdx.y == 0 && c < cols) exps[c] = e;
    }
    __syncthreads();
    // 16 lanes per output row, 4 values each; 16 rows per pass
    const int q = (threadIdx.x & 15) * 4;
    for (int cc = threadIdx.x >> 4; cc < 64; cc += 16) {
        if (c0 + cc >= cols || r0 + q >= ldk) continue;
        const int e = se[cc];
        f16x4 hi, lo;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            _Float16 h, l;
            split1(tile[q + i][cc], e, h, l);
            hi[i] = h;
            lo[i] = l;
        }
        const int j = r0 + q;
        _Float16 *p = out + (size_t)(c0 + cc) * ldk * 2 + (j >> 5) * 64 + (j & 31);
        *reinterpret_cast<f16x4 *>(p) = hi;
        *reinterpret_cast<f16x4 *>(p + 32) = lo;
    }
}

// ------------------------------------------------------------------ the product

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xC07F); }  // lgkmcnt(0) only

#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t BufResH;
__device__ __forceinline__ BufResH buf_res_h(const _Float16 *base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)bytes, 0x00020000);
}
#else
typedef const _Float16 *BufResH;
__device__ inline BufResH buf_res_h(const _Float16 *base, unsigned) { return base; }
#endif

__device__ __forceinline__ void dma16_h(BufResH r, unsigned voff, unsigned soff, void *l) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)l, 16, (int)voff,
                                             (int)soff, 0, 0);
#endif
}

// 128 x 256 output tiles, 8 waves of 64 x 64 (2 x 2 blocks of v_mfma_f32_32x32x16_f16, main and cross
// accumulators), K in steps of 32 (one 128-byte row of hi and lo per operand row) through three LDS
// stages of 48 KB filled by direct-to-LDS buffer loads. In step k the fragments of its second half are
// read while its first half is multiplied; then, once the wave's loads of step k + 1 have landed, one
// barrier makes every wave's visible and frees stage k, and the loads of step k + 3 and the fragment
// reads of step k + 1's first half go out under the second half's MFMAs: no LDS or memory latency stands
// between MFMAs except at a tile's start. Workgroup -> (split, tile): the splits of K (few tiles: dW
// products) write partial sums that hgemm_sum_kernel adds in order.
constexpr int HM = 128, HN = 256, HSTAGE = (HM + HN) * 128, HLOADS = (HM + HN) / 64;  // a load: 8 rows a wave

// LDS position of 16-byte chunk c of a 128-byte row r (as the int8 product: no bank conflicts)
__device__ __forceinline__ int hswz(int r, int c) { return c ^ ((r >> 1) & 7); }

struct HgemmArgs {
    const _Float16 *a, *b;
    const int *ea, *eb;
    int m, n, ldk, steps, splits;  // K steps in all; the splits of them
    float *c;
    int ldc, add;
    float *part;  // splits > 1: [splits][m][n]
};

template <int LEFT>
__device__ __forceinline__ void half_schedule() {
    // 8 fragment reads of the next half and up to 6 loads between 12 MFMAs
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
    if constexpr (LEFT > 0) __builtin_amdgcn_sched_group_barrier(0x020, LEFT / 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    if constexpr (LEFT > 0) __builtin_amdgcn_sched_group_barrier(0x020, LEFT - LEFT / 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
}

__global__ __launch_bounds__(512, 1) void hgemm_kernel(HgemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) char hsm[];
    const int tiles_n = (p.n + HN - 1) / HN, tiles_m = (p.m + HM - 1) / HM, tiles = tiles_m * tiles_n;
    const int total = tiles * p.splits;
    // XCD x (workgroups x mod 8) takes the x-th eighth of the items; rows fastest in groups of 8
    int t = blockIdx.x;
    if (total % 8 == 0) t = (t & 7) * (total >> 3) + (t >> 3);
    const int sp = t / tiles;
    t -= sp * tiles;
    const int span = 8 * tiles_n, g = t / span, rem = t - g * span, rows = min(8, tiles_m - g * 8);
    const int m0 = (g * 8 + rem % rows) * HM, n0 = (rem / rows) * HN;
    const int k0 = (int)((long long)p.steps * sp / p.splits), k1 = (int)((long long)p.steps * (sp + 1) / p.splits);

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const unsigned ldb = (unsigned)p.ldk * 4u;  // bytes per operand row
    const BufResH ra = buf_res_h(p.a + (size_t)m0 * p.ldk * 2, (unsigned)min(HM, p.m - m0) * ldb);
    const BufResH rb = buf_res_h(p.b + (size_t)n0 * p.ldk * 2, (unsigned)min(HN, p.n - n0) * ldb);
    unsigned voff[HLOADS];
#pragma unroll
    for (int i = 0; i < HLOADS; i++) {
        const int r = (i * 8 + wave) * 8 + (lane >> 3), rr = i < HM / 64 ? r : r - HM;
        voff[i] = (unsigned)rr * ldb + (unsigned)hswz(rr, lane & 7) * 16u;
    }
    auto issue = [&](int i, int k, int stage) {
        dma16_h(i < HM / 64 ? ra : rb, voff[i], (unsigned)k * 128u, hsm + stage * HSTAGE + (i * 8 + wave) * 1024);
    };
    const int fr = lane & 31, fc = lane >> 5;
    struct Frags {
        f16x8 ah[2], al[2], bh[2], bl[2];
    };
    auto frag = [&](int row, int c, const char *base) {
        return *reinterpret_cast<const f16x8 *>(base + row * 128 + hswz(row, c) * 16);
    };
    auto read = [&](Frags &f, int stage, int ks) {
        const char *la = hsm + stage * HSTAGE, *lb = la + HM * 128;
        const int c = ks * 2 + fc;
#pragma unroll
        for (int i = 0; i < 2; i++) f.ah[i] = frag(wm * 64 + i * 32 + fr, c, la);
#pragma unroll
        for (int j = 0; j < 2; j++) f.bh[j] = frag(wn * 64 + j * 32 + fr, c, lb);
#pragma unroll
        for (int j = 0; j < 2; j++) f.bl[j] = frag(wn * 64 + j * 32 + fr, c + 4, lb);
#pragma unroll
        for (int i = 0; i < 2; i++) f.al[i] = frag(wm * 64 + i * 32 + fr, c + 4, la);
    };
    f32x16 acc[2][2], crs[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = crs[i][j] = f32x16{};
    auto mul = [&](const Frags &f) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bh[j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) crs[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bl[j], crs[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) crs[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.al[i], f.bh[j], crs[i][j], 0, 0, 0);
    };

    // loads past the last step read the last step's lines again (in bounds, unused)
#pragma unroll
    for (int s = 0; s < 3; s++)
#pragma unroll
        for (int i = 0; i < HLOADS; i++) issue(i, min(k0 + s, k1 - 1), s);
    wait_vm<2 * HLOADS>();
    AVA_ISSUE_FENCE();
    __builtin_amdgcn_s_barrier();
    AVA_ISSUE_FENCE();
    Frags f0, f1;
    read(f0, 0, 0);
    int stage = 0;
    for (int k = k0; k < k1; k++) {
        const int next = stage == 2 ? 0 : stage + 1;
        read(f1, stage, 1);
        mul(f0);
        half_schedule<0>();
        __builtin_amdgcn_sched_barrier(0);  // the waits come after the first half's MFMAs
        wait_lgkm0();         // this wave has read all of stage k
        wait_vm<HLOADS>();    // its loads of step k + 1 have landed (those of k + 2 may be in flight)
        AVA_ISSUE_FENCE();
        __builtin_amdgcn_s_barrier();
        AVA_ISSUE_FENCE();
        read(f0, next, 0);
#pragma unroll
        for (int i = 0; i < HLOADS; i++) issue(i, min(k + 3, k1 - 1), stage);
        mul(f1);
        half_schedule<HLOADS>();
        stage = next;
    }
    wait_vm<0>();  // no load into LDS outlives the workgroup

    // block (i, j): register r is row 32 i + 8 (r >> 2) + 4 (lane >> 5) + (r & 3), column 32 j + (lane & 31).
    // Every access goes through a resource over the tile's existing rows (the range check drops the rows past
    // m; a lane's column past n takes an offset past the range), so the tail needs no branch. The wave's 64 row
    // exponents sit in one register, lane l row l's; block row i's reach one register by a bpermute (lane 16 q +
    // z: row 32 i + 8 (z >> 2) + (z & 3) + 4 (q >> 1)) and each output register's by a DPP row broadcast.
    const bool part = p.splits > 1, add = !part && p.add;
    const unsigned ldo4 = (unsigned)(part ? p.n : p.ldc) * 4u;
    float *out = (part ? p.part + (size_t)sp * p.m * p.n : p.c) + (size_t)m0 * (ldo4 / 4);
    const BufRes rc = buf_res(out, (unsigned)min(HM, p.m - m0) * ldo4);
    const int z = lane & 15, q = lane >> 4;
    unsigned voc[2];
    int eb[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int col = n0 + wn * 64 + j * 32 + fr;
        voc[j] = col < p.n ? (unsigned)(wm * 64 + fc * 4) * ldo4 + (unsigned)col * 4u : 0x80000000u;
        eb[j] = p.eb[min(col, p.n - 1)];
    }
    const int ex = p.ea[min(m0 + wm * 64 + lane, p.m - 1)];
    auto row_exp = [&](int e, int r) {
        switch (r) {
#define AVA_BC(R) \
    case R: return __builtin_amdgcn_mov_dpp(e, 0x150 + R, 0xf, 0xf, true);
            AVA_BC(0) AVA_BC(1) AVA_BC(2) AVA_BC(3) AVA_BC(4) AVA_BC(5) AVA_BC(6) AVA_BC(7)
            AVA_BC(8) AVA_BC(9) AVA_BC(10) AVA_BC(11) AVA_BC(12) AVA_BC(13) AVA_BC(14)
#undef AVA_BC
            default: return __builtin_amdgcn_mov_dpp(e, 0x150 + 15, 0xf, 0xf, true);
        }
    };
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int er = __builtin_amdgcn_ds_bpermute((32 * i + 8 * (z >> 2) + (z & 3) + 4 * (q >> 1)) << 2, ex);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            float old[16];
            auto soff = [&](int r) { return (unsigned)(i * 32 + (r >> 2) * 8 + (r & 3)) * ldo4; };
            // (the range check sees the lane's offset only: the row's goes into it)
            if (add) {
#pragma unroll
                for (int r = 0; r < 16; r++) old[r] = load_f32(rc, voc[j] + soff(r), 0);
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                // (an infinity is in the main sum; its rest, inf - inf, made the cross sum NaN)
                const float s = acc[i][j][r], x = fmaf(crs[i][j][r], 1.0f / LO_SCALE, s);
                float v = ldexpf(fabsf(s) < INFINITY ? x : s, row_exp(er, r) + eb[j]);
                if (add) v = old[r] + v;
                store_f32(rc, voc[j] + soff(r), 0, v);
            }
        }
    }
}

// C (+)= the splits' partial sums, added in order; V floats a thread.
template <int V>
__global__ __launch_bounds__(256) void hgemm_sum_kernel(const float *__restrict__ part, int splits, int m, int n,
                                                        float *__restrict__ c, int ldc, int add) {
    typedef float fv __attribute__((ext_vector_type(V)));
    const size_t mn = (size_t)m * n / V;
    const fv *pv = reinterpret_cast<const fv *>(part);
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < mn; i += (size_t)gridDim.x * 256) {
        fv v = pv[i];
        for (int s = 1; s < splits; s++) v += pv[(size_t)s * mn + i];
        const unsigned e = (unsigned)i * V, r = e / (unsigned)n;
        fv *o = reinterpret_cast<fv *>(c + (size_t)r * ldc + (e - r * (unsigned)n));
        *o = add ? *o + v : v;
    }
}

}  // namespace

namespace ava {

// Few tiles: K in up to 16 parts of at least 8 steps, as many as fill the 256 CUs.
constexpr int SPLIT_ITEMS = 256;
int hgemm_splits(int m, int n, int k) {
    const int tiles = ceil_div(m, HM) * ceil_div(n, HN), steps = hgemm_ldk(k) / 32;
    return std::max(1, std::min({SPLIT_ITEMS / tiles, steps / 8, 16}));
}
size_t hgemm_part_max() { return (size_t)SPLIT_ITEMS * HM * HN; }

int hgemm_split_rows(const float *x, int rows, int cols, int ld, void *planes, int *exps, hipStream_t st) {
    const int ldk = hgemm_ldk(cols);
    auto go = [&](auto one, auto four, auto eight, auto any) {
        if (ldk <= 1024) one<<<ceil_div(rows, 4), 256, 0, st>>>(x, rows, cols, ld, ldk, (_Float16 *)planes, exps);
        else if (ldk <= 4096) four<<<rows, 256, 0, st>>>(x, rows, cols, ld, ldk, (_Float16 *)planes, exps);
        else if (ldk <= 8192) eight<<<rows, 256, 0, st>>>(x, rows, cols, ld, ldk, (_Float16 *)planes, exps);
        else any<<<rows, 256, 0, st>>>(x, rows, cols, ld, ldk, (_Float16 *)planes, exps);
    };
    if (cols % 4 == 0 && ld % 4 == 0 && (uintptr_t)x % 16 == 0)
        go(split_rows_kernel<true, 1, 4>, split_rows_kernel<true, 4, 4>, split_rows_kernel<true, 4, 8>,
           split_rows_kernel<true, 4, 0>);
    else
        go(split_rows_kernel<false, 1, 4>, split_rows_kernel<false, 4, 4>, split_rows_kernel<false, 4, 8>,
           split_rows_kernel<false, 4, 0>);
    AVA_LAUNCHED("split_rows");
    return AVA_OK;
}

size_t hgemm_part_floats(int rows, int cols) { return (size_t)ceil_div(rows, SPLIT_ROWS) * cols; }

int hgemm_split_cols(const float *x, int rows, int cols, int ld, void *planes, int *exps, float *part, hipStream_t st) {
    const int ldk = hgemm_ldk(rows), np = ceil_div(rows, SPLIT_ROWS);
    col_max_kernel<<<dim3(ceil_div(cols, 64), np), 256, 0, st>>>(x, rows, cols, ld, part);
    split_cols_kernel<<<dim3(ceil_div(cols, 64), ceil_div(ldk, 64)), 256, 0, st>>>(x, rows, cols, ld, ldk, part, np,
                                                                                 (_Float16 *)planes, exps);
    AVA_LAUNCHED("split_cols");
    return AVA_OK;
}

int hgemm(const HgemmOp &a, const HgemmOp &b, int m, int n, int k, float *c, int ldc, bool add, float *part,
          size_t part_floats, hipStream_t st) {
    const int splits = hgemm_splits(m, n, k);
    AVA_REQUIRE(splits == 1 || part_floats >= (size_t)splits * m * n, AVA_ERR_SHAPE,
                "hgemm: %zu floats of scratch, %d splits of %d x %d", part_floats, splits, m, n);
    const HgemmArgs p{(const _Float16 *)a.planes, (const _Float16 *)b.planes, a.exps, b.exps, m, n, hgemm_ldk(k),
                      hgemm_ldk(k) / 32, splits, c, ldc, add ? 1 : 0, part};
    if (int r = lds_opt_in((const void *)hgemm_kernel, 3 * HSTAGE)) return r;
    hgemm_kernel<<<ceil_div(m, HM) * ceil_div(n, HN) * splits, 512, 3 * HSTAGE, st>>>(p);
    AVA_LAUNCHED("hgemm");
    if (splits > 1) {
        const bool v4 = n % 4 == 0 && ldc % 4 == 0 && (uintptr_t)c % 16 == 0 && (uintptr_t)part % 16 == 0;
        if (v4)
            hgemm_sum_kernel<4><<<std::min(2048, ceil_div((long)m * n, 1024)), 256, 0, st>>>(part, splits, m, n, c, ldc, p.add);
        else
            hgemm_sum_kernel<1><<<std::min(2048, ceil_div((long)m * n, 256)), 256, 0, st>>>(part, splits, m, n, c, ldc, p.add);
        AVA_LAUNCHED("hgemm_sum");
    }
    return AVA_OK;
}

}  // namespace ava
