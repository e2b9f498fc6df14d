"""The backward kernels (ava_lif_scan_bwd, ava_kwta_relu2_bwd, ava_mem_scan_bwd, ava_dense_back)
against the oracle's backward (itself pinned by autograd in test_oracle_backward.py), through the
C ABI on the GPU.

Bars: the LIF backward replays the forward with the same rounding and walks back in the oracle's
order, every operation rounded alone on both sides, so it is bit-exact; so are relu²'s backward and
the dense mix's sums over blocks. The dense weights' gradients (f32 partial sums against float64) and
the memory backward (f32 on the GPU, float64 in the oracle) meet 1e-5 relative (of each output's
largest magnitude), 1e-4 over 2048 steps.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def rel(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


def lif_inputs(seed, B, T, D, levels, signed):
    rng = np.random.default_rng(seed)
    cur = (rng.normal(size=(B, T, D)) * 1.2).astype(np.float32)
    ps = np.concatenate([rng.uniform(0.15, 0.95, D), rng.uniform(0.6, 1.4, D), rng.uniform(0.8, 0.99, D),
                         rng.uniform(0.02, 0.5, D)]).astype(np.float32)
    v0 = rng.normal(size=(B, D)).astype(np.float32)
    hi = 1 if (levels == 1 or not signed) else 2
    s0 = rng.integers(0 if not signed else -hi, hi + 1, (B, D)).astype(np.float32)
    a0 = rng.uniform(0, 1, (B, D)).astype(np.float32)
    g = rng.normal(size=(B, T, D)).astype(np.float32)
    gv = rng.normal(size=(B, D)).astype(np.float32)
    ga = rng.normal(size=(B, D)).astype(np.float32)
    return cur, ps, v0, s0, a0, g, gv, ga


def run_lif(cur, ps, v0, s0, a0, g, gv, ga, levels, signed, alif, slope, rg):
    from ava_amd import ops
    st = ops.LifState(dev(v0), dev(s0), dev(a0))
    return {k: host(v) for k, v in ops.lif_gen_bwd(dev(cur), dev(ps), dev(g), init=st, g_vT=dev(gv),
                                                    g_aT=dev(ga) if alif else None, levels=levels, signed=signed,
                                                    alif=alif, slope=slope, reset_grad=rg).items()}


@pytest.mark.parametrize("T", [1, 5, 16, 77])
@pytest.mark.parametrize("levels,signed", [(2, True), (1, True), (1, False)])
@pytest.mark.parametrize("alif", [True, False])
@pytest.mark.parametrize("rg", [False, True])
@pytest.mark.parametrize("D", [40, 64])
def test_lif_bwd(T, levels, signed, alif, rg, D):
    """Segment edges: T below, at and above the 16-step segment (77 = a short first segment + 4), on a
    ragged last wave (D=40) and on whole waves of one stream (D=64)."""
    slope = 0.5 if rg else 2.0
    x = lif_inputs(T * 7 + levels + 2 * alif + 4 * rg + D, 3, T, D, levels, signed)
    print(f"lif_bwd T={T} D={D} levels={levels} signed={signed} alif={alif} rg={rg}", flush=True)
    o = O.lif_bwd(x[0], x[1], x[5], x[2], x[3], x[4], x[6], x[7] if alif else None, levels=levels, signed=signed,
                  alif=alif, slope=slope, reset_grad=rg)
    gpu = run_lif(*x, levels, signed, alif, slope, rg)
    for k in ("dI", "dv0", "dbeta") + (("da0", "drho", "dgain") if alif else ()):
        assert np.array_equal(gpu[k], o[k]), (k, rel(gpu[k], o[k]))


@pytest.mark.parametrize("rg", [False, True])
def test_lif_bwd_large_values(rg):
    """Membranes past the range of the short reciprocal (1e9) in single segments and lanes, thresholds and traces past
    the counted spikes' (third wave; its theta 1e9, rho above 1), slopes on both sides of 1e6: the oracle's bits from
    the one-lane walk, and the segments' form within its usual rounding."""
    B, T, D = 2, 70, 192
    for slope in (2.0, 3e6):
        x = list(lif_inputs(31 + rg, B, T, D, 2, True))
        x[0][0, 20, 3] = 4e9
        x[0][1, 40, 70:80] = -7e11
        x[1][D + 130] = 1e9  # theta
        x[1][2 * D + 140] = 1.25  # rho
        o = O.lif_bwd(x[0], x[1], x[5], x[2], x[3], x[4], x[6], x[7], levels=2, signed=True, alif=True, slope=slope,
                      reset_grad=rg)
        gpu = run_lif(*x, 2, True, True, slope, rg)
        from ava_amd import ops
        st = ops.LifState(dev(x[2]), dev(x[3]), dev(x[4]))
        seg = ops.lif_gen_bwd(dev(x[0]), dev(x[1]), dev(x[5]), init=st, g_vT=dev(x[6]), g_aT=dev(x[7]), slope=slope,
                              reset_grad=rg, segments=True)
        for k in ("dI", "dv0", "dbeta", "da0", "drho", "dgain"):
            assert np.array_equal(gpu[k], o[k], equal_nan=True), (slope, k, rel(gpu[k], o[k]))
            # per value: the walk's own rounding over 70 steps (a few ulp each), relative to the largest of its chain
            d = np.abs(host(seg[k]) - o[k])
            top = np.max(np.abs(o[k]), axis=1, keepdims=True) if k == "dI" else np.abs(o[k]) + 1e-3 * np.max(np.abs(o[k]))
            assert np.all(d <= 1e-4 * top + 1e-30), (slope, k, float(np.max(d / (top + 1e-30))))


@pytest.mark.parametrize("levels,signed", [(1, True), (1, False), (2, True)])
def test_lif_bwd_many_chains(levels, signed):
    """More chains than three waves a SIMD hold (256 x 1024 on 256 CUs): one level's spikes are formed again on the way
    back instead of kept. The oracle's bits, with the reset gradient (which reads them)."""
    B, T, D = 256, 19, 1024
    x = lif_inputs(61 + levels, B, T, D, levels, signed)
    print(f"lif_bwd many chains levels={levels} signed={signed}", flush=True)
    o = O.lif_bwd(x[0], x[1], x[5], x[2], x[3], x[4], x[6], x[7], levels=levels, signed=signed, alif=True, slope=2.0,
                  reset_grad=True)
    gpu = run_lif(*x, levels, signed, True, 2.0, True)
    for k in ("dI", "dv0", "da0", "dbeta", "drho", "dgain"):
        assert np.array_equal(gpu[k], o[k]), (k, rel(gpu[k], o[k]))


def test_lif_bwd_long():
    """config[1]'s sequence length and width (T 2048, D 2048) on 8 streams, int2 with ALIF and the
    reset gradient."""
    B, T, D = 8, 2048, 2048
    x = lif_inputs(5, B, T, D, 2, True)
    print(f"lif_bwd long B={B} T={T} D={D}", flush=True)
    o = O.lif_bwd(x[0], x[1], x[5], x[2], x[3], x[4], x[6], x[7], levels=2, signed=True, alif=True, slope=0.5,
                  reset_grad=True)
    gpu = run_lif(*x, 2, True, True, 0.5, True)
    for k in ("dI", "dv0", "da0", "dbeta", "drho", "dgain"):
        e = rel(gpu[k], o[k])
        print(f"  {k}: rel {e:.2e}, bit-identical {np.mean(gpu[k] == o[k]):.4f}", flush=True)
        assert np.array_equal(gpu[k], o[k]), (k, e)


def run_lif_seg(cur, ps, v0, s0, a0, g, gv, ga, levels, signed, alif, slope, rg):
    from ava_amd import ops
    st = ops.LifState(dev(v0), dev(s0), dev(a0))
    return {k: host(v) for k, v in ops.lif_gen_bwd(dev(cur), dev(ps), dev(g), init=st, g_vT=dev(gv),
                                                    g_aT=dev(ga) if alif else None, levels=levels, signed=signed,
                                                    alif=alif, slope=slope, reset_grad=rg, segments=True).items()}


@pytest.mark.parametrize("T", [1, 33, 200])
@pytest.mark.parametrize("levels,signed", [(2, True), (1, True), (1, False)])
@pytest.mark.parametrize("alif", [True, False])
@pytest.mark.parametrize("rg", [False, True])
@pytest.mark.parametrize("D", [40, 64])
def test_lif_bwd_segments(T, levels, signed, alif, rg, D):
    """ava_lif_scan_bwd_segments against the oracle's walk (which the one-lane kernel equals bit for bit):
    one step, a 32-step segment and a 1-step one, seven segments the last of them short. The segments'
    affine functions associate the backward sums differently: within 2e-6 of each output's largest
    value here. D=40 parks the states from the general scan, D=64 from the buffer-resource one."""
    slope = 0.5 if rg else 2.0
    x = lif_inputs(T * 11 + levels + 2 * alif + 4 * rg + D, 3, T, D, levels, signed)
    print(f"lif_bwd segments T={T} D={D} levels={levels} signed={signed} alif={alif} rg={rg}", flush=True)
    o = O.lif_bwd(x[0], x[1], x[5], x[2], x[3], x[4], x[6], x[7] if alif else None, levels=levels, signed=signed,
                  alif=alif, slope=slope, reset_grad=rg)
    gpu = run_lif_seg(*x, levels, signed, alif, slope, rg)
    for k in ("dI", "dv0", "dbeta") + (("da0", "drho", "dgain") if alif else ()):
        e = rel(gpu[k], o[k])
        assert e < 2e-6, (k, e)


def test_lif_bwd_segments_long():
    """The training step's shape (4 streams x 1024 channels, T 2048: 64 segments per chain), int2 with
    ALIF and the reset gradient, against the oracle's walk."""
    B, T, D = 4, 2048, 1024
    x = lif_inputs(6, B, T, D, 2, True)
    print(f"lif_bwd segments long B={B} T={T} D={D}", flush=True)
    o = O.lif_bwd(x[0], x[1], x[5], x[2], x[3], x[4], x[6], x[7], levels=2, signed=True, alif=True, slope=0.5,
                  reset_grad=True)
    gpu = run_lif_seg(*x, 2, True, True, 0.5, True)
    for k in ("dI", "dv0", "da0", "dbeta", "drho", "dgain"):
        e = rel(gpu[k], o[k])
        print(f"  {k}: rel {e:.2e}", flush=True)
        assert e < 1e-5, (k, e)


@pytest.mark.parametrize("slope", [-0.5, -0.25, 0.0])
def test_lif_bwd_segments_any_slope(slope):
    """The training step's form takes any slope (ava_train_new does not bound it): with a negative one 1 + slope |x| may be 0,
    whose surrogate is an infinity and not NaN. One 32-step segment: the oracle's bits."""
    import ctypes as C
    from ava_amd import _lib
    B, T, D = 2, 32, 64
    f = getattr(_lib.lib(), "_ZN3ava16lif_scan_bwd_segEPKfiiiS1_S1_S1_S1_iiifiS1_S1_S1_PfS2_S2_S2_S2_S2_S2_mS1_P12ihipStream_t")
    cur, ps, v0, s0, a0, g, _, _ = lif_inputs(8, B, T, D, 1, False)
    ps[:D], ps[D:2 * D] = 0.5, 1.0
    v0[:], s0[:] = 0.0, 0.0
    cur[:, :, :8] = 0.0
    cur[:, T - 1, :4] = 3.0  # x = v - theta = 2: 1 + slope |x| = 0 at slope -0.5
    cur[:, T - 1, 4:8] = 5.0  # 4: at slope -0.25
    o = O.lif_bwd(cur, ps, g, v0, s0, a0, levels=1, signed=False, alif=False, slope=slope)
    d = [dev(x) for x in (cur, ps, v0, s0, a0, g)]
    out = [torch.empty((B, T, D), device="cuda")] + [torch.empty((B, D), device="cuda") for _ in range(5)]
    nb = _lib.lib().ava_lif_scan_bwd_segments_workspace(B, T, D)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    p = lambda t: C.c_void_p(t.data_ptr())
    f.restype = C.c_int
    f.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int] + [C.c_void_p] * 4 + [C.c_int] * 3 + [C.c_float, C.c_int] + \
        [C.c_void_p] * 10 + [C.c_size_t, C.c_void_p, C.c_void_p]
    rc = f(p(d[0]), B, T, D, p(d[1]), p(d[2]), p(d[3]), p(d[4]), 1, 0, 0, slope, 0, p(d[5]), None, None,
           *(p(x) for x in out), p(ws), nb // 4, None, _lib.current_stream())
    assert rc == 0
    want = o["dI"]
    if slope < 0:
        assert np.isinf(want[:, T - 1]).any()
    assert np.array_equal(host(out[0]), want, equal_nan=True)


def test_kwta_relu2_bwd():
    from ava_amd import ops
    rng = np.random.default_rng(3)
    n, h, k = 2048, 4096, 1024
    u = rng.normal(size=(n, h)).astype(np.float32)
    u[:, 100:110] = u[:, 0:10]  # repeated values
    ga = rng.normal(size=(n, h)).astype(np.float32)
    a, kth = ops.kwta_relu(dev(u), k, relu2=True)
    gu = host(ops.kwta_relu2_bwd(dev(u), kth, dev(ga)))
    ref = O.kwta_relu2_bwd(u, host(kth), ga)
    assert np.array_equal(gu, ref)
    assert np.array_equal(host(kth), O.kwta(u, k)[1])  # the same threshold the oracle selects


@pytest.mark.parametrize("i", [0, 3, 7])
def test_dense_back(i):
    from ava_amd import ops
    rng = np.random.default_rng(i)
    L, M = 8, 1 << 20
    S = rng.normal(size=(L + 1, M)).astype(np.float32)
    G = rng.normal(size=(L, M)).astype(np.float32)
    wf = rng.normal(size=L * (L + 3) // 2).astype(np.float32)
    out, dw = ops.dense_back(dev(S), dev(G), dev(wf), dev(G[i]), col=i + 1, i0=i, L=L, nd=i + 2)
    ro, rdw = O.dense_back(S, G, wf, G[i], col=i + 1, i0=i, L=L, nd=i + 2)
    assert np.array_equal(host(out), ro)
    assert rel(host(dw), rdw) < 1e-5
    e, _ = ops.dense_back(dev(S), dev(G), dev(wf), dev(np.zeros(M, np.float32)), col=0, i0=0, L=L, nd=0)
    assert np.array_equal(host(e), O.dense_back(S, G, wf, np.zeros(M, np.float32), col=0, i0=0, L=L, nd=0)[0])


def mem_inputs(seed, BH, T, g, hs=64):
    rng = np.random.default_rng(seed)

    def unit(x):
        return (x / np.linalg.norm(x, axis=-1, keepdims=True)).astype(np.float32)

    q, k, e = (unit(rng.normal(size=(BH, T, hs))) for _ in range(3))
    v = rng.normal(size=(BH, T, hs)).astype(np.float32)
    la = np.log(rng.uniform(0.85, 0.999, (BH, T, g))).astype(np.float32)
    b = rng.uniform(0.1, 1.9, (BH, T, g)).astype(np.float32)
    F0 = (rng.normal(size=(BH, hs, hs)) * 0.3).astype(np.float32)
    S0 = (rng.normal(size=(BH, hs, hs)) * 0.1).astype(np.float32)
    dy = rng.normal(size=(BH, T, hs)).astype(np.float32)
    dF = (rng.normal(size=(BH, hs, hs)) * 0.2).astype(np.float32)
    dS = (rng.normal(size=(BH, hs, hs)) * 0.2).astype(np.float32)
    return q, k, e, v, la, b, F0, S0, dy, dF, dS


def run_mem(x, m, cap, init=True):
    from ava_amd import ops
    q, k, e, v, la, b, F0, S0, dy, dF, dS = x
    o = ops.mem_gen_bwd(*(dev(z) for z in (q, k, e, v, la, b, dy)), m=m, cap=cap,
                        F0=dev(F0) if init else None, S0=dev(S0) if (init and m) else None,
                        dF_T=dev(dF) if init else None, dS_T=dev(dS) if (init and m) else None)
    return {n: host(t) for n, t in o.items()}


MEM_OUT = ("dq", "dk", "de", "dv", "dla", "db", "dF0")


@pytest.mark.parametrize("T", [1, 4, 37])
@pytest.mark.parametrize("g", [64, 1])
@pytest.mark.parametrize("m", [0.0, 0.5])
@pytest.mark.parametrize("cap", [1e5, 0.6])
def test_mem_bwd(T, g, m, cap):
    """Group edges (T below, at and off the 4-step checkpoint), per-channel and per-head gates,
    momentum, and a bound that holds on many elements (cap 0.6)."""
    x = mem_inputs(T + g + int(10 * m) + int(cap < 1), 6, T, g)
    print(f"mem_bwd T={T} g={g} m={m} cap={cap}", flush=True)
    o = O.mem_rec_bwd(*x[:6], x[8], m=m, cap=cap, F0=x[6], S0=x[7] if m else None, dF_T=x[9],
                      dS_T=x[10] if m else None)
    gpu = run_mem(x, m, cap)
    for n in MEM_OUT + (("dS0",) if m else ()):
        e = rel(gpu[n], o[n])
        assert e < 1e-5, (n, e)


def test_mem_bwd_zero_state():
    x = mem_inputs(41, 4, 19, 64)
    o = O.mem_rec_bwd(*x[:6], x[8], m=0.5)
    gpu = run_mem(x, 0.5, 1e5, init=False)
    for n in MEM_OUT + ("dS0",):
        assert rel(gpu[n], o[n]) < 1e-5, n


def test_mem_bwd_long():
    """The block stack's sequence length (T 2048) with per-channel gates and momentum 0.5 on 16 heads.
    float32 against float64 over 2048 steps of a recurrence whose state decays by alpha ~ 0.85-0.999:
    the gradients meet 1e-4 relative."""
    x = mem_inputs(77, 16, 2048, 64)
    print("mem_bwd long BH=16 T=2048", flush=True)
    o = O.mem_rec_bwd(*x[:6], x[8], m=0.5, F0=x[6], S0=x[7], dF_T=x[9], dS_T=x[10])
    gpu = run_mem(x, 0.5, 1e5)
    for n in MEM_OUT + ("dS0",):
        e = rel(gpu[n], o[n])
        print(f"  {n}: rel {e:.2e}", flush=True)
        assert e < 1e-4, (n, e)


def test_mem_bwd_many_heads():
    """512 heads: one workgroup per head and 16 columns per wave (fewer heads take four workgroups per
    head, a wave's 4 columns each, and add the rows' sums of the four in a second kernel)."""
    x = mem_inputs(91, 512, 9, 64)
    print("mem_bwd BH=512 T=9", flush=True)
    o = O.mem_rec_bwd(*x[:6], x[8], m=0.5, F0=x[6], S0=x[7], dF_T=x[9], dS_T=x[10])
    gpu = run_mem(x, 0.5, 1e5)
    for n in MEM_OUT + ("dS0",):
        e = rel(gpu[n], o[n])
        assert e < 1e-5, (n, e)


def clear_heads(x, m, cap):
    """The heads none of whose float64 states comes within 3e-7 of the bound before it is applied (a few
    float32 roundings of a value of 0.6): there float32 decides the bound as float64 does."""
    q, k, e, v, la, b, F, S = (z.astype(np.float64) for z in x[:8])
    margin = np.full(q.shape[0], np.inf)
    S = S if m else 0.0 * S
    for t in range(q.shape[1]):
        a, bt = np.exp(la[:, t]), b[:, t]
        r = np.einsum("hi,hij->hj", e[:, t], F)
        S = m * S + (bt * k[:, t])[:, :, None] * v[:, t][:, None] - (a * bt * e[:, t])[:, :, None] * r[:, None]
        P = a[:, :, None] * F + S
        margin = np.minimum(margin, np.abs(np.abs(P) - cap).min(axis=(1, 2)))
        F = np.clip(P, -cap, cap)
    return margin > 3e-7


@pytest.mark.parametrize("BH,T", [(16, 33), (32, 16), (33, 33), (65, 17), (96, 18), (97, 17), (129, 47), (193, 16),
                                  (512, 32), (530, 33)])
@pytest.mark.parametrize("g,m", [(64, 0.5), (1, 0.0)])
@pytest.mark.parametrize("cap", [1e5, 0.6])
def test_mem_bwd_walk_shapes(BH, T, g, m, cap):
    """Each split of a head's columns over workgroups (on 256 CUs up to 16, 96, 192 heads, more; from
    512 and past 32 steps the two walks one after the other), chunks of 16 steps whole and
    short, with the bound never and often reached (the reverse walk's second form and the masked rows)."""
    x = mem_inputs(BH + T + g, BH, T, g)
    print(f"mem_bwd BH={BH} T={T} g={g} m={m} cap={cap}", flush=True)
    o = O.mem_rec_bwd(*x[:6], x[8], m=m, cap=cap, F0=x[6], S0=x[7] if m else None, dF_T=x[9],
                      dS_T=x[10] if m else None)
    gpu = run_mem(x, m, cap)
    ok = clear_heads(x, m, cap)
    assert np.mean(ok) > 0.5, np.mean(ok)
    for n in MEM_OUT + (("dS0",) if m else ()):
        e = rel(gpu[n][ok], o[n][ok])
        assert e < 1e-5, (n, e)


# outputs on inputs of their layout: the carried gradients; each on its own input; turned round; on dy
ALIASES = [{"dF0": "dF_T", "dS0": "dS_T"}, {"dF0": "F0", "dS0": "S0"},
           {"dq": "q", "dk": "k", "de": "e", "dv": "v", "dla": "la", "db": "b"},
           {"dq": "k", "dk": "e", "de": "v", "dv": "q", "dla": "b", "db": "la"}, {"dv": "dy"}, {"dq": "dy", "dv": "k"}]


@pytest.mark.parametrize("alias", ALIASES)
@pytest.mark.parametrize("BH,T,g,m", [(6, 37, 64, 0.5), (6, 37, 1, 0.0), (70, 18, 64, 0.5), (130, 33, 1, 0.5)])
@pytest.mark.parametrize("cap", [1e5, 0.6])
def test_mem_bwd_in_place(alias, BH, T, g, m, cap):
    """Outputs on the inputs' buffers, through the C entry (the wrapper allocates its own): the bits of a call
    with buffers of its own, with and without elements at the bound."""
    import ctypes as C
    from ava_amd import _lib
    names = ("q", "k", "e", "v", "la", "b", "F0", "S0", "dy", "dF_T", "dS_T")
    x = mem_inputs(BH + T + g, BH, T, g)
    print(f"mem_bwd in place {alias} BH={BH} T={T} g={g} m={m} cap={cap}", flush=True)
    want = run_mem(x, m, cap)
    i = {n: dev(z) for n, z in zip(names, x)}
    like = {"dla": "la", "db": "b", "dF0": "F0", "dS0": "S0"}
    o = {n: i[alias[n]] if n in alias else torch.empty_like(i[like.get(n, "q")])
         for n in ("dq", "dk", "de", "dv", "dla", "db", "dF0", "dS0")}
    L = _lib.lib()
    nb = L.ava_mem_scan_bwd_workspace(BH, T, int(m != 0))
    work = torch.empty(nb, dtype=torch.uint8, device="cuda")
    p = lambda t: C.c_void_p(t.data_ptr())
    s = lambda n: p(i[n]) if m else None
    _lib.check(L.ava_mem_scan_bwd(p(i["q"]), p(i["k"]), p(i["e"]), p(i["v"]), p(i["la"]), p(i["b"]), BH, T, 64, g, m,
                                  cap, p(i["F0"]), s("S0"), p(i["dy"]), p(i["dF_T"]), s("dS_T"), p(o["dq"]), p(o["dk"]),
                                  p(o["de"]), p(o["dv"]), p(o["dla"]), p(o["db"]), p(o["dF0"]),
                                  p(o["dS0"]) if m else None, p(work), nb, _lib.current_stream()), "ava_mem_scan_bwd")
    for n in MEM_OUT + (("dS0",) if m else ()):
        assert np.array_equal(host(o[n]), want[n]), n


@pytest.mark.parametrize("BH,T,g,m", [(6, 37, 64, 0.5), (130, 18, 1, 0.0)])
@pytest.mark.parametrize("cap", [1e5, 0.6])
def test_mem_bwd_off_16_bytes(BH, T, g, m, cap):
    """Inputs and outputs one float past a 16-byte boundary: the bits of aligned ones."""
    x = mem_inputs(BH + T + g, BH, T, g)
    print(f"mem_bwd off 16 bytes BH={BH} T={T} g={g} m={m} cap={cap}", flush=True)
    want = run_mem(x, m, cap)
    import ctypes as C
    from ava_amd import _lib
    L = _lib.lib()

    def off(n):
        t = torch.empty(n + 1, dtype=torch.float32, device="cuda")[1:]
        assert t.data_ptr() % 16 == 4
        return t

    i = [off(z.size).copy_(dev(z).view(-1)) for z in x]
    o = {n: off(want[n].size) for n in MEM_OUT + (("dS0",) if m else ())}
    nb = L.ava_mem_scan_bwd_workspace(BH, T, int(m != 0))
    work = torch.empty(nb, dtype=torch.uint8, device="cuda")
    p = lambda t: C.c_void_p(t.data_ptr())
    q, k, e, v, la, b, F0, S0, dy, dF, dS = (p(t) for t in i)
    _lib.check(L.ava_mem_scan_bwd(q, k, e, v, la, b, BH, T, 64, g, m, cap, F0, S0 if m else None, dy, dF,
                                  dS if m else None, p(o["dq"]), p(o["dk"]), p(o["de"]), p(o["dv"]), p(o["dla"]),
                                  p(o["db"]), p(o["dF0"]), p(o["dS0"]) if m else None, p(work), nb,
                                  _lib.current_stream()), "ava_mem_scan_bwd")
    for n in o:
        assert np.array_equal(host(o[n]), want[n].reshape(-1)), n


def test_wrappers_ignore_the_default_dtype():
    """The wrappers allocate float32 whatever torch's default dtype is (a float64 default once gave
    float64 output buffers that the kernels, writing float32, left mostly unwritten)."""
    old = torch.get_default_dtype()
    torch.set_default_dtype(torch.float64)
    try:
        x = lif_inputs(9, 2, 3, 8, 2, True)
        o = O.lif_bwd(x[0], x[1], x[5], x[2], x[3], x[4], x[6], x[7], slope=2.0)
        gpu = run_lif(*x, 2, True, True, 2.0, False)
        for k in ("dI", "dv0", "da0", "dbeta", "drho", "dgain"):
            assert gpu[k].dtype == np.float32 and np.array_equal(gpu[k], o[k]), k
    finally:
        torch.set_default_dtype(old)
