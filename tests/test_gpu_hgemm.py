"""The training step's f32 products on the f16 matrix cores (ava::hgemm and its split passes), called by symbol,
against float64.

Bars, from the form: an operand's two terms leave at most 2^-23 of a value (2^-51 of its row's largest for values
far below it), the dropped term product is at most 2^-22 of a product, and every f32 addition rounds by 2^-24 of a partial
sum. So per element the error is at most (2^-21 + (K + parts) 2^-24) sum |a b| + 2^-51 (max|a| sum |b| + max|b| sum |a|);
in the 2-norm, over values without a common sign, at most 2^-22 + 2^-24 sqrt(K / 16) of the result's (the operands'
errors at their largest, one independent rounding per matrix instruction of 16 products)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

VP, I = C.c_void_p, C.c_int


class Op(C.Structure):
    _fields_ = [("planes", VP), ("exps", VP)]


def fn(name, args, res=I):
    from ava_amd import _lib
    f = getattr(_lib.lib(), name)
    f.argtypes, f.restype = args, res
    return f


def stream():
    from ava_amd import _lib
    return _lib.current_stream()


def split(x, cols):
    """The operand x [rows][K], or with cols x [K][rows] (K down its columns); x may be a view with a row stride."""
    rows, k = (x.shape[1], x.shape[0]) if cols else x.shape
    ldk = (k + 63) // 64 * 64
    planes = torch.full((rows * ldk * 4,), 0x7f, dtype=torch.uint8, device="cuda")
    exps = torch.empty(rows, dtype=torch.int32, device="cuda")
    if cols:
        part = torch.empty(fn("_ZN3ava17hgemm_part_floatsEii", [I, I], C.c_size_t)(k, rows), device="cuda")
        f = fn("_ZN3ava16hgemm_split_colsEPKfiiiPvPiPfP12ihipStream_t", [VP, I, I, I, VP, VP, VP, VP])
        assert f(x.data_ptr(), k, rows, x.stride(0), planes.data_ptr(), exps.data_ptr(), part.data_ptr(), stream()) == 0
    else:
        f = fn("_ZN3ava16hgemm_split_rowsEPKfiiiPvPiP12ihipStream_t", [VP, I, I, I, VP, VP, VP])
        assert f(x.data_ptr(), rows, k, x.stride(0), planes.data_ptr(), exps.data_ptr(), stream()) == 0
    return planes, exps


def product(a, b, a_cols=False, b_cols=False, add=None, ldc=None):
    """a [m][k] times b [n][k]^T (float32, CUDA), each handed over as it lies or transposed (its split_cols form)."""
    m, k = a.shape
    n = b.shape[0]
    pa, ea = split(a.t().contiguous() if a_cols else a, a_cols)
    pb, eb = split(b.t().contiguous() if b_cols else b, b_cols)
    ldc = ldc or n
    c = torch.full((m, ldc), 7.0, device="cuda")
    if add is not None:
        c[:, :n] = add
    parts = fn("_ZN3ava12hgemm_splitsEiii", [I, I, I])(m, n, k)
    part = torch.full((parts * m * n if parts > 1 else 1,), float("nan"), device="cuda")
    f = fn("_ZN3ava5hgemmERKNS_7HgemmOpES2_iiiPfibS3_mP12ihipStream_t",
           [C.POINTER(Op), C.POINTER(Op), I, I, I, VP, I, C.c_bool, VP, C.c_size_t, VP])
    oa, ob = Op(pa.data_ptr(), ea.data_ptr()), Op(pb.data_ptr(), eb.data_ptr())
    assert f(C.byref(oa), C.byref(ob), m, n, k, c.data_ptr(), ldc, add is not None, part.data_ptr(), part.numel(),
             stream()) == 0
    torch.cuda.synchronize()
    assert torch.all(c[:, n:] == 7.0)  # nothing past a row's n columns
    return c[:, :n], parts


def f64(x):
    return x.cpu().double()


def check(a, b, c, parts, add=None):
    a, b, c = f64(a), f64(b), f64(c)
    k = a.shape[1]
    want = a @ b.t() + (f64(add) if add is not None else 0.0)
    s = a.abs() @ b.abs().t() + (f64(add).abs() if add is not None else 0.0)
    low = a.abs().amax(1, keepdim=True) * b.abs().sum(1) + a.abs().sum(1, keepdim=True) * b.abs().amax(1)
    tol = (2.0**-21 + (k + parts + 1) * 2.0**-24) * s + 2.0**-51 * low + 1e-37
    assert torch.all((c - want).abs() <= tol), float(((c - want).abs() / tol).max())
    rel = float((c - want).norm() / want.norm().clamp_min(1e-300))
    print(f"{tuple(a.shape)} x {tuple(b.shape)}, {parts} parts: relative 2-norm {rel:.2e}", flush=True)
    return rel, want


def bar(k):
    return 2.0**-22 + 2.0**-24 * (max(k, 16) / 16) ** 0.5


def rnd(seed, *shape):
    return torch.from_numpy(np.random.default_rng(seed).standard_normal(shape, dtype=np.float32)).cuda()


# tiles whole and ragged (128 x 256), K at and off the 64-value blocks, K cut into parts with a short last one, each
# width of the row split (1024, 4096, 8192, more) and widths off 4
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (128, 256, 64), (129, 257, 65), (64, 1000, 1024), (255, 40, 1030),
                                   (300, 700, 4096), (32, 130, 4100), (70, 60, 8192), (65, 33, 8207), (1100, 1300, 96)])
@pytest.mark.parametrize("a_cols,b_cols", [(False, False), (True, False), (False, True), (True, True)])
def test_product_matches_float64(m, n, k, a_cols, b_cols):
    a, b = rnd(m + k, m, k), rnd(n + k + 1, n, k)
    c, parts = product(a, b, a_cols, b_cols)
    rel, _ = check(a, b, c, parts)
    assert rel < bar(k)


@pytest.mark.parametrize("m,n,k,ldc", [(130, 260, 128, 264), (200, 96, 4096, 96), (33, 70, 2050, 81)])
def test_product_adds_into_wider_rows(m, n, k, ldc):
    a, b, add = rnd(1, m, k), rnd(2, n, k), 3.0 * rnd(3, m, n)
    c, parts = product(a, b, add=add, ldc=ldc)
    rel, _ = check(a, b, c, parts, add)
    assert rel < bar(k)


def operands(kind, m=512, n=768, k=1024):
    a, b = rnd(11, m, k), rnd(12, n, k)
    g = np.random.default_rng(13)
    u = lambda *s: torch.from_numpy(g.random(s, dtype=np.float32)).cuda()
    if kind == "binades":
        return a * torch.exp2((40.0 * (u(m, 1) - 0.5)).floor()), b * torch.exp2((40.0 * (u(n, 1) - 0.5)).floor())
    if kind.startswith("lognormal"):
        sg = float(kind.split()[1])
        return a.sign() * torch.exp(sg * rnd(14, m, k)), b.sign() * torch.exp(sg * rnd(15, n, k))
    if kind.startswith("outlier"):  # one element of each row far above the others, meeting zeros
        a[:, 7] *= float(kind.split()[1])
        b[:, 7] = 0.0
    if kind == "spikes":
        a = a.sign() * torch.floor(1.0 + 2.0 * u(m, k)) * (u(m, k) < 0.05)
    if kind == "relu2":
        a = torch.where(a > 0.67, a * a, torch.zeros_like(a))
    return a.contiguous(), b.contiguous()


@pytest.mark.parametrize("kind", ["normal", "binades", "lognormal 1", "lognormal 2", "outlier 1e4", "outlier 1e6",
                                  "outlier 1e8", "spikes", "relu2"])
@pytest.mark.parametrize("cols", [False, True])
def test_no_further_from_float64_than_an_f32_product(kind, cols):
    a, b = operands(kind)
    c, parts = product(a, b, cols, cols)
    rel, want = check(a, b, c, parts)
    lib = float((f64(a @ b.t()) - want).norm() / want.norm())
    print(f"{kind}: relative 2-norm {rel:.2e}, the library's f32 product {lib:.2e}", flush=True)
    assert rel <= lib


def test_zero_rows_subnormals_and_extremes():
    """Rows of zeros give zeros; rows near either end of f32's range keep their values."""
    a, b = rnd(21, 160, 128), rnd(22, 96, 128)
    a[5] = 0.0
    b[9] = 0.0
    a[17] *= 2.0**-140  # subnormal
    a[18] *= 2.0**120
    b[11] *= 2.0**-20
    for cols in (False, True):
        c, parts = product(a, b, cols, cols)
        check(a, b, c, parts)
        assert torch.all(c[5] == 0.0) and torch.all(c[:, 9] == 0.0)


@pytest.mark.parametrize("cols", [False, True])
@pytest.mark.parametrize("k", [96, 2048])
def test_infinities_and_nan_as_in_an_f32_product(cols, k):
    """An infinity or NaN reaches its own row or column only, as the infinity (of its sign) or NaN that a product of the
    values gives, also with values beside it that f16 would not hold (1e6; a value more than 2^39 below its row's largest
    counts as zero to an infinity it meets); opposite infinities and infinity times zero give NaN."""
    a, b = rnd(31, 140, k), rnd(32, 270, k)
    b[:, 5] = torch.where(b[:, 5] > 0, 1.0, -2.0)  # no second term
    a[3, 5] = float("inf")
    a[4, 5], a[4, 6] = float("-inf"), 1e6
    a[5, 7] = float("nan")
    a[6, 5], a[6, 8] = float("inf"), float("-inf")
    b[10, 5] = 0.0
    b[20, 9] = float("inf")
    b[21, 9] = float("nan")
    a[7, 9] = 0.0
    c, parts = product(a, b, cols, cols)
    got, want = f64(c), f64(a) @ f64(b).t()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert inf.any() and torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], want[inf])
    keep_a = torch.isfinite(a).all(1)
    keep_b = torch.isfinite(b).all(1)
    assert torch.isfinite(got[keep_a.cpu()][:, keep_b.cpu()]).all()
    check(a[keep_a], b[keep_b], c[keep_a][:, keep_b], parts)
