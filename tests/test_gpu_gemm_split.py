"""Large fp32 products (operands split into three bf16 parts, six matrix products) against 64-bit sums.

Bound on the error: that of the fp32 matrix-unit kernels on the same operands, measured as 1.79e-8 sqrt(K) (relative 2-norm,
normal operands, K 128 to 4096). Ordinary sums stay under two thirds of it (0.57e-8 sqrt(K) measured); parts of a tile that
are computed again on fp32 matrix units are allowed twice it."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT
from frankentorch_amd.device import EPI_BIAS, EPI_GELU, EPI_GELU_TANH, EPI_RESIDUAL, DeviceBuffer

pytestmark = pytest.mark.gpu

# ragged tiles in both directions with K no multiple of 32; whole tiles; few tiles and a deep K (the K range is split);
# tall and narrow; K shorter than a run of the split; 64 x 128 tiles, whole and with the K range split in seven
SHAPES = [(4097, 3077, 1001), (4096, 3072, 768), (1030, 770, 20003), (20011, 1000, 520), (2048, 2304, 3072), (2331, 768, 768), (768, 768, 2331)]


def _gemm(hip, m, n, k, a, b, trans_a=False, trans_b=False, **kw):
    dc = DeviceBuffer((m, n), np.float32)
    bias, res = kw.pop("bias", None), kw.pop("residual", None)
    up = lambda x: None if x is None else DeviceBuffer.from_host(x)
    hip.gemm(hip.gemm_desc(m, n, k, trans_a=trans_a, trans_b=trans_b, epilogue=kw.pop("epilogue", 0)), up(a), up(b), dc, up(bias), up(res),
             kw.pop("alpha", 1.0))
    return dc.to_host()


def _rel(got, ref):
    return np.linalg.norm(got.astype(np.float64) - ref) / np.linalg.norm(ref)


def _bound(k, again=False):
    return (2.0 if again else 2.0 / 3.0) * 1.79e-8 * np.sqrt(k)


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
def test_split_product_forms(hip, m, n, k, form):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32)
    rows = np.unique(np.r_[np.arange(0, m, 97), m - 17 : m])
    ref = a[rows].astype(np.float64) @ b.T.astype(np.float64)
    got = _gemm(hip, m, n, k, np.ascontiguousarray(a.T) if form == "tn" else a, b if form == "nt" else np.ascontiguousarray(b.T),
                trans_a=form == "tn", trans_b=form == "nt")
    assert _rel(got[rows], ref) <= _bound(k)


@pytest.mark.parametrize("m,n,k", [(661, 2304, 640), (1159, 1280, 640), (2257, 640, 640)])
def test_split_product_before_the_one_for_little_work(hip, m, n, k):
    """Both take products of 1.5 to 2 GFLOP against [n, k] weights; the split one has the smaller error, 0.57e-8 sqrt(K) measured (four fp32
    chains a product: 0.9e-8 sqrt(K))."""
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32)
    rows = np.arange(0, m, 97)
    assert _rel(_gemm(hip, m, n, k, a, b, trans_b=True)[rows], a[rows].astype(np.float64) @ b.T.astype(np.float64)) <= 0.7e-8 * np.sqrt(k)


@pytest.mark.parametrize("m,n,k", [(4096, 3072, 768), (2048, 768, 11008), (2331, 768, 768), (768, 768, 50257)])
@pytest.mark.parametrize("kind", ["one sign", "relu", "one term"])
def test_split_product_of_other_operands(hip, m, n, k, kind):
    """Operands of one sign would show a drift of the sums, half-empty ones an error that does not shrink with the number of
    terms (fp32 kernels: 1.35e-8 and 1.27e-8 sqrt(k) up to K 4096). A single term shows the products that are left out: one
    rounding (2^-24) and less than 2^-24 left out."""
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32)
    if kind == "one sign":
        a, b = np.abs(a), np.abs(b)
    elif kind == "relu":
        a = np.maximum(a, 0)
    else:
        col = rng.integers(0, k, m)
        keep = a[np.arange(m), col]
        a = np.zeros((m, k), np.float32)
        a[np.arange(m), col] = keep
    got = _gemm(hip, m, n, k, a, b, trans_b=True)
    rows = np.arange(0, m, 41)
    ref = a[rows].astype(np.float64) @ b.T.astype(np.float64)
    if kind == "one term":
        assert np.abs(got[rows] - ref).max(initial=0, where=ref == 0) == 0
        assert (np.abs(got[rows] - ref) <= 2.0 ** -23 * np.abs(ref)).all()
    else:
        assert _rel(got[rows], ref) <= 2.0 / 3.0 * 1.27e-8 * np.sqrt(k)


@pytest.mark.parametrize("m,n,k", [(4097, 3077, 1001), (1030, 770, 20003), (2331, 768, 768), (768, 768, 2331)])
@pytest.mark.parametrize("epilogue,alpha", [(EPI_BIAS, 1.0), (EPI_BIAS | EPI_GELU, 1.0), (EPI_BIAS | EPI_GELU_TANH, 1.0), (EPI_BIAS | EPI_RESIDUAL, -0.5)])
def test_split_product_epilogues(hip, m, n, k, epilogue, alpha):
    rng = np.random.default_rng(7)
    a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32) * np.float32(k ** -0.5)
    bias, res = rng.standard_normal(n, np.float32), rng.standard_normal((m, n), np.float32)
    plain = _gemm(hip, m, n, k, a, b, trans_b=True).astype(np.float64) * alpha + bias
    got = _gemm(hip, m, n, k, a, b, trans_b=True, epilogue=epilogue, alpha=alpha, bias=bias, residual=res if epilogue & EPI_RESIDUAL else None)
    if epilogue & EPI_GELU:
        from scipy.special import erf
        plain = plain * 0.5 * (1 + erf(plain / np.sqrt(2)))
    if epilogue & EPI_GELU_TANH:
        plain = 0.5 * plain * (1 + np.tanh(np.sqrt(2 / np.pi) * (plain + 0.044715 * plain ** 3)))
    if epilogue & EPI_RESIDUAL:
        plain = plain + res
    assert np.abs(got - plain).max() <= 4e-6  # a few roundings of values up to 8


@pytest.mark.parametrize("m,n,k", [(4096, 3072, 768), (768, 768, 2331)])
def test_split_product_values_the_parts_cannot_hold(hip, m, n, k):
    """Infinities, NaN, floats that round up to a bf16 infinity, overflowing products and magnitudes whose low bits lie below
    the bf16 subnormals: what fp32 arithmetic gives."""
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32)
    a[5, 7], a[6, 8], a[600, 9], b[40, 11], b[41, 12] = np.inf, -np.inf, np.nan, np.inf, np.nan
    a[700], b[500] = 0, 0
    a[700, k - 3], b[500, k - 3] = np.finfo(np.float32).max, np.float32(0.5)
    a[701] = a[702] * np.float32(1e-36)
    a[703] *= np.float32(1e30)
    b[600] *= np.float32(1e30)
    got = _gemm(hip, m, n, k, a, b, trans_b=True)
    with np.errstate(all="ignore"):
        for r in (5, 6, 600, 700, 701, 703, 704):
            ref = (a[r].astype(np.float64) * b.astype(np.float64)).sum(1)
            want = ref.astype(np.float32)
            if r == 703:  # terms of 1e60 and either sign: the order of the sum decides which infinity it ends at
                assert not np.isfinite(got[r, 600])
                want[600] = got[r, 600]
            assert np.array_equal(np.isnan(got[r]), np.isnan(want)), r
            fine = np.isfinite(want)
            assert np.array_equal(got[r][~fine & ~np.isnan(want)], want[~fine & ~np.isnan(want)]), r
            scale = np.abs(a[r].astype(np.float64)) @ np.abs(b.astype(np.float64)).T
            # 2^-24 per rounding of a running sum, one for four k at most, and the subnormal spacing
            ok = np.abs(got[r].astype(np.float64) - ref)[fine] <= (k / 4 * 2.0 ** -24 * scale[fine] + k * 2.0 ** -149)
            assert ok.all(), (r, int((~ok).sum()))
    assert got[700, 500] == np.float32(np.finfo(np.float32).max) * np.float32(0.5)


# either side of the limits on operands (2^-110 and 2^53) and on sums (2^-100)
@pytest.mark.parametrize("small,large", [(-120, 60), (-128, 20), (-140, 40), (-100, 23), (0, 25), (3, 48), (0, 53), (-105, 48), (-60, -45), (-104, 0)])
def test_split_product_small_beside_large(hip, small, large):
    """A row whose low bits (or all of them) lie below the bf16 subnormals, times columns large enough to bring the sums back:
    the same bound as for ordinary operands (the sums of a subnormal row too: its floats are exact)."""
    m, n, k = 2048, 2304, 768
    rng = np.random.default_rng(small + large + 500)
    a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32)
    a[11] = np.ldexp(a[11], small)
    b[100:160] = np.ldexp(b[100:160], large)
    got = _gemm(hip, m, n, k, a, b, trans_b=True).astype(np.float64)
    for rows, cols in ((slice(11, 12), slice(100, 160)), (slice(0, 11), slice(90, 170)), (slice(11, 12), slice(160, 400))):
        ref = a[rows].astype(np.float64) @ b[cols].T.astype(np.float64)
        floor = np.sqrt(ref.size) * 2.0 ** -126  # results that are subnormal themselves
        assert np.linalg.norm(got[rows, cols] - ref) <= _bound(k, True) * np.linalg.norm(ref) + floor


def test_split_product_cancelling_to_the_lowest_bits(hip):
    """Two products that cancel but for bits far below bf16's: what is left is the exact difference, for operands small enough
    that their lower parts are subnormal too."""
    m, n, k = 2048, 2304, 768
    a, b = np.zeros((m, k), np.float32), np.zeros((n, k), np.float32)
    cases = [(2.0 ** -130, 2.0 ** -5, 2.0 ** 23), (2.0 ** -130, 2.0 ** -5, 2.0 ** 40), (2.0 ** -109, 2.0 ** -23, 2.0 ** 40), (2.0 ** -112, 2.0 ** -20, 2.0 ** 20),
             (1.0, 2.0 ** -23, 1.0), (2.0 ** 40, 2.0 ** -23, 2.0 ** -20)]
    for i, (x, d, y) in enumerate(cases):
        a[5 + 70 * i, 0], a[5 + 70 * i, 41] = x * (1 + d), -x
        b[7 + 70 * i, 0] = b[7 + 70 * i, 41] = y
    got = _gemm(hip, m, n, k, a, b, trans_b=True)
    for i, (x, d, y) in enumerate(cases):
        assert got[5 + 70 * i, 7 + 70 * i] == np.float32(x * d * y), (i, x, d, y)


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("m,n,k,off,pad", [(1030, 772, 1280, 4, 8), (1029, 771, 1283, 1, 3), (4097, 2001, 333, 3, 5)])
def test_split_product_of_operands_inside_larger_ones(hip, m, n, k, off, pad, form):
    """Row pitches, bases that are no multiple of 16 bytes, a pitched residual: NaN beside the operands, and nothing written
    beside C."""
    rng = np.random.default_rng(m)
    a, b, bias = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32), rng.standard_normal(n, np.float32)

    def inside(x, fill):
        store = np.full(off + x.shape[0] * (x.shape[1] + pad), fill, np.float32)
        store[off:].reshape(x.shape[0], -1)[:, : x.shape[1]] = x
        return store

    def rows_of(store, shape):
        return store[off:].reshape(shape[0], shape[1] + pad)

    sa, sb = a.T if form == "tn" else a, b if form == "nt" else b.T
    res = rng.standard_normal((m, n), np.float32)
    da, db, dres, dc = (DeviceBuffer.from_host(x) for x in (inside(sa, np.nan), inside(sb, np.nan), inside(res, np.nan), inside(np.full((m, n), 7, np.float32), 7.0)))
    desc = hip.gemm_desc(m, n, k, trans_a=form == "tn", trans_b=form == "nt", lda=sa.shape[1] + pad, ldb=sb.shape[1] + pad, ldc=n + pad,
                         epilogue=EPI_BIAS | EPI_RESIDUAL)
    hip.gemm(desc, da.view(off), db.view(off), dc.view(off), DeviceBuffer.from_host(bias), dres.view(off))
    out = dc.to_host()
    got = rows_of(out, (m, n))
    rows = np.unique(np.r_[np.arange(0, m, 97), m - 17 : m])
    ref = a[rows].astype(np.float64) @ b.T.astype(np.float64) + bias + res[rows]
    assert _rel(got[rows, :n], ref) <= _bound(k)
    assert np.all(got[:, n:] == 7.0) and np.all(out[:off] == 7.0)


def test_split_product_is_repeatable_and_padding_is_not_read_into_it(hip):
    m, n, k = 4097, 3077, 1001
    rng = np.random.default_rng(4)
    a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32)
    first = _gemm(hip, m, n, k, a, b, trans_b=True)
    _gemm(hip, m + 64, n, k, np.full((m + 64, k), np.nan, np.float32), b, trans_b=True)  # leaves NaN in the scratch memory
    assert np.array_equal(first, _gemm(hip, m, n, k, a, b, trans_b=True))


ROUTE_SHAPES = [(2048, 2304, 768), (4096, 3072, 256), (2050, 1540, 288), (2331, 768, 768), (768, 768, 2331), (8192, 768, 3072), (3072, 768, 8192)]


def route_products(hip):
    """Every seventh row of the products, for this process's setting of FT_HIP_GEMM_SPLIT, with what they should be."""
    for m, n, k in ROUTE_SHAPES:
        rng = np.random.default_rng(m + 2 * n + k)
        a, b = rng.standard_normal((m, k), np.float32), rng.standard_normal((n, k), np.float32)
        rows = np.arange(0, m, m // 64)
        ref = a[rows].astype(np.float64) @ b.T.astype(np.float64)
        for form in ("nt", "nn", "tn"):
            got = _gemm(hip, m, n, k, np.ascontiguousarray(a.T) if form == "tn" else a, b if form == "nt" else np.ascontiguousarray(b.T),
                        trans_a=form == "tn", trans_b=form == "nt")
            yield "%s_%d_%d_%d" % (form, m, n, k), got[rows], ref
    rows, vocab, d = 1000, 20000, 512  # with row maxima
    rng = np.random.default_rng(9)
    x, w = rng.standard_normal((rows, d), np.float32), rng.standard_normal((vocab, d), np.float32)
    logits, best = DeviceBuffer((rows, vocab)), DeviceBuffer((rows,))
    hip.linear_argmax(DeviceBuffer.from_host(x), DeviceBuffer.from_host(w), rows, vocab, d, logits, best, DeviceBuffer((hip.linear_argmax_workspace_floats(rows, vocab),)))
    got = logits.to_host()
    assert np.array_equal(best.to_host(), np.argmax(got, axis=1).astype(np.float32))
    yield "argmax", got[::20], x[::20].astype(np.float64) @ w.T.astype(np.float64)


CHILD = """
import sys
sys.path[:0] = [%(root)r, %(root)r + "/tests"]
import numpy as np
from frankentorch_amd import device as hip
import test_gpu_gemm_split as t
np.savez(sys.argv[1], **{name: got for name, got, _ in t.route_products(hip)})
"""


def test_which_kernels_run(hip, tmp_path):
    """With the split product switched off (a child process: the switch is read once) the same calls run on the fp32 kernels, as
    batches and captures without scratch do: both are near the 64-bit product, and not one has the other's bits."""
    path = str(tmp_path / "fp32.npz")
    subprocess.run([sys.executable, "-c", CHILD % {"root": ROOT}, path], check=True, timeout=110, env=dict(os.environ, FT_HIP_GEMM_SPLIT="0"))
    fp32 = np.load(path)
    for name, got, ref in route_products(hip):
        k = int(name.rsplit("_", 1)[1]) if "_" in name else 512
        assert _rel(got, ref) <= _bound(k), name
        assert _rel(fp32[name], ref) <= _bound(k, True), name
        assert not np.array_equal(got, fp32[name]), name
