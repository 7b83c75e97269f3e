"""float64 products of middling size (K split over a workgroup's wavefronts) against extended-precision sums of sampled rows.
Bound: chains of at most K / 16 matrix instructions of four k each, one of which loses 0.9 of 2^-53, relative 2-norm on normal operands
under 2^-53 sqrt(K) / 2 + 2^-53; few tiles are held to more below."""
import numpy as np
import pytest

from frankentorch_amd.device import EPI_BIAS, EPI_GELU, EPI_RESIDUAL, DeviceBuffer

pytestmark = pytest.mark.gpu


def _run(hip, m, n, k, form, batch=1, epilogue=0, alpha=1.0, pad=0):
    rng = np.random.default_rng(m * 7 + n * 3 + k + batch)
    ta, tb = form[0] == "t", form[1] == "t"
    a, b = rng.standard_normal((batch, k, m + pad) if ta else (batch, m, k + pad)), rng.standard_normal((batch, n, k + pad) if tb else (batch, k, n + pad))
    bias, res = rng.standard_normal(n), rng.standard_normal((batch, m, n))
    up = DeviceBuffer.from_host
    c = DeviceBuffer((batch, m, n), np.float64)
    desc = hip.gemm_desc(m, n, k, trans_a=ta, trans_b=tb, batch=batch, epilogue=epilogue)
    desc.lda, desc.ldb, desc.stride_a, desc.stride_b = a.shape[2], b.shape[2], a[0].size, b[0].size
    hip.gemm(desc, up(a), up(b), c, up(bias) if epilogue & EPI_BIAS else None, up(res) if epilogue & EPI_RESIDUAL else None, alpha)
    a = np.swapaxes(a[:, :, :m], 1, 2) if ta else a[:, :, :k]
    b = np.swapaxes(b[:, :, :k], 1, 2) if tb else b[:, :, :n]
    rows = np.unique(np.r_[np.arange(0, m, max(1, m // 7)), m - 1])
    got = c.to_host().reshape(batch, m, n)
    ref = alpha * np.matmul(a[:, rows].astype(np.longdouble), b.astype(np.longdouble)) if m * n * k * batch < 4e7 else \
        alpha * np.stack([[(x.astype(np.longdouble)[:, None] * y).sum(0) for x in xs] for xs, y in zip(a[:, rows[-2:]], b)])
    if ref.shape[1] != len(rows):
        rows = rows[-2:]
    if epilogue & EPI_BIAS:
        ref = ref + bias
    if epilogue & EPI_RESIDUAL:
        ref = ref + res[:, rows]
    return got[:, rows], ref


# one tile and less, K shorter than a group and than a group a wavefront, every remainder of K modulo 8 in each form, odd pitches
# (rows that are not 16-byte aligned), column tiles that are no multiple of eight, eight wavefronts and four, the longest K of each, past which other kernels run
@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 2), (3, 5, 7), (32, 32, 8), (33, 31, 9), (64, 70, 64), (40, 300, 131), (100, 33, 1021), (17, 290, 2047), (600, 650, 13),
                                   (1021, 1000, 30), (515, 777, 252), (700, 801, 2557), (1030, 1060, 831), (64, 64, 1536), (64, 64, 2000), (300, 900, 1600), (300, 900, 1602)])
def test_against_extended_precision(hip, form, m, n, k):
    got, ref = _run(hip, m, n, k, form)
    err = np.linalg.norm((got - ref).astype(np.float64)) / np.linalg.norm(ref.astype(np.float64))
    assert err <= 2.0 ** -53 * (1 + np.sqrt(k) / 2)


# one tile, eight wavefronts and four with up to 512 tiles, K in whole groups and ragged, the longest K of each
@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
@pytest.mark.parametrize("m,n,k", [(32, 32, 1000), (64, 600, 1500), (17, 290, 2047), (64, 64, 1300), (300, 900, 1300), (512, 1010, 2001), (128, 2080, 1024)])
def test_few_tiles_have_short_chains(hip, form, m, n, k):
    """Chains of at most 18 matrix instructions (9.6e-17 sqrt(18 / 2), measured on the matrix unit) and K / 256 additions of their results
    (4.5e-17 sqrt(additions / 2), the mean rounding of one) and of up to eight wavefronts, a fifth and the spread over the outputs looked at on top."""
    got, ref = _run(hip, m, n, k, form)
    bound = 1.2 * np.hypot(9.6e-17 * 3, 4.5e-17 * np.sqrt((k / 256 + 8) / 2)) * (1 + 3 / np.sqrt(2 * ref.size))
    assert np.linalg.norm((got - ref).astype(np.float64)) <= bound * np.sqrt(ref.size * k)


@pytest.mark.parametrize("form", ["nt", "nn", "tn"])
def test_batches_pitches_and_epilogues(hip, form):
    for m, n, k, batch, epilogue, alpha, pad in ((65, 90, 100, 1, EPI_BIAS | EPI_RESIDUAL, 1.0, 1), (40, 50, 64, 5, EPI_BIAS, 1.0, 0), (130, 70, 37, 40, EPI_RESIDUAL, -0.5, 3)):
        got, ref = _run(hip, m, n, k, form, batch, epilogue, alpha, pad)
        assert np.linalg.norm((got - ref).astype(np.float64)) <= 2.0 ** -53 * (2 + np.sqrt(k) / 2) * np.linalg.norm(ref.astype(np.float64))
    plain, _ = _run(hip, 65, 90, 100, form, epilogue=EPI_BIAS)
    gelu, _ = _run(hip, 65, 90, 100, form, epilogue=EPI_BIAS | EPI_GELU)
    from scipy.special import erf
    assert np.max(np.abs(gelu - 0.5 * plain * (1 + erf(plain / np.sqrt(2))))) <= 1e-14 * np.max(np.abs(plain))


def test_values_past_the_edges_stay_out(hip):
    """Infinities in the last row of K's remainder of one operand meet zeros of the other only where the caller put them."""
    a, b = np.ones((40, 13)), np.ones((50, 13))
    a[7, 12] = np.inf
    c = DeviceBuffer((40, 50), np.float64)
    hip.gemm(hip.gemm_desc(40, 50, 13, trans_b=True), DeviceBuffer.from_host(a), DeviceBuffer.from_host(b), c)
    out = c.to_host()
    assert np.isposinf(out[7]).all() and np.array_equal(np.delete(out, 7, axis=0), np.full((39, 50), 13.0))
