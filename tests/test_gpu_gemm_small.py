"""Products of few rows or little work (K split over a workgroup's four or eight wavefronts, operands turned into the MFMA layout through LDS)
against 64-bit sums. Error on normal operands, whose sums have the size sqrt(K): chains of at most 24 MFMAs of four k each (5.0e-8 sqrt(24 / 2), measured on
the matrix unit), whose results are added one after another, at most K / 128 of them a wavefront, and then over the wavefronts
(2.4e-8 sqrt(additions / 2): the mean rounding of an addition); a fifth is allowed on top, and three standard deviations of a root mean
square over few outputs."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT
from frankentorch_amd.device import EPI_BIAS, EPI_GELU, EPI_RESIDUAL, DeviceBuffer

pytestmark = pytest.mark.gpu


def _close(got, ref, k, alpha=1.0):
    bound = 1.2 * np.hypot(5.0e-8 * np.sqrt(24 / 2), 2.4e-8 * np.sqrt((k / 128 + 4) / 2)) * (1 + 3 / np.sqrt(2 * ref.size))
    return np.linalg.norm(got - ref) <= bound * abs(alpha) * np.sqrt(ref.size * k)


def _run(hip, m, n, k, trans_b, batch=1, epilogue=0, alpha=1.0, pad=0):
    rng = np.random.default_rng(m * 7 + n * 3 + k + batch)
    a, b = rng.standard_normal((batch, m, k + pad), np.float32), rng.standard_normal((batch, n, k + pad) if trans_b else (batch, k, n + pad), np.float32)
    bias, res = rng.standard_normal(n, np.float32), rng.standard_normal((batch, m, n), np.float32)
    up = DeviceBuffer.from_host
    c = DeviceBuffer((batch, m, n))
    desc = hip.gemm_desc(m, n, k, trans_b=trans_b, batch=batch, epilogue=epilogue)
    desc.lda, desc.ldb, desc.stride_a, desc.stride_b = k + pad, (k if trans_b else n) + pad, a[0].size, b[0].size
    hip.gemm(desc, up(a), up(b), c, up(bias) if epilogue & EPI_BIAS else None, up(res) if epilogue & EPI_RESIDUAL else None, alpha)
    ref = alpha * (a[:, :, :k].astype(np.float64) @ (np.swapaxes(b[:, :, :k], 1, 2) if trans_b else b[:, :, :n]).astype(np.float64))
    if epilogue & EPI_BIAS:
        ref = ref + bias
    if epilogue & EPI_RESIDUAL:
        ref = ref + res
    return c.to_host().reshape(ref.shape).astype(np.float64), ref


# tiles of one row and one column; ragged tiles; column tiles that are no multiple of eight (the XCD order's last run); wavefronts
# without a group of k (K 272 over eight), partly filled slots, six slots (K 768, 3072), four wavefronts (many tiles), two row tiles
# (1536 tiles and more, with an odd number of row tiles), two column tiles as well (3072 and more, an odd number of them) and three row
# tiles (6000 and more), the largest single row and the LM head's shape with few rows; a K walked in many passes
NT = [(1, 1, 256), (1, 17, 272), (16, 16, 256), (17, 33, 464), (37, 768, 3072), (5, 3072, 768), (64, 768, 1040), (37, 2304, 768), (128, 1016, 384),
      (400, 2304, 768), (333, 1536, 512), (49, 8200, 256), (65, 10000, 768), (1, 50257, 768), (33, 20000, 272), (200, 3793, 272), (65, 20003, 256), (41, 33009, 272),
      (37, 3072, 768), (200, 3072, 768), (64, 5000, 992), (64, 512, 16384), (128, 128, 40000)]


@pytest.mark.parametrize("m,n,k", NT)
def test_rows_times_rows(hip, m, n, k):
    got, ref = _run(hip, m, n, k, True)
    assert _close(got, ref, k)


@pytest.mark.parametrize("m,n,k", [(400, 2304, 768), (130, 1036, 400), (1600, 1152, 384), (300, 512, 1536), (64, 3072, 768)])
def test_rows_times_columns(hip, m, n, k):
    got, ref = _run(hip, m, n, k, False)
    assert _close(got, ref, k)


@pytest.mark.parametrize("trans_b,m,n,k", [(True, 37, 200, 512), (True, 70, 333, 256), (False, 200, 260, 512)])
def test_batches_pitches_and_epilogues(hip, trans_b, m, n, k):
    for batch, epilogue, alpha, pad in ((1, EPI_BIAS | EPI_RESIDUAL, 1.0, 4), (5, EPI_BIAS, 1.0, 0), (3, EPI_RESIDUAL, -0.5, 8)):
        got, ref = _run(hip, m, n, k, trans_b, batch, epilogue, alpha, pad)
        assert _close(got, ref, k, alpha)
    plain, _ = _run(hip, m, n, k, trans_b, epilogue=EPI_BIAS)
    gelu, _ = _run(hip, m, n, k, trans_b, epilogue=EPI_BIAS | EPI_GELU)
    from scipy.special import erf
    ref = 0.5 * plain * (1 + erf(plain / np.sqrt(2)))
    assert np.max(np.abs(gelu - ref)) <= 1e-6 * np.max(np.abs(ref))


CHILD = """
import sys
sys.path[:0] = [%(root)r, %(root)r + "/tests"]
import numpy as np
from frankentorch_amd import device as hip
import test_gpu_gemm_small as t
np.savez(sys.argv[1], **{str(i): t._run(hip, *s, True)[0] for i, s in enumerate(t.LONG)})
"""
LONG = [(64, 128, 131072), (16, 256, 131072), (64, 128, 98304), (1, 128, 131072)]


def test_longest_reductions(hip, tmp_path):
    """Few tiles and a K past the limit run on the kernels that cut K over workgroups, as they do with these kernels switched off (a child
    process: the switch is read once); on this side of it they do not. Error: the large tiles' 1.8e-8 sqrt(K) at the most."""
    path = str(tmp_path / "large.npz")
    subprocess.run([sys.executable, "-c", CHILD % {"root": ROOT}, path], check=True, timeout=110, env=dict(os.environ, FT_HIP_GEMM_SMALL="0"))
    large = np.load(path)
    for i, (m, n, k) in enumerate(LONG):
        got, ref = _run(hip, m, n, k, True)
        assert np.linalg.norm(got - ref) <= 1.8e-8 * np.sqrt(k) * np.linalg.norm(ref)
        assert np.array_equal(got, large[str(i)]) == (i < 2), (m, n, k)
