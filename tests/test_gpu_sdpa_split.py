"""Attention on the bf16 matrix units (Q, K, V and the weights split into three bf16 parts) against 64-bit attention.

Bound on the error: that of the fp32 matrix-unit kernels on the same operands, at most 2.0e-8 sqrt(keys) + 1.2e-7 (relative
2-norm, normal operands, measured from 64 to 2048 keys; 1.6e-8 sqrt(keys) + 0.5e-7 here)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT
from frankentorch_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu


def _inputs(heads, group, sq, sk, d, seed=1):
    rng = np.random.default_rng(seed + heads * 7 + sq * 31 + sk)
    return (rng.standard_normal((heads, sq, d), np.float32), rng.standard_normal((heads // group, sk, d), np.float32),
            rng.standard_normal((heads // group, sk, d), np.float32))


def _run(hip, q, k, v, causal, scale=None):
    heads, sq, d = q.shape
    hkv, sk = k.shape[:2]
    out = DeviceBuffer(q.shape)
    scale = 1.0 / np.sqrt(d) if scale is None else scale
    hip.sdpa_forward(hip.sdpa_desc_gqa(1, heads, hkv, sq, sk, d, d, causal), scale, *(DeviceBuffer.from_host(x) for x in (q, k, v)), out)
    return out.to_host().reshape(q.shape)


def _ref(q, k, v, causal, scale=None):
    scale = 1.0 / np.sqrt(q.shape[1]) if scale is None else scale
    with np.errstate(all="ignore"):
        s = (q.astype(np.float64) @ k.astype(np.float64).T) * scale
        if causal:
            s[np.arange(s.shape[0])[:, None] < np.arange(s.shape[1])] = -np.inf
        w = np.exp(s - s.max(axis=1, keepdims=True))
        return (w / w.sum(axis=1, keepdims=True)) @ v.astype(np.float64)


def _rel(got, ref):
    return np.linalg.norm(got - ref) / np.linalg.norm(ref)


# head size 64 on 256 queries a workgroup: one stage of 64 keys and its remainders, three stages, two query blocks, grouped heads;
# on 128 queries and two key halves: halves that are empty (32 keys and fewer), a half with one key, ragged blocks, a long cache;
# head size 128: 32-key stages, ragged ends, short last block, fewer keys than queries
@pytest.mark.parametrize("heads,group,sq,sk,d,causal", [
    (300, 1, 256, 64, 64, False), (300, 4, 250, 65, 64, False), (300, 1, 255, 191, 64, False), (260, 1, 511, 129, 64, True), (96, 4, 300, 300, 64, True),
    (40, 1, 250, 32, 64, False), (70, 1, 129, 33, 64, False), (70, 7, 131, 97, 64, True), (12, 1, 777, 777, 64, True), (16, 4, 700, 1500, 64, False), (9, 1, 1100, 1, 64, False), (96, 1, 127, 127, 64, True),
    (3, 1, 257, 257, 128, True), (2, 2, 300, 2049, 128, False), (5, 1, 33, 161, 128, False), (40, 4, 520, 191, 128, True), (4, 1, 200, 320, 128, True)])
def test_against_64_bit(hip, heads, group, sq, sk, d, causal):
    q, k, v = _inputs(heads, group, sq, sk, d)
    out = _run(hip, q, k, v, causal)
    for h in sorted({0, heads // 2, heads - 1}):
        assert _rel(out[h], _ref(q[h], k[h // group], v[h // group], causal)) <= 2.0e-8 * np.sqrt(sk) + 1.2e-7, "head %d" % h
    if causal:
        assert np.array_equal(out[:, 0], np.repeat(v[:, 0], group, axis=0))


@pytest.mark.parametrize("d,heads,sq,sk", [(64, 300, 256, 200), (64, 40, 300, 200), (128, 7, 300, 200)])
@pytest.mark.parametrize("causal", [False, True])
def test_operands_the_parts_cannot_stand_for(hip, d, heads, sq, sk, causal):
    """Each head has one kind of them: the rows that it reaches are computed on fp32 matrix units."""
    q, k, v = _inputs(heads, 1, sq, sk, d)
    q[0], k[0, 3, 5] = np.abs(q[0]), -np.inf       # a key that nobody looks at
    v[1] *= np.float32(2.0 ** -112)                # third parts below the bf16 subnormals
    v[1, 7] = 0.0
    k[2] *= np.float32(2.0 ** 60)                  # scores of 2^60 and more: one key takes everything
    q[3, 100] *= np.float32(2.0 ** 70)
    v[4, 9, 3] = np.float32(3.4e38)                # rounds to infinity in bf16
    v[5, 20, 2] = np.nan                           # reaches the rows that see key 20, one column of them
    out = _run(hip, q, k, v, causal)
    with np.errstate(all="ignore"):
        for h in range(6):
            ref = _ref(q[h], k[h], v[h], causal)
            got = out[h].astype(np.float64)
            if h == 5:
                first = 20 if causal else 0
                assert np.isnan(got[first:, 2]).all() and np.isfinite(np.delete(got, 2, axis=1)).all()
                ok = np.arange(d) != 2
                got, ref = got[:, ok], ref[:, ok]
            assert np.isfinite(got).all(), "head %d" % h
            top = np.abs(ref).max()  # (norms of values near the ends of the range would leave it)
            # scores of 2^60 carry an error of 2^36: two keys that are close exchange their places now and then
            rows = np.linalg.norm(got / top - ref / top, axis=1) <= 5e-6 * np.linalg.norm(ref / top, axis=1)
            assert rows.mean() >= (0.97 if h in (2, 3) else 1.0), "head %d: %d rows" % (h, (~rows).sum())
    ref = _ref(q[heads - 1], k[heads - 1], v[heads - 1], causal)
    assert _rel(out[heads - 1], ref) <= 2.0e-8 * np.sqrt(sk) + 1.2e-7


@pytest.mark.parametrize("d,heads,sq,sk", [(64, 300, 256, 80), (64, 40, 300, 200), (128, 7, 300, 200)])
@pytest.mark.parametrize("values", [1.0, 2.0 ** 60, 2.0 ** 125])
def test_weights_below_the_parts(hip, d, heads, sq, sk, values):
    """The key that takes all weight has values of zero, and the others lie 60 to 87 nats lower: nothing but their weights, down to 2^-126,
    makes up the outputs. The scores are exact, so a weight carries the rounding of its exponent of at most 128 (2^-18) and of log2(e)
    (128 x 2^-26), times ln 2, and an ulp: 4e-6; a sum of one sign no more, and a few ulp of its own."""
    rng = np.random.default_rng(sk)
    q, k = np.zeros((heads, sq, d), np.float32), np.zeros((heads, sk, d), np.float32)
    q[:, :, 0] = 8.0
    top = np.linspace(61, 86.5, heads)[rng.permutation(heads)]
    k[:, :, 0] = -np.round((top[:, None] + rng.random((heads, sk)) * 0.5) * 64) / 64
    k[:, 3, 0] = 0.0
    v = ((0.5 + 0.5 * rng.random((heads, sk, d))) * values).astype(np.float32)
    v[:, 3] = 0.0
    out = _run(hip, q, k, v, False, scale=0.125)
    for h in np.argsort(top)[::max(1, heads // 12)].tolist() + [int(np.argmax(top))]:
        ref = _ref(q[h], k[h], v[h], False, 0.125)
        assert np.max(np.abs(out[h] / ref - 1)) <= 5e-6, "%.1f nats" % top[h]


@pytest.mark.parametrize("d,heads", [(64, 300), (128, 4)])
def test_scales_beyond_the_range_stay_on_fp32_units(hip, d, heads):
    q, k, v = _inputs(heads, 1, 256, 200, d)
    q *= np.float32(2.0 ** -60)
    out = _run(hip, q, k, v, True, scale=2.0 ** 57)
    assert _rel(out[0], _ref(q[0], k[0], v[0], True, 2.0 ** 57)) <= 1e-6


CHILD = """
import sys
sys.path[:0] = [%(root)r, %(root)r + "/tests"]
import numpy as np
from frankentorch_amd import device as hip
import test_gpu_sdpa_split as t
np.savez(sys.argv[1], **{str(i): t._run(hip, *t._inputs(h, 1, sq, sk, 64), causal) for i, (h, sq, sk, causal, _) in enumerate(t.SHORT)})
"""
# heads, queries, keys, causal, on bf16 units
SHORT = [(300, 64, 64, False, False), (260, 33, 33, True, False), (1024, 20, 128, True, False), (32, 300, 40, False, True), (260, 100, 64, True, False),
         (70, 250, 32, False, True), (96, 300, 40, False, True), (128, 600, 64, False, True), (300, 64, 65, False, True), (96, 65, 65, False, True)]


def test_few_keys_stay_on_fp32_units(hip, tmp_path):
    """Up to 64 keys of head size 64 and up to 128 queries run on bf16 units where all blocks run at once; the others give the bits that they give
    with that kernel switched off (a child process: the switch is read once). Error: theirs, at most
    2.5e-8 sqrt(keys) + 1.4e-7 (3.05e-7 measured for 64 keys, 1.6e-7 for 16)."""
    path = str(tmp_path / "fp32.npz")
    subprocess.run([sys.executable, "-c", CHILD % {"root": ROOT}, path], check=True, timeout=110, env=dict(os.environ, FT_HIP_SDPA_SPLIT="0"))
    fp32 = np.load(path)
    for i, (heads, sq, sk, causal, split) in enumerate(SHORT):
        q, k, v = _inputs(heads, 1, sq, sk, 64)
        out = _run(hip, q, k, v, causal)
        assert np.array_equal(out, fp32[str(i)]) != split, SHORT[i]
        for h in (0, heads - 1):
            assert _rel(out[h], _ref(q[h], k[h], v[h], causal)) <= 2.5e-8 * np.sqrt(sk) + 1.4e-7
