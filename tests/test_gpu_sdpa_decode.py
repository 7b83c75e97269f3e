"""Attention of a few new tokens against a K/V cache (the key-split kernel): edges of the 32-key tiles and of the shares, row
counts around the 16- and 32-row tiles, grouped heads, masks of every alignment. Against the CPU checker, fp32 <= 2e-5."""
import math

import numpy as np
import pytest

from conftest import TOL_GEMM_F32, rel_err
from frankentorch_amd import synth
from frankentorch_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu

# (batch, h_q, h_kv, seq_q, seq_k, d)
SHAPES = [(1, 1, 1, 1, 1, 64), (2, 4, 4, 1, 31, 32), (1, 8, 2, 4, 32, 64), (1, 8, 2, 4, 33, 128), (2, 17, 1, 1, 64, 32), (1, 8, 1, 4, 65, 64),
          (1, 6, 2, 8, 130, 128), (1, 33, 1, 1, 97, 64), (3, 32, 8, 1, 397, 128), (1, 4, 1, 8, 1027, 64), (1, 8, 8, 2, 4099, 128), (1, 9, 1, 8, 200, 32),
          # more than 16 rows on a K/V head and more than 2048 keys: tiles of 32 rows; more heads than 128, either side of that line
          (1, 32, 1, 1, 2500, 32), (1, 17, 1, 2, 2049, 128), (1, 24, 1, 3, 3000, 64), (1, 24, 1, 3, 2048, 64), (5, 32, 8, 5, 500, 64), (5, 32, 32, 8, 513, 64)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("mask_kind", ["none", "shared", "per_head"])
def test_few_queries_against_a_cache(hip, oracle, shape, mask_kind):
    batch, hq, hkv, sq, sk, d = shape
    q, k, v = (synth.normal(51, t, s) for t, s in (("q", (batch, hq, sq, d)), ("k", (batch, hkv, sk, d)), ("v", (batch, hkv, sk, d))))
    scale = np.float32(1.0 / math.sqrt(d))
    mask = np.zeros((sq, sk), np.float32)
    if mask_kind != "none":
        mshape = (sq, sk) if mask_kind == "shared" else (batch * hq, sq, sk)
        mask = synth.normal(51, "mask", mshape, 0.0, 0.5)
        mask[synth.uniform(51, "hide", mshape) < 0.3] = -np.inf
        mask[..., : sk // 2] = -np.inf  # whole shares without a visible key
        mask[..., sk - 1] = 0.25
        if sk > 40:
            mask[..., 0, :] = -np.inf   # a row with nothing visible is NaN

    def run(kk, vv, heads_kv):
        bufs = [DeviceBuffer.from_host(t) for t in (q, kk, vv, mask)]
        out = DeviceBuffer.from_host(np.full(q.shape, 7.0, np.float32))
        desc = hip.sdpa_desc_gqa(batch, hq, heads_kv, sq, sk, d, d, False)
        if mask_kind == "none":
            hip.sdpa_forward(desc, scale, bufs[0], bufs[1], bufs[2], out)
        else:
            hip.sdpa_forward_masked(desc, scale, bufs[0], bufs[1], bufs[2], bufs[3], 0 if mask.ndim == 2 else sq * sk, out)
        return out.to_host()

    got, ref = run(k, v, hkv), oracle.sdpa_forward_masked_gqa(q, k, v, scale, mask)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    if ok.any():
        assert rel_err(got[ok], ref[ok]) <= TOL_GEMM_F32
    expanded = run(np.repeat(k, hq // hkv, axis=1), np.repeat(v, hq // hkv, axis=1), hq)
    assert np.array_equal(got.view(np.uint32), expanded.view(np.uint32))


def _strided(hip, batch, hq, hkv, sq, sk, d, q, k, v, scale, mask=None, dtype=np.float32):
    """q, k, v are (buffer, batch stride, head stride, row stride, offset) in elements; the output is contiguous."""
    from frankentorch_amd import _lib
    a = _lib.SdpaDesc()
    a.num_bh, a.heads, a.seq_q, a.seq_k, a.d_k, a.d_v = batch * hq, hq, sq, sk, d, d
    for n, t in (("q", q), ("k", k), ("v", v)):
        for f, x in zip(("batch", "head", "row"), t[1:4]):
            setattr(a, "%s_%s_stride" % (n, f), x)
    a.o_batch_stride, a.o_head_stride, a.o_row_stride = hq * sq * d, sq * d, d
    a.causal, a.kv_group = 0, hq // hkv if hq != hkv else 0
    out = DeviceBuffer.from_host(np.full((batch, hq, sq, d), 7.0, dtype))
    ptrs = [t[0].view(t[4]) for t in (q, k, v)]
    if mask is None:
        hip.sdpa_forward(a, scale, *ptrs, out)
    else:
        hip.sdpa_forward_masked(a, scale, *ptrs, DeviceBuffer.from_host(mask), 0, out)
    return out.to_host()


@pytest.mark.parametrize("sk", [1, 70, 300])
@pytest.mark.parametrize("reverse", [False, True])
def test_caches_as_they_lie_in_memory(hip, oracle, sk, reverse):
    """Caches stored [batch, key, head, d] with room for more keys, read forwards and from the last key back (negative row
    strides), beside NaN in everything that is not part of the problem."""
    batch, hq, hkv, sq, d, room, pad = 2, 8, 4, 2, 64, 13, 8
    q, k, v = (synth.normal(52, t, s) for t, s in (("q", (batch, hq, sq, d)), ("k", (batch, hkv, sk, d)), ("v", (batch, hkv, sk, d))))
    row, bat = hkv * (d + pad), (sk + room) * hkv * (d + pad)
    views = []
    for t in (k, v):
        store = np.full((batch, sk + room, hkv, d + pad), np.nan, np.float32)
        store[:, :sk, :, :d] = t.transpose(0, 2, 1, 3)[:, ::-1] if reverse else t.transpose(0, 2, 1, 3)
        views.append((DeviceBuffer.from_host(store), bat, d + pad, -row if reverse else row, (sk - 1) * row if reverse else 0))
    qs = np.full((batch, sq, hq, d + 4), np.nan, np.float32)
    qs[..., :d] = q.transpose(0, 2, 1, 3)
    qv = (DeviceBuffer.from_host(qs), sq * hq * (d + 4), d + 4, hq * (d + 4), 0)
    got = _strided(hip, batch, hq, hkv, sq, sk, d, qv, *views, np.float32(0.125))
    ref = oracle.sdpa_forward_masked_gqa(q, k, v, np.float32(0.125), np.zeros((sq, sk), np.float32))
    assert rel_err(got, ref) <= TOL_GEMM_F32


@pytest.mark.parametrize("sk", [1, 31, 33, 64, 300, 1030])
@pytest.mark.parametrize("d,masked", [(128, False), (128, True), (64, True), (32, True)])
def test_non_finite_values_at_the_last_key(hip, oracle, sk, d, masked):
    """The last K/V row also stands in for the keys past it in its 32-key tile: an infinite value there is infinite in the output
    (its weight is positive), not NaN; a NaN key is NaN everywhere; scales of either sign and zero."""
    batch, hq, hkv, sq = 1, 4, 2, 2
    for scale in (0.125, 0.0, -0.125):
        for what in ("value", "key"):
            q, k, v = (synth.normal(54, t, s) for t, s in (("q", (batch, hq, sq, d)), ("k", (batch, hkv, sk, d)), ("v", (batch, hkv, sk, d))))
            if what == "value":
                v[0, 0, -1, 3], v[0, 1, -1, 5] = np.inf, -np.inf
            else:
                k[0, 0, -1, 7] = np.nan
            views = [(DeviceBuffer.from_host(t), hkv * sk * d, sk * d, d, 0) for t in (k, v)]
            mask = synth.normal(54, "m", (sq, sk), 0.0, 0.5) if masked else None
            got = _strided(hip, batch, hq, hkv, sq, sk, d, (DeviceBuffer.from_host(q), hq * sq * d, sq * d, d, 0), *views, np.float32(scale), mask)
            ref = oracle.sdpa_forward_masked_gqa(q, k, v, np.float32(scale), mask if masked else np.zeros((sq, sk), np.float32))
            fine = np.isfinite(ref)
            assert np.array_equal(got[~fine], ref[~fine], equal_nan=True), (scale, what)
            if fine.any():
                assert rel_err(got[fine], ref[fine]) <= TOL_GEMM_F32


@pytest.mark.parametrize("sq,d,masked,dtype", [(2, 64, True, np.float32), (70, 128, False, np.float32), (70, 64, True, np.float32), (70, 64, False, np.float64)])
def test_a_cache_read_backwards_on_the_other_kernels(hip, oracle, sq, d, masked, dtype):
    """Negative row strides where the tiled kernels' unsigned lane offsets cannot go: the general kernel answers."""
    batch, hq, hkv, sk = 1, 4, 2, 77
    q, k, v = (synth.normal(53, t, s, dtype=dtype) for t, s in (("q", (batch, hq, sq, d)), ("k", (batch, hkv, sk, d)), ("v", (batch, hkv, sk, d))))
    views = [(DeviceBuffer.from_host(np.ascontiguousarray(t[:, :, ::-1])), hkv * sk * d, sk * d, -d, (sk - 1) * d) for t in (k, v)]
    mask = synth.normal(53, "m", (sq, sk), 0.0, 0.5, dtype=dtype) if masked else None
    got = _strided(hip, batch, hq, hkv, sq, sk, d, (DeviceBuffer.from_host(q), hq * sq * d, sq * d, d, 0), *views, dtype(0.125), mask, dtype)
    ref = oracle.sdpa_forward_masked_gqa(q, k, v, dtype(0.125), mask if masked else np.zeros((sq, sk), dtype))
    assert rel_err(got, ref) <= (TOL_GEMM_F32 if dtype == np.float32 else 1e-12)
