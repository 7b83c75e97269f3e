"""Scratch memory of the split product and of few-query attention: a captured graph owns its own, whatever else runs meanwhile;
a call that gets none falls back to the kernels that need none."""
import ctypes as C
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from conftest import ROOT, TOL_GEMM_F32, rel_err
from frankentorch_amd import _lib, fused, synth
from frankentorch_amd.device import DeviceBuffer, Stream

pytestmark = pytest.mark.gpu


class Hip:
    """The runtime's capture calls, through the library that links against it."""

    def __getattr__(self, name):
        def call(*a):
            rc = getattr(_lib.load(), name)(*a)
            assert rc == 0, (name, rc)
        return call


rt = Hip()


class Graph:
    def __init__(self, stream, launch):
        graph, self.exec = C.c_void_p(), C.c_void_p()
        rt.hipStreamBeginCapture(C.c_void_p(stream.handle), 1)  # thread-local mode
        launch(stream.handle)
        rt.hipStreamEndCapture(C.c_void_p(stream.handle), C.byref(graph))
        rt.hipGraphInstantiate(C.byref(self.exec), graph, None, None, C.c_size_t(0))
        rt.hipGraphDestroy(graph)

    def replay(self, stream):
        rt.hipGraphLaunch(self.exec, C.c_void_p(stream.handle))

    def free(self):
        rt.hipGraphExecDestroy(self.exec)


class Decode:
    """Eight query heads on two K/V heads, one new token, 1500 keys: several shares of the keys."""

    def __init__(self, hip, seed, sk=1500):
        self.q, self.k, self.v = (DeviceBuffer.from_host(synth.normal(seed, n, s)) for n, s in (("q", (2, 8, 1, 64)), ("k", (2, 2, sk, 64)), ("v", (2, 2, sk, 64))))
        self.out, self.hip = DeviceBuffer((2, 8, 1, 64)), hip
        self.desc = hip.sdpa_desc_gqa(2, 8, 2, 1, sk, 64, 64, False)

    def launch(self, stream):
        self.hip.sdpa_forward(self.desc, 0.125, self.q, self.k, self.v, self.out, stream)


class Product:
    def __init__(self, hip, seed, m=2048, n=2304, k=768):
        self.a, self.b = (DeviceBuffer.from_host(synth.normal(seed, n_, s)) for n_, s in (("a", (m, k)), ("b", (n, k))))
        self.out, self.hip = DeviceBuffer((m, n)), hip
        self.desc = hip.gemm_desc(m, n, k, trans_b=True)

    def launch(self, stream):
        self.hip.gemm(self.desc, self.a, self.b, self.out, stream=stream)


def _eager(hip, op, stream):
    op.launch(stream.handle)
    stream.synchronize()
    return op.out.to_host().view(np.uint32)


@pytest.mark.parametrize("kind", [Decode, Product])
def test_graphs_of_one_capture_stream_replay_beside_each_other(hip, kind):
    """Two graphs captured on one warm stream, replayed on two others while the capture stream runs the same calls eagerly on
    other operands: every result has the bits of the same call alone."""
    home, side = Stream(), (Stream(), Stream())
    ops, third = [kind(hip, 70 + i) for i in range(2)], kind(hip, 79)
    want, want3 = [_eager(hip, op, home) for op in ops], _eager(hip, third, home)
    held = [hip.gemm_workspace_info()[0]]
    graphs = []
    for op in ops:
        graphs.append(Graph(home, op.launch))
        held.append(hip.gemm_workspace_info()[0])
    assert held[0] < held[1] < held[2]  # a block of its own each
    for _ in range(4):
        for _ in range(5):
            for g, s in zip(graphs, side):
                g.replay(s)
            third.launch(home.handle)
        hip.synchronize()
        for op, w in zip(ops, want):
            assert np.array_equal(op.out.to_host().view(np.uint32), w)
        assert np.array_equal(third.out.to_host().view(np.uint32), want3)
        _eager(hip, third, side[0])  # and eager work between the replays
    for g in graphs:
        g.free()
    assert hip.gemm_workspace_info()[0] >= held[2]  # what a caller's graph was given stays


def test_threads_on_one_stream(hip):
    """Calls of several threads on one stream share its block: no thread's kernels come between another's two launches."""
    s = Stream()
    ops = [kind(hip, 90 + i) for i in range(2) for kind in (Product, Decode)]
    want = [_eager(hip, op, s) for op in ops]
    failed = []

    def work(op):
        try:
            for _ in range(25):
                op.launch(s.handle)
        except Exception as e:  # noqa: BLE001 - reported below
            failed.append(e)

    for _ in range(3):
        threads = [threading.Thread(target=work, args=(op,)) for op in ops]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        s.synchronize()
        assert not failed
        for op, w in zip(ops, want):
            assert np.array_equal(op.out.to_host().view(np.uint32), w)


def test_a_capture_without_a_warm_stream_gives_the_same_bits(hip):
    op, s = Product(hip, 75), Stream()
    want = _eager(hip, op, Stream())
    g = Graph(s, op.launch)
    for _ in range(3):
        g.replay(s)
        hip.synchronize()
        assert np.array_equal(op.out.to_host().view(np.uint32), want)
        _eager(hip, op, s)
    g.free()


def test_a_larger_product_beside_a_live_graph(hip):
    """The stream's own block is outgrown and replaced; the graph does not notice, and tensors made afterwards are not written."""
    s, op = Stream(), Product(hip, 76)
    want = _eager(hip, op, s)
    g = Graph(s, op.launch)
    ret0 = hip.gemm_workspace_info()[1]
    big = Product(hip, 77, m=4097, n=3077, k=1001)
    _eager(hip, big, s)
    assert hip.gemm_workspace_info()[1] > ret0
    canaries = [DeviceBuffer.from_host(np.full((rows, 1024), 7.0, np.float32)) for rows in (4096, 8192, 16384, 32768)]
    for _ in range(3):
        g.replay(s)
        hip.synchronize()
        assert np.array_equal(op.out.to_host().view(np.uint32), want)
        _eager(hip, big, s)
    for t in canaries:
        assert np.all(t.to_host() == 7.0)
    g.free()


def test_an_encoder_gives_its_graph_scratch_back(hip):
    batch, seq, d, f = 2, 1024, 512, 2048
    rng = np.random.default_rng(3)
    w = lambda *s: (rng.standard_normal(s) * 0.02).astype(np.float32)
    layer = dict(ln1_w=np.ones(d, np.float32), ln1_b=w(d), wq=w(d, d), bq=w(d), wk=w(d, d), bk=w(d), wv=w(d, d), bv=w(d), wo=w(d, d), bo=w(d),
                 ln2_w=np.ones(d, np.float32), ln2_b=w(d), w1=w(f, d), b1=w(f), w2=w(d, f), b2=w(d))
    enc = fused.EncoderHip(d, 8, f, [layer], 1e-5, causal=True)
    x, out = DeviceBuffer.from_host(w(batch * seq, d)), DeviceBuffer((batch * seq, d))
    enc.forward_dev(x, out, batch, seq)
    want, before = out.to_host(), hip.gemm_workspace_info()
    for _ in range(3):
        enc.forward_dev(x, out, batch, seq, graph=True)
        assert np.array_equal(out.to_host(), want)
    assert hip.gemm_workspace_info()[0] > before[0]
    del enc
    assert hip.gemm_workspace_info() == before


def test_the_per_thread_stream_is_given_none(hip):
    """hipStreamPerThread is one handle for a different stream in every thread: no block may be kept under it."""
    per_thread = C.c_void_p(2)
    before = hip.gemm_workspace_info()[0]
    for op in (Decode(hip, 80), Product(hip, 81, m=2048, n=2048)):
        want = _eager(hip, op, Stream())
        mid = hip.gemm_workspace_info()[0]
        op.launch(per_thread.value)
        hip.synchronize()
        assert rel_err(op.out.to_host(), want.view(np.float32)) <= TOL_GEMM_F32
        # (the fp32 product may take split-tile accumulators, 128 x 128 floats twice a workgroup)
        assert hip.gemm_workspace_info()[0] - mid <= 512 * 2 * 128 * 128 * 4
    assert hip.gemm_workspace_info()[0] >= before


def test_trim_gives_the_streams_blocks_back(hip):
    s, op = Stream(), Product(hip, 82, m=4096, n=4096, k=1024)
    want = _eager(hip, op, s)
    live, _ = hip.gemm_workspace_info()
    assert _lib.load().fth_pool_trim() == 0
    after, retired = hip.gemm_workspace_info()
    assert after <= live - 2 * 6 * 4096 * 1024
    assert np.array_equal(_eager(hip, op, s), want)


def test_a_refused_allocation_leaves_no_error_behind(hip):
    t = C.c_void_p()
    assert _lib.load().fth_tensor_alloc(C.c_int64(1 << 30), C.c_int64(1 << 20), C.byref(t)) != 0
    x = DeviceBuffer.from_host(np.ones(1000, np.float32))
    hip.add(x, x, x, 1000)  # its launch check would report the refusal
    assert np.all(x.to_host() == 2.0)


CHILD = """
import sys
sys.path[:0] = [%(root)r, %(root)r + "/tests"]
import numpy as np
from frankentorch_amd import device as hip
import test_gpu_stream_scratch as t
s = t.Stream()
np.savez(sys.argv[1], *[t._eager(hip, op, s) for op in (t.Decode(hip, 70), t.Product(hip, 70)) for _ in range(2)], live=hip.gemm_workspace_info()[0])
"""


@pytest.mark.parametrize("knob", ["0", "2"])
def test_without_scratch_the_other_kernels_answer(hip, tmp_path, knob):
    """FT_HIP_STREAM_SCRATCH: 0 gives none, 2 lets the driver refuse every allocation."""
    path = str(tmp_path / "out.npz")
    subprocess.run([sys.executable, "-c", CHILD % {"root": ROOT}, path], check=True, timeout=100, env=dict(os.environ, FT_HIP_STREAM_SCRATCH=knob))
    got = np.load(path)
    s = Stream()
    for i, op in enumerate((Decode(hip, 70), Product(hip, 70))):
        want = _eager(hip, op, s).view(np.float32)
        assert np.array_equal(got["arr_%d" % (2 * i)], got["arr_%d" % (2 * i + 1)])
        assert rel_err(got["arr_%d" % (2 * i)].view(np.float32), want) <= TOL_GEMM_F32
    assert got["live"] <= 512 * 2 * 128 * 128 * 4


CAPTURE_CHILD = """
import sys
sys.path[:0] = [%(root)r, %(root)r + "/tests"]
import numpy as np
from frankentorch_amd import device as hip
import test_gpu_stream_scratch as t
out = {}
for name, kind in (("decode", t.Decode), ("product", t.Product)):
    op, s = kind(hip, 70), t.Stream()
    out[name + "_eager"] = t._eager(hip, op, s)
    g = t.Graph(s, op.launch)
    for i in range(3):
        g.replay(s)
        s.synchronize()
        out[name + "_%%d" %% i] = op.out.to_host()
        t._eager(hip, op, s)
np.savez(sys.argv[1], **out)
"""


def test_a_capture_that_is_given_none(hip, tmp_path):
    """FT_HIP_STREAM_SCRATCH=3: eager calls have their scratch, the capture does not and records the other kernels, whose own
    workspace no eager call has sized."""
    path = str(tmp_path / "out.npz")
    subprocess.run([sys.executable, "-c", CAPTURE_CHILD % {"root": ROOT}, path], check=True, timeout=100, env=dict(os.environ, FT_HIP_STREAM_SCRATCH="3"))
    got = np.load(path)
    for name, kind in (("decode", Decode), ("product", Product)):
        want = _eager(hip, kind(hip, 70), Stream())
        assert np.array_equal(got[name + "_eager"], want)
        for i in range(3):
            assert rel_err(got["%s_%d" % (name, i)], want.view(np.float32)) <= TOL_GEMM_F32
            assert np.array_equal(got["%s_%d" % (name, i)], got[name + "_0"])
        assert not np.array_equal(got[name + "_0"].view(np.uint32), want)  # other kernels, other rounding
