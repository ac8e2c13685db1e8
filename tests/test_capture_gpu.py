"""Projections captured into a HIP graph through the context's public compute stream
(h3_hip_compute_stream): a graph must not hold a workspace of the context, which later
calls use and, growing it, free."""
import ctypes as C
import math

import numpy as np
import pytest

from h3cli_amd import synth
from h3cli_amd.runtime import Gpu
from tests.helpers import bf16
from tests.test_block_gpu import q8_weight, synthetic_q8

pytestmark = pytest.mark.gpu


class Graph:
    """What the calls inside `with` launch on the context's stream, captured."""

    def __init__(self, gpu):
        self.hip = C.CDLL("libamdhip64.so.7")
        self.stream = C.c_void_p(gpu.lib.h3_hip_compute_stream(gpu.handle))
        self.graph, self.exec = C.c_void_p(), C.c_void_p()

    def call(self, name, *args):
        status = getattr(self.hip, name)(*args)
        assert status == 0, (name, status)

    def __enter__(self):
        self.call("hipStreamBeginCapture", self.stream, 1)   # thread-local
        return self

    def __exit__(self, *exc):
        self.call("hipStreamEndCapture", self.stream, C.byref(self.graph))
        if not exc[0]:
            self.call("hipGraphInstantiate", C.byref(self.exec), self.graph, None, None, C.c_size_t(0))

    def launch(self):
        self.call("hipGraphLaunch", self.exec, self.stream)

    def close(self):
        if self.exec:
            self.call("hipGraphExecDestroy", self.exec)
        self.call("hipGraphDestroy", self.graph)


@pytest.mark.parametrize("m,k,n,group,eager", [
    (300, 4096, 512, 0, "shares="),          # BF16, split over K
    (300, 4096, 512, 4096, "shares="),       # W8A16 per channel
    (300, 4096, 512, 64, "shares="),
    (3300, 1024, 5120, 64, "converted"),     # W8A16, the weight converted first
])
def test_captured_projection_holds_no_workspace(m, k, n, group, eager):
    print(f"[capture] m={m} k={k} n={n} group={group}", flush=True)
    with Gpu() as g:
        x = synth.normal_bf16(m, m * k)
        if group:
            codes, scales = synthetic_q8(m + n, n, k, group)
            w = q8_weight(g, codes, scales, n, k, group)
            wide = np.repeat(scales.reshape(n, -1), group, axis=1)[:, :k]
            wv = bf16(synth.f32_to_bf16(codes.reshape(n, k).astype(np.float32) * wide))
        else:
            bits = synth.normal_bf16(m + 1, n * k, scale=1 / math.sqrt(k))
            w, wv = g.from_bf16(bits), bf16(bits).reshape(n, k)
        tx, out, other = g.from_bf16(x), g.empty(m * n), g.empty(m * n)
        # A larger projection, which needs more of every workspace.
        big = [g.empty(1100 * 8192), g.empty(1100 * 5120)]
        codes, scales = synthetic_q8(1, 5120, 8192, 64)
        big_q8, big_bf16 = q8_weight(g, codes, scales, 5120, 8192, 64), g.empty(5120 * 8192)

        def linear(dst, src, weight, *shape):
            g.check(g.lib.h3_gpu_linear_bf16(g.handle, dst.handle, src.handle, weight.handle, None, *shape), "linear")

        g.begin()
        linear(other, tx, w, m, k, n)      # warm: the workspaces are there and large enough
        assert eager in g.last_kernel(), g.last_kernel()
        g.submit()
        graph = Graph(g)
        g.begin()
        with graph:
            linear(out, tx, w, m, k, n)
            captured = g.last_kernel()
        assert "shares=" not in captured and "converted" not in captured, captured
        rows = np.unique(np.r_[0:m:37, m - 1])
        xv = bf16(x).reshape(m, k)[rows].astype(np.float64)
        want = xv @ wv.T.astype(np.float64)
        bound = 2.0 ** -8 * np.abs(want) + k * 2.0 ** -24 * (np.abs(xv) @ np.abs(wv).T)
        first = None
        for _ in range(3):
            for t in big + [big_bf16]:
                g.check(g.lib.h3_hip_fill_normal_bf16(g.handle, t.handle, 3, C.c_float(1.0), t.elements), "fill")
            linear(big[1], big[0], big_bf16, 1100, 8192, 5120)
            linear(big[1], big[0], big_q8, 1100, 8192, 5120)
            g.check(g.lib.h3_hip_fill_normal_bf16(g.handle, out.handle, 4, C.c_float(1.0), m * n), "fill")
            graph.launch()
            g.submit()
            got = out.read()
            assert np.all(np.abs(bf16(got).reshape(m, n)[rows] - want) <= bound)
            first = got if first is None else first
            assert np.array_equal(got, first)
            g.begin()
        g.submit()
        graph.close()


def test_mlp_is_refused_while_capturing():
    """Its intermediates need memory; the refusal leaves the capture and the context whole."""
    m, k, hidden, n = 300, 512, 384, 256
    with Gpu() as g:
        tx, w1, w2 = (g.from_bf16(synth.normal_bf16(i, c, scale=0.05))
                      for i, c in ((1, m * k), (2, 2 * hidden * k), (3, n * hidden)))
        out = g.empty(m * n)
        args = (g.handle, out.handle, tx.handle, w1.handle, w2.handle, m, k, hidden, n)
        g.begin()
        g.check(g.lib.h3_gpu_mlp_bf16(*args), "mlp")
        g.submit()
        want = out.read()
        graph = Graph(g)
        g.begin()
        with graph:
            assert not g.lib.h3_gpu_mlp_bf16(*args)
            assert "captured" in g.error()
        graph.close()
        g.cancel()
        g.begin()
        g.check(g.lib.h3_gpu_mlp_bf16(*args), "mlp")
        g.submit()
        assert np.array_equal(out.read(), want)
