"""GPU: dense calls under stream capture (sili_forward_dense recorded into a
graph).  A capture records work that has not run when the call returns, so it
must leave the layer's copies of a store as they were, read nothing that is not
there, and keep what it recorded alive: column-block copies that an update made
stale, copies of another split, work-item tables that no call has built yet.
Every replay is checked, with eager calls and updates between the replays."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_capi import Api, _ptr
from tests.test_gpu_parity import _edge_block4_layer

pytestmark = pytest.mark.gpu


class Calls:
    """Forward passes of one layer on a stream of their own: eager and captured."""

    def __init__(self, hip, L, n_in, n_out, most):
        self.api, self.L, self.h = Api(hip.LIB_PATH), L, C.c_void_p(L.handle)
        self.n_in, self.n_out = n_in, n_out
        self.x, self.y, self.st = C.c_void_p(), C.c_void_p(), C.c_void_p()
        self.rt("sili_device_alloc", self.h, most * n_in * 4, C.byref(self.x))
        self.rt("sili_device_alloc", self.h, most * n_out * 4, C.byref(self.y))
        self.rt("hipStreamCreate", C.byref(self.st))
        self.graphs = []

    def rt(self, name, *args):  # (the HIP runtime that the library is linked to)
        self.api.ck(getattr(self.api.L, name)(*args))

    def forward(self, B):
        self.rt("sili_forward_dense", self.h, self.x, B, self.y, self.st)

    def capture(self, B, mode=0):
        g, run = C.c_void_p(), C.c_void_p()
        self.rt("hipStreamBeginCapture", self.st, mode)
        self.forward(B)
        self.rt("hipStreamEndCapture", self.st, C.byref(g))
        self.rt("hipGraphInstantiate", C.byref(run), g, None, None, C.c_size_t(0))
        self.graphs.append((g, run))
        return lambda: self.rt("hipGraphLaunch", run, self.st)

    def result(self, call, x):
        y = np.full((x.shape[0], self.n_out), np.nan, np.float32)
        self.rt("sili_memcpy_h2d", self.h, self.x, _ptr(x), x.nbytes)
        self.rt("sili_memcpy_h2d", self.h, self.y, _ptr(y), y.nbytes)
        call()
        self.rt("hipStreamSynchronize", self.st)
        self.rt("sili_memcpy_d2h", self.h, _ptr(y), self.y, y.nbytes)
        return y

    def close(self):
        for g, run in self.graphs:
            self.rt("hipGraphExecDestroy", run)
            self.rt("hipGraphDestroy", g)
        self.rt("hipStreamDestroy", self.st)
        for p in (self.x, self.y):
            self.rt("sili_device_free", self.h, p)


def close_to(got, want, what):
    # the fp32 bar, 1e-5 of the summed magnitudes, which are at least the largest output
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-5 * np.abs(want).max(), err_msg=what)


N_IN, N_OUT, B = 16387, 70, 136  # an operand of 8.9 MB: passes over 5 scattered and 2 block4 copies


def twins(hip):
    """Two equal layers with scattered synapses and tiles."""
    br, bc, tiles, ptrs, cols, q, vs = _edge_block4_layer(N_IN, N_OUT, 17, density=0.03)
    out = []
    for _ in range(2):
        L = hip.SparseLinearLayer(N_IN, N_OUT, 8 * len(cols) + 64 * len(br) + 4096)
        L.load_weights(ptrs, cols, q)
        L.load_block4_tiles(br, bc, tiles)
        L.set_value_scales(vs)
        L.get_value_scales()  # the binding hands pending setters on
        out.append(L)
    return out


def test_captured_forward_around_updates(hip, monkeypatch):
    L, plain = twins(hip)
    rng = np.random.default_rng(5)
    calls = Calls(hip, L, N_IN, N_OUT, B)

    def inputs():
        return rng.normal(size=(B, N_IN)).astype(np.float32)

    def want(x):
        monkeypatch.setenv("SILI_COLBLOCK", "0")
        y = plain.forward_dense(x)
        monkeypatch.delenv("SILI_COLBLOCK")
        return y

    def update():
        x, g = inputs(), rng.normal(size=(B, N_OUT)).astype(np.float32)
        before = want(x)
        for layer in (L, plain):
            layer.forward_dense(x)
            layer.backward_dense(g, 0.05)
        assert np.abs(want(x) - before).max() > 1e-3 * np.abs(before).max()  # the update shows

    def check(call, what):
        x = inputs()
        close_to(calls.result(call, x), want(x), what)

    eager = lambda: calls.forward(B)
    update()
    update()  # by now the copies know their places
    first = calls.capture(B)  # the copies are stale
    check(eager, "eager after a capture that followed an update")
    check(first, "replay")
    update()
    check(first, "replay after an update")
    check(eager, "eager after an update")
    second = calls.capture(B)  # the copies hold the store's values
    for turn in range(3):
        check(second, f"replay {turn}")
        check(eager, f"eager {turn}")
        update()
        check(second, f"replay after update {turn}")
        check(first, f"first graph after update {turn}")
    calls.close()


def test_captured_copies_outlive_another_split(hip):
    """Copies in 5 blocks, recorded; then a batch that takes 3; then the graph."""
    L, _ = twins(hip)
    rng = np.random.default_rng(6)
    calls = Calls(hip, L, N_IN, N_OUT, B)
    x = rng.normal(size=(B, N_IN)).astype(np.float32)
    want = calls.result(lambda: calls.forward(B), x)
    replay = calls.capture(B)
    for other in (72, 101):
        small = rng.normal(size=(other, N_IN)).astype(np.float32)
        calls.result(lambda: calls.forward(other), small)
        close_to(calls.result(replay, x), want, f"replay after batch {other}")
    calls.close()


@pytest.mark.parametrize("cold", [37, 72, 101])
def test_capture_of_a_batch_that_never_ran(hip, cold):
    """Only the workspaces are there: neither the copies of this batch's split
    nor the short rows' table may be built."""
    L, plain = twins(hip)
    rng = np.random.default_rng(7)
    calls = Calls(hip, L, N_IN, N_OUT, B)
    calls.result(lambda: calls.forward(B), rng.normal(size=(B, N_IN)).astype(np.float32))
    x = rng.normal(size=(cold, N_IN)).astype(np.float32)
    replay = calls.capture(cold)
    want = plain.forward_dense(x)
    close_to(calls.result(replay, x), want, "replay")
    close_to(calls.result(lambda: calls.forward(cold), x), want, "eager")
    close_to(calls.result(replay, x), want, "replay")
    calls.close()


def test_relaxed_capture_builds_a_stream_copy(hip, monkeypatch):
    """A relaxed capture (mode 2) may allocate and wait on other streams: the
    stream copy of batch 8 is built beside it, on the layer's stream."""
    L, plain = twins(hip)
    rng = np.random.default_rng(9)
    calls = Calls(hip, L, N_IN, N_OUT, B)
    calls.result(lambda: calls.forward(B), rng.normal(size=(B, N_IN)).astype(np.float32))
    x = rng.normal(size=(8, N_IN)).astype(np.float32)
    want = plain.forward_dense(x)
    monkeypatch.setenv("SILI_B1_STREAM", "2")
    replay = calls.capture(8, 2)
    assert L.info()["stream_shadow"] == 1
    for _ in range(3):
        close_to(calls.result(replay, x), want, "replay")
        close_to(calls.result(lambda: calls.forward(8), x), want, "eager")
    calls.close()


def test_capture_before_the_short_rows_are_split(hip):
    n_in, n_out = 300, 6000
    rng = np.random.default_rng(8)
    keep = rng.random((n_in, n_out)) < 0.02
    ptrs = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    cols = np.nonzero(keep)[1].astype(np.int32)
    L = hip.SparseLinearLayer(n_in, n_out, len(cols))
    L.load_weights(ptrs, cols, rng.normal(size=len(cols)).astype(np.float32))
    calls = Calls(hip, L, n_in, n_out, 128)
    calls.result(lambda: calls.forward(128), rng.normal(size=(128, n_in)).astype(np.float32))
    x = rng.normal(size=(37, n_in)).astype(np.float32)
    replay = calls.capture(37)
    assert L.info()["short_rows_shadow"] == 0
    want = calls.result(lambda: calls.forward(37), x)
    assert L.info()["short_rows_shadow"] >= 1024  # the case is one of those
    close_to(calls.result(replay, x), want, "replay")
    calls.close()
