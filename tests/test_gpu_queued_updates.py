"""GPU: copies of a store's values that a call builds on the layer's own stream
while optimizer steps are still queued on the caller's: the call comes after
those steps on its stream, so it has to multiply by their result."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_capi import Api, _ptr
from tests.test_gpu_stream import kernel_counts

pytestmark = pytest.mark.gpu

N, STEPS, TRAIN_B = 8192, 60, 136  # (a workspace that has to grow waits for everything)


# (batch, the gather it takes): a stream copy; a stream copy in column blocks or
# passes; column-block copies (an operand of 4.4 MB)
@pytest.mark.parametrize("B,scope", [(1, "stream"), (8, "stream"), (136, "gather")])
def test_copy_waits_for_queued_updates(hip, monkeypatch, B, scope):
    monkeypatch.setenv("SILI_MFMA24", "0")
    rng = np.random.default_rng(B)
    keep = rng.random((N, N)) < 0.02
    ptrs = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    cols = np.nonzero(keep)[1].astype(np.int32)
    w = rng.normal(size=len(cols)).astype(np.float32)
    x, g = rng.normal(size=(136, N)).astype(np.float32), rng.normal(size=(136, N)).astype(np.float32)
    api = Api(hip.LIB_PATH)
    rt = lambda name, *args: api.ck(getattr(api.L, name)(*args))
    got = []
    for wait in (True, False):
        L = hip.SparseLinearLayer(N, N, len(cols))
        L.load_weights(ptrs, cols, w)
        h, st = C.c_void_p(L.handle), C.c_void_p()
        rt("hipStreamCreate", C.byref(st))
        dev = {}
        for k, n in (("x", x.size), ("g", g.size), ("y", x.size), ("dx", x.size)):
            dev[k] = C.c_void_p()
            rt("sili_device_alloc", h, 4 * n, C.byref(dev[k]))
        rt("sili_memcpy_h2d", h, dev["x"], _ptr(x), x.nbytes)
        rt("sili_memcpy_h2d", h, dev["g"], _ptr(g), g.nbytes)

        def update():
            rt("sili_backward_dense", h, dev["x"], dev["g"], TRAIN_B, dev["dx"], None, None, 0.05, st)

        def forward():
            rt("sili_forward_dense", h, dev["x"], B, dev["y"], st)

        update()  # its set-up waits
        rt("hipStreamSynchronize", st)
        for _ in range(STEPS):
            update()
        if wait:
            rt("hipStreamSynchronize", st)
        forward()
        rt("hipStreamSynchronize", st)
        y = np.empty((B, N), np.float32)
        rt("sili_memcpy_d2h", h, _ptr(y), dev["y"], y.nbytes)
        counts = kernel_counts(hip, L, forward)
        assert any(k.startswith("fwd:" + scope) for k in counts), counts
        got.append((y, L.export_scattered()["val"]))
        for p in dev.values():
            rt("sili_device_free", h, p)
        rt("hipStreamDestroy", st)
    (want, codes), (y, codes2) = got
    assert np.array_equal(codes, codes2)
    # the fp32 bar, 1e-5 of the summed magnitudes, which are at least the largest output
    np.testing.assert_allclose(y, want, rtol=0, atol=1e-5 * np.abs(want).max())
