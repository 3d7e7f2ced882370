"""GPU: batches that are no multiple of 4 in the float4 kernels (the dense
gathers, the fused grad-input + grad-W, the block4 gather and grad-W, the
column-block passes, the sparse-input paths), whose last chunk of batch columns
reads on into the next feature's row: every remainder, at the chunk sizes'
edges, against the oracle, with infinities and NaN in single features that must
not reach their neighbours' results."""
import ctypes as C

import numpy as np
import pytest

from oracle import HostLayer
from tests.test_gpu_capi import Api, _ptr
from tests.test_gpu_parity import _edge_block4_layer
from tests.util import assert_close_terms

pytestmark = pytest.mark.gpu

BATCHES = [2, 3, 5, 7, 9, 17, 33, 37, 63, 65, 127, 129, 255, 511, 515]


@pytest.fixture(scope="module")
def layers(hip):
    out = {}
    # mixed stores with edge tiles; a wide one (column-block passes from batch 64 on)
    for n_in, n_out, density in ((61, 83, 0.3), (16387, 70, 0.03)):
        br, bc, tiles, ptrs, cols, q, vs = _edge_block4_layer(n_in, n_out, 17, density=density)
        H = HostLayer(n_in, n_out).load_csr(ptrs, cols, w=q).load_tiles(br, bc, tiles).set_scales(vs)
        L = hip.SparseLinearLayer(n_in, n_out, len(cols) + 16 * len(br) + 64)
        L.load_weights(ptrs, cols, q)
        L.load_block4_tiles(br, bc, tiles)
        L.set_value_scales(vs)
        L.get_value_scales()  # the binding hands pending setters on
        out[n_in] = (H, L)
    return out


def step(hip, L, H, x, g):
    """y, dx, gw of one forward and backward through the C entry points."""
    api = Api(hip.LIB_PATH)
    h, B = C.c_void_p(L.handle), x.shape[0]
    sizes = dict(x=x.size, g=g.size, y=g.size, dx=x.size, gs=int(H.row_elem_start[-1]), gb=16 * H.n_tiles)
    dev = {}
    for k, n in sizes.items():
        dev[k] = C.c_void_p()
        api.ck(api.L.sili_device_alloc(h, 4 * n, C.byref(dev[k])))
    got = {k: np.zeros(n, np.float32) for k, n in sizes.items()}
    try:
        api.ck(api.L.sili_memcpy_h2d(h, dev["x"], _ptr(x), x.nbytes))
        api.ck(api.L.sili_memcpy_h2d(h, dev["g"], _ptr(g), g.nbytes))
        st = api.L.sili_stream(h)
        api.ck(api.L.sili_forward_dense(h, dev["x"], B, dev["y"], st))
        api.ck(api.L.sili_backward_dense(h, None, dev["g"], B, dev["dx"], dev["gs"], dev["gb"], 0.0, st))
        api.ck(api.L.sili_synchronize(h))
        for k in got:
            api.ck(api.L.sili_memcpy_d2h(h, _ptr(got[k]), dev[k], got[k].nbytes))
    finally:
        for p in dev.values():
            api.ck(api.L.sili_device_free(h, p))
    return got["y"].reshape(B, -1), got["dx"].reshape(B, -1), got["gs"], got["gb"]


@pytest.mark.parametrize("finite", [True, False])
@pytest.mark.parametrize("B", BATCHES)
def test_odd_batch_step_matches_oracle(hip, layers, B, finite):
    rng = np.random.default_rng(B)
    for n_in, (H, L) in layers.items():
        x = rng.normal(size=(B, n_in)).astype(np.float32)
        g = rng.normal(size=(B, H.n_out)).astype(np.float32)
        if not finite:  # the first batch rows: what the feature before reads past its end
            x[:3, 5::9] = np.inf
            x[1, 6::11] = np.nan
            g[:3, 4::9] = -np.inf
        y, dx, gs, gb = step(hip, L, H, x, g)
        with np.errstate(all="ignore"):
            assert_close_terms(y, H.forward_dense(x), H.forward_dense(x, absmode=True), f"y {n_in} B{B}")
            assert_close_terms(dx, H.backward_dense(x, g)[0], H.backward_dense(x, g, absmode=True)[0], f"dx {n_in} B{B}")
            want, bound = H.sampled_gradw(x, g), H.sampled_gradw(x, g, absmode=True)
            assert_close_terms(gs, want[0], bound[0], f"grad-W {n_in} B{B}")
            assert_close_terms(gb, want[1], bound[1], f"block4 grad-W {n_in} B{B}")
