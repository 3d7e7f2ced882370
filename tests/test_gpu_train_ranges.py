"""GPU: the optimizer update's fast steps (train.hip) against the oracle's
IEEE restatement where they can go wrong: every remainder of the step groups
(8, 4, 1), tile counts around a wave's 16 and a block's 64, edge tiles and
rows, and operands outside the fast step's range (zero, tiny, huge and
non-finite second moments and step numerators), which must take the step as
written.  Value and tile bytes are equal; dx is within the fp32 bar."""
import numpy as np
import pytest

from test_gpu_train import _sorted_tiles, gpu_layer
from train_util import add_tiles, b4_reserve_like_device, dx_bound, dx_bound_tiles, host_layer, make_train_case
from util import assert_close_terms

pytestmark = pytest.mark.gpu

BATCHES = [1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 37]


def batch_inputs(rng, B, n_in, n_out, kind):
    x = rng.normal(size=(B, n_in)).astype(np.float32)
    dy = rng.normal(size=(B, n_out)).astype(np.float32)
    if kind == "zeros":  # gated inputs and gradients: zero moments and numerators
        x[rng.random(x.shape) < 0.6] = 0.0
        dy[rng.random(dy.shape) < 0.6] = 0.0
    elif kind == "tiny":  # products down to the subnormals
        x *= np.float32(10.0) ** rng.integers(-24, 1, x.shape).astype(np.float32)
        dy *= np.float32(10.0) ** rng.integers(-24, 1, dy.shape).astype(np.float32)
    elif kind == "huge":  # squares that overflow
        dy *= np.float32(10.0) ** rng.integers(0, 22, dy.shape).astype(np.float32)
    elif kind == "nonfinite":
        x[rng.random(x.shape) < 0.02] = np.inf
        dy[rng.random(dy.shape) < 0.02] = np.nan
    return x, dy


def check(L, H, x, dy, lr, kind, tiles, what):
    bound = dx_bound(H, dy, lr) + (dx_bound_tiles(H, dy, lr) if tiles else 0.0)
    L.forward_dense(x)
    dxg = L.backward_dense(dy, lr)
    with np.errstate(all="ignore"):
        dxh, _, _ = H.backward_train(x, dy, lr)
    assert np.array_equal(L.export_scattered()["val"], H.val[:H.nnz]), what + ": value bytes"
    if tiles:
        ex = L.export_block4()
        gt = _sorted_tiles(ex["br"], ex["bc"], ex["tiles"], H.n_out)
        ht = _sorted_tiles(H.tile_br, H.tile_bc, H.tiles[:16 * H.n_tiles], H.n_out)
        assert all(np.array_equal(a, b) for a, b in zip(gt, ht)), what + ": tile bytes"
    if kind != "nonfinite":
        assert_close_terms(dxg, dxh, bound, what + ": dx")


@pytest.mark.parametrize("kind", ["normal", "zeros", "tiny", "huge", "nonfinite"])
@pytest.mark.parametrize("trainable", [False, True])
def test_scattered_update_ranges(hip, kind, trainable):
    for B in BATCHES:
        c = make_train_case(24, 150, 0.6, 40 + B, os_trainable=trainable)
        c["imp"][c["rng"].random(len(c["imp"])) < 0.3] = 0.0
        H, L = host_layer(c), gpu_layer(hip, c)
        for step in range(2):
            x, dy = batch_inputs(c["rng"], B, 24, 150, kind)
            check(L, H, x, dy, 0.05, kind, False, f"{kind} batch {B} step {step}")


# (tiles per block row, columns past the last full tile, rows)
SHAPES = [(1, 0, 8), (15, 0, 8), (16, 3, 8), (17, 0, 7), (63, 1, 8), (64, 0, 5), (65, 2, 8), (130, 0, 8)]


@pytest.mark.parametrize("kind", ["normal", "zeros", "tiny", "huge", "nonfinite"])
@pytest.mark.parametrize("shape", SHAPES)
def test_block4_update_ranges(hip, kind, shape):
    nt, extra, n_in = shape
    n_out = 4 * nt + extra
    for B in (1, 4, 7, 12, 37):
        c = add_tiles(make_train_case(n_in, n_out, 0.0, 60 + B, empty_rows=n_in), tile_density=1.1, seed=nt)
        H, L = host_layer(c), gpu_layer(hip, c, extra=16 * len(c["br"]))
        H.load_tiles(c["br"], c["bc"], c["tiles"])
        L.load_block4_tiles(c["br"], c["bc"], c["tiles"])
        b4_reserve_like_device(L, H, 64 + 16 * len(c["br"]))
        x, dy = batch_inputs(c["rng"], B, n_in, n_out, kind)
        check(L, H, x, dy, 0.05, kind, True, f"{kind} {shape} batch {B}")


@pytest.mark.parametrize("B", [1, 2, 3])
@pytest.mark.parametrize("rank", [1, 2, 3, 4])
def test_block4_few_steps(hip, monkeypatch, rank, B):
    """Batches of 1 to 3 (a slot a lane): every rank, output scales that train,
    rows past a block's 16 tiles, an edge tile and an edge row."""
    import test_gpu_train as T
    opts = dict(rank=rank, os_trainable=True, imp_scales=True, tile_density=0.7)
    monkeypatch.setattr(T, "B4_CASES", [(39, 150, 0.01, 70 + 3 * rank + B, B, 0.3, opts, "plain")])
    T.test_block4_update_matches_oracle(hip, 0)
