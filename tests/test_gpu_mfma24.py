"""GPU: the gathers on the 2:4 sparse matrix cores (csrc/mfma24.hip) against
the oracle (linear_disldo.hpp:68-126 and its transpose) where they can go
wrong: rows and columns that fill no tile of 32 or block of 128 (512 columns a
turn), empty rows, groups of 4 columns with 3 and 4 entries (the overflow list)
up to full rows, batches around the operand tiles (10 and 21 for the pieces as
columns, 32, 64, 128 a chunk), inputs over the whole float range (tiny ones that
take the products, large and non-finite ones that leave them, scales that cancel),
and the copy's life: built late, dropped when values or structure change, its
memory, stores and captured calls that stay with the other kernels."""
import ctypes as C

import numpy as np
import pytest

from oracle import HostLayer
from tests.test_gpu_capi import Api, _ptr
from tests.test_gpu_stream import kernel_counts
from tests.util import assert_close_terms

pytestmark = pytest.mark.gpu


def case(n_in, n_out, density, seed, full=True):
    rng = np.random.default_rng(seed)
    keep = rng.random((n_in, n_out)) < density
    keep[1::7] = False                # empty inputs
    keep[:, 3::11] = False            # empty outputs
    if full and n_in > 8:
        keep[4], keep[:, 5] = True, True  # a full row and column: groups of 4
    cols = np.nonzero(keep)[1].astype(np.int32)
    ptrs = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return ptrs, cols, rng.normal(0, 0.5, len(cols)).astype(np.float32)


def make(hip, n_in, n_out, density, seed, scales, full=True):
    ptrs, cols, q = case(n_in, n_out, density, seed, full)
    H = HostLayer(n_in, n_out).load_csr(ptrs, cols, w=q)
    L = hip.SparseLinearLayer(n_in, n_out, 4 * len(cols) + 4096)
    L.load_weights(ptrs, cols, q)
    if scales:
        rng = np.random.default_rng(seed + 1)
        vs = rng.uniform(0.5, 1.5, n_in).astype(np.float32)
        os_ = rng.uniform(0.5, 1.5, n_out).astype(np.float32)
        H.set_scales(vs, os_)
        L.set_value_scales(vs)
        L.set_output_scales(os_)
    return H, L


def check(hip, H, L, x, dy, what, mfma=True):
    got = {}
    counts = kernel_counts(hip, L, lambda: got.update(y=L.forward_dense(x), dx=L.backward_dense(dy, 0.0)))
    assert counts.get("fwd:mfma24", 0) == mfma and counts.get("bwd:mfma24", 0) == mfma, (what, counts)
    with np.errstate(all="ignore"):
        assert_close_terms(got["y"], H.forward_dense(x), H.forward_dense(x, absmode=True), f"fwd {what}")
        assert_close_terms(got["dx"], H.backward_dense(x, dy)[0], H.backward_dense(x, dy, absmode=True)[0], f"bwd {what}")
    return got


# (n_in, n_out, density, scales): both directions run, so each pair is a row and a column count
SHAPES = [(1, 1, 1.0, False), (31, 129, 0.5, True), (33, 512, 0.1, False), (700, 513, 0.1, True),
          (100, 1030, 1.0, True), (2500, 67, 0.02, False)]


@pytest.mark.parametrize("B", [2, 8, 10, 11, 21, 22, 32, 33, 37, 64, 65, 96, 128, 129, 300])
@pytest.mark.parametrize("shape", SHAPES)
def test_mfma24_matches_oracle(hip, monkeypatch, shape, B):
    monkeypatch.setenv("SILI_MFMA24", "2")
    H, L = make(hip, *shape[:3], B + shape[1], shape[3])
    rng = np.random.default_rng(B)
    # magnitudes over 40 octaves: every piece of the split counts
    x = (rng.normal(size=(B, shape[0])) * 2.0 ** rng.integers(-20, 20, (B, 1))).astype(np.float32)
    dy = (rng.normal(size=(B, shape[1])) * 2.0 ** rng.integers(-20, 20, (B, 1))).astype(np.float32)
    check(hip, H, L, x, dy, f"{shape} B{B}")


@pytest.mark.parametrize("B", [8, 16, 32, 64, 128])
def test_mfma24_more_tiles_than_units(hip, monkeypatch, B):
    """Enough rows for two row tiles a wave, and many turns of columns."""
    monkeypatch.setenv("SILI_MFMA24", "2")
    H, L = make(hip, 150, 70001, 0.03, B, True)
    rng = np.random.default_rng(B)
    check(hip, H, L, rng.normal(size=(B, 150)).astype(np.float32), rng.normal(size=(B, 70001)).astype(np.float32), f"B{B}")


@pytest.mark.parametrize("B", [8, 16, 37, 128])
@pytest.mark.parametrize("kind", ["nonfinite", "tiny"])
def test_mfma24_inputs_without_a_split(hip, monkeypatch, kind, B):
    monkeypatch.setenv("SILI_MFMA24", "2")
    H, L = make(hip, 300, 400, 0.2, 5, True)
    rng = np.random.default_rng(B)
    x, dy = rng.normal(size=(B, 300)).astype(np.float32), rng.normal(size=(B, 400)).astype(np.float32)
    fine = (x.copy(), dy.copy())
    if kind == "nonfinite":
        x[B // 2, 17], x[0, 40], dy[B - 1, 399] = np.inf, -np.inf, np.nan
    else:
        x *= np.float32(1e-36)
        dy *= np.float32(1e-36)
    got = check(hip, H, L, x, dy, f"{kind} B{B}")
    if kind == "tiny":  # products of normal numbers near the smallest: 24 bits still
        for k, want, bound in (("y", H.forward_dense(x), H.forward_dense(x, absmode=True)),
                               ("dx", H.backward_dense(x, dy)[0], H.backward_dense(x, dy, absmode=True)[0])):
            # a sum of n <= 400 roundings of half an ulp each, and of subnormals' steps
            assert np.all(np.abs(got[k] - want) <= 400 * (2.0 ** -24 * bound + 2.0 ** -149)), k
    check(hip, H, L, *fine, f"after {kind} B{B}")


@pytest.mark.parametrize("B", [8, 16, 37, 64, 150])
@pytest.mark.parametrize("kind", ["large x", "large dy", "scales", "octaves", "zero scales"])
def test_mfma24_ranges(hip, monkeypatch, kind, B):
    """Finite results whose way there could leave the range: inputs near the
    largest float under small scales, scales that cancel each other, batch rows
    of every magnitude down to the subnormals, scales of 0."""
    monkeypatch.setenv("SILI_MFMA24", "2")
    H, L = make(hip, 300, 400, 0.2, 5, False)
    rng = np.random.default_rng(B)
    x, dy = rng.normal(size=(B, 300)).astype(np.float32), rng.normal(size=(B, 400)).astype(np.float32)
    vs, os_ = rng.uniform(0.5, 1.5, 300).astype(np.float32), rng.uniform(0.5, 1.5, 400).astype(np.float32)
    if kind == "large x":  # sums of up to 300 terms of 6 * 3e37 * 0.007 at most, larger by 1 / 0.003 without the output's scale
        x[::3] = rng.uniform(-3e37, 3e37, x[::3].shape)
        x[0, 3], os_ = 0.0, os_ * np.float32(0.003)
    elif kind == "large dy":
        dy[1::3] = rng.uniform(-3e37, 3e37, dy[1::3].shape)
        dy[1, 3], vs = -0.0, vs * np.float32(0.003)
    elif kind == "scales":  # an input times its own scale alone is subnormal, or infinite
        x, dy = x * np.float32(1e-15), dy * np.float32(1e15)
        vs, os_ = vs * np.float32(1e-27), os_ * np.float32(1e27)
    elif kind == "octaves":
        x = np.ldexp(x, np.linspace(-146, 60, B).astype(int)[:, None]).astype(np.float32)
        dy = np.ldexp(dy, np.linspace(-146, 60, B).astype(int)[:, None]).astype(np.float32)
    else:
        vs[::2], os_[::3] = 0.0, 0.0
    H.set_scales(vs, os_)
    L.set_value_scales(vs)
    L.set_output_scales(os_)
    got = check(hip, H, L, x, dy, f"{kind} B{B}")
    assert all(np.all(np.isfinite(v)) for v in got.values())
    for k, want, bound in (("y", H.forward_dense(x), H.forward_dense(x, absmode=True)),
                           ("dx", H.backward_dense(x, dy)[0], H.backward_dense(x, dy, absmode=True)[0])):
        # sums of n <= 400 terms: half an ulp each for the weight's two products, the input's and the
        # sum's on either side, and a step of the subnormals
        lim = 400 * 4 * (2.0 ** -24 * bound.astype(np.float64) + 2.0 ** -149)
        assert np.all(np.abs(got[k].astype(np.float64) - want) <= lim), k


@pytest.mark.parametrize("B", [8, 37, 150])
def test_mfma24_one_row_without_a_split(hip, monkeypatch, B):
    """Only the batch row that holds the input leaves the products: the others'
    outputs are the same bits as without it."""
    monkeypatch.setenv("SILI_MFMA24", "2")
    H, L = make(hip, 300, 400, 0.2, 5, True)
    rng = np.random.default_rng(B)
    x, dy = rng.normal(size=(B, 300)).astype(np.float32), rng.normal(size=(B, 400)).astype(np.float32)
    fine = check(hip, H, L, x, dy, f"fine B{B}")
    row = B // 2
    x[row, 17], dy[row, 20] = np.inf, np.nan
    got = check(hip, H, L, x, dy, f"one row B{B}")
    for k in got:
        others = np.arange(B) != row
        assert np.array_equal(got[k][others].view(np.uint32), fine[k][others].view(np.uint32)), k
        assert not np.all(np.isfinite(got[k][row])), k


def test_mfma24_copy_follows_changes(hip, monkeypatch):
    monkeypatch.setenv("SILI_MFMA24", "2")
    L = make(hip, 700, 1000, 0.1, 3, True)[1]
    rng = np.random.default_rng(4)
    x, dy = rng.normal(size=(48, 700)).astype(np.float32), rng.normal(size=(48, 1000)).astype(np.float32)

    def agree(what):
        got = {}
        for mode in "20":
            monkeypatch.setenv("SILI_MFMA24", mode)
            got[mode] = L.forward_dense(x), L.backward_dense(dy, 0.0)
        for a, b in zip(got["2"], got["0"]):
            np.testing.assert_allclose(a, b, rtol=1e-5, atol=1e-4, err_msg=what)

    agree("loaded")
    L.backward_dense(dy, 0.05)
    agree("after an update")
    cr, cc = rng.integers(0, 700, 2000).astype(np.int32), rng.integers(0, 1000, 2000).astype(np.int32)
    L.synapto_step(0.2, cr, cc, rng.normal(0, 0.3, 2000).astype(np.float32))
    agree("after a synaptogenesis step")
    L.set_value_scales(rng.uniform(0.5, 1.5, 700).astype(np.float32))
    agree("after new scales")


def test_mfma24_is_built_when_it_pays(hip, monkeypatch):
    """The default: other kernels until the copy has paid for itself, again
    after an update, and never on a layer too small for it or with an output of
    so many entries past the second of a group that one wave would be at it for
    longer than the other kernels take."""
    monkeypatch.delenv("SILI_MFMA24", raising=False)
    H, L = make(hip, 1000, 8192, 0.3, 6, False, full=False)
    rng = np.random.default_rng(7)
    x, dy = rng.normal(size=(128, 1000)).astype(np.float32), rng.normal(size=(128, 8192)).astype(np.float32)
    used = [kernel_counts(hip, L, lambda: L.forward_dense(x)).get("fwd:mfma24", 0) for _ in range(60)]
    assert used[0] == 0 and used[-1] == 1 and sorted(used) == used, used
    assert_close_terms(L.forward_dense(x), H.forward_dense(x), H.forward_dense(x, absmode=True), "built")
    L.backward_dense(dy, 0.05)
    assert "fwd:mfma24" not in kernel_counts(hip, L, lambda: L.forward_dense(x))
    uneven = make(hip, 1000, 8192, 0.3, 6, False)[1]
    assert all("fwd:mfma24" not in kernel_counts(hip, uneven, lambda: uneven.forward_dense(x)) for _ in range(60))
    small = make(hip, 300, 400, 0.2, 5, False)[1]
    xs = rng.normal(size=(64, 300)).astype(np.float32)
    assert all("fwd:mfma24" not in kernel_counts(hip, small, lambda: small.forward_dense(xs)) for _ in range(20))


def test_mfma24_copy_gives_its_memory_back(hip, monkeypatch):
    """A copy of 50 MB and more that an update drops before it has paid is freed;
    one that is too large a part of the free memory is not built."""
    lib = C.CDLL(hip.LIB_PATH)

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    monkeypatch.delenv("SILI_MFMA24", raising=False)
    L = make(hip, 2048, 65536, 0.1, 9, False, full=False)[1]
    rng = np.random.default_rng(9)
    x, dy = rng.normal(size=(128, 2048)).astype(np.float32), rng.normal(size=(128, 65536)).astype(np.float32)
    L.forward_dense(x)
    L.backward_dense(dy, 0.01)  # the optimizer's state
    for _ in range(30):
        if kernel_counts(hip, L, lambda: L.forward_dense(x)).get("fwd:mfma24"):
            break
    else:
        pytest.fail("no copy was built")
    held = free()
    for _ in range(10):  # (the runtime gives freed memory back some calls later)
        L.backward_dense(dy, 0.01)
        kernel_counts(hip, L, lambda: L.forward_dense(x))
        if free() - held > 45 << 20:
            break
    assert free() - held > 45 << 20
    monkeypatch.setenv("SILI_MFMA24_FREE_PCT", "0")
    for _ in range(60):
        assert "fwd:mfma24" not in kernel_counts(hip, L, lambda: L.forward_dense(x))


def test_mfma24_leaves_repeatable_stores_alone(hip, monkeypatch):
    """A store built for bitwise repeats gives the same bits on every call."""
    monkeypatch.delenv("SILI_MFMA24", raising=False)
    monkeypatch.setenv("SILI_SPLIT_COMBINE", "1")
    L = make(hip, 1000, 8192, 0.3, 6, False, full=False)[1]
    rng = np.random.default_rng(7)
    x = rng.normal(size=(128, 1000)).astype(np.float32)
    y = L.forward_dense(x)
    for _ in range(60):
        assert np.array_equal(L.forward_dense(x).view(np.uint32), y.view(np.uint32))
    assert "fwd:mfma24" not in kernel_counts(hip, L, lambda: L.forward_dense(x))


def test_mfma24_leaves_what_a_captured_call_needs(hip, monkeypatch):
    """A batch that ran twice before it is captured: the captured call takes the
    other kernels, whose first use builds and waits, so the first of those runs
    took them too, although another batch had the copy built by then.  The graph
    is replayed on new inputs between eager calls."""
    monkeypatch.delenv("SILI_MFMA24", raising=False)
    api = Api(hip.LIB_PATH)
    H, L = make(hip, 1000, 8192, 0.3, 6, False, full=False)
    rng = np.random.default_rng(8)
    xw = rng.normal(size=(128, 1000)).astype(np.float32)
    for _ in range(60):
        L.forward_dense(xw)
    assert kernel_counts(hip, L, lambda: L.forward_dense(xw)).get("fwd:mfma24", 0) == 1
    B, h = 64, C.c_void_p(L.handle)
    x, y, st, graph, run = (C.c_void_p() for _ in range(5))
    rt = lambda name, *args: api.ck(getattr(api.L, name)(*args))  # the HIP runtime that the library is linked to
    rt("sili_device_alloc", h, B * 1000 * 4, C.byref(x))
    rt("sili_device_alloc", h, B * 8192 * 4, C.byref(y))
    rt("hipStreamCreate", C.byref(st))
    got = np.empty((B, 8192), np.float32)

    def forward():
        rt("sili_forward_dense", h, x, B, y, st)

    def result(call):
        v = rng.normal(size=(B, 1000)).astype(np.float32)
        got[:] = np.nan
        rt("sili_memcpy_h2d", h, x, _ptr(v), v.nbytes)
        rt("sili_memcpy_h2d", h, y, _ptr(got), got.nbytes)
        call()
        rt("hipStreamSynchronize", st)
        rt("sili_memcpy_d2h", h, _ptr(got), y, got.nbytes)
        assert_close_terms(got, H.forward_dense(v), H.forward_dense(v, absmode=True), "replay")

    assert "fwd:mfma24" not in kernel_counts(hip, L, lambda: result(forward))
    assert kernel_counts(hip, L, lambda: result(forward)).get("fwd:mfma24", 0) == 1
    rt("hipStreamBeginCapture", st, 0)
    forward()
    rt("hipStreamEndCapture", st, C.byref(graph))
    rt("hipGraphInstantiate", C.byref(run), graph, None, None, C.c_size_t(0))
    for _ in range(3):
        result(lambda: rt("hipGraphLaunch", run, st))
        result(forward)
    rt("hipGraphExecDestroy", run)
    rt("hipGraphDestroy", graph)
    rt("hipStreamDestroy", st)
    rt("sili_device_free", h, x)
    rt("sili_device_free", h, y)
