"""The work a user has the sparse layer do, as measurable cases.

Each case is one pass through the public entry points -- the C ABI of
include/sili_hip.h on device buffers, or the numpy methods of
SparseLinearLayer where `"api"` says "numpy" -- on seeded inputs of the shapes
that bench.py, the tests and the reference's layers use:

decode    forward only: a folded transformer stack decoding tokens, or one layer
step      forward + grad-input + nnz-sampled grad-W (learning_rate 0)
sparse    forward on an energy-gated sparse input + grad-input; skewed rows
block4    the `step` on 4x4 tiles
train     forward + backward with the optimizer update, scattered or block4
synapto   one bulk prune/regrow/rebuild step and the forward pass after it
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import sili__new_amd as sili

DEV = "cuda:0"
CELLS_AT_ONCE = 1 << 26


# ---- cases ------------------------------------------------------------------

def listed():
    return [
        # one layer, one token: the smallest call, where launches and latency count
        dict(name="decode_4096_b1", kind="decode", n_in=4096, n_out=4096, density=0.05, batch=1, api="device"),
        # the q/k/v/o shape of a 40-block folded transformer stack at 10 % density:
        # a single token, a small and a large token batch
        dict(name="decode_folded_b1", kind="decode", n_in=5120, n_out=204800, density=0.1, batch=1, api="device"),
        dict(name="decode_folded_b8", kind="decode", n_in=5120, n_out=204800, density=0.1, batch=8, api="device"),
        dict(name="decode_folded_b128", kind="decode", n_in=5120, n_out=204800, density=0.1, batch=128, api="device"),
        # sizes and a batch that divide by nothing
        dict(name="step_odd_b37", kind="step", n_in=3001, n_out=5003, density=0.04, batch=37, api="device"),
        # bench.py's default layer
        dict(name="step_8192_b64", kind="step", n_in=8192, n_out=8192, density=0.02, batch=64, api="device"),
        # the same layer as FoldedLayer calls it: numpy arrays in and out
        dict(name="numpy_8192_b64", kind="step", n_in=8192, n_out=8192, density=0.02, batch=64, api="numpy"),
        # energy-gated inputs (10 % active) over power-law rows
        dict(name="sparse_16384_b32", kind="sparse", n_in=16384, n_out=16384, density=0.01, active=0.1, batch=32),
        # 4x4 tiles at 3 % block density: forward, grad-input, grad-W of every slot
        dict(name="block4_16384_b256", kind="block4", n_in=16384, n_out=16384, density=0.03, batch=256),
        # a training step of each store
        dict(name="train_8192_b64", kind="train", store="scattered", n_in=8192, n_out=8192, density=0.02, batch=64),
        dict(name="train_block4_b256", kind="train", store="block4", n_in=16384, n_out=16384, density=0.03, batch=256),
        # structure learning: prune 1 %, regrow as many, rebuild; then the next forward
        dict(name="synapto_16384", kind="synapto", n_in=16384, n_out=16384, density=0.03, batch=32),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _side(rng, lo, hi):
    """A layer width: mostly arbitrary, sometimes a round one."""
    n = int(_log(rng, lo, hi))
    return max(lo, n // 64 * 64) if rng.random() < 0.4 else n


def _batch(rng, hi):
    """A batch: any number, or a power of two as often."""
    b = int(_log(rng, 1, hi + 1))
    return 1 << int(math.log2(b) + 0.5) if rng.random() < 0.5 and 1 << int(math.log2(b) + 0.5) <= hi else b


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "step", "step", "sparse", "block4", "train", "train", "synapto"])
    if kind == "decode":
        n_in, n_out = _side(rng, 512, 16384), _side(rng, 512, 200000)
        density = round(_log(rng, 0.01, 0.15), 4)
        density = round(min(density, 9e7 / (n_in * n_out)), 5)
        return dict(kind=kind, n_in=n_in, n_out=n_out, density=density, batch=_batch(rng, 128), api="device")
    if kind == "step":
        n_in, n_out = _side(rng, 512, 16384), _side(rng, 512, 16384)
        return dict(kind=kind, n_in=n_in, n_out=n_out, density=round(_log(rng, 0.005, 0.06), 4), batch=_batch(rng, 128),
                    api=rng.choice(["device", "device", "device", "numpy"]))
    if kind == "sparse":
        n_in, n_out = _side(rng, 2048, 16384), _side(rng, 2048, 16384)
        return dict(kind=kind, n_in=n_in, n_out=n_out, density=round(_log(rng, 0.005, 0.03), 4),
                    active=round(_log(rng, 0.005, 0.3), 4), batch=_batch(rng, 64))
    n_in, n_out = 4 * _side(rng, 256, 4096), 4 * _side(rng, 256, 4096)
    if kind == "train" and rng.random() < 0.6:
        return dict(kind=kind, store="scattered", n_in=n_in, n_out=n_out, density=round(_log(rng, 0.005, 0.04), 4),
                    batch=_batch(rng, 128))
    if kind == "synapto":
        return dict(kind=kind, n_in=n_in, n_out=n_out, density=round(_log(rng, 0.01, 0.04), 4), batch=_batch(rng, 64))
    c = dict(kind=kind, n_in=n_in, n_out=n_out, density=round(_log(rng, 0.01, 0.03), 4), batch=_batch(rng, 256))
    if kind == "train":
        c["store"] = "block4"
    return c


# ---- seeded inputs -----------------------------------------------------------

FP4_LEVELS = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
FP4_EDGES = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)  # a tie goes to the larger magnitude


def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + stream) % (1 << 62))
    return g


def _fp4_codes(q):
    """E2M1 codes (sign << 3 | magnitude; a zero has code 0) of float32 values."""
    edges = torch.tensor(FP4_EDGES, device=q.device, dtype=torch.float32)
    mag = torch.bucketize(q.abs(), edges, right=True)
    return (mag + 8 * ((q < 0) & (mag > 0))).to(torch.uint8)


def _fp4_values(codes):
    levels = torch.tensor(FP4_LEVELS, device=codes.device, dtype=torch.float64)
    c = codes.long()
    return levels[c & 7] * torch.where(c >= 8, -1.0, 1.0).to(torch.float64)


def _zipf_rows(n, mean, longest, gen):
    """Row lengths with a Zipf (exponent 1.2) tail, rescaled to `mean`."""
    k = torch.arange(1, longest + 1, device=DEV, dtype=torch.float64)
    cdf = torch.cumsum(k ** -1.2, 0)
    u = torch.rand(n, generator=gen, device=DEV, dtype=torch.float64) * cdf[-1]
    ln = (torch.searchsorted(cdf, u) + 1).double()
    return (ln * (mean * n / ln.sum())).clamp(1.0, float(longest))


def _scattered(case, seed):
    """A scattered layer: row starts, columns (ascending per row), FP4 codes and
    per-row scales; weights ~N(0, 0.02), or for `decode` its tails, as magnitude
    pruning leaves them."""
    n_in, n_out, d = case["n_in"], case["n_out"], case["density"]
    g = _gen(seed, 1)
    prob = torch.full((n_in,), float(d), device=DEV)
    if case["kind"] == "sparse":
        prob = (_zipf_rows(n_in, d * n_out, max(2, n_out // 4), g) / n_out).float()
    rows, cols, step = [], [], max(1, CELLS_AT_ONCE // n_out)
    for r0 in range(0, n_in, step):
        p = prob[r0:r0 + step, None]
        r, c = torch.nonzero(torch.rand(p.shape[0], n_out, generator=g, device=DEV) < p, as_tuple=True)
        rows.append((r + r0).int())
        cols.append(c.int())
    rows, cols = torch.cat(rows), torch.cat(cols)
    ptrs = torch.zeros(n_in + 1, dtype=torch.int32, device=DEV)
    ptrs[1:] = torch.cumsum(torch.bincount(rows.long(), minlength=n_in), 0).int()
    if case["kind"] == "decode":
        t = 1.0 - d * (1.0 - torch.rand(len(rows), generator=g, device=DEV))
        w = 0.02 * math.sqrt(2.0) * torch.erfinv(t.clamp(max=1.0 - 1e-7))
        w = torch.where(torch.rand(len(rows), generator=g, device=DEV) < 0.5, w, -w)
    else:
        w = 0.02 * torch.randn(len(rows), generator=g, device=DEV)
    top = torch.zeros(n_in, device=DEV).scatter_reduce_(0, rows.long(), w.abs(), "amax")
    scale = torch.where(top > 0, top / 6.0, torch.ones_like(top))
    codes = _fp4_codes(w / scale[rows.long()])
    return dict(ptrs=ptrs, rows=rows, cols=cols, codes=codes, scale=scale)


def _tiles(case, seed):
    """Distinct random 4x4 tiles in (block row, block column) order, every slot
    live; slot lj*4+li of a tile is row 4*br+li, column 4*bc+lj."""
    nbr, nbc = case["n_in"] // 4, case["n_out"] // 4
    g = _gen(seed, 1)
    pos = torch.nonzero(torch.rand(nbr, nbc, generator=g, device=DEV) < case["density"])
    br, bc = pos[:, 0].int(), pos[:, 1].int()
    slot = torch.arange(16, device=DEV)
    rows = (4 * br.long()[:, None] + slot % 4).reshape(-1)
    cols = (4 * bc.long()[:, None] + slot // 4).reshape(-1)
    w = 0.02 * torch.randn(len(rows), generator=g, device=DEV)
    top = torch.zeros(case["n_in"], device=DEV).scatter_reduce_(0, rows, w.abs(), "amax")
    scale = torch.where(top > 0, top / 6.0, torch.ones_like(top))
    codes = _fp4_codes(w / scale[rows])
    return dict(br=br, bc=bc, rows=rows.int(), cols=cols.int(), codes=codes, scale=scale)


def _is_block4(case):
    return case["kind"] in ("block4", "synapto") or case.get("store") == "block4"


def _weights(case, seed):
    return _tiles(case, seed) if _is_block4(case) else _scattered(case, seed)


def _activations(case, seed):
    """x [batch, n_in] and the upstream gradient g [batch, n_out], ~N(0, 1); a
    sparse input is |N(0, 1)| at its active positions, with its CSR form."""
    gen, b = _gen(seed, 2), case["batch"]
    g = torch.randn(b, case["n_out"], generator=gen, device=DEV)
    x = torch.randn(b, case["n_in"], generator=gen, device=DEV)
    if case["kind"] != "sparse":
        return dict(x=x, g=g)
    keep = torch.rand(b, case["n_in"], generator=gen, device=DEV) < case["active"]
    x = torch.where(keep, x.abs(), torch.zeros_like(x))
    ptrs = torch.zeros(b + 1, dtype=torch.int32, device=DEV)
    ptrs[1:] = torch.cumsum(keep.sum(1), 0).int()
    idx = torch.nonzero(keep)[:, 1].int()
    return dict(x=x, g=g, x_ptrs=ptrs, x_idx=idx, x_vals=x[keep])


def _gradw_room(case):
    """Floats of the grad-W buffer: the expected synapse count and its spread.
    The buffer's end, past the layer's synapses, stays zero."""
    return int(1.02 * case["density"] * case["n_in"] * case["n_out"]) + 16384


CANDIDATE_LISTS = 48


def _prune_count(n):
    return int(math.floor(0.01 * n + 0.5))


def _candidates(case, n, seed):
    """The host's regrowth proposals, a list of positions and initial values per
    step (twice as many as a step grows)."""
    gen, m = _gen(seed, 3), 2 * _prune_count(n) + 64
    shape = (CANDIDATE_LISTS, m)
    r = torch.randint(case["n_in"], shape, generator=gen, device=DEV, dtype=torch.int32)
    c = torch.randint(case["n_out"], shape, generator=gen, device=DEV, dtype=torch.int32)
    v = 0.01 * torch.randn(shape, generator=gen, device=DEV)
    return r, c, v


# ---- the C ABI -----------------------------------------------------------------

_lib = None
_stream = None


def _abi():
    global _lib
    if _lib is None:
        lib, vp, i64 = C.CDLL(sili.LIB_PATH), C.c_void_p, C.c_int64
        lib.sili_last_error.restype = C.c_char_p
        lib.sili_set_value_scale.argtypes = [vp, vp]
        lib.sili_forward_dense.argtypes = [vp, vp, i64, vp, vp]
        lib.sili_forward_sparse.argtypes = [vp, vp, vp, vp, i64, i64, vp, vp]
        lib.sili_backward_dense.argtypes = [vp, vp, vp, i64, vp, vp, vp, C.c_float, vp]
        lib.sili_synapto_step.argtypes = [vp, C.c_float, vp, vp, vp, vp, i64, C.c_int, vp]
        _lib = lib
    return _lib


def _check(rc):
    if rc:
        raise RuntimeError(_abi().sili_last_error().decode())


def _on():
    """The one stream that the program issues its work on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return C.c_void_p(_stream.cuda_stream)


# ---- one case --------------------------------------------------------------------

def prepare(case, seed):
    w = _weights(case, seed)
    n = len(w["codes"])
    layer = sili.SparseLinearLayer(case["n_in"], case["n_out"], n)
    if _is_block4(case):
        # low nibble the weight, high nibble importance code 1: every slot live
        tiles = (w["codes"] | 16).cpu().numpy()
        layer.load_block4_tiles(w["br"].cpu().numpy(), w["bc"].cpu().numpy(), tiles)
    else:
        layer.load_weight_bytes(w["ptrs"].cpu().numpy(), w["cols"].cpu().numpy(), (w["codes"] << 4).cpu().numpy())
    scale = w["scale"].cpu().numpy()
    a = _activations(case, seed)
    s = dict(case=case, layer=layer, h=C.c_void_p(layer.handle), n=n)
    if case.get("api") == "numpy":
        layer.set_value_scales(scale)
        s.update(x=a["x"].cpu().numpy(), g=a["g"].cpu().numpy())
    else:
        _check(_abi().sili_set_value_scale(s["h"], scale.ctypes.data_as(C.c_void_p)))
        b = case["batch"]
        s.update(a, y=torch.empty(b, case["n_out"], device=DEV), stream=_on())
        if case["kind"] in ("step", "sparse", "block4", "train"):
            s["dx"] = torch.empty(b, case["n_in"], device=DEV)
        if case["kind"] in ("step", "block4"):
            s["gw"] = torch.zeros(_gradw_room(case), device=DEV)
        if case["kind"] == "sparse":
            s["nnz_x"] = len(a["x_vals"])
        if case["kind"] == "synapto":
            r, c, v = _candidates(case, n, seed)
            s.update(cand=(r.cpu().numpy(), c.cpu().numpy(), v.cpu().numpy()), at=0)
        if case["kind"] == "train":
            layer.seed_stochastic_rounding(int(seed) & 0xFFFFFFFF)
    torch.cuda.synchronize()
    return s


def _p(t):
    return C.c_void_p(t.data_ptr())


def run(s):
    case, kind, b, h = s["case"], s["case"]["kind"], s["case"]["batch"], s["h"]
    if case.get("api") == "numpy":
        y = s["layer"].forward_dense(s["x"])
        return y, s["layer"].backward_dense(s["g"], 0.0)
    lib, st = _abi(), s["stream"]
    if kind == "synapto":
        r, c, v = (a[s["at"]] for a in s["cand"])
        s["at"] = (s["at"] + 1) % CANDIDATE_LISTS
        stats = np.zeros(7, np.int64)
        _check(lib.sili_synapto_step(h, 0.01, r.ctypes.data, c.ctypes.data, v.ctypes.data, None, r.size, 1,
                                     stats.ctypes.data))
        _check(lib.sili_forward_dense(h, _p(s["x"]), b, _p(s["y"]), st))
        return s["y"], stats
    if kind == "sparse":
        _check(lib.sili_forward_sparse(h, _p(s["x_ptrs"]), _p(s["x_idx"]), _p(s["x_vals"]), s["nnz_x"], b, _p(s["y"]),
                                       st))
        _check(lib.sili_backward_dense(h, _p(s["x"]), _p(s["g"]), b, _p(s["dx"]), None, None, 0.0, st))
        return s["y"], s["dx"]
    _check(lib.sili_forward_dense(h, _p(s["x"]), b, _p(s["y"]), st))
    if kind == "decode":
        return s["y"]
    # the backward reads the input that the forward kept, except at batch 1, where none is kept
    x = _p(s["x"]) if b == 1 else None
    if kind == "train":
        # the optimizer update with the layer's defaults; dx is taken over the updated weights
        _check(lib.sili_backward_dense(h, x, _p(s["g"]), b, _p(s["dx"]), None, None, 0.01, st))
        return s["y"], s["dx"]
    gws, gwb = (None, _p(s["gw"])) if kind == "block4" else (_p(s["gw"]), None)
    _check(lib.sili_backward_dense(h, x, _p(s["g"]), b, _p(s["dx"]), gws, gwb, 0.0, st))
    return s["y"], s["dx"], s["gw"]


def work(case):
    n_in, n_out, b, kind = case["n_in"], case["n_out"], case["batch"], case["kind"]
    nnz = case["density"] * n_in * n_out
    # a scattered synapse: a value byte and an index byte; a tile: 16 value bytes and an index byte
    weights = (17 / 16 if _is_block4(case) else 2) * nnz + 4 * n_in
    fwd = 4.0 * b * (n_in + n_out)
    if kind == "decode":
        return dict(bytes=weights + fwd, flops=2 * nnz * b)
    if kind == "synapto":
        # the stores read and written, the candidates, and the forward pass
        return dict(bytes=3 * weights + 0.02 * 12 * nnz + fwd, flops=2 * nnz * b)
    both = 2 * fwd + weights
    if kind == "sparse":
        x = case["active"] * b * n_in
        return dict(bytes=weights + 8 * x + 4.0 * b * n_out + fwd, flops=2 * nnz * b * (1 + case["active"]))
    if kind == "train":
        # per synapse and batch step: forward, grad-input and gradient products, and
        # the importance average, step, clip and rounding (about 14 operations)
        return dict(bytes=both + nnz, flops=20 * nnz * b)
    gw = 0.0 if case.get("api") == "numpy" else 1.0
    return dict(bytes=both + 4 * gw * nnz, flops=(4 + 2 * gw) * nnz * b)


def tolerance(case):
    """Sums of float32 products in any order: 6e-8 to 2.1e-7 off 64 bits over
    these row lengths, so four times that.  A training step's codes depend on no
    sum, its scales on sums held in 64 bits."""
    return {"rel": 1e-6, "max": 4e-5}


def _dense(case, w):
    out = torch.zeros(case["n_in"], case["n_out"], dtype=torch.float64, device=DEV)
    out[w["rows"].long(), w["cols"].long()] = _fp4_values(w["codes"]) * w["scale"].double()[w["rows"].long()]
    return out


def _after_synapto(case, w, seed):
    """The weights one step later: the 1 % smallest |w| (ties by row, then
    column) pruned; the first as many candidates grown that are distinct and
    held no synapse before the step."""
    rows, cols, n = w["rows"].long(), w["cols"].long(), len(w["codes"])
    k = _prune_count(n)
    mag = (_fp4_values(w["codes"]).float() * w["scale"][rows]).abs()
    key = (mag.view(torch.int32).long() << 31) | (rows * case["n_out"] + cols)
    gone = torch.sort(key).indices[:k]
    dense = _dense(case, w)
    taken = torch.zeros(case["n_in"] * case["n_out"], dtype=torch.bool, device=DEV)
    taken[rows * case["n_out"] + cols] = True
    dense[rows[gone], cols[gone]] = 0.0
    r, c, v = (t[0] for t in _candidates(case, n, seed))
    flat = (r.long() * case["n_out"] + c.long()).cpu().numpy()
    first = np.zeros(len(flat), bool)
    first[np.unique(flat, return_index=True)[1]] = True
    good = np.nonzero(first & ~taken[torch.from_numpy(flat).to(DEV)].cpu().numpy())[0][:k]
    at = torch.from_numpy(good).to(DEV)
    r, c, v = r[at].long(), c[at].long(), v[at]
    dense[r, c] = _fp4_values(_fp4_codes(v / w["scale"][r])) * w["scale"].double()[r]
    return dense


def exact(case, seed):
    w, a = _weights(case, seed), _activations(case, seed)
    x, g = a["x"].double(), a["g"].double()
    kind = case["kind"]
    if kind == "synapto":
        return x @ _after_synapto(case, w, seed), None
    dense = _dense(case, w)
    y = x @ dense
    if kind == "decode":
        return y
    if kind == "train":
        return y, None  # dx follows a chain of rounded weight steps
    dx = g @ dense.T
    if kind == "sparse" or case.get("api") == "numpy":
        return y, dx
    del dense
    gw = torch.zeros(_gradw_room(case), dtype=torch.float64, device=DEV)
    gw[:len(w["codes"])] = (x.T @ g)[w["rows"].long(), w["cols"].long()]
    return y, dx, gw
