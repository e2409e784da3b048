"""pkv_linear_forward, the small decoder's products with the row-wise steps around them, against the
same steps in float64, at the edges of its tiles: 16 rows x 64 columns a workgroup, depths of 16 to
1,536 in steps of 128. A float32 product of n terms summed in any order is within n * 2^-24 of the
sum of its terms' magnitudes; the norm's rows add 4e-7 of theirs."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from paged_kv_serving_amd import _native

pytestmark = pytest.mark.gpu

P, I64, I32, F32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int32, ctypes.c_float
ADD, SWIGLU, ROPE_APPEND, LOGITS = range(4)


class Linear(ctypes.Structure):
    """struct pkv_linear (include/pkv.h)."""

    _fields_ = [
        ("input", P), ("weights", P), ("norm_weight", P), ("output", P), ("input_stride", I64), ("weight_stride", I64),
        ("output_stride", I64), ("rows", I64), ("kind", I32), ("cols", I32), ("depth", I32), ("eps", F32),
        ("row_index", P), ("input_rows", I64), ("positions", P), ("slots", P), ("cos_table", P), ("sin_table", P),
        ("table_rows", I64), ("key_pool", P), ("value_pool", P), ("num_slots", I64), ("num_heads", I32),
        ("head_dim", I32), ("pool_dtype", I32),
    ]  # fmt: skip


def _call(device, **fields) -> int:
    """The library's return code; tensors are passed by address."""
    args = Linear(**{k: v.data_ptr() if isinstance(v, torch.Tensor) else v for k, v in fields.items()})
    rc = _native.library().pkv_linear_forward(ctypes.addressof(args), device.index, None)
    torch.cuda.synchronize()
    return rc


def _inputs(device, rows, depth, cols, transposed=False):
    rng = np.random.default_rng(rows + depth + cols)
    x = rng.standard_normal((rows, depth)).astype(np.float32)
    w = rng.standard_normal((cols, depth) if transposed else (depth, cols)).astype(np.float32)
    g = rng.standard_normal(depth).astype(np.float32)
    return rng, x, w, g, *(torch.from_numpy(a).to(device) for a in (x, w, g))


def _normed(x, g):
    x64 = x.astype(np.float64)
    return x64 / np.sqrt(np.mean(x64**2, axis=1, keepdims=True) + 1e-5) * g


def _bound(x, w):
    return (x.shape[1] * 2.0**-24 + 4e-7) * (np.abs(x) @ np.abs(w))


SIZES = [(1, 16, 1), (15, 128, 63), (16, 144, 64), (17, 320, 65), (33, 1536, 130), (128, 256, 256)]


@pytest.mark.parametrize(("rows", "depth", "cols"), SIZES)
def test_add_swiglu_and_logits(device, rows, depth, cols) -> None:
    _, x, w, _, dx, dw, _ = _inputs(device, rows, depth, cols)
    hidden = torch.ones((rows, cols + 3), device=device)
    assert _call(device, kind=ADD, input=dx, input_stride=depth, rows=rows, depth=depth, cols=cols, weights=dw,
                 weight_stride=cols, output=hidden, output_stride=cols + 3) == 0  # fmt: skip
    got = hidden.cpu().numpy()
    assert np.all(np.abs(got[:, :cols] - (1 + x.astype(np.float64) @ w)) <= _bound(x, w) + 2.0**-24 * np.abs(got[:, :cols]))
    assert np.all(got[:, cols:] == 1)

    _, x, w, g, dx, dw, dg = _inputs(device, rows, depth, 2 * cols)
    out = torch.zeros((rows, cols), device=device)
    assert _call(device, kind=SWIGLU, input=dx, input_stride=depth, rows=rows, depth=depth, cols=cols, weights=dw,
                 weight_stride=2 * cols, output=out, output_stride=cols, norm_weight=dg, eps=1e-5) == 0  # fmt: skip
    n = _normed(x, g)
    gate, up = n @ w[:, :cols], n @ w[:, cols:]
    silu = gate / (1 + np.exp(-np.clip(gate, -60, 60)))
    slack = _bound(n, w)  # silu's slope stays below 1.1
    tol = 1.1 * slack[:, :cols] * np.abs(up) + np.abs(silu) * slack[:, cols:] + 1e-6 * np.abs(silu * up) + 1e-9
    assert np.all(np.abs(out.cpu().numpy() - silu * up) <= tol + 1.1 * slack[:, :cols] * slack[:, cols:])

    rng, x, w, g, dx, dw, dg = _inputs(device, rows, depth, cols, transposed=True)
    wanted = rng.integers(0, rows, 18)
    wanted[3] = rows  # outside the input: a row of zeros
    out = torch.full((18, cols), 7.0, device=device)
    assert _call(device, kind=LOGITS, input=dx, input_stride=depth, rows=18, depth=depth, cols=cols, weights=dw,
                 weight_stride=depth, output=out, output_stride=cols, norm_weight=dg, eps=1e-5, input_rows=rows,
                 row_index=torch.from_numpy(wanted).to(device)) == 0  # fmt: skip
    got, n = out.cpu().numpy(), _normed(x, g)
    assert np.all(got[3] == 0)
    assert _call(device, kind=LOGITS, input=dx, input_stride=depth, rows=18, depth=depth, cols=cols, weights=dw,
                 weight_stride=depth, output=out, output_stride=cols, norm_weight=dg, eps=0.0, input_rows=rows,
                 row_index=torch.from_numpy(wanted).to(device)) == 0  # fmt: skip
    assert np.all(out.cpu().numpy()[3] == 0)  # also without an eps: no 0 / 0
    keep = np.arange(18) != 3
    want = n[wanted[keep]] @ w.T
    assert np.all(np.abs(got[keep] - want) <= _bound(n[wanted[keep]], w.T))


@pytest.mark.parametrize("pool", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize(("rows", "heads", "dim", "depth"), [(1, 1, 32, 32), (17, 3, 32, 96), (33, 4, 64, 256), (16, 8, 32, 256)])
def test_rope_append(device, pool, rows, heads, dim, depth) -> None:
    """q to the output, k and v to their slots; a slot outside the pool and a position outside the
    tables write nothing there. Odd head counts put two parts of q | k | v in one column tile."""
    model = heads * dim
    rng, x, w, g, dx, dw, dg = _inputs(device, rows, depth, 3 * model)
    positions, slots = rng.integers(0, 50, rows), rng.permutation(rows + 5)[:rows]
    if rows > 2:
        positions[1], slots[2] = 50, -1
    angles = rng.standard_normal((50, dim // 2))
    cos, sin = np.cos(angles).astype(np.float32), np.sin(angles).astype(np.float32)
    on = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    keys, values = (torch.zeros((rows + 5, model), dtype=pool, device=device) for _ in range(2))
    out = torch.zeros((rows, 3 * model), device=device)
    assert _call(device, kind=ROPE_APPEND, input=dx, input_stride=depth, rows=rows, depth=depth, cols=3 * model,
                 weights=dw, weight_stride=3 * model, output=out, output_stride=3 * model, norm_weight=dg, eps=1e-5,
                 positions=on(positions), slots=on(slots), cos_table=on(cos), sin_table=on(sin), table_rows=50,
                 key_pool=keys, value_pool=values, num_slots=rows + 5, num_heads=heads, head_dim=dim,
                 pool_dtype=int(pool == torch.bfloat16)) == 0  # fmt: skip
    n = _normed(x, g)
    y, slack = n @ w, _bound(n, w)
    parts = [y[:, i * model : (i + 1) * model].reshape(rows, heads, dim) for i in range(3)]
    tols = [slack[:, i * model : (i + 1) * model].reshape(rows, heads, dim) for i in range(3)]
    safe = np.minimum(positions, 49)
    c, s = cos[safe][:, None].astype(np.float64), sin[safe][:, None].astype(np.float64)
    half = dim // 2
    want, tol = [], []
    for i in range(2):
        lo, hi = parts[i][..., :half], parts[i][..., half:]
        want.append(np.concatenate([lo * c - hi * s, hi * c + lo * s], -1))
        both = tols[i][..., :half] + tols[i][..., half:] + 3e-7 * (np.abs(lo) + np.abs(hi))
        tol.append(np.concatenate([both, both], -1))
    got = out.cpu().numpy()
    live = positions < 50
    assert np.all(np.abs(got[live, :model].reshape(-1, heads, dim) - want[0][live]) <= tol[0][live])
    assert np.all(got[~live] == 0) and np.all(got[:, model:] == 0)
    step = 2.0**-8 if pool == torch.bfloat16 else 0.0
    for held, w64, t in ((keys, want[1], tol[1]), (values, parts[2], tols[2])):
        held = held.float().cpu().numpy().reshape(-1, heads, dim)
        stored = live & (slots >= 0)
        assert np.all(np.abs(held[slots[stored]] - w64[stored]) <= t[stored] + step * np.abs(w64[stored]))
        rest = np.setdiff1d(np.arange(rows + 5), slots[stored])
        assert np.all(held[rest] == 0)


def test_refused_arguments(device) -> None:
    """Depths that are no multiple of 16 or past the limit, head_dim 128, overlapping strides."""
    x = torch.zeros((4, 64), device=device)
    base = dict(kind=ADD, input=x, input_stride=64, rows=4, depth=64, cols=64, weights=x, weight_stride=64, output=x,
                output_stride=64)  # fmt: skip
    assert _call(device, **{**base, "rows": 0}) == 0
    assert _call(device, **{**base, "depth": 40}) == -2
    assert _call(device, **{**base, "depth": 1552, "input_stride": 1552}) == -2
    assert _call(device, **{**base, "input_stride": 60}) == -1
    assert _call(device, **{**base, "output_stride": 60}) == -1
    assert _call(device, **{**base, "kind": LOGITS}) == -1  # no norm weight
    assert _call(device, **{**base, "kind": ROPE_APPEND, "norm_weight": x, "head_dim": 128}) == -2
    assert _call(device, **{**base, "kind": 9, "norm_weight": x}) == -1
