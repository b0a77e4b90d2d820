"""The batched step's column kernels at the edges of their workgroups and
chunks: plx_spread_cols (four samples a lane, or one where the batch is no
multiple of four or a column is not 16-byte aligned), plx_scatter_batch, and
plx_reduce_cols (16 units a workgroup, 64 samples a chunk) -- the same bits
as the sums in sample order."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from plastax_amd import _lib
from test_gpu_parity import _equal

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _pointers(tensors):
    return (ctypes.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("batch", [1, 3, 4, 63, 64, 65, 128, 258])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 1000])
def test_columns_spread_scatter_and_reduce(n: int, batch: int, offset: int) -> None:
    rng = np.random.default_rng(1000 * n + batch)
    print(f"columns {n} batch {batch} offset {offset}", flush=True)
    ncols = _lib.PLX_MAX_BATCH_COLS if n == 17 else 3
    cols = [(rng.standard_normal(n) * 10.0 ** rng.integers(-3, 4)).astype(np.float32) for _ in range(ncols)]
    cols[0][0] = np.inf
    src = [torch.from_numpy(c).to(DEV) for c in cols]
    out = [torch.zeros(n * batch + offset, device=DEV)[offset:] for _ in cols]
    src_p, out_p = _pointers(src), _pointers(out)  # (kept: an address alone would not keep the arrays)
    _lib.call("plx_spread_cols", n, batch, ncols, ctypes.addressof(src_p), ctypes.addressof(out_p), None)
    for c, o in zip(cols, out):
        assert _equal(o.cpu().numpy(), np.repeat(c, batch)), "spread"

    k = max(1, n // 3)
    ids = rng.permutation(n)[:k].astype(np.int32)
    x = rng.standard_normal((batch, k)).astype(np.float32)
    ids_d, x_d = torch.from_numpy(ids).to(DEV), torch.from_numpy(x).to(DEV)
    _lib.call("plx_scatter_batch", k, batch, ids_d.data_ptr(), x_d.data_ptr(), out[0].data_ptr(), None)
    want = np.repeat(cols[0], batch).reshape(n, batch)
    want[ids] = x.T
    assert _equal(out[0].cpu().numpy(), want.ravel()), "scatter"

    for shift in range(3):  # every mode in every place
        rows = [rng.standard_normal((n, batch)).astype(np.float32) for _ in cols]
        modes = [(j + shift) % 3 for j in range(ncols)]  # MEAN, SUM, FIRST
        for o, r in zip(out, rows):
            o.copy_(torch.from_numpy(r.ravel()))
        red = [torch.zeros(n, device=DEV) for _ in cols]
        arr = (ctypes.c_int32 * ncols)(*modes)
        red_p = _pointers(red)
        _lib.call("plx_reduce_cols", n, batch, ncols, ctypes.addressof(arr), ctypes.addressof(out_p),
                  ctypes.addressof(red_p), None)
        for mode, r, got in zip(modes, rows, red):
            s = r[:, 0].copy()
            if mode != 2:
                for b in range(1, batch):
                    s += r[:, b]
            if mode == 0:
                s /= np.float32(batch)
            assert _equal(got.cpu().numpy(), s), f"reduce mode {mode}"


def test_columns_of_more_lanes_than_a_launch() -> None:
    """A column of more than 2^32 values (one lane each: an odd batch), and
    more units than one reduction launch takes."""
    free, _ = torch.cuda.mem_get_info(DEV)
    if free < 60 << 30:
        pytest.skip("needs two 17 GB columns")
    n, batch, part = 1_048_577, 4099, 8192
    col = (torch.arange(n, device=DEV) % 8191).float()
    out = torch.zeros((n, batch), device=DEV)
    src_p, out_p = _pointers([col]), _pointers([out])
    print(f"columns {n} batch {batch}", flush=True)
    _lib.call("plx_spread_cols", n, batch, 1, ctypes.addressof(src_p), ctypes.addressof(out_p), None)
    for u in range(0, n, part):
        assert bool((out[u : u + part] == col[u : u + part, None]).all()), f"spread, units {u} .."
    ids = torch.randperm(n, device=DEV).to(torch.int32)
    x = torch.empty((batch, n), device=DEV)
    k = torch.arange(n, device=DEV)
    for b in range(0, batch, 64):
        bs = torch.arange(b, min(b + 64, batch), device=DEV)
        x[b : b + 64] = ((k[None] * 31 + bs[:, None] * 7) % 65521).float()
    _lib.call("plx_scatter_batch", n, batch, ids.data_ptr(), x.data_ptr(), out.data_ptr(), None)
    for u in range(0, n, part):
        assert torch.equal(out[ids[u : u + part].long()], x[:, u : u + part].t()), f"scatter, inputs {u} .."
    del out, x
    n = (1 << 28) + 17
    cols = (torch.arange(2 * n, device=DEV) % 4093).float()
    red = [torch.zeros(n, device=DEV) for _ in range(3)]
    modes = (ctypes.c_int32 * 3)(0, 1, 2)  # MEAN, SUM, FIRST
    src_p, red_p = _pointers([cols] * 3), _pointers(red)
    print(f"reduction of {n} units", flush=True)
    _lib.call("plx_reduce_cols", n, 2, 3, ctypes.addressof(modes), ctypes.addressof(src_p), ctypes.addressof(red_p),
              None)
    both = cols[::2] + cols[1::2]
    for got, want in zip(red, (both / 2, both, cols[::2])):
        assert torch.equal(got, want)
