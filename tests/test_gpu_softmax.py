"""Softmax cross-entropy at the edges of its two forms (plx_loss_softmax_ce):
one workgroup per sample up to PLX_SOFTMAX_ONE outputs, a workgroup per
256-output piece beyond; whole and broken pieces, one sample and several,
against the oracle bit for bit (each piece's sum and the sum over the pieces
keep their order). Inputs with a tied maximum, -inf and, for the maximum's
scan, NaN."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from plastax_amd import _lib
from plastax_amd.step import softmax_partials
from test_gpu_parity import _equal, _first_diff

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("special", [None, "tied", "inf", "nan"])
@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("n", [1, 37, 64, 255, 257, 1023, 1025, 4095, 4096, 4097, 65537])
def test_softmax_forms_match_the_oracle(oracle, n: int, batch: int, special) -> None:
    rng = np.random.default_rng(n + batch)
    units = n + 5
    ids = rng.permutation(units)[:n].astype(np.int32)
    act = (rng.standard_normal((units, batch)) * 3).astype(np.float32)
    if special == "tied":
        act[ids[rng.integers(0, n, 3)]] = 11.0
    elif special == "inf":
        act[ids[n // 2]] = -np.inf
    elif special == "nan":
        act[ids[n // 2]] = np.nan
    t = rng.random((batch, n)).astype(np.float32)
    t /= t.sum(1, keepdims=True)
    dev = [torch.from_numpy(v).to(DEV) for v in (ids, act, t)]
    seed = torch.zeros((units, batch), device=DEV)
    losses = torch.empty(batch, device=DEV)
    parts = softmax_partials(n, batch, DEV)
    print(f"softmax n {n} batch {batch} {special}", flush=True)
    _lib.call("plx_loss_softmax_ce", n, dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr(), seed.data_ptr(),
              None if parts is None else parts.data_ptr(), losses.data_ptr(), batch, None)
    torch.cuda.synchronize()
    got_seed, got_loss = seed.cpu().numpy(), losses.cpu().numpy()
    lib = oracle.load()
    for b in range(batch):
        a, tb = np.ascontiguousarray(act[:, b]), np.ascontiguousarray(t[b])
        want, terms = np.zeros(n, np.float32), np.zeros(n, np.float32)
        f32 = [v.ctypes.data_as(ctypes.POINTER(ctypes.c_float)) for v in (a, tb, want, terms)]
        at = ids.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))
        val = np.float32(lib.ox_loss_softmax_ce(f32[0], at, n, f32[1], f32[2], f32[3], 256))
        col = np.ascontiguousarray(got_seed[ids, b])
        if special == "nan":  # (a NaN's payload is nobody's contract)
            assert np.array_equal(col, want, equal_nan=True) and np.array_equal(got_loss[b], val, equal_nan=True)
            continue
        assert _equal(col, want), f"sample {b}: seed {_first_diff(col, want)}"
        assert _equal(got_loss[b : b + 1], np.asarray([val])), f"sample {b}: loss {got_loss[b]!r} {val!r}"
