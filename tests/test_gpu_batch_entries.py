"""plx_forward_batch and plx_backward_batch called on descriptors of their
own: every monoid, rows of no entries and around a 64-entry chunk and a
256-entry window, in sample groups (255 rows) and a wave per row (256), with
each way an entry is named and skipped -- a tombstone at its position
(``dead``), a liveness byte in list order (``live``), a position table
(``pos``) -- and constant map factors, bit for bit with the fold in order."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from plastax_amd import _lib
from test_gpu_parity import _equal

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
OPS = {0: np.add, 1: np.multiply, 2: np.maximum, 3: np.minimum}
IDENT = {0: 0.0, 1: 1.0, 2: -np.inf, 3: np.inf}
WAYS = ["plain", "dead", "live", "pos", "pos dead", "pos live dead", "w const", "x const dead"]


def _rows(rng: np.random.Generator, nrows: int) -> np.ndarray:
    lens = rng.integers(0, 12, nrows)
    lens[: 12] = [0, 1, 7, 8, 15, 16, 63, 64, 65, 130, 257, 300]
    return rng.permutation(lens)


@pytest.mark.parametrize("batch", [66, 132])
@pytest.mark.parametrize("monoid", [0, 1, 2, 3])
@pytest.mark.parametrize("nrows", [255, 256])
def test_batched_entries_match_the_fold_in_order(nrows: int, monoid: int, batch: int) -> None:
    rng = np.random.default_rng(1000 * nrows + 10 * monoid + batch)
    lens = _rows(rng, nrows)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n_ent, n_units = int(ptr[-1]), 300
    other = rng.integers(0, n_units, n_ent).astype(np.int32)
    unit = rng.permutation(n_units)[:nrows].astype(np.int32)
    weight = (rng.standard_normal(n_ent) + 1.0).astype(np.float32)
    dead = (rng.random(n_ent) < 0.3).astype(np.uint8)
    live = (rng.random(n_ent) < 0.7).astype(np.uint8)
    pos = rng.permutation(n_ent).astype(np.int32)
    x = rng.standard_normal((n_units, batch)).astype(np.float32)
    acc0 = rng.standard_normal((n_units, batch)).astype(np.float32)
    dev = {k: torch.from_numpy(v).to(DEV) for k, v in dict(
        ptr=ptr, other=other, unit=unit, weight=weight, dead=dead, live=live, pos=pos, x=x,
        level=np.zeros(n_units, np.int32), is_input=np.zeros(n_units, np.uint8)).items()}
    op = OPS[monoid]
    for direction in ("forward", "backward"):
        for way in WAYS:
            if direction == "forward" and ("pos" in way or "live" in way):
                continue
            print(f"{direction} rows {nrows} monoid {monoid} batch {batch} {way}", flush=True)
            at = pos if "pos" in way else np.arange(n_ent)
            gone = np.zeros(n_ent, bool)
            if "dead" in way:
                gone |= dead[at] != 0
            if "live" in way:
                gone |= live == 0
            wv = np.full(n_ent, np.float32(1.5)) if "w const" in way else weight[at]
            want = acc0.copy()
            for r in range(nrows):
                s = np.full(batch, np.float32(IDENT[monoid]))
                for e in range(ptr[r], ptr[r + 1]):
                    if not gone[e]:
                        xv = np.float32(0.75) if "x const" in way else x[other[e]]
                        s = op(s, wv[e] * xv)
                want[unit[r]] = op(acc0[unit[r]], s)
            acc = torch.from_numpy(acc0).to(DEV)
            d = _lib.plx_forward_desc() if direction == "forward" else _lib.plx_bwd_batch_desc()
            d.nrows, d.monoid = nrows, monoid
            d.row_unit, d.row_ptr = dev["unit"].data_ptr(), dev["ptr"].data_ptr()
            d.weight, d.acc = dev["weight"].data_ptr(), acc.data_ptr()
            d.dead = dev["dead"].data_ptr() if "dead" in way else None
            d.fin.level, d.fin.is_input, d.fin.fin_level = dev["level"].data_ptr(), dev["is_input"].data_ptr(), 1
            if "w const" in way:
                d.map.flags, d.map.w = _lib.PLX_MAP_W_CONST, 1.5
            if "x const" in way:
                d.map.flags, d.map.x = _lib.PLX_MAP_X_CONST, 0.75
            if direction == "forward":
                d.src, d.x = dev["other"].data_ptr(), dev["x"].data_ptr()
                _lib.call("plx_forward_batch", d, batch, None)
            else:
                d.batch = batch
                d.dst, d.g = dev["other"].data_ptr(), dev["x"].data_ptr()
                d.pos = dev["pos"].data_ptr() if "pos" in way else None
                d.live = dev["live"].data_ptr() if "live" in way else None
                _lib.call("plx_backward_batch", d, None)
            torch.cuda.synchronize()
            assert _equal(acc.cpu().numpy(), want), way
