"""The generic fold's blocks (plx_gen_fold): map values evaluated side by side
and folded per row in order. Rows per workgroup 1, 3 and 64's neighbourhood,
rows longer than a window of entries, empty rows, tombstones inside rows, one
to eight components with every monoid -- bit for bit with the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import nets
import plastax_amd as px
import plastax_amd.numpy as jnp
from plastax_amd import _lib
from test_gpu_parity import assert_same_state

pytestmark = pytest.mark.gpu

SRC = 1500
COLS = tuple(px.FieldSpec.float32(f"part{k}") for k in range(7))


class _Eight(px.ForwardPass):
    combine = (px.monoid.sum_, px.monoid.max_, px.monoid.min_, px.monoid.prod, px.monoid.sum_, px.monoid.max_,
               px.monoid.sum_, px.monoid.min_)

    def map(self, u, dst, src, c, cid, g):
        w, x = c[px.WEIGHT, cid], u[px.ACTIVATION, src]
        return (w * x, w, x, jnp.float32(1.0) + w * jnp.float32(0.01), jnp.float32(1.0), jnp.abs(w) * x, jnp.abs(w),
                w * x)

    def apply(self, u, i, g, acc):
        return px.UnitWrite.of((px.ACTIVATION, jnp.tanh(acc[0])), *((f, acc[k + 1]) for k, f in enumerate(COLS)))


class _One(px.ForwardPass):
    combine = (px.monoid.sum_,)

    def map(self, u, dst, src, c, cid, g):
        return (jnp.abs(c[px.WEIGHT, cid]) * jnp.tanh(u[px.ACTIVATION, src]),)

    def apply(self, u, i, g, acc):
        return px.UnitWrite.of((px.ACTIVATION, jnp.tanh(acc[0])))


class _Prune(px.PruneConn):
    def predicate(self, u, c, cid, g):
        h = c[px.FROM_ID, cid] * jnp.int32(7) + c[px.TO_ID, cid] * jnp.int32(13)
        return (h % jnp.int32(5)) == jnp.int32(0)


@pytest.mark.parametrize("prune", [False, True])
@pytest.mark.parametrize("fwd", [_One(), _Eight()])
@pytest.mark.parametrize("width", [1, 3, 700, 2049, 5000])
def test_generic_fold_blocks_match_the_oracle(oracle, width: int, fwd, prune: bool) -> None:
    rng = np.random.default_rng(width)
    total = 20000
    cut = np.sort(rng.integers(0, total, width - 1)) if width > 1 else np.zeros(0, np.int64)
    lens = np.minimum(np.diff(np.concatenate([[0], cut, [total]])), SRC)
    lens[0] = 1301
    if width > 3:
        lens[2] = 0
    src = np.concatenate([rng.choice(SRC, n, replace=False) for n in lens]).astype(np.int32)
    dst = (SRC + np.repeat(np.arange(width), lens)).astype(np.int32)
    w = (rng.standard_normal(src.size) * 0.1).astype(np.float32)
    body = dict(forward_pass=fwd, extra_unit_fields=COLS)
    if prune:
        body["prune_conn"] = _Prune()
    net = type("Net", (px.Network,), body)
    static, state = px.NetworkBuilder.from_edges(
        net, SRC + width, src, dst, weights=w, input_ids=np.arange(SRC), output_ids=np.arange(SRC, SRC + width),
        globals_=None, device="cuda")
    o = nets.oracle_for(oracle, net, static, state)
    step = px.make_step(net, static)
    for k in range(2):
        x = rng.standard_normal(SRC).astype(np.float32)
        print(f"generic fold width {width} prune {prune} step {k}", flush=True)
        state = step(state, px.StepInputs(x)).state
        o.step(x)
        torch.cuda.synchronize()
        assert_same_state(static, state, o, f"step {k}")


def test_generic_fold_of_more_rows_than_a_launch() -> None:
    """2^30 rows and some, at 64 a workgroup of 256 lanes: every row's
    accumulator takes its fold (no entries: the identity, 2 here)."""
    dev = torch.device("cuda", 0)
    n = (1 << 30) + 130
    if torch.cuda.mem_get_info(dev)[0] < 40 << 30:
        pytest.skip("needs three 4 GB columns")
    print(f"generic fold of {n} rows", flush=True)
    units = torch.arange(n, dtype=torch.int32, device=dev)
    ptr = torch.zeros(n + 1, dtype=torch.int32, device=dev)
    acc = (units % 1021).float()
    ids = torch.zeros(4, dtype=torch.int32, device=dev)
    d = _lib.plx_gen_fold_desc()
    d.nrows, d.ncomp, d.num_units, d.batch, d.prog.nout = n, 1, n, 1, 1
    d.monoid[0], d.identity[0], d.acc[0] = 1, 2.0, acc.data_ptr()  # product
    d.row_unit, d.row_ptr, d.from_id = units.data_ptr(), ptr.data_ptr(), ids.data_ptr()
    _lib.call("plx_gen_fold", d, None)
    want = (units % 1021).float() * 2.0
    assert torch.equal(acc, want)
