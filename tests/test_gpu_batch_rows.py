"""The batched step at the edges of its levels' dispatch: 255 and 256 rows
(sample groups, a wave per row), batches around a wave's samples (one and four
per lane), forward rows of 1 to 399 entries (16, 64, 65 and 128 among them),
backward rows of at most 9 and the outputs' empty ones, with and without
tombstones inside them -- bit for bit with the batched oracle. (Empty forward
rows, long backward rows and the other monoids: test_gpu_batch_entries.)"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import nets
import plastax_amd as px
import plastax_amd.numpy as jnp
from test_gpu_parity import _equal, assert_same_state

pytestmark = pytest.mark.gpu

N_IN = 400


class _Prune(px.PruneConn):
    def predicate(self, u, c, cid, g):
        h = c[px.FROM_ID, cid] * jnp.int32(7) + c[px.TO_ID, cid] * jnp.int32(13)
        return (h % jnp.int32(9)) == jnp.int32(0)


@pytest.mark.parametrize("prune", [False, True])
@pytest.mark.parametrize("batch", [1, 5, 16, 64, 65, 128, 132, 258])
@pytest.mark.parametrize("hidden", [255, 256])
def test_batched_levels_match_the_oracle(oracle, hidden: int, batch: int, prune: bool) -> None:
    from oracle import batched as ob

    fwd = nets.MaxForward() if batch == 5 else nets.TanhForward()
    base = nets.make_trained_net("BR", fwd, nets.TanhBackward(), px.optim.momentum(1e-2, 0.9, nets.GRAD_PRE_ACT),
                                 px.Propagation.TOPOLOGICAL)
    body = {"batch_reduction": px.MeanFloatFirstRest()}
    if prune:
        body["prune_conn"] = _Prune()
    net = type("Net", (base,), body)
    rng = np.random.default_rng(hidden + batch)
    lens = rng.integers(1, 30, hidden)
    lens[:5] = [16, 64, 65, 399, 128]
    src = [rng.choice(N_IN, n, replace=False) for n in lens]
    dst = [np.full(n, N_IN + j) for j, n in enumerate(lens)]
    for j in range(9):  # the output level: few, long rows
        src.append(N_IN + rng.choice(hidden, 200 if j else hidden, replace=False))
        dst.append(np.full(src[-1].size, N_IN + hidden + j))
    src, dst = np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32)
    w = (rng.standard_normal(src.size) * 0.2).astype(np.float32)
    n = N_IN + hidden + 9
    static, state = px.NetworkBuilder.from_edges(net, n, src, dst, weights=w, input_ids=np.arange(N_IN),
                                                 output_ids=np.arange(n - 9, n), globals_=None, device="cuda")
    o = nets.oracle_for(oracle, net, static, state)
    orc = ob.OracleBatch(o, batch)
    step = px.make_step(net, static, batch_size=batch)
    for k in range(2):
        x = rng.standard_normal((batch, N_IN)).astype(np.float32)
        t = rng.standard_normal((batch, 9)).astype(np.float32)
        print(f"batched level {hidden} batch {batch} prune {prune} step {k}", flush=True)
        res = step(state, px.StepInputs(x, t))
        state = res.state
        lo = orc.step(x, t)
        torch.cuda.synchronize()
        assert _equal(np.float32([float(res.loss)]), np.float32([lo])), f"loss at step {k}"
        assert_same_state(static, state, o, f"step {k}")
