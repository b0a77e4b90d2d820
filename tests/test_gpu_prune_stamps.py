"""PruneConn's launch over the whole slab and per bucket: an edge killed while
its bucket holds Adam's step count as one number keeps that count in its own
column. Buckets that share the count take one launch, buckets with counts of
their own (another number, one per edge) one each; a bucket without live edges
has no say, and capacities that are no multiple of four put padding between
the buckets -- every column, the counts at the killed slots among them, against
the oracle."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

import nets
import plastax_amd as px
import plastax_amd.numpy as jnp
from plastax_amd import grow, synth
from test_gpu_parity import assert_same_state

pytestmark = pytest.mark.gpu


class _Prune(px.PruneConn):
    def predicate(self, u, c, cid, g):
        h = c[px.FROM_ID, cid] * jnp.int32(7) + c[px.TO_ID, cid] * jnp.int32(13) + g["step"]
        return (h % jnp.int32(23)) == jnp.int32(0)


# Per bucket: one count, "edge" (a count per edge) or None (no live edge); and
# the launches of a step.
STARTS = {
    "shared": ([3, 3, 3, 3], 1),
    "shared, first and last empty": ([None, 5, 5, None], 1),
    "two counts": ([3, 7, 7, 3], 4),
    "two counts, one bucket empty": ([9, None, 2, 2], 4),
    "a count per edge": ([4, "edge", 4, None], 4),
    "a count per edge everywhere": (["edge", "edge", "edge", None], 1),
}


@pytest.mark.parametrize("mode", ["tiled", "churn"])
@pytest.mark.parametrize("start", list(STARTS))
def test_killed_edges_keep_their_step_count(oracle, monkeypatch, start: str, mode: str) -> None:
    counts, launches = STARTS[start]
    base = nets.make_trained_net("PS", nets.TanhForward(), nets.TanhBackward(), px.optim.adam(1e-2, nets.GRAD_PRE_ACT),
                                 px.Propagation.TOPOLOGICAL)

    class Net(base):
        prune_conn = _Prune()

    e = synth.c2_topological(seed=6, scale=512, layers=5)
    g = {"step": np.int32(0)}
    static, state = px.NetworkBuilder.from_edges(Net, e.num_units, e.src, e.dst, weights=e.weight,
                                                 input_ids=e.input_ids, output_ids=e.output_ids, globals_=g,
                                                 capacity_headroom=0.1, device="cuda")
    rng = np.random.default_rng(len(start))
    buckets = []
    for b, (bucket, count) in enumerate(zip(state.conns, counts)):
        cap = bucket["dead"].numel() // 4 * 4 - 4 + b  # b past a multiple of four
        assert int((bucket["dead"][cap:] == 0).sum()) == 0  # (headroom only is cut off)
        new = {name: col[:cap].clone() for name, col in bucket.items()}
        if count is None:
            new["dead"].fill_(1)
        elif count == "edge":
            new["opt/t"].copy_(torch.from_numpy(rng.integers(1, 9, cap).astype(np.float32)))
        else:
            new["opt/t"].fill_(float(count))
        buckets.append(new)
    static = dataclasses.replace(static, level_capacities=tuple(b["dead"].numel() for b in buckets))
    state.conns = tuple(buckets)
    o = nets.oracle_for(oracle, Net, static, state)
    step = px.make_step(Net, static)
    step.arena_mode = mode
    if mode == "churn":
        o.tile = None
    seen = []
    site_eval = grow.Kernels.site_eval
    monkeypatch.setattr(grow.Kernels, "site_eval", lambda self, *a, **k: (seen.append(k["n"]), site_eval(self, *a, **k))[1])
    for k in range(4):
        state.globals_ = o.globals_ = {"step": np.int32(k)}
        x = rng.standard_normal(e.input_ids.size).astype(np.float32)
        t = rng.standard_normal(e.output_ids.size).astype(np.float32)
        print(f"stamps {start} {mode} step {k}", flush=True)
        seen.clear()
        state = step(state, px.StepInputs(x, t)).state
        assert len(seen) == launches, seen
        o.step(x, t)
        assert_same_state(static, state, o, f"step {k}")
