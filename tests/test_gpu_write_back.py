"""Columns copied back into their logical slots (plx_write_slots,
plx_fill_live) against numpy: counts around a workgroup's span, aligned and
unaligned columns (the four- and one-position forms), byte and 4-byte columns,
slots outside the bucket, a count on the device, columns of killed edges; and a
net's logical view read after every step and after several, with kills in
between, against the oracle."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import nets
import plastax_amd as px
import plastax_amd.numpy as jnp
from plastax_amd import _lib, synth
from test_gpu_parity import assert_same_state

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [1, 3, 4, 255, 1023, 1024, 1025, 8191, 70001])
def test_write_slots_matches_numpy(n: int, shift: int) -> None:
    rng = np.random.default_rng(n + shift)
    room = (n + 3) // 4 * 4
    limit = n + 50
    slot = np.full(shift + room, -1, np.int32)
    slot[shift : shift + n] = rng.permutation(limit)[:n]
    slot[shift + n // 2] = -1
    f, g = (rng.standard_normal(shift + room).astype(np.float32) for _ in range(2))
    u = rng.integers(0, 2, shift + room).astype(np.uint8)
    dead = rng.integers(0, 2, shift + room).astype(np.uint8)
    live = max(n - 2, 0)
    count = max(n - 1, 1)
    want = [np.zeros(limit, np.float32), np.zeros(limit, np.float32), np.zeros(limit, np.uint8),
            np.zeros(limit, np.uint8)]
    for p in range(count):
        s = slot[shift + p]
        if s < 0:
            continue
        want[0][s] = f[shift + p]
        want[2][s] = u[shift + p]
        if p >= live or dead[shift + p]:
            want[1][s] = g[shift + p]
            want[3][s] = dead[shift + p]
    ts = [torch.from_numpy(v).to(DEV) for v in (slot, f, g, u, dead)]
    out = [torch.from_numpy(np.zeros_like(v)).to(DEV) for v in want]
    n_dev = torch.tensor([count], dtype=torch.int32, device=DEV)
    at = [t.data_ptr() + shift * t.element_size() for t in ts]
    src = (ctypes.c_void_p * 4)(at[1], at[2], at[3], at[4])
    dst = (ctypes.c_void_p * 4)(*[t.data_ptr() for t in out])
    size = (ctypes.c_int32 * 4)(4, 4, 1, 1)
    print(f"write slots n {n} shift {shift}", flush=True)
    _lib.call("plx_write_slots", n, n_dev.data_ptr(), at[0], limit, 4, ctypes.addressof(src), ctypes.addressof(dst),
              ctypes.addressof(size), 0b1010, at[4], live, None)
    fill = torch.zeros(shift + room, device=DEV)
    _lib.call("plx_fill_live", n, at[4], 2.5, fill.data_ptr(), None)
    torch.cuda.synchronize()
    for got, ref in zip(out, want):
        assert np.array_equal(got.cpu().numpy(), ref)
    assert np.array_equal(fill.cpu().numpy()[:n], np.where(dead[shift : shift + n] == 0, np.float32(2.5), 0))


class _Prune(px.PruneConn):
    def predicate(self, u, c, cid, g):
        h = c[px.FROM_ID, cid] * jnp.int32(7) + c[px.TO_ID, cid] * jnp.int32(13) + g["step"]
        return (h % jnp.int32(61)) == jnp.int32(0)


@pytest.mark.parametrize("mode", ["tiled", "churn"])
@pytest.mark.parametrize("every", [1, 3])
def test_logical_view_after_kills_matches_the_oracle(oracle, mode: str, every: int) -> None:
    base = nets.make_trained_net("WB", nets.TanhForward(), nets.TanhBackward(), px.optim.adam(1e-2, nets.GRAD_PRE_ACT),
                                 px.Propagation.TOPOLOGICAL)

    class Net(base):
        prune_conn = _Prune()

    e = synth.c2_topological(seed=2, scale=256, layers=4)
    g = {"step": np.int32(0)}
    static, state = px.NetworkBuilder.from_edges(Net, e.num_units, e.src, e.dst, weights=e.weight,
                                                 input_ids=e.input_ids, output_ids=e.output_ids, globals_=g,
                                                 capacity_headroom=0.3, device="cuda")
    o = nets.oracle_for(oracle, Net, static, state)
    step = px.make_step(Net, static)
    step.arena_mode = mode
    if mode == "churn":
        o.tile = None
    rng = np.random.default_rng(3)
    for k in range(7):
        state.globals_ = o.globals_ = {"step": np.int32(k // 2 if k % 2 else k)}
        x = rng.standard_normal(e.input_ids.size).astype(np.float32)
        t = rng.standard_normal(e.output_ids.size).astype(np.float32)
        state = step(state, px.StepInputs(x, t)).state
        o.step(x, t)
        if k % every == every - 1:
            print(f"write back {mode} step {k}", flush=True)
            assert_same_state(static, state, o, f"step {k}")


@pytest.mark.parametrize("strided", [("weight",), ("dead", "opt/t"), ("dead", "weight", "opt/m", "opt/v", "opt/t")])
def test_logical_columns_that_are_strided_views(oracle, strided: tuple[str, ...]) -> None:
    """A caller's bucket columns that are strided views (the host-built layout
    reads any): the copy back follows their strides and leaves the storage
    between their elements alone."""
    base = nets.make_trained_net("WS", nets.TanhForward(), nets.TanhBackward(), px.optim.adam(1e-2, nets.GRAD_PRE_ACT),
                                 px.Propagation.TOPOLOGICAL)

    class Net(base):
        prune_conn = _Prune()

    e = synth.c2_topological(seed=4, scale=512, layers=3)
    g = {"step": np.int32(0)}
    static, state = px.NetworkBuilder.from_edges(Net, e.num_units, e.src, e.dst, weights=e.weight,
                                                 input_ids=e.input_ids, output_ids=e.output_ids, globals_=g,
                                                 capacity_headroom=0.3, device="cuda")
    o = nets.oracle_for(oracle, Net, static, state)
    buckets, between = [], []
    for bucket in state.conns:
        new = dict(bucket)
        for name in strided:
            room = torch.full((2 * bucket[name].numel(),), 77, dtype=bucket[name].dtype, device=DEV)
            new[name] = room[::2].copy_(bucket[name])
            between.append(room[1::2])
        buckets.append(new)
    state.conns = tuple(buckets)
    step = px.make_step(Net, static)
    step.layout_build = "host"
    rng = np.random.default_rng(5)
    for k in range(3):
        state.globals_ = o.globals_ = {"step": np.int32(k)}
        x = rng.standard_normal(e.input_ids.size).astype(np.float32)
        t = rng.standard_normal(e.output_ids.size).astype(np.float32)
        print(f"write back, strided {strided}, step {k}", flush=True)
        state = step(state, px.StepInputs(x, t)).state
        o.step(x, t)
        assert_same_state(static, state, o, f"step {k}")
        assert all(bool((gap == 77).all()) for gap in between)
