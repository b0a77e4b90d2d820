"""The forward sweep's block sizes (fwd_block_rows): levels of few rows get
blocks of fewer rows. Each level width crosses a line of that rule (one row a
block, one workgroup per CU, eight rows a block, two workgroups per CU); rows
of no, one, odd and several thousand edges (more than one window of a block).
Bit for bit with the oracle: every row folds its edges in slot order whatever
block it is in."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import nets
import plastax_amd as px
from test_gpu_parity import assert_same_state

pytestmark = pytest.mark.gpu

SRC = 6000


def _ragged(width: int, total: int, seed: int):
    """SRC inputs -> width units; row lengths random, some empty, the first
    row longer than a window of positions where the total allows."""
    rng = np.random.default_rng(seed)
    cut = np.sort(rng.integers(0, total, width - 1)) if width > 1 else np.zeros(0, np.int64)
    lens = np.diff(np.concatenate([[0], cut, [total]]))
    lens[0] = min(max(int(lens[0]), 5003), SRC)
    lens = np.minimum(lens, SRC)
    if width > 3:
        lens[2] = 0
    src = np.concatenate([rng.choice(SRC, n, replace=False) for n in lens]).astype(np.int32)
    dst = (SRC + np.repeat(np.arange(width), lens)).astype(np.int32)
    w = (rng.standard_normal(src.size) * 0.1).astype(np.float32)
    return src, dst, w


class _Sum(px.Network):
    forward_pass = nets.TanhForward()


class _Max(px.Network):
    forward_pass = nets.MaxForward()


@pytest.mark.parametrize("net", [_Sum, _Max])
@pytest.mark.parametrize("width", [1, 2, 10, 255, 257, 2047, 2049, 4096, 4097])
def test_blocks_of_few_rows_match_the_oracle(oracle, net, width: int) -> None:
    src, dst, w = _ragged(width, 30000, width)
    static, state = px.NetworkBuilder.from_edges(
        net, SRC + width, src, dst, weights=w, input_ids=np.arange(SRC), output_ids=np.arange(SRC, SRC + width),
        globals_=None, device="cuda")
    o = nets.oracle_for(oracle, net, static, state)
    step = px.make_step(net, static)
    rng = np.random.default_rng(1)
    for k in range(2):
        x = rng.standard_normal(SRC).astype(np.float32)
        print(f"forward split width {width} step {k}", flush=True)
        state = step(state, px.StepInputs(x)).state
        o.step(x)
        torch.cuda.synchronize()
        assert_same_state(static, state, o, f"step {k}")
