"""The copy back into the logical buckets, host side (no kernel runs: the
library is a stand-in): a copy that fails is due again at the next read, on
either layout; a tiled arena's view read while another device is current is
copied on the arena's."""

from __future__ import annotations

import types

import pytest
import torch

from plastax_amd import _lib
from plastax_amd._churn import ChurnArena
from plastax_amd._layout import Arena
from plastax_amd.state import NetworkState


class _StandIn:
    """Counts plx_write_slots calls; the one numbered ``fail`` returns an error."""

    def __init__(self) -> None:
        self.writes, self.fail = 0, -1

    def plx_write_slots(self, *args):
        self.writes += 1
        return int(self.writes - 1 == self.fail)

    def plx_last_error(self):
        return b"stand-in"


def _state(monkeypatch, cls) -> tuple[NetworkState, Arena, _StandIn]:
    lib = _StandIn()
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: types.SimpleNamespace(cuda_stream=0))
    dtypes = dict(from_id=torch.int32, to_id=torch.int32, weight=torch.float32, dead=torch.uint8)
    conns = tuple({k: torch.zeros(8, dtype=t) for k, t in dtypes.items()} for _ in range(3))
    arena = cls.__new__(cls)
    arena.device = torch.device("cuda", 0)
    arena.cols = {k: torch.zeros(32, dtype=t) for k, t in dtypes.items()}
    arena.slot = torch.arange(32, dtype=torch.int32)
    arena.bases, arena.caps, arena.lives = [0, 8, 16], [8] * 3, [8] * 3
    arena.live_dev = [torch.tensor([8], dtype=torch.int32)] * 3
    arena.t_name, arena.t_now, arena._written = None, [], set()
    state = NetworkState({"level": torch.zeros(4, dtype=torch.int32)}, conns, None)
    state._arena = arena
    return state, arena, lib


@pytest.mark.parametrize("cls", [Arena, ChurnArena])
@pytest.mark.parametrize("columns", [{"weight"}, {"dead"}, None])
def test_a_failed_copy_back_is_due_again(monkeypatch, cls, columns) -> None:
    state, arena, lib = _state(monkeypatch, cls)
    if cls is ChurnArena and columns == {"dead"}:  # (kills alone take a path of their own)
        monkeypatch.setattr(arena, "_write_kills", lambda conns, written: [
            _lib.check(lib.plx_write_slots(), "kills") for _ in conns], raising=False)
    state._mark_ahead(columns)
    lib.fail = 1
    with pytest.raises(_lib.PlxError):
        state.conns
    lib.writes, lib.fail = 0, -1
    state.conns
    assert lib.writes == 3  # every bucket again
    state.conns
    assert lib.writes == 3  # and then the view is in step
    assert arena._written == set()


def test_the_copy_back_runs_on_the_arenas_device(monkeypatch) -> None:
    state, arena, lib = _state(monkeypatch, Arena)
    current = [1]
    monkeypatch.setattr(torch.cuda, "current_device", lambda: current[-1])

    class On:
        def __init__(self, device) -> None:
            self.index = torch.device(device).index

        def __enter__(self) -> None:
            current.append(self.index)

        def __exit__(self, *exc) -> None:
            current.pop()

    monkeypatch.setattr(torch.cuda, "device", On)
    on = []
    monkeypatch.setattr(lib, "plx_write_slots", lambda *args: on.append(current[-1]) or 0, raising=False)
    state._mark_ahead({"weight"})
    state.conns
    assert on == [0, 0, 0] and current == [1] and arena._written == set()
