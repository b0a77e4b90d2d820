"""The radix passes of plx_sort at the edges of their waves' and tiles' spans
and of their two forms (each scatter reads the digit table itself up to 256
tiles; beyond, the table is scanned), with counts on the device below the
bound (tiles without an element; none at all): the stable order, and the list
past the count as it was."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from test_gpu_growth import _kernels

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
FORM = 256 * 4096  # the largest bound whose table each scatter reads


@pytest.mark.parametrize("spread", [1, 3, 100000])
@pytest.mark.parametrize("n_max,count", [
    (1025, 1025), (4096, 4095), (4097, 1), (4097, 4097), (5000, 0), (8192, 255), (8192, 257), (70000, 4352),
    (270336, 266240), (FORM, 300001), (FORM, FORM), (FORM + 1, FORM + 1), (FORM + 4097, 5000),
])
def test_radix_passes_sort_stably(n_max: int, count: int, spread: int) -> None:
    rng = np.random.default_rng(n_max + count + spread)
    print(f"radix sort {count} of {n_max}, keys below {spread}", flush=True)
    k = _kernels()
    size = n_max + 7
    hi, lo = (rng.integers(0, spread, size).astype(np.int32) for _ in range(2))
    vals = rng.permutation(size)[:n_max].astype(np.int32)
    vals[count:] = 2_000_000_000  # no element of the columns
    hi_t, lo_t, v_t = (torch.from_numpy(a).to(DEV) for a in (hi, lo, vals))
    n_dev = torch.tensor([count], dtype=torch.int32, device=DEV)
    k.sort(v_t, n_max, [(0, 17, lo_t, None), (0, 32, hi_t, None)], n_dev=n_dev)
    got = v_t.cpu().numpy()
    head = vals[:count]
    assert np.array_equal(got[:count], head[np.lexsort((lo[head], hi[head]))])
    assert np.array_equal(got[count:], vals[count:]), "past the count"
