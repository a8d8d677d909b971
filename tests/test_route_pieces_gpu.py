"""The device route at the edges of its pieces.

A wavefront holds its pairs in pieces of 512, eight consecutive pairs a lane;
up to 2048 pairs take four wavefronts of one piece, more take sixteen of eight
(a second round past 65536 pairs).  Ids start at any element of their tensor.
Reference: torch's stable argsort of the keys.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from mlx_iqk_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", (torch.int32, torch.int64))
@pytest.mark.parametrize("P", (1, 7, 8, 9, 511, 512, 513, 2047, 2048, 2049, 8191, 8193, 65535, 65536, 65537, 140001))
@pytest.mark.parametrize("E,ppx,skip", [(1, 1, 0), (3, 3, 1), (257, 6, 3)])
def test_route_matches_a_stable_argsort(device, dtype, P, E, ppx, skip):
    print(f"route pieces {dtype} P={P} E={E} ppx={ppx} skip={skip}", flush=True)
    rng = np.random.default_rng(P + E)
    ids = rng.integers(0, E, P + skip)
    ids[rng.random(P + skip) < 0.05] = E  # beyond the stack
    ids[-1] = -1
    got = kernels.route_ids(torch.from_numpy(ids).to(device, dtype)[skip:], E, 1, ppx)
    key = torch.from_numpy(np.where((ids >= 0) & (ids < E), ids, 0)[skip:]).to(device)
    valid = torch.from_numpy(((ids >= 0) & (ids < E))[skip:]).to(device)
    order = torch.argsort(key, stable=True)
    offs = torch.zeros(E + 1, dtype=torch.int64, device=device)
    offs[1:] = torch.cumsum(torch.bincount(key, minlength=E), 0)
    n_x = (P + ppx - 1) // ppx
    assert torch.equal(got[0].long(), offs)
    assert torch.equal(got[1].long(), torch.where(valid, torch.arange(P, device=device) // ppx, n_x)[order])
    assert torch.equal(got[2].long(), order)
