"""The GPU pack at other widths and wire alignments.

A block copies its wire rows 16 bytes at a time from a 4-byte aligned start and
hands half a 256-weight block to a thread: rows of one block, widths that do
not divide a block's items, rows of many blocks, and wire that starts 4, 8 or
12 bytes past a 16-byte boundary.  The bytes are ``format.pack``'s.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import wirepack
from mlx_iqk_amd import format as fmt
from mlx_iqk_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("member", fmt.MEMBERS)
@pytest.mark.parametrize("n,rows", [(256, 4), (256, 516), (768, 12), (5120, 68), (16384, 8)])
@pytest.mark.parametrize("skip", (0, 4, 8, 12))
def test_pack_is_format_pack(device, member, n, rows, skip):
    wire = np.ascontiguousarray(wirepack.random_wire(member, rows, n, seed=n + skip, scales="sweep"))
    room = torch.zeros(wire.size + 16, dtype=torch.uint8, device=device)
    view = room[skip:skip + wire.size].view(wire.shape)
    view.copy_(torch.from_numpy(wire))
    got = kernels.pack(member, view, n)
    for k, v in fmt.pack(member, wire, n).items():
        assert np.array_equal(got[k].cpu().numpy().view(np.uint8), np.ascontiguousarray(v).view(np.uint8)), k
