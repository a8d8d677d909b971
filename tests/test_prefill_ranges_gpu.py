"""Row ranges of a prefill call against the full call, bit for bit, where the
call is large enough for the 128-slot tiles and where its blocks route for
themselves: a call's tile forms sum an element in different orders, so the
full call and its ranges have to choose the same one.
"""

from __future__ import annotations

import pytest
import torch

import wirepack
from mlx_iqk_amd import format as fmt
from mlx_iqk_amd import kernels
from mlx_iqk_amd.nn import IqkSwitchLinear

pytestmark = pytest.mark.gpu


def _module(member, experts, out, n, device):
    """Every four rows drawn from 512 random ones."""
    pool = torch.from_numpy(wirepack.random_wire(member, 512, n, seed=out, scales="serving")).to(device)
    g = torch.Generator(device=device).manual_seed(experts)
    pick = torch.randint(128, (experts * out // 4,), generator=g, device=device)
    module = IqkSwitchLinear(member, experts, out, n, device=device)
    module.load_wire(pool.view(128, -1)[pick].view(experts * out, -1))
    return module


def _ranges_concatenate(module, x, ids, widths):
    full = module.prefill(x, ids)
    start = 0
    for rows in widths:
        part = module.sorted_matmul_range(x, ids, start, rows)
        assert torch.equal(part.view(torch.int16), full[..., start:start + rows].contiguous().view(torch.int16)), (start, rows)
        start += rows
    assert start == module.out_features


# pairs of an expert: last 128-slot tiles of 1 .. 16 slots (few-slot tiles of
# the 64-slot cut), of 65 .. 80 (a 64-slot tile and a few-slot one), between
# and full; experts of few pairs and none
COUNTS = [1408, 1409, 1416, 1424, 1425, 1440, 1472, 1473, 1480, 1488, 1489, 5, 0, 70]


@pytest.mark.parametrize("member", fmt.MEMBERS)
@pytest.mark.parametrize("n", kernels.SUPPORTED_IN_FEATURES)
def test_ranges_of_a_call_of_wide_tiles(device, member, n):
    """The full 4096 rows lie above the wide tiles' line, each range's own
    work below it."""
    print(f"wide ranges {member} n={n}", flush=True)
    pairs = sum(COUNTS)
    assert pairs >= 160 * len(COUNTS) and 8 * pairs < 3 * 512 * 128 <= 16 * pairs
    module = _module(member, len(COUNTS), 4096, n, device)
    g = torch.Generator(device=device).manual_seed(n)
    ids = torch.repeat_interleave(torch.arange(len(COUNTS)), torch.tensor(COUNTS)).to(device)
    ids = ids[torch.randperm(pairs, generator=g, device=device)]
    x = torch.randn((pairs, 1, n), generator=g, device=device).to(torch.float16)
    _ranges_concatenate(module, x, ids, (2048, 1024, 512, 256, 128, 64, 32, 16, 8, 8))


@pytest.mark.parametrize("member", fmt.MEMBERS)
def test_ranges_on_both_sides_of_own_routing(device, member):
    """700 pairs over 256 experts: a range of up to 1024 of the 2048 rows
    stays below 1536 blocks, the full call does not."""
    print(f"own-routing ranges {member}", flush=True)
    module = _module(member, 256, 2048, 2048, device)
    g = torch.Generator(device=device).manual_seed(1)
    ids = torch.randint(0, 256, (700,), generator=g, device=device)
    ids[:90] = 3
    x = torch.randn((700, 1, 2048), generator=g, device=device).to(torch.float16)
    _ranges_concatenate(module, x, ids, (1024, 512, 256, 128, 64, 32, 32))


@pytest.mark.parametrize("member", fmt.MEMBERS)
def test_ranges_that_route_for_themselves_of_a_call_of_wide_tiles(device, member):
    """1024 pairs through 49152 rows lie above the wide tiles' line; a range of
    1024 rows is one launch, last tiles of 52, 3 and 9 slots among its tiles."""
    print(f"own-routing ranges of a wide call {member}", flush=True)
    module = _module(member, 3, 49152, 2048, device)
    counts = [500, 515, 9]
    assert sum(counts) * (49152 // 256) >= 3 * 512 * 128
    g = torch.Generator(device=device).manual_seed(5)
    ids = torch.repeat_interleave(torch.arange(3), torch.tensor(counts)).to(device)[torch.randperm(1024, generator=g, device=device)]
    x = torch.randn((1024, 1, 2048), generator=g, device=device).to(torch.float16)
    _ranges_concatenate(module, x, ids, (1024, 16384, 8192, 16384, 4096, 2048, 1024))
