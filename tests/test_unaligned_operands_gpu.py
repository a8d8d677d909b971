"""Operands that start inside a larger allocation, at an odd element: they are
contiguous, so every route takes them as they are, and the loads of 8 and 16
bytes then cross their natural alignment.  Outputs equal, bit for bit, those of
the same values in allocations of their own.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import wirepack
from mlx_iqk_amd import format as fmt
from mlx_iqk_amd import kernels
from mlx_iqk_amd.nn import IqkSwitchLinear

pytestmark = pytest.mark.gpu
_SIGNED = {torch.uint32: torch.int32, torch.uint16: torch.int16}


def _odd(t: torch.Tensor) -> torch.Tensor:
    """t's values in a contiguous tensor that starts one element into its storage."""
    s = t.view(_SIGNED.get(t.dtype, t.dtype))
    room = torch.zeros(s.numel() + 2, dtype=s.dtype, device=s.device)
    view = room[1:-1].view(s.shape).copy_(s).view(t.dtype)
    assert view.is_contiguous() and view.data_ptr() % 16 == t.element_size()
    return view


def _module(member, experts, out, n, device):
    wire = wirepack.random_wire(member, experts * out, n, seed=out, scales="serving")
    module = IqkSwitchLinear(member, experts, out, n, device=device)
    module.load_wire(torch.from_numpy(wire).to(device))
    return module


def _same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("member", fmt.MEMBERS)
@pytest.mark.parametrize("n", kernels.SUPPORTED_IN_FEATURES)
@pytest.mark.parametrize("wide", (False, True))
def test_activations_and_ids(device, member, n, wide):
    """Decode, the prefill in one launch and behind a route (pieces of 512
    ids in registers and not), tiles of every form, the sorted forms."""
    print(f"unaligned operands {member} n={n} wide={wide}", flush=True)
    experts, out = 5, 48
    module = _module(member, experts, out, n, device)
    g = torch.Generator(device=device).manual_seed(n)
    dtype = torch.int64 if wide else torch.int32
    for pairs, decode in ((7, True), (48, True), (70, False), (700, False), (2600, False)):
        x = torch.randn((pairs, 1, n), generator=g, device=device).to(torch.float16)
        ids = torch.randint(0, experts, (pairs,), generator=g, device=device)
        ids[:pairs // 2] = 0  # tiles of 64 slots, and of fewer
        ids = ids.to(dtype)
        call = module.gemv if decode else module.prefill
        assert _same(call(_odd(x), _odd(ids)), call(x, ids)), pairs
        if decode and member in kernels.IQ2_MEMBERS and not wide:
            ids, order = torch.sort(ids)
            toks = order.to(torch.int32)
            for form in (module.gemv_sorted, module.gemv_union):
                assert _same(form(_odd(x.view(pairs, n)), _odd(ids), _odd(toks)), form(x.view(pairs, n), ids, toks))


# few-slot tiles of 8 and 16, tiles of 32 and 64; behind them the counts of a
# call of 128-slot tiles and its rests
COUNTS = {"tiles": (256, [3, 12, 30, 64, 70]), "wide": (4096, [1410, 1424, 1440, 1500, 1473, 1536, 1664, 1664, 1290])}


@pytest.mark.parametrize("member", fmt.MEMBERS)
@pytest.mark.parametrize("n", kernels.SUPPORTED_IN_FEATURES)
@pytest.mark.parametrize("form", sorted(COUNTS))
def test_streams_activations_and_lists(device, member, n, form):
    """The contraction on every stream plane at an odd element too (the byte
    planes at an odd address)."""
    print(f"unaligned streams {member} n={n} {form}", flush=True)
    out, counts = COUNTS[form]
    P = sum(counts)
    assert form != "wide" or (P >= 160 * len(counts) and 16 * P >= 3 * 512 * 128)
    module = _module(member, len(counts), out, n, device)
    rng = np.random.default_rng(P)
    x = torch.from_numpy(rng.standard_normal((301, n)).astype(np.float16)).to(device)
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    lists = [torch.from_numpy(a).to(device) for a in (offs, rng.integers(0, 301, P).astype(np.int32),
                                                     rng.permutation(P).astype(np.int32))]
    streams = module._streams()
    shape = (module.member, len(counts), out)
    want = kernels.fused_matmul(shape[0], x, streams, *shape[1:], *lists)
    got = kernels.fused_matmul(shape[0], _odd(x), [_odd(s) for s in streams], *shape[1:], *(_odd(a) for a in lists))
    assert _same(got, want)
    assert bool(torch.isfinite(want).all())
