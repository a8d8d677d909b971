"""Prefill and verify calls whose operands are already in the kernels' layout
go to the launch binding in one call; every other form takes the general
route.  Both give the same bits, and the binding refuses what the entry points
refuse.
"""

from __future__ import annotations

import ctypes
import itertools

import numpy as np
import pytest
import torch

import wirepack
from mlx_iqk_amd import _native, build, kernels, nn
from mlx_iqk_amd import format as fmt
from mlx_iqk_amd.nn import IqkSwitchLinear


def test_the_binding_refuses_as_the_entry_points():
    if not build.HIP_LIB.is_file():
        build.build_hip()
    _native.load()
    fast = _native.launcher()
    assert fast is not None
    streams = _native.pointer_array([16] * 5)
    addr = ctypes.addressof(streams)
    good = [0, 4096, 32, 8, 16, 4, addr, 5, 0, 32, 16, 0, 8, 1, 2, 16, 16, 0]
    assert fast.prefill(*good[:5], 3, *good[6:]) == _native.ERR_ARGUMENT  # a pair names a row past x
    for at, bad, code in ((3, 4097, _native.ERR_ARGUMENT), (10, 0, _native.ERR_ARGUMENT),
                          (12, -1, _native.ERR_ARGUMENT), (12, 1 << 31, _native.ERR_ARGUMENT),
                          (13, 0, _native.ERR_ARGUMENT), (13, 1 << 40, _native.ERR_ARGUMENT),
                          (14, 0, _native.ERR_ARGUMENT)):
        assert fast.prefill(*good[:at], bad, *good[at + 1:]) == code
    for at, bad in ((0, 1 << 31), (7, 1 << 32)):
        with pytest.raises(OverflowError):
            fast.prefill(*good[:at], bad, *good[at + 1:])
    good = [1, 0, 4096, 32, 8, 16, 4, addr, 5, 16, 16, 3, 16, 0]
    for at, bad, code in ((1, 7, _native.ERR_MEMBER), (1, 2, _native.ERR_MEMBER), (2, 3072, _native.ERR_GEOMETRY),
                          (5, 0, _native.ERR_ARGUMENT), (8, 4, _native.ERR_ARGUMENT), (10, 0, _native.ERR_ARGUMENT)):
        for union in (0, 1):
            assert fast.sorted(union, *good[1:at], bad, *good[at + 1:]) == code
    for at, bad in ((1, 1 << 31), (8, 1 << 32), (11, -1), (11, 1 << 32)):
        with pytest.raises(OverflowError):
            fast.sorted(*good[:at], bad, *good[at + 1:])
    with pytest.raises(TypeError):
        fast.prefill(0)
    with pytest.raises(TypeError):
        fast.sorted(0)


def test_pairs_per_x_row_is_the_broadcast():
    """Over every small pair of shapes: a number exactly where the broadcast
    gives pair p the activation row p // number and keeps the pairs' shape."""
    shapes = [s for r in range(4) for s in itertools.product((1, 2, 3), repeat=r)]
    for batch, xbatch in itertools.product(shapes, shapes):
        got = nn._pairs_per_x_row(xbatch, batch)
        try:
            keeps = torch.broadcast_shapes(xbatch, batch) == batch
        except RuntimeError:
            keeps = False
        if not keeps:
            assert got is None
            continue
        row = np.broadcast_to(np.arange(np.prod(xbatch, dtype=int)).reshape(xbatch), batch).reshape(-1)
        if got is not None:
            assert (row == np.arange(row.size) // got).all()
        else:  # no number of consecutive pairs a row fits
            assert not any((row == np.arange(row.size) // n).all() for n in range(1, row.size + 1))


@pytest.mark.parametrize("member", fmt.MEMBERS)
@pytest.mark.parametrize("form", ("gemv_sorted", "gemv_union"))
def test_sorted_forms_name_a_wrong_operand_before_the_device(member, form):
    """A module in host memory refuses operands that disagree as one on a GPU
    does, and only then its own streams."""
    module = IqkSwitchLinear(member, 4, 32, 2048)
    call, x, ids = getattr(module, form), torch.zeros((2, 2048), dtype=torch.float16), torch.zeros(4, dtype=torch.int32)
    with pytest.raises(nn.IqkRuntimeError, match="toks carries 3 rows for 4 pairs"):
        call(x, ids, ids[:3])
    with pytest.raises(RuntimeError, match="is invalid for input of size"):
        call(x[:, :100], ids, ids)
    with pytest.raises(kernels.IqkKernelError, match="must live on a GPU"):
        call(x, ids, ids)


def _module(member, experts, out, n, device):
    wire = wirepack.random_wire(member, experts * out, n, seed=out, scales="serving")
    module = IqkSwitchLinear(member, experts, out, n, device=device)
    module.load_wire(torch.from_numpy(wire).to(device))
    return module


def _same(a, b):
    return a.shape == b.shape and torch.equal(a.view(torch.int16), b.view(torch.int16))


# x's batch shape, its rows a pair, the ids' shape, whether the call is direct
FORMS = [((21, 1), 1, (21, 4), True), ((21, 4), 1, (21, 4), True), ((84,), 1, (84,), True), ((1, 1), 3, (21, 4), True),
         ((), 2, (70,), True), ((5, 1, 1), 1, (5, 3, 7), True), ((5, 3, 1), 1, (5, 3, 7), True),
         ((1, 4), 1, (21, 4), False), ((21, 4), 1, (1, 4), False), ((2, 21, 1), 1, (21, 4), False)]


@pytest.mark.gpu
@pytest.mark.parametrize("member", fmt.MEMBERS)
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("wide", (False, True))
def test_prefill_direct_equals_the_general_route(device, monkeypatch, member, form, wide):
    xb, M, ib, direct = form
    print(f"direct prefill {member} {form} wide={wide}", flush=True)
    experts, out, n = 5, 64, 2048
    module = _module(member, experts, out, n, device)
    rng = np.random.default_rng(len(xb) + M)
    ids = rng.integers(0, experts, ib)
    ids.reshape(-1)[::17] = experts  # names no expert: NaN rows
    x = torch.from_numpy(rng.standard_normal((*xb, M, n)).astype(np.float16)).to(device)
    sel = torch.from_numpy(ids).to(device, torch.int64 if wide else torch.int32)
    calls = []
    inner = kernels.prefill_checked
    monkeypatch.setattr(kernels, "prefill_checked", lambda *a: calls.append(1) or inner(*a))
    got, part = module.prefill(x, sel), module.sorted_matmul_range(x, sel, 16, 32)
    assert len(calls) == (2 if direct else 0)
    monkeypatch.setattr(kernels, "prefill_checked", lambda *a: False)
    assert _same(got, module.prefill(x, sel)) and _same(part, module.sorted_matmul_range(x, sel, 16, 32))
    # other layouts and types: the general route, the same bits
    monkeypatch.setattr(kernels, "prefill_checked", inner)
    strided = torch.empty((*x.shape[:-1], 2 * n), dtype=x.dtype, device=device)[..., ::2].copy_(x)
    assert _same(got, module.prefill(strided, sel)) and _same(got, module.prefill(x.float(), sel))


@pytest.mark.gpu
@pytest.mark.parametrize("member", fmt.MEMBERS[:2])
@pytest.mark.parametrize("union", (False, True))
@pytest.mark.parametrize("pairs", (1, 7, 48))
def test_sorted_direct_equals_the_general_route(device, monkeypatch, member, union, pairs):
    print(f"direct sorted {member} union={union} pairs={pairs}", flush=True)
    experts, out, n = 5, 64, 4096
    module = _module(member, experts, out, n, device)
    rng = np.random.default_rng(pairs)
    ids = torch.from_numpy(np.sort(rng.integers(0, experts + 1, pairs))).to(device, torch.int32)
    toks = torch.from_numpy(rng.integers(0, 9, pairs)).to(device, torch.int32)  # row 8 is past x
    x = torch.from_numpy(rng.standard_normal((8, n)).astype(np.float16)).to(device)
    form = module.gemv_union if union else module.gemv_sorted
    got = form(x, ids, toks)
    monkeypatch.setattr(kernels, "gemv_sorted_checked", lambda *a: False)
    assert _same(got, form(x, ids, toks))
    monkeypatch.undo()
    assert _same(got, form(x.float(), ids.to(torch.int64), toks.to(torch.int64)))


@pytest.mark.gpu
def test_prefill_direct_replays_in_a_graph(device):
    print("direct prefill graph", flush=True)
    experts, out, n = 5, 64, 2048
    module = _module("iq2_ks", experts, out, n, device)
    x = torch.randn((21, 1, 1, n), device=device).to(torch.float16)
    ids = torch.randint(0, experts, (21, 4), device=device)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        module(x, ids)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = module(x, ids)
    for _ in range(3):
        x.copy_(torch.randn(x.shape, device=device).to(torch.float16))
        ids.copy_(torch.randint(0, experts, ids.shape, device=device))
        graph.replay()
        assert _same(y, module(x, ids))
        torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("member,n", [("iq2_ks", 4096), ("iq2_k", 4096), ("iq2_k", 2048), ("iq1_s_r4", 2048)])
@pytest.mark.parametrize("pairs,experts", [(1, 1), (63, 512), (64, 3), (511, 2), (512, 256), (513, 9), (1023, 512),
                                           (1024, 5), (1024, 513), (1025, 5)])
@pytest.mark.parametrize("wide", (False, True))
def test_blocks_find_the_pairs_the_route_lists(device, monkeypatch, member, n, pairs, experts, wide):
    """Around the limits of the one-launch form (1024 pairs, 512 experts): the
    outputs of the routed form, with ids that name no expert."""
    print(f"own routing {member} n={n} pairs={pairs} experts={experts} wide={wide}", flush=True)
    module = _module(member, experts, 48, n, device)
    rng = np.random.default_rng(pairs + experts)
    ids = np.minimum(rng.geometric(0.02 if experts > 100 else 0.3, pairs) - 1, experts - 1)  # some experts with many
    bad = (experts, -1) + (((1 << 32) + 1, -(1 << 63)) if wide else (2**31 - 1, -(2**31)))
    for at, b in zip(rng.choice(pairs, min(len(bad), pairs // 2), replace=False), bad):
        ids[at] = b
    sel = torch.from_numpy(ids).to(device, torch.int64 if wide else torch.int32)
    x = torch.from_numpy(rng.standard_normal((pairs, 1, n)).astype(np.float16)).to(device)
    got = module.prefill(x, sel)
    monkeypatch.setattr(kernels, "prefill_checked", lambda *a: False)
    assert _same(got, module.prefill(x, sel))
    assert torch.equal(torch.isnan(got).all(-1).reshape(-1), (sel < 0) | (sel >= experts))


def _pool_module(member, experts, out, n, device):
    """Every four rows drawn from 512 random ones."""
    pool = torch.from_numpy(wirepack.random_wire(member, 512, n, seed=out, scales="serving")).to(device)
    g = torch.Generator(device=device).manual_seed(experts)
    pick = torch.randint(128, (experts * out // 4,), generator=g, device=device)
    module = IqkSwitchLinear(member, experts, out, n, device=device)
    module.load_wire(pool.view(128, -1)[pick].view(experts * out, -1))
    return module


@pytest.mark.gpu
@pytest.mark.parametrize("member", fmt.MEMBERS)
@pytest.mark.parametrize("out,tokens,top_k,experts,own", [
    (272, 86, 6, 40, True), (272, 170, 6, 300, True),  # two column blocks, the second of 16 rows; two pieces of pairs
    (2048, 32, 6, 200, True), (2048, 193, 1, 200, False),  # 192 and 193 tiles of eight column blocks: by pairs
    (2048, 170, 6, 176, True), (2048, 170, 6, 177, False),  # by experts, pairs sharing activation rows
])
@pytest.mark.parametrize("wide", (False, True))
def test_own_routing_over_column_blocks(device, monkeypatch, member, out, tokens, top_k, experts, own, wide):
    """The one-launch form over several column blocks and pairs that share an
    activation row, on both sides of its 1536 blocks: the routed form's
    outputs, its workspace written by the routed form alone."""
    print(f"own routing {member} out={out} {tokens}x{top_k} of {experts} wide={wide}", flush=True)
    pairs, n = tokens * top_k, 2048
    assert own == (min(pairs, -(-pairs // 64) + experts) * -(-out // 256) <= 1536)
    module = _pool_module(member, experts, out, n, device)
    g = torch.Generator(device=device).manual_seed(pairs)
    x = torch.randn((tokens, 1, 1, n), generator=g, device=device).to(torch.float16)
    ids = torch.randint(0, experts, (tokens, top_k), generator=g, device=device)
    ids[::3, 0] = 1  # an expert of many pairs
    ids[tokens // 2, -1] = experts
    sel = ids.to(torch.int64 if wide else torch.int32)
    got = module.prefill(x, sel)
    chk, work = module._checked(), torch.full((2 * pairs + experts + 1,), -7, dtype=torch.int32, device=device)
    y = torch.empty_like(got)
    rc = _native.launcher().prefill(_native.MEMBER_IDS[member], n, out, experts, x.data_ptr(), tokens, chk.ptrs_addr,
                                    chk.count, 0, out, sel.data_ptr(), wide, pairs, 1, top_k, work.data_ptr(),
                                    y.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and _same(y, got)
    assert bool((work == -7).all()) == own
    monkeypatch.setattr(kernels, "prefill_checked", lambda *a: False)
    assert _same(got, module.prefill(x, sel))
    assert torch.equal(torch.isnan(got).all(-1).squeeze(-1), sel == experts)
