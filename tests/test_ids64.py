"""64-bit expert ids, read by the decode and route kernels themselves.

An int64 id equal to an int32 one selects the same expert, bit for bit in the
result; one outside [0, num_experts) -- also one whose low 32 bits name an
expert -- selects none: a NaN row on the decode, no activation row in the
route.  The pair counts reach each dispatch form of the decode (16-row and
32-row workgroups, two row blocks, two and three pairs a workgroup) and the
path for out_features that are not a multiple of 32.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import wirepack
from mlx_iqk_amd import _native, build, kernels
from mlx_iqk_amd import format as fmt
from mlx_iqk_amd.nn import IqkSwitchLinear


def test_the_entry_points_refuse_bad_arguments():
    if not build.HIP_LIB.is_file():
        build.build_hip()
    lib = _native.load()
    ptrs = (ctypes.c_void_p * 5)(*([16] * 5))
    assert lib.iqk_gemv_ids64(9, 4096, 32, 4, 16, ptrs, 5, 16, 1, 1, 16, None) == _native.ERR_MEMBER
    assert lib.iqk_gemv_ids64(0, 1024, 32, 4, 16, ptrs, 5, 16, 1, 1, 16, None) == _native.ERR_GEOMETRY
    assert lib.iqk_gemv_ids64(0, 4096, 32, 4, 16, ptrs, 5, None, 1, 1, 16, None) == _native.ERR_ARGUMENT
    assert lib.iqk_gemv_ids64(0, 4096, 32, 4, 16, ptrs, 4, 16, 1, 1, 16, None) == _native.ERR_ARGUMENT
    assert lib.iqk_gemv_ids64(0, 4096, 32, 4, 16, ptrs, 5, 16, 2, 3, 16, None) == _native.ERR_ARGUMENT
    assert lib.iqk_gemv_ids64(0, 4096, 32, 4, 16, ptrs, 5, 16, 1, 0, 16, None) == _native.OK
    assert lib.iqk_route_ids64(None, 4, 8, 1, 1, 4, 16, 16, 16, None) == _native.ERR_ARGUMENT
    assert lib.iqk_route_ids64(16, 4, 4097, 1, 1, 4, 16, 16, 16, None) == _native.ERR_ARGUMENT
    assert lib.iqk_route_ids64(16, 4, 8, 1, 1, 3, 16, 16, 16, None) == _native.ERR_ARGUMENT


def test_the_public_launchers_still_refuse_int64_ids():
    ids = torch.zeros(4, dtype=torch.int64)
    with pytest.raises(kernels.IqkKernelError):
        kernels.route(ids, 8)
    with pytest.raises(kernels.IqkKernelError):
        kernels.gemv("iq2_ks", torch.zeros(1, 4096, dtype=torch.float16), [], ids, 4, 8, 32)


_BAD = (-1, 1 << 32, (1 << 32) + 3, -(1 << 63), (1 << 63) - 1)


def _ids(rng, experts, shape, bad):
    ids = rng.integers(0, experts, shape)
    if bad:
        flat = ids.reshape(-1)
        at = rng.choice(flat.size, min(flat.size, len(_BAD) + 1), replace=False)
        for i, b in zip(at, (experts, *_BAD)):
            flat[i] = b
    return ids


@pytest.mark.gpu
@pytest.mark.parametrize("member", fmt.MEMBERS)
@pytest.mark.parametrize("out", (48, 256, 2048))
@pytest.mark.parametrize("tokens,top_k", [(1, 6), (8, 7), (24, 4), (24, 6), (80, 2)])
@pytest.mark.parametrize("bad", (False, True))
def test_decode_reads_int64_ids(device, member, out, tokens, top_k, bad):
    print(f"ids64 decode {member} out={out} {tokens}x{top_k} bad={bad}", flush=True)
    experts, n = 7, 2048
    rng = np.random.default_rng(tokens * top_k)
    wire = wirepack.random_wire(member, experts * out, n, seed=out, scales="serving")
    module = IqkSwitchLinear(member, experts, out, n, device=device)
    module.load_wire(torch.from_numpy(wire).to(device))
    ids = _ids(rng, experts, (tokens, top_k), bad)
    x = torch.from_numpy(rng.standard_normal((tokens, 1, 1, n)).astype(np.float16)).to(device)
    got = module.gemv(x, torch.from_numpy(ids).to(device))
    narrow = np.where((ids >= 0) & (ids < experts), ids, -1).astype(np.int32)
    want = module.gemv(x, torch.from_numpy(narrow).to(device))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    invalid = torch.from_numpy(narrow < 0).to(device)
    assert torch.isnan(got[invalid]).all() and torch.isfinite(got[~invalid]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("P,E,M,ppx", [(1, 1, 1, 1), (300, 8, 3, 1), (12288, 256, 1, 6), (16385, 4096, 1, 1)])
def test_route_reads_int64_ids(device, P, E, M, ppx):
    print(f"ids64 route P={P} E={E} M={M} ppx={ppx}", flush=True)
    ids = _ids(np.random.default_rng(P), E, P, bad=P > 10)
    n_x = ((P + ppx - 1) // ppx) * M
    narrow = np.where((ids >= 0) & (ids < E), ids, -1).astype(np.int32)
    got = kernels.route_ids(torch.from_numpy(ids).to(device), E, M, ppx, n_x)
    want = kernels.route(torch.from_numpy(narrow).to(device), E, M, ppx, n_x)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
