"""The gate/up dgrad with a split reduction (hmoe_gate_up_dgrad_split) and the un-permute that adds its parts."""
import numpy as np
import pytest
import torch

from tests.util import f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,d,h,parts", [([1, 0, 255, 256, 257], 8, 72, 2), ([300, 40, 0, 129], 264, 536, 3),
                                              ([64] * 8, 520, 1024, 4), ([7], 16, 24, 2)])
def test_split_dgrad(counts, d, h, parts):
    """Every part is the product over its own k range, and their sum the whole product within the fp32 bound
    2 K 2^-24 sum |a b| (products of bf16 values are exact in fp32)."""
    from trenowanie_generatora_obrazkow_amd import ops
    E, M = len(counts), sum(counts)
    g = torch.Generator().manual_seed(M + d)
    dgu = torch.randn(M, 2 * h, generator=g).bfloat16()
    wgu = torch.randn(E, d, 2 * h, generator=g).bfloat16()
    c = torch.tensor(counts, dtype=torch.int32, device="cuda")
    got = ops.gate_up_dgrad(dgu.cuda(), wgu.cuda(), c, M, parts=parts)
    assert got.shape == (parts, M, d)
    kper = -(-(-(-2 * h // 32)) // parts) * 32
    a, w = f32(dgu).astype(np.float64), f32(wgu).astype(np.float64)
    whole = f32(ops.gate_up_dgrad(dgu.cuda(), wgu.cuda(), c, M))
    for e, r0 in enumerate(np.cumsum([0] + counts[:-1])):
        r = slice(r0, r0 + counts[e])
        bound = 2 * (2 * h) * 2.0 ** -24 * (np.abs(a[r]) @ np.abs(w[e]).T)
        for q in range(parts):
            k = slice(q * kper, (q + 1) * kper)
            assert (np.abs(f32(got[q, r]) - a[r, k] @ w[e][:, k].T) <= bound).all(), (e, q)
        assert (np.abs(f32(got.sum(0)[r]) - whole[r]) <= 2 * bound).all(), e


@pytest.mark.parametrize("T,d,E,k,parts", [(33, 264, 5, 2, 2), (7, 2056, 20, 3, 4)])
def test_unpermute_adds_parts(T, d, E, k, parts):
    from trenowanie_generatora_obrazkow_amd import ops
    g = torch.Generator().manual_seed(T)
    dxs = torch.randn(parts, T * k, d, generator=g).cuda()
    inv = torch.randperm(T * k, generator=g).int().cuda()
    inv[3] = -1  # a slot routed nowhere
    dl, wr = torch.randn(T, E, generator=g).cuda(), torch.randn(E, d, generator=g).bfloat16().cuda()
    for args in ({}, dict(dlogits=dl, wr=wr)):
        got = ops.unpermute_bwd(dxs, inv, T, k, **args)
        want = ops.unpermute_bwd(dxs.double().sum(0).float(), inv, T, k, **args)
        assert ((got.float() - want.float()).abs() <= 2 ** -7 * want.float().abs() + 1e-5).all()


def test_parts_rule():
    from trenowanie_generatora_obrazkow_amd import _lib
    parts = _lib.lib().hmoe_gate_up_dgrad_parts
    assert parts(32768, 16, 1536, 4096) == 1  # the large tiles fill the chip
    assert parts(4096, 8, 1024, 2048) == 3 and parts(9003, 12, 760, 1352) == 2
    assert parts(4096, 8, 1024, 256) == 1 and parts(0, 8, 1024, 2048) == 1  # too short a reduction; no rows
