"""The one-call experts (hmoe_moe_experts) where act goes from the gate/up GEMM to the down GEMM in blocked rows,
against the same GEMMs called one by one with act in rows: the same products, so bit-identical.  Both tile sizes, bf16,
fp16 and int8 weights, hidden widths off a 32-wide k-slice (and below one), ragged, empty and few-row experts, row
blocks shared by experts, M off a whole block, and invalid ids."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ids(T, k, E, kind, g):
    if kind == "even":  # exactly T k / E rows each
        return (torch.arange(T * k) % E).view(T, k).int()
    p = torch.tensor([0.0 if e == 1 else 2.0 ** (-e) for e in range(E)])  # expert 1 has no rows, the last ones few
    flat = torch.multinomial(p / p.sum(), T * k, replacement=True, generator=g)
    if kind == "invalid":
        flat[::7] = -1
    return flat.view(T, k).int()


@pytest.mark.parametrize("tile", ["L", "S"])
@pytest.mark.parametrize("weights", ["bf16", "fp16", "int8", "int8_fp16"])
@pytest.mark.parametrize("T,d,E,k,h,kind", [(512, 256, 4, 1, 320, "even"), (513, 272, 4, 2, 336, "skew"),
                                            (700, 512, 6, 2, 16, "skew"), (641, 144, 5, 1, 1040, "invalid"),
                                            (130, 256, 2, 1, 112, "skew")])
def test_experts_match_op_by_op(tile, weights, T, d, E, k, h, kind, monkeypatch):
    from trenowanie_generatora_obrazkow_amd import ops
    print(f"act blocked {tile} {weights} T={T} d={d} E={E} k={k} h={h} {kind}", flush=True)
    monkeypatch.setenv("HMOE_GEMM_TILE", tile)
    dev = torch.device("cuda")
    dt = torch.float16 if "fp16" in weights else torch.bfloat16
    g = torch.Generator().manual_seed(T + h)
    x = torch.randn(T, d, generator=g).to(dt).to(dev)
    ids = _ids(T, k, E, kind, g).to(dev)
    tw = torch.rand(T, k, generator=g).to(dev)
    if weights.startswith("int8"):
        wgu, wd = (torch.randint(-127, 128, s, generator=g, dtype=torch.int8).to(dev) for s in ((E, d, 2 * h), (E, h, d)))
        wgu_s, wd_s = (torch.rand(s, generator=g).mul_(2e-3).bfloat16().to(dev) for s in ((E, 2 * h), (E, d)))
    else:
        wgu, wd = (torch.randn(s, generator=g).mul_(s[1] ** -0.5).to(dt).to(dev) for s in ((E, d, 2 * h), (E, h, d)))
        wgu_s = wd_s = None
    y, inv, _ = ops.moe_experts(x, ids, tw, wgu, wd, wgu_s, wd_s)
    disp = ops.dispatch(ids, E, topk_w=tw, dtype=dt)
    act, _ = ops.gate_up_swiglu(x, wgu, disp.counts, T * k, a_idx=disp.a_idx, wgu_s=wgu_s)
    ref, _ = ops.down_scatter(act, wd, disp.counts, T * k, disp.w_sorted, disp.order, wd_s=wd_s)
    assert torch.equal(inv, disp.inv_pos)
    rows = (inv >= 0).nonzero().flatten()  # (rows of invalid ids are not written)
    assert torch.equal(y.view(T * k, d)[rows].view(torch.int16), ref.view(T * k, d)[rows].view(torch.int16))
    assert ref[rows].float().abs().max() > 0
