"""The few-rows GEMM kernel (csrc/gemm_few.h) against the persistent kernel, which the oracle tests pin: both run the same
MFMAs in the same k order and round at the same places, so the results are equal bit for bit.  Sizes sit at the edges of
its tiles (32, 64 and 128 rows; 128 and 256 columns), with empty experts, experts of several m-tiles, k-slices fewer than
the ring holds, ragged K and N, and row strides above the widths; the tile that the rule takes for them is checked."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows per expert, columns, K, and the tile rows (negative: the persistent kernel's) that the rule takes for the products to N columns
# with 16-bit and int8 weights, and for gate/up to N hidden columns with either
EDGE32 = [0, 1, 31, 32, 33, 0, 64, 5, 97, 0, 0]
CASES = {
    "one-expert": ([40], 136, 72, (32, 32, 32, 32)),
    "32-row-edges": (EDGE32, 264, 744, (32, 32, 32, 32)),
    "32-row-edges-short-k": (EDGE32, 1024, 24, (32, 32, 32, 32)),
    "few-rows-many-experts": ([0] * 100 + [1, 0, 2] + [0] * 153, 512, 544, (32, 32, 32, 32)),
    "64-row-edges": ([0, 1, 63, 64, 65, 2, 0, 130] * 8, 520, 544, (64, 64, 64, 64)),
    "64-row-skew": ([600] + [3] * 60 + [0, 0, 0], 1976, 40, (64, 64, 64, 64)),
    "256-experts": ([4, 0, 9, 7] * 64, 272, 96, (32, 32, 64, 64)),
    "128-row-edges": ([127, 128, 129, 0, 1, 64, 65, 200] * 4, 1928, 520, (128, 128, 128, 128)),
    "128-row-skew": ([1100] + [50] * 30 + [0], 1976, 520, (128, 128, 128, 128)),
    "128-row-short-k": ([1100] + [50] * 30 + [0], 1544, 64, (64, 64, 128, 128)),
    "257-experts": ([2, 1, 0] * 85 + [3, 1], 528, 136, (-128, -128, -256, -256)),  # past the kernel's expert limit
}


def _inputs(counts, dt, K, gen):
    E, M = len(counts), sum(counts)
    T = max(M // 2, 1)
    c = torch.tensor(counts, dtype=torch.int32)
    x = torch.randn(T, K, generator=gen).to(dt)
    a_idx = torch.randint(0, T, (M,), generator=gen).int()
    y_idx = torch.randperm(M, generator=gen).int()
    return E, M, c.cuda(), x.cuda(), a_idx.cuda(), y_idx.cuda(), torch.rand(M, generator=gen).to(dt).cuda()


def _weights(E, K, N, dt, quant, gen):
    if not quant:
        return (torch.randn(E, K, N, generator=gen) * K ** -0.5).to(dt).cuda(), None
    q = torch.randint(-128, 128, (E, K, N), generator=gen, dtype=torch.int8).cuda()
    s = (torch.rand(E, N, generator=gen) * 0.02 + 1e-3).to(torch.bfloat16 if quant == "bf16" else torch.float32)
    return q, s.cuda()


@pytest.mark.parametrize("dt,quant", [(torch.bfloat16, None), (torch.float16, None), (torch.bfloat16, "bf16"),
                                      (torch.float16, "fp32")])
@pytest.mark.parametrize("case", CASES)
def test_bit_identical_to_persistent(case, dt, quant, monkeypatch):
    from trenowanie_generatora_obrazkow_amd import _lib, ops
    counts, N, K, tiles = CASES[case]
    N = -(-N // 16) * 16 if quant else N
    tile = _lib.lib().hmoe_forward_tile
    w_dt = _lib.dt(torch.int8 if quant else dt)
    got = tile(sum(counts), len(counts), K, N, 0, w_dt), tile(sum(counts), len(counts), K, N, 1, w_dt)
    assert got == (tiles[1::2] if quant else tiles[::2])
    print(f"few rows {case} {dt} quant={quant}", flush=True)
    gen = torch.Generator().manual_seed(len(case) + K)
    E, M, c, x, a_idx, y_idx, scale = _inputs(counts, dt, K, gen)
    w, ws = _weights(E, K, N, dt, quant, gen)
    wgu, gs = _weights(E, K, 2 * N, dt, quant, gen)
    xs = x[a_idx.long()].contiguous()
    # the same operands with row strides above their widths
    xw, ww = (torch.zeros(*t.shape[:-1], t.shape[-1] + 16, dtype=t.dtype, device="cuda") for t in (x, w))
    xw[:, :K], ww[..., :N] = x, w
    yw = torch.zeros(M, N + 24, dtype=dt, device="cuda")

    def run():
        return [ops.grouped_mm(x, w, c, M, a_idx=a_idx, y_idx=y_idx, scale=scale, w_scale=ws),
                ops.grouped_mm(xs, w, c.long(), M, scale=scale.float(), w_scale=ws),
                ops.down_scatter(xs, w, c, M, scale, y_idx, wd_s=ws)[0],
                ops.gate_up_swiglu(x, wgu, c, M, a_idx=a_idx, wgu_s=gs)[0],
                ops.gate_up_swiglu(xs, wgu, c, M, wgu_s=gs)[0],
                ops.grouped_mm(xw[:, :K], ww[..., :N], c, M, a_idx=a_idx, y_idx=y_idx, scale=scale, w_scale=ws,
                               out=yw[:, :N]).contiguous(),
                ops.gate_up_swiglu(xw[:, :K], wgu, c, M, a_idx=a_idx, wgu_s=gs)[0]]

    got = run()
    assert (yw[:, N:] == 0).all()
    monkeypatch.setenv("HMOE_GEMM_TILE", "S")
    assert tile(M, E, K, N, 0, w_dt) == -128 and tile(M, E, K, N, 1, w_dt) == -128
    want = run()
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), f"{case}: call {i}"


@pytest.mark.parametrize("counts,M", [([70, 85, 15, 40], 90), ([3] * 100 + [90], 311), ([5, 40, 64, 64, 1, 2], 170)])
def test_counts_beyond_the_rows(counts, M, monkeypatch):
    """Counts that name more rows than there are: each expert's rows below M are its own, as in the persistent kernel."""
    from trenowanie_generatora_obrazkow_amd import ops
    print(f"few rows, counts of {sum(counts)} rows, M={M}", flush=True)
    gen = torch.Generator().manual_seed(M)
    E, K, N = len(counts), 96, 264
    c = torch.tensor(counts, dtype=torch.int32).cuda()
    x = torch.randn(M, K, generator=gen).bfloat16().cuda()
    w = (torch.randn(E, K, N, generator=gen) * K ** -0.5).bfloat16().cuda()
    got = ops.grouped_mm(x, w, c, M)
    monkeypatch.setenv("HMOE_GEMM_TILE", "S")
    assert torch.equal(got.view(torch.int16), ops.grouped_mm(x, w, c, M).view(torch.int16))
    start = 0
    for e, n in enumerate(counts):
        r = slice(start, min(start + n, M))
        start = min(start + n, M)
        ref = x[r].float() @ w[e].float()
        assert ((got[r].float() - ref).abs() <= 2 ** -8 * ref.abs() + 1e-4).all(), e
