"""The BailingMoeV2 block as one C call (hmoe_moe_block) against its entry points one by one: the same bits, with and
without the side stream, from several threads, and when x's stream is not the default one."""
import threading

import pytest
import torch

from tests.test_gpu_poziomka import _make_block

pytestmark = pytest.mark.gpu


def _op_by_op(m, x, monkeypatch):
    from trenowanie_generatora_obrazkow_amd import ops
    monkeypatch.setattr(ops, "probe", {})  # a set probe takes the entry points one by one
    try:
        return m(x)
    finally:
        monkeypatch.setattr(ops, "probe", None)


@pytest.mark.parametrize("d,h,E,k,sh,T", [(256, 64, 16, 4, 64, 1), (264, 80, 32, 4, 40, 7), (512, 96, 64, 6, 96, 333),
                                          (2048, 320, 128, 8, 320, 64)])
def test_block_call_bit_exact(oracle, d, h, E, k, sh, T, monkeypatch):
    d16 = -(-d // 16) * 16  # int8 rows come in 16s
    m = _make_block(oracle, d16, h, E, k, 8, 2, sh, seed=T).cuda()
    x = torch.randn(T, d16, generator=torch.Generator().manual_seed(T)).bfloat16().cuda()
    want = _op_by_op(m, x, monkeypatch)
    for overlap in (True, False):
        m.overlap_shared = overlap
        assert torch.equal(m(x).view(torch.int16), want.view(torch.int16)), overlap


def test_block_call_bf16_experts(oracle, monkeypatch):
    m = _make_block(oracle, 256, 64, 16, 4, 8, 2, 64, seed=3)
    m._wgu, m._wd = ((w.float() * s.float().unsqueeze(1)).bfloat16() for w, s in ((m._wgu, m._wgu_s), (m._wd, m._wd_s)))
    m._wgu_s = m._wd_s = None
    m = m.cuda()
    x = torch.randn(50, 256, generator=torch.Generator().manual_seed(4)).bfloat16().cuda()
    assert torch.equal(m(x).view(torch.int16), _op_by_op(m, x, monkeypatch).view(torch.int16))


def test_block_call_threads_and_streams(oracle):
    """Threads on streams of their own share the device's side stream and events; every call's x is written on its own
    stream just before the call and overwritten right after it."""
    m = _make_block(oracle, 512, 96, 64, 6, 8, 2, 96, seed=9).cuda()
    gen = torch.Generator().manual_seed(5)
    xs = [torch.randn(200, 512, generator=gen).bfloat16().cuda() for _ in range(3)]
    want = [m(x) for x in xs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            x = torch.empty_like(xs[i])
            for _ in range(20):
                x.copy_(xs[i])
                y = m(x)
                x.zero_()
                torch.cuda.current_stream().synchronize()
                if not torch.equal(y, want[i]):
                    bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
