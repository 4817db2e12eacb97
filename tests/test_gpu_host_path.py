"""The native host path: threads that share a stream (and its workspace), gradients that arrive in odd layouts and types."""
import threading

import pytest
import torch

from helpers import make_qkv, uniform_block_mask

pytestmark = pytest.mark.gpu


@pytest.fixture
def deterministic():
    import fa2_custom_mask as fm
    before = fm.set_deterministic(True)
    yield
    fm.set_deterministic(before)


def test_threads_on_one_stream(dev, deterministic):
    """Four threads train on the default stream at the same time; each result equals the same step made alone (the
    backward keeps delta in the workspace between its launches)."""
    import fa2_custom_mask as fm
    cases = []
    for i in range(4):
        q, k, v, do = [x.to(dev) for x in make_qkv(1, 2, 700 + 64 * i, 64, torch.float16, 700 + i, n=4)]
        mask = uniform_block_mask(1, 1, -(-q.shape[2] // 64), 0.5, 710 + i).to(dev)
        for x in (q, k, v):
            x.requires_grad_(True)
        cases.append((q, k, v, do, mask))

    def step(case):
        q, k, v, do, mask = case
        o = fm.flash_attention_custom_mask(q, k, v, mask, 0.125)
        return torch.autograd.grad(o, (q, k, v), do)

    alone = [step(c) for c in cases]
    torch.cuda.synchronize()
    got = [[] for _ in cases]
    threads = [threading.Thread(target=lambda i=i: got[i].extend(step(cases[i]) for _ in range(20))) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for ref, runs in zip(alone, got):
        assert len(runs) == 20
        for run in runs:
            assert all(torch.equal(a, b) for a, b in zip(run, ref))


@pytest.mark.parametrize("D", [32, 64])
def test_gradients_in_odd_layouts(dev, deterministic, D):
    """An expanded gradient (from a sum), one in another type (fp32 results), and the LSE as a second output."""
    import fa2_custom_mask as fm
    q, k, v = [x.to(dev).requires_grad_(True) for x in make_qkv(1, 2, 200, D, torch.float16, 720)]
    mask = uniform_block_mask(1, 1, 4, 0.6, 721).to(dev)
    ref = torch.autograd.grad(fm.flash_attention_custom_mask(q, k, v, mask, 0.2), (q, k, v), torch.ones_like(q))
    got = torch.autograd.grad(fm.flash_attention_custom_mask(q, k, v, mask, 0.2).sum(), (q, k, v))
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, mask, 0.2, out_fp32=True)
    assert o.dtype == torch.float32 and o.shape == q.shape and not lse.requires_grad
    got32 = torch.autograd.grad(o, (q, k, v), torch.ones_like(o))
    for a, b, c in zip(ref, got, got32):
        assert torch.equal(a, b) and a.dtype == c.dtype == torch.float16
        assert float((a.float() - c.float()).norm() / a.float().norm()) < 2e-3      # o is rounded to fp16 once or not at all
    q1, k1, v1 = q.detach(), k.detach().requires_grad_(True), v.detach()
    only_k = torch.autograd.grad(fm.flash_attention_custom_mask(q1, k1, v1, mask, 0.2), k1, torch.ones_like(q))[0]
    assert torch.equal(only_k, ref[1])
