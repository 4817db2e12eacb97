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


def test_reorder_beside_training_on_one_stream(dev, deterministic):
    """One thread reorders tokens (sizes that grow, so its workspace is replaced) while two train on the same stream: the
    gradients equal those of the step made alone."""
    import fa2_custom_mask as fm
    q, k, v, do = [x.to(dev) for x in make_qkv(1, 4, 900, 64, torch.float16, 730, n=4)]
    mask = uniform_block_mask(1, 1, 15, 0.5, 731).to(dev)
    for x in (q, k, v):
        x.requires_grad_(True)

    def step():
        o = fm.flash_attention_custom_mask(q, k, v, mask, 0.125)
        return torch.autograd.grad(o, (q, k, v), do)

    alone = step()
    torch.cuda.synchronize()
    runs, moved = [], []

    def reorder():
        for heads in range(1, 41):
            x = torch.randn(1, heads, 2 * 3 * 64, 64, device=dev, dtype=torch.float16)
            plan = {"permute": [torch.full((heads,), 4, device=dev)]}
            y = fm.inv_permute_attn_triton(fm.permute_qkv_triton(x.clone(), x.clone(), x.clone(), plan, 0, 2, 3, 64, 0)[0], plan, 0, 2, 3, 64, 0)
            moved.append(torch.equal(x, y))

    threads = [threading.Thread(target=reorder)]
    threads += [threading.Thread(target=lambda: runs.extend(step() for _ in range(40))) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert len(runs) == 80 and len(moved) == 40 and all(moved)
    for run in runs:
        assert all(torch.equal(a, b) for a, b in zip(run, alone))


@pytest.mark.parametrize("elementwise", [False, True])
def test_column_lists(dev, deterministic, elementwise):
    """A forward with an elementwise mask that is never followed by a backward makes row lists only; the first backward
    makes the column lists, on whatever thread and stream it runs, and the next forward with the mask finds them."""
    import fa2_custom_mask as fm
    from fa2_custom_mask.utils import lists_cache
    q, k, v, do = [x.to(dev) for x in make_qkv(1, 2, 200, 64, torch.float16, 760, n=4)]
    for x in (q, k, v):
        x.requires_grad_(True)
    mask = uniform_block_mask(1, 1, 4, 0.6, 761).to(dev)
    if elementwise:
        mask = mask.repeat_interleave(64, 2).repeat_interleave(64, 3)[:, :, :200, :200].tril().contiguous()
    o = fm.flash_attention_custom_mask(q, k, v, mask, 0.2)
    assert lists_cache.get(mask, 200, False) is not None and (lists_cache.get(mask, 200, True) is None) == elementwise
    got = []
    thread = threading.Thread(target=lambda: got.extend(torch.autograd.grad(o, (q, k, v), do, retain_graph=True)))
    thread.start()
    thread.join()
    assert lists_cache.get(mask, 200, True) is not None
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    fresh = mask.clone()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        o2 = fm.flash_attention_custom_mask(q, k, v, fresh, 0.2)
    again = torch.autograd.grad(o2, (q, k, v), do)                        # lists made on the side stream
    at_hand = torch.autograd.grad(fm.flash_attention_custom_mask(q, k, v, mask, 0.2), (q, k, v), do)
    torch.cuda.synchronize()
    lists_cache.clear()
    rebuilt = torch.autograd.grad(o, (q, k, v), do)
    torch.cuda.synchronize()
    o_ref, _, *ref = fm.attention_forward_backward(q.detach(), k.detach(), v.detach(), mask, 0.2, do)
    assert torch.equal(o.detach(), o_ref)
    for grads in (got, again, at_hand, rebuilt):
        assert all(torch.equal(a, b) for a, b in zip(grads, ref))


def test_mask_written_before_the_backward_is_refused(dev):
    import fa2_custom_mask as fm
    q, k, v = [x.to(dev).requires_grad_(True) for x in make_qkv(1, 1, 128, 64, torch.float16, 740)]
    mask = uniform_block_mask(1, 1, 2, 1.0, 741).to(dev)
    o = fm.flash_attention_custom_mask(q, k, v, mask, 0.2)
    mask[0, 0, 0, 1] = False
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.backward(torch.ones_like(o))


def test_transforms_are_refused(dev):
    """vmap and forward-mode differentiation of the autograd function have no rule and raise."""
    import fa2_custom_mask as fm
    import torch.autograd.forward_ad as fwad
    q, k, v = [x.to(dev).requires_grad_(True) for x in make_qkv(1, 1, 128, 64, torch.float16, 750)]
    mask = uniform_block_mask(1, 1, 2, 1.0, 751).to(dev)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda x: fm.flash_attention_custom_mask(x, k, v, mask, 0.2))(torch.stack([q, q]))
    with pytest.raises((RuntimeError, NotImplementedError)):
        with fwad.dual_level():
            fm.flash_attention_custom_mask(fwad.make_dual(q, torch.ones_like(q)), k, v, mask, 0.2)
