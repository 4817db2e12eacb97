"""Scores that are not finite reach the forward's results: one NaN in a key or a query, one infinite score, in launches
whose row lists one workgroup walks and in launches that share them, where the shares' sums are merged.  The rows that
are not finite are those of the plain softmax over the kept keys; all others agree with it."""
import pytest
import torch

from helpers import make_qkv

pytestmark = pytest.mark.gpu

MAXABS = {torch.float16: 2e-2, torch.bfloat16: 3e-2}


def poisoned(what, q, k):
    """q, k of head 0 with one value that is not finite."""
    q, k = q.clone(), k.clone()
    if what == "key":
        k[0, 0, 70, 3] = float("nan")
    elif what == "query":
        q[0, 0, 130, 3] = float("nan")
    else:                                    # an overflowed activation: scores of both infinite signs
        k[0, 0, 70, 3] = float("inf")
    return q, k


def check(dev, H, N, D, dtype, elementwise, what):
    import fa2_custom_mask as fm
    q, k, v = make_qkv(1, H, N, D, dtype, 900 + N + D)
    q, k = poisoned(what, q, k)
    nb = -(-N // 64)
    tiles = torch.ones(nb, nb, dtype=torch.bool).tril()
    dense = tiles.repeat_interleave(64, 0).repeat_interleave(64, 1)[:N, :N]
    if elementwise:
        dense = dense & torch.ones(N, N, dtype=torch.bool).tril()
    mask = dense if elementwise else tiles
    sc = D ** -0.5
    o, lse = fm.flash_attention_custom_mask_lse(q.to(dev), k.to(dev), v.to(dev), mask[None, None].to(dev), sc)
    torch.cuda.synchronize()
    o, lse = o.cpu().double(), lse.cpu().double()
    s = (q[0, 0].double() @ k[0, 0].double().T * sc).masked_fill(~dense, float("-inf"))
    ref, ref_lse = torch.softmax(s, -1) @ v[0, 0].double(), torch.logsumexp(s, -1)
    bad = ~torch.isfinite(ref).all(-1)
    assert 0 < int(bad.sum()) < N
    assert torch.equal(torch.isnan(o[0, 0]), bad[:, None].expand(N, D))
    assert torch.equal(torch.isfinite(lse[0, 0]), ~bad)
    assert float((o[0, 0] - ref)[~bad].abs().max()) <= MAXABS[dtype]
    assert float((lse[0, 0] - ref_lse)[~bad].abs().max()) <= 2e-3
    assert bool(torch.isfinite(o[:, 1:]).all()) and bool(torch.isfinite(lse[:, 1:]).all())


# D = 128 and 256, row lists shared (2 heads) and not (1100 row blocks): elementwise masks, ragged lengths, block masks
@pytest.mark.parametrize("what", ["key", "query", "inf"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D,H,N,elementwise", [(128, 2, 1024, True), (128, 2, 1000, False), (128, 100, 704, True), (128, 100, 700, False),
                                               (256, 2, 1024, False), (256, 2, 1000, True), (256, 100, 704, False)])
def test_row_blocks_of_wavefront_pairs(dev, D, H, N, elementwise, dtype, what):
    check(dev, H, N, D, dtype, elementwise, what)


# D = 64: ranges of workgroups (row blocks inside a range, and shared by several), ranges of wavefronts, a wavefront per
# row block, long row blocks cut; D = 128: ranges of workgroups
@pytest.mark.parametrize("what", ["key", "query", "inf"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D,H,N,elementwise", [(64, 2, 704, False), (64, 1, 4096, False), (64, 2, 1000, True), (64, 66, 2000, False),
                                               (64, 160, 1300, False), (128, 2, 1024, False), (128, 1, 2048, False)])
def test_ranges_and_row_blocks(dev, D, H, N, elementwise, dtype, what):
    check(dev, H, N, D, dtype, elementwise, what)


# D = 64: ranges of workgroups (more row blocks than the kernel for short lists takes)
@pytest.mark.parametrize("what", ["key", "query", "inf"])
@pytest.mark.parametrize("N,elementwise", [(8256, False), (8300, True)])
def test_ranges_of_long_heads(dev, N, elementwise, what):
    check(dev, 1, N, 64, torch.float16, elementwise, what)
