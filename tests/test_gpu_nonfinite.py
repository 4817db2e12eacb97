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
    assert bool(torch.isnan(lse[0, 0])[torch.isnan(ref_lse)].all())          # (-inf would say that there is no key)
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


# D = 64: pairs of wavefronts (one share, four), ranges of wavefronts, a wavefront per row block, long row blocks cut; D = 128:
# shared lists of block masks
@pytest.mark.parametrize("what", ["key", "query", "inf"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D,H,N,elementwise", [(64, 2, 704, False), (64, 1, 4096, False), (64, 2, 1000, True), (64, 66, 2000, False),
                                               (64, 160, 1300, False), (128, 2, 1024, False), (128, 1, 2048, False)])
def test_ranges_and_row_blocks(dev, D, H, N, elementwise, dtype, what):
    check(dev, H, N, D, dtype, elementwise, what)


# D = 64: ranges of workgroups (more row blocks than the kernel for short lists takes)
@pytest.mark.parametrize("what", ["key", "query", "inf"])
@pytest.mark.parametrize("H,N,elementwise,dtype", [(1, 8256, False, torch.float16), (1, 8300, True, torch.float16), (3, 8300, False, torch.bfloat16)])
def test_ranges_of_long_heads(dev, H, N, elementwise, dtype, what):
    check(dev, H, N, 64, dtype, elementwise, what)


# Keys whose scores are -inf for every query (a bias column of K that Q picks up): half of every tile, the first tiles of every
# row, all keys but one of a row block.  A wavefront's first tile, half tile or share may then hold nothing else: the result is
# the softmax over the other keys, and not a number (lse -inf) where there are none, however the launch splits its lists.
#   D = 64: pairs of wavefronts (4, with 4 shares, 2), ranges of workgroups, of wavefronts, row blocks; D = 128 and 256: shared
#   lists, whole ones, ragged lengths
@pytest.mark.parametrize("hidden", ["first halves", "second halves", "first tiles", "all but one"])
@pytest.mark.parametrize("dtype,out_fp32", [(torch.float16, False), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("D,H,N", [(64, 3, 1000), (64, 1, 4096), (64, 16, 3072), (64, 1, 8300), (64, 12, 8192), (64, 160, 1300),
                                   (128, 2, 1024), (128, 100, 700), (256, 2, 1024), (256, 2, 1000), (256, 100, 704)])
def test_scores_of_minus_infinity(dev, D, H, N, dtype, out_fp32, hidden):
    import fa2_custom_mask as fm
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, D, dtype, 950 + N + D)]
    key = torch.arange(N, device=dev)
    if hidden == "all but one":
        gone = key != N - 5
    else:
        gone = {"first halves": key % 64 < 32, "second halves": key % 64 >= 32, "first tiles": key < 192}[hidden]
    q[..., 0] = 1.0
    k[..., 0] = 0.0
    k[:, :, gone, 0] = float("-inf")
    nb = -(-N // 64)
    tiles = torch.ones(nb, nb, dtype=torch.bool, device=dev).tril()
    keep = tiles.repeat_interleave(64, 0).repeat_interleave(64, 1)[:N, :N]
    sc = D ** -0.5
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, tiles[None, None], sc, out_fp32=out_fp32)
    for h in sorted({0, H - 1}):
        s = (q[0, h].double() @ k[0, h].double().T * sc).masked_fill(~keep, float("-inf"))
        ref, ref_lse = torch.softmax(s, -1) @ v[0, h].double(), torch.logsumexp(s, -1)
        none = torch.isnan(ref).all(-1)
        assert torch.equal(torch.isnan(o[0, h]), none[:, None].expand(N, D))
        assert torch.equal(lse[0, h] == float("-inf"), none) and not bool(torch.isnan(lse[0, h]).any())
        assert float((o[0, h] - ref)[~none].abs().max()) <= MAXABS[dtype]
        assert float((lse[0, h] - ref_lse)[~none].abs().max()) <= (2e-3 if out_fp32 or dtype == torch.float16 else 2.0 ** -8)


# A value of V that is not finite reaches the rows that keep its key, in its column, and no others: launches whose first tiles take
# the numerators in two parts (D = 128: two groups of wavefronts, one; D = 256: whole lists, shared ones), and others.
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("dtype,out_fp32", [(torch.float16, False), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("D,H,N", [(64, 2, 704), (128, 2, 1500), (128, 8, 2304), (128, 100, 700), (256, 2, 1000), (256, 1, 2048), (256, 100, 704)])
def test_values_that_are_not_finite(dev, D, H, N, dtype, out_fp32, value):
    import fa2_custom_mask as fm
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, D, dtype, 970 + N + D)]
    q = q * 0.25                                  # (no numerator of a kept key is rounded to 0)
    nb = -(-N // 64)
    tiles = torch.ones(nb, nb, dtype=torch.bool, device=dev).tril()
    tiles[nb // 2, : nb // 2] = False             # a row block that keeps its own tile only
    key = [3, N // 2, N - 2]
    for i, x in enumerate(key):
        v[0, 0, x, 5 + i] = value
    o, _ = fm.flash_attention_custom_mask_lse(q, k, v, tiles[None, None], D ** -0.5, out_fp32=out_fp32)
    keep = tiles.repeat_interleave(64, 0).repeat_interleave(64, 1)[:N, :N]
    s = (q[0, 0].double() @ k[0, 0].double().T * D ** -0.5).masked_fill(~keep, float("-inf"))
    ref = torch.softmax(s, -1) @ torch.nan_to_num(v[0, 0].double(), nan=0.0, posinf=0.0, neginf=0.0)
    want = torch.zeros_like(ref, dtype=torch.bool)
    for i, x in enumerate(key):
        want[:, 5 + i] = keep[:, x]
    got = o[0, 0].double()
    assert bool(torch.isfinite(got)[~want].all()) and float((got - ref)[~want].abs().max()) <= MAXABS[dtype]
    assert bool((torch.isnan(got[want]) if value != value else got[want] == value).all())
    assert bool(torch.isfinite(o[:, 1:]).all())
