"""Forward at sizes the CPU oracle does not finish in seconds (N up to 19 000, up to 8 heads), over mask structures
that put the kept-tile list of a head into every regime of the forward's range splitting: ranges far shorter than a
row block, several row blocks per range, rows of wildly different lengths, heads without tiles, lists shared by all
heads or one per head.  The bar is the naive masked matmul + softmax of the reference's own check
(kernel-test.py:36-39) evaluated in fp32 by torch on the GPU, in row chunks; that evaluation is itself held against
the CPU oracle on a small case below.

Tolerances: rel-L2 of O 1e-3 (3e-3 where O is typed bf16: the cast of an exact result alone is 1.7e-3), LSE within
2e-3, rows without kept tiles give O = 0 and LSE = -inf exactly."""
import numpy as np
import pytest
import torch

from helpers import fwd_route_d64
from oracle import bsattn_oracle as orc

pytestmark = pytest.mark.gpu

KINDS = ["uniform", "causal", "band", "skew", "blocks", "fewrows", "dense", "stripes"]


def make_mask(rs, Hm, nb):
    kind = str(rs.choice(KINDS))
    g = torch.Generator().manual_seed(int(rs.randint(1 << 30)))
    keep = float(rs.choice([0.01, 0.03, 0.05, 0.1, 0.15, 0.25, 0.35, 0.5, 0.75, 0.9, 1.0]))
    m = torch.rand(1, Hm, nb, nb, generator=g) < keep
    i = torch.arange(nb)
    if kind == "causal":
        m &= torch.tril(torch.ones(nb, nb, dtype=torch.bool))
    elif kind == "band":
        w = int(rs.randint(1, max(2, nb // 3)))
        m = ((i[:, None] - i[None, :]).abs() <= w).expand(1, Hm, nb, nb).clone()
    elif kind == "skew":          # the keep probability of a row varies over orders of magnitude; some rows full, some empty
        p = torch.rand(1, Hm, nb, 1, generator=g) ** 4
        m = torch.rand(1, Hm, nb, nb, generator=g) < p
        full = torch.rand(1, Hm, nb, 1, generator=g) < 0.05
        empty = torch.rand(1, Hm, nb, 1, generator=g) < 0.1
        m = (m | full) & ~empty
    elif kind == "blocks":        # block-diagonal super blocks
        s = int(rs.randint(2, max(3, nb // 2)))
        m = ((i // s)[:, None] == (i // s)[None, :]).expand(1, Hm, nb, nb).clone()
    elif kind == "fewrows":       # one row block in twelve keeps anything
        rows = torch.rand(1, Hm, nb, 1, generator=g) < 0.08
        m = (torch.rand(1, Hm, nb, nb, generator=g) < max(keep, 0.3)) & rows
    elif kind == "dense":
        m = torch.ones(1, Hm, nb, nb, dtype=torch.bool)
    elif kind == "stripes":       # the same column blocks in every row, plus the diagonal
        cols = torch.rand(1, Hm, 1, nb, generator=g) < keep
        m = cols.expand(1, Hm, nb, nb).clone() | torch.eye(nb, dtype=torch.bool)
    if Hm > 1 and rs.rand() < 0.3:
        m[:, int(rs.randint(Hm))] = False       # a head that keeps nothing
    return kind, keep, m


def naive_forward(q, k, v, mask, sc, chunk=2048):
    """softmax(q k^T sc, masked) v and its log-sum-exp in fp32, `chunk` rows at a time; mask [1, H|1, nb, nb]."""
    B, H, N, D = q.shape
    o = torch.empty(B, H, N, D, device=q.device, dtype=torch.float32)
    lse = torch.empty(B, H, N, device=q.device, dtype=torch.float32)
    for b in range(B):
        for h in range(H):
            mh = mask[0, h if mask.shape[1] > 1 else 0]
            kf, vf = k[b, h].float(), v[b, h].float()
            for r0 in range(0, N, chunk):
                r1 = min(N, r0 + chunk)
                s = (q[b, h, r0:r1].float() @ kf.T) * sc
                mm = mh[r0 // 64:(r1 + 63) // 64].repeat_interleave(64, 0)[: r1 - r0].repeat_interleave(64, 1)[:, :N]
                s = s.masked_fill(~mm, float("-inf"))
                l = torch.logsumexp(s, dim=-1)
                none = torch.isinf(l)
                p = torch.exp(s - torch.where(none, torch.zeros_like(l), l)[:, None])
                o[b, h, r0:r1] = torch.where(none[:, None], torch.zeros_like(p), p) @ vf
                lse[b, h, r0:r1] = l
    return o, lse


def rel_l2(x, ref):
    x, ref = x.double(), ref.double()
    return float((x - ref).norm() / max(float(ref.norm()), 1e-30))


def test_naive_forward_agrees_with_the_oracle(dev):
    rs = np.random.RandomState(7)
    H, nb = 2, 5
    N = nb * 64 - 9
    _, _, mask = make_mask(rs, H, nb)
    mask[0, 0, 2] = False                                  # a row block without kept tiles
    g = torch.Generator().manual_seed(7)
    q, k, v = [torch.randn(1, H, N, 64, generator=g).half() for _ in range(3)]
    o, lse = naive_forward(q.to(dev), k.to(dev), v.to(dev), mask.to(dev), 0.125, chunk=128)
    o_r, lse_r = orc.naive_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(),
                                     orc.expand_block_mask(mask.numpy())[..., :N, :N], 0.125, return_lse=True)
    fin = np.isfinite(lse_r)
    assert not fin.all() and np.array_equal(np.isfinite(lse.cpu().numpy()), fin)
    assert np.abs(lse.cpu().numpy()[fin] - lse_r[fin]).max() <= 1e-5
    assert np.abs(o.cpu().numpy() - o_r).max() <= 1e-5


@pytest.mark.parametrize("seed", range(96))
def test_forward_against_naive(dev, seed):
    import fa2_custom_mask as fm
    rs = np.random.RandomState(seed)
    D = int(rs.choice([64, 64, 64, 128]))
    dtype = torch.float16 if rs.rand() < 0.6 else torch.bfloat16
    H = int(rs.choice([1, 1, 1, 2, 3, 4, 8]))
    nb = int(rs.randint(8, 300 if H <= 2 else 160))
    N = nb * 64 - (int(rs.randint(1, 64)) if rs.rand() < 0.15 else 0)
    Hm = H if rs.rand() < 0.5 else 1
    kind, keep, mask = make_mask(rs, Hm, nb)
    out_fp32 = bool(rs.rand() < 0.5)
    print(dict(seed=seed, D=D, dtype=str(dtype), H=H, N=N, Hm=Hm, kind=kind, keep=keep, out_fp32=out_fp32,
               tiles=int(mask.sum())), flush=True)
    g = torch.Generator().manual_seed(seed)
    q, k, v = [torch.randn(1, H, N, D, generator=g).to(dtype).to(dev) for _ in range(3)]
    sc = 1.0 / np.sqrt(D)
    md = mask.to(dev)
    o_ref, lse_ref = naive_forward(q, k, v, md, sc)
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, md, sc, out_fp32=out_fp32)
    torch.cuda.synchronize()
    assert o.dtype == (torch.float32 if out_fp32 else dtype)
    assert bool(torch.isfinite(o).all())
    none = torch.isinf(lse_ref)
    assert torch.equal(torch.isinf(lse), none)
    assert bool((o[none] == 0).all())
    if (~none).any():
        assert float((lse[~none] - lse_ref[~none]).abs().max()) <= 2e-3
    bar = 3e-3 if (dtype == torch.bfloat16 and not out_fp32) else 1e-3
    assert rel_l2(o, o_ref) <= bar


# About as many row blocks as wavefronts: ranges of single wavefronts, whose last row block is walked before the first one.  Sizes
# at both ends of that regime (0.75 to 1.5 row blocks per wavefront, from 1 on below 32 and above 300 row blocks), inside it and just outside it,
# ranges that lie in one row block, end with one, and span several; bounds as above.
@pytest.mark.parametrize("B,H,N,dtype,out_fp32,seed", [
    (1, 25, 4096, torch.float16, False, 0), (1, 24, 4096, torch.bfloat16, True, 1), (1, 24, 4033, torch.bfloat16, False, 2),
    (1, 16, 8160, torch.float16, True, 3), (2, 23, 4096, torch.float16, False, 4), (2, 8, 8192, torch.bfloat16, True, 5),
    (1, 23, 8192, torch.float16, False, 6), (1, 12, 16100, torch.bfloat16, False, 7), (1, 47, 4064, torch.float16, True, 8),
    (1, 20, 4096, torch.float16, False, 0), (1, 27, 8192, torch.float16, False, 6), (1, 16, 16100, torch.bfloat16, False, 7)])
def test_ranges_of_wavefronts(dev, B, H, N, dtype, out_fp32, seed):
    import fa2_custom_mask as fm
    rs = np.random.RandomState(100 + seed)
    g = torch.Generator(device=dev).manual_seed(seed)
    nb = (N + 63) // 64
    per_wavefront = B * H * nb / (8 * torch.cuda.get_device_properties(0).multi_processor_count)
    route = "workgroups" if per_wavefront < 0.75 else "wavefronts" if per_wavefront < 1.5 else "rows"
    assert fwd_route_d64(B, H, N) == route
    q, k, v = [torch.randn(B, H, N, 64, generator=g, device=dev).to(dtype) for _ in range(3)]
    bar = 3e-3 if (dtype == torch.bfloat16 and not out_fp32) else 1e-3
    for step in range(3):
        kind, keep, mask = make_mask(rs, H if step == 1 else 1, nb)
        md = mask.to(dev)
        print(dict(kind=kind, keep=keep, tiles=int(mask.sum())), flush=True)
        o_ref, lse_ref = naive_forward(q, k, v, md, 0.125)
        o, lse = fm.flash_attention_custom_mask_lse(q, k, v, md, 0.125, out_fp32=out_fp32)
        none = torch.isinf(lse_ref)
        assert torch.equal(torch.isinf(lse), none) and bool((o[none] == 0).all()) and bool(torch.isfinite(o).all())
        if (~none).any():
            assert float((lse[~none] - lse_ref[~none]).abs().max()) <= 2e-3
        assert rel_l2(o, o_ref) <= bar
        again, _ = fm.flash_attention_custom_mask_lse(q, k, v, md, 0.125, out_fp32=out_fp32)
        assert route == "workgroups" or torch.equal(o, again)                       # (a wavefront's order is fixed)
    if N <= 4096 and B == 1:                               # elementwise: a window of tokens
        i = torch.arange(N, device=dev)
        d = i[:, None] - i[None, :]
        tokens = ((d >= 0) & (d < N // 3))[None, None]
        o = fm.flash_attention_custom_mask(q, k, v, tokens, 0.125)
        for h in (0, H - 1):
            s = (q[0, h].float() @ k[0, h].float().T * 0.125).masked_fill(~tokens[0, 0], float("-inf"))
            assert rel_l2(o[0, h], torch.softmax(s, -1) @ v[0, h].float()) <= (3e-3 if dtype == torch.bfloat16 else 1e-3)


# Few row blocks at D = 64: shares of a list that meet in the launch, two, three or four at most, of at least 8 tiles (bf16 from 56 row
# blocks on: of one).  Row block r keeps r tiles (modulo the row blocks), so that every length is there, none and all among them.
@pytest.mark.parametrize("H,N,dtype,out_fp32", [(1, 1536, torch.float16, False), (1, 3600, torch.bfloat16, True), (1, 5120, torch.float16, True),
                                               (1, 5100, torch.bfloat16, False), (2, 4096, torch.float16, False), (1, 8190, torch.bfloat16, True)])
def test_shares_of_every_length(dev, H, N, dtype, out_fp32):
    import fa2_custom_mask as fm
    assert fwd_route_d64(1, H, N) == "pairs"
    nb = (N + 63) // 64
    g = torch.Generator(device=dev).manual_seed(N)
    q, k, v = [torch.randn(1, H, N, 64, generator=g, device=dev).to(dtype) for _ in range(3)]
    order = torch.rand(nb, nb, generator=g, device=dev).argsort(1).argsort(1)
    mask = (order < ((torch.arange(nb, device=dev) * 7) % (nb + 1))[:, None])[None, None]
    mask[0, 0, 3] = True
    mask[0, 0, 4] = False
    o_ref, lse_ref = naive_forward(q, k, v, mask, 0.125)
    bar = 3e-3 if (dtype == torch.bfloat16 and not out_fp32) else 1e-3
    none = torch.isinf(lse_ref)
    first = None
    for step in range(4):
        o, lse = fm.flash_attention_custom_mask_lse(q, k, v, mask, 0.125, out_fp32=out_fp32)
        assert torch.equal(torch.isinf(lse), none) and bool((o[none] == 0).all())
        assert rel_l2(o, o_ref) <= bar and float((lse[~none] - lse_ref[~none]).abs().max()) <= 2e-3
        assert first is None or torch.equal(o, first)
        first = o
    tokens = mask.repeat_interleave(64, 2).repeat_interleave(64, 3)[..., :N, :N].clone()
    tokens[0, 0, 1::2, ::3] = False                        # words: partly set tiles
    o = fm.flash_attention_custom_mask(q, k, v, tokens, 0.125)
    for h in (0, H - 1):
        s = (q[0, h].float() @ k[0, h].float().T * 0.125).masked_fill(~tokens[0, 0], float("-inf"))
        p = torch.nan_to_num(torch.softmax(s, -1), nan=0.0)
        assert rel_l2(o[0, h], p @ v[0, h].float()) <= (3e-3 if dtype == torch.bfloat16 else 1e-3)


# Ranges of workgroups and short lists of like length: a workgroup takes a row block, or a part of one of those that are left (three heads:
# none, one and two: parts; the numbers of tiles lie on both sides of the lines).  Rows without tiles; uneven lists, which stay on the ranges:
# growing ones, some of all tiles, long and short ones in turn (which heads are taken: own_rows_check.cpp).
@pytest.mark.parametrize("H,N,tiles,dtype", [(3, 10048, 20, torch.float16), (3, 10048, 63, torch.bfloat16), (3, 10048, 66, torch.float16),
                                             (2, 16100, 5, torch.float16), (1, 12000, 4, torch.bfloat16), (1, 12000, 30, torch.float16),
                                             (2, 9024, 24, torch.float16), (2, 9000, 50, torch.bfloat16), (2, 11000, 16, torch.float16),
                                             (1, 17536, 28, torch.float16), (1, 20000, 40, torch.bfloat16), (3, 9300, 30, torch.bfloat16)])
@pytest.mark.parametrize("kind", ["even", "causal", "holes", "whole", "turns"])
def test_row_blocks_of_workgroups(dev, H, N, tiles, dtype, kind):
    import fa2_custom_mask as fm
    assert fwd_route_d64(1, H, N) == "workgroups"
    nb = (N + 63) // 64
    g = torch.Generator(device=dev).manual_seed(tiles)
    q, k, v = [torch.randn(1, H, N, 64, generator=g, device=dev).to(dtype) for _ in range(3)]
    mask = torch.rand(1, H if kind == "holes" else 1, nb, nb, generator=g, device=dev) < tiles / nb
    i = torch.arange(nb, device=dev)
    if kind == "causal":
        mask &= i[:, None] >= i[None, :]
    if kind == "holes":
        mask &= (i % 5 != 0)[:, None]
        mask[0, 0] &= (i < 3)[:, None]                     # a head with three lists
    if kind == "whole":
        mask[..., [1, nb // 2, nb - 1], :] = True
        mask[..., 0] = True
    if kind == "turns":
        mask[..., ::2, nb // 16:] = False
    o_ref, lse_ref = naive_forward(q, k, v, mask, 0.125)
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, mask, 0.125)
    none = torch.isinf(lse_ref)
    assert torch.equal(torch.isinf(lse), none) and bool((o[none] == 0).all())
    assert rel_l2(o, o_ref) <= (3e-3 if dtype == torch.bfloat16 else 1e-3) and float((lse[~none] - lse_ref[~none]).abs().max()) <= 2e-3


# The same for elementwise masks: a window of tokens, whose lists but the first ones are of like length, and one whose first tokens and
# last keep all others.
@pytest.mark.parametrize("kind", ["window", "window and whole rows"])
@pytest.mark.parametrize("H,N,tokens,dtype", [(1, 12000, 1000, torch.float16), (3, 9300, 1500, torch.bfloat16), (2, 9024, 1400, torch.float16)])
def test_row_blocks_of_workgroups_elementwise(dev, H, N, tokens, dtype, kind):
    import fa2_custom_mask as fm
    assert fwd_route_d64(1, H, N) == "workgroups"
    g = torch.Generator(device=dev).manual_seed(tokens)
    q, k, v = [torch.randn(1, H, N, 64, generator=g, device=dev).to(dtype) for _ in range(3)]
    i = torch.arange(N, device=dev)
    mask = (i[:, None] - i[None, :]).abs() < tokens
    if kind != "window":
        mask[:70] = True
        mask[-1] = True
    o = fm.flash_attention_custom_mask(q, k, v, mask[None, None], 0.125)
    for h in (0, H - 1):
        s = (q[0, h].float() @ k[0, h].float().T * 0.125).masked_fill(~mask, float("-inf"))
        assert rel_l2(o[0, h], torch.softmax(s, -1) @ v[0, h].float()) <= (3e-3 if dtype == torch.bfloat16 else 1e-3)
