"""The ways the forward at D = 64 splits a launch (ranges of workgroups, ranges of wavefronts, whole row blocks), and
sequence lengths that are not a multiple of 64, whose last tile must touch nothing beyond the tensors.  Against the CPU
oracle on sampled heads."""
import numpy as np
import pytest
import torch

from oracle import bsattn_oracle as orc
from helpers import make_qkv, uniform_block_mask, errors, f32, same_up_to_rounding, fwd_route_d64

pytestmark = pytest.mark.gpu

MAXABS = {torch.float16: 2e-2, torch.bfloat16: 3e-2}
RELL2 = {torch.float16: 1e-3, torch.bfloat16: 3e-3}          # bf16-typed results: rounding an exact one costs 1.7e-3


def block_mask(nb, keep, seed):
    m = uniform_block_mask(1, 1, nb, keep, seed)
    m[0, 0, nb // 3, :] = False                              # a row block without kept tiles
    m[0, 0, nb // 2, :] = True                               # a full one: ranges end inside it
    m[0, 0, :, nb - 1] |= torch.arange(nb) % 2 == 0          # the last, partly filled column
    return m


# wavefronts of the GPU: 2048.  2048 row blocks: ranges of wavefronts, each a whole number of row blocks on average;
# 2080 and 2400: ranges that cut row blocks; 3200: whole row blocks; 8 ragged row blocks of 4 heads: pairs of wavefronts; 130 of 3
# heads: ranges of workgroups
@pytest.mark.parametrize("B,H,N", [(2, 16, 4096), (1, 40, 3300), (1, 24, 6337), (4, 40, 1250), (1, 4, 449), (1, 3, 8300)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("elementwise", [False, True])
def test_modes(dev, B, H, N, dtype, elementwise):
    import fa2_custom_mask as fm
    assert fwd_route_d64(B, H, N) == {4096: "wavefronts", 3300: "wavefronts", 6337: "wavefronts", 1250: "rows", 449: "pairs", 8300: "workgroups"}[N]
    nb = -(-N // 64)
    q, k, v = make_qkv(B, H, N, 64, dtype, 500 + N)
    block = block_mask(nb, 0.3, 501 + N)
    dense = torch.from_numpy(orc.expand_block_mask(block.numpy())[..., :N, :N].copy())
    if elementwise:
        i = torch.arange(N)
        dense = dense & ((i[:, None] - i[None, :]) % 7 != 0)
        dense[0, 0, 5, :] = False                            # a query without keys
    mask = dense if elementwise else block
    o, lse = fm.flash_attention_custom_mask_lse(q.to(dev), k.to(dev), v.to(dev), mask.to(dev), 0.125)
    torch.cuda.synchronize()
    assert o.shape == (B, H, N, 64) and lse.shape == (B, H, N) and bool(torch.isfinite(o.float()).all())
    for b, h in ((0, 0), (B - 1, H - 1)):
        sl = (slice(b, b + 1), slice(h, h + 1))
        o_ref, lse_ref = orc.naive_attention(f32(q[sl]), f32(k[sl]), f32(v[sl]), dense.numpy(), 0.125, return_lse=True)
        ma, rl = errors(o[sl], o_ref)
        assert ma <= MAXABS[dtype] and rl <= RELL2[dtype], (b, h, ma, rl)
        fin = np.isfinite(lse_ref)
        got = lse[sl].cpu().numpy()
        assert np.array_equal(np.isfinite(got), fin) and np.abs(got[fin] - lse_ref[fin]).max() <= 2e-3


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("N", [1, 63, 130, 191])
@pytest.mark.parametrize("contiguous_rows", [True, False])
def test_nothing_beyond_the_last_token_is_touched(dev, D, N, contiguous_rows):
    """q, k, v, dO are the first N rows of larger tensors that hold NaN behind them: a value read from there would
    reach a result (even with weight zero)."""
    import fa2_custom_mask as fm
    B, H = 1, 3
    pad = 64 - N % 64
    row = D if contiguous_rows else D + 8
    g = torch.Generator().manual_seed(600 + N)
    big = torch.full((4, B, H, N + pad, row), float("nan"))
    big[:, :, :, :N, :D] = torch.randn(4, B, H, N, D, generator=g)
    q, k, v, do = big.half().to(dev)[:, :, :, :N, :D].unbind(0)
    nb = -(-N // 64)
    block = uniform_block_mask(1, 1, nb, 0.7, 601 + N)
    dense = orc.expand_block_mask(block.numpy())[..., :N, :N]
    sc = D ** -0.5
    res = fm.attention_forward_backward(q, k, v, block.to(dev), sc, do, out_fp32=True)
    torch.cuda.synchronize()
    o_ref, lse_ref = orc.naive_attention(f32(q), f32(k), f32(v), dense, sc, return_lse=True)
    dq, dk, dv = orc.attention_backward(f32(q), f32(k), f32(v), dense, sc, f32(do))[:3]
    for name, got, ref in zip(("o", "lse", "dq", "dk", "dv"), res, (o_ref, lse_ref, dq, dk, dv)):
        ma, rl = errors(got, ref)
        assert ma <= 2e-2 and (rl <= 1e-3 or ma <= 1e-5), (name, ma, rl)     # (a zero gradient has no relative error)


# D = 128, elementwise masks and ragged lengths: single groups of wavefronts (504 and 512 row blocks), two groups (32, 6 and 81), whose lists are
# shared by up to 4 workgroups.  Backward: lists of 13 and 16 tiles shared at D = 64 and 256.
@pytest.mark.parametrize("H,N,D", [(8, 4000, 128), (8, 4090, 128), (2, 1000, 128), (3, 100, 128), (1, 5184, 128), (8, 777, 64),
                                   (2, 1000, 64), (8, 777, 256), (2, 1000, 256), (12, 1400, 256)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("elementwise", [False, True])
@pytest.mark.parametrize("out_fp32", [False, True])
def test_shared_lists(dev, H, N, D, dtype, elementwise, out_fp32):
    import fa2_custom_mask as fm
    nb = -(-N // 64)
    q, k, v, do = make_qkv(1, H, N, D, dtype, 800 + N, n=4)
    block = block_mask(nb, 0.3, 801 + N)
    dense = torch.from_numpy(orc.expand_block_mask(block.numpy())[..., :N, :N].copy())
    if elementwise:
        i = torch.arange(N)
        dense = dense & (i[:, None] - i[None, :] < N // 3) & ((i[:, None] - i[None, :]) % 7 != 0)
        dense[0, 0, 5, :] = False
    mask = dense if elementwise else block
    sc = D ** -0.5
    res = fm.attention_forward_backward(q.to(dev), k.to(dev), v.to(dev), mask.to(dev), sc, do.to(dev), out_fp32=out_fp32)
    torch.cuda.synchronize()
    sl = (slice(None), slice(H - 1, H))
    o_ref, lse_ref = orc.naive_attention(f32(q[sl]), f32(k[sl]), f32(v[sl]), dense.numpy(), sc, return_lse=True)
    # fp32 results: P and dS have 16 bits; 16-bit ones are rounded once more (bf16: 2^-9 for O, the gradients' P and dS too)
    rel = 1e-3 if out_fp32 or dtype == torch.float16 else 3e-3
    ma, rl = errors(res[0][sl], o_ref)
    assert ma <= MAXABS[dtype] and rl <= rel, (ma, rl)
    fin = np.isfinite(lse_ref)
    lse = res[1][sl].cpu().numpy()
    assert np.array_equal(np.isfinite(lse), fin) and np.abs(lse[fin] - lse_ref[fin]).max() <= 2e-3
    if N <= 1400:
        grads = orc.attention_backward(f32(q[sl]), f32(k[sl]), f32(v[sl]), dense.numpy(), sc, f32(do[sl]))[:3]
        for name, got, ref in zip(("dq", "dk", "dv"), res[2:], grads):
            ma, rl = errors(got[sl], ref)
            assert rl <= (2e-3 if rel == 1e-3 else 1e-2), (name, ma, rl)


def long_row_masks(nb, H):
    """Block masks [1, H, nb, nb] with row blocks that are much longer than the others (ROWS_MODE cuts them)."""
    g = torch.Generator().manual_seed(77)
    m = torch.rand(1, H, nb, nb, generator=g) < 0.06
    m[:, :, :, 1] = True
    m[0, 0, :4] = True                                       # the rows of leading text tokens
    m[0, 1] = False
    m[0, 1, nb // 2] = True                                  # one full row block, nothing else
    m[0, 2] = False
    m[0, 2, torch.arange(nb) % 4 == 1] = True                # a quarter of the row blocks full, the others empty
    m[0, 3, nb - 1] = True                                   # the last, partly filled row block
    m[0, 3, 0, :25] = True                                   # (25 tiles: the shortest that is cut)
    m[0, 4] = True                                           # no row block longer than the others
    return m


# 3240 and 3264 row blocks: one wavefront takes one; the long ones are cut
@pytest.mark.parametrize("H,N,elementwise", [(60, 3450, False), (60, 3450, True), (24, 8704, False)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_long_row_blocks(dev, H, N, dtype, elementwise):
    import fa2_custom_mask as fm
    nb = -(-N // 64)
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, 64, dtype, 600 + N)]
    block = long_row_masks(nb, H)
    mask = block.to(dev)
    if elementwise:
        i = torch.arange(N, device=dev)
        mask = mask.repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N] & ((i[:, None] - i[None, :]) % 7 != 0)
    call = lambda: fm.flash_attention_custom_mask_lse(q, k, v, mask, 0.125)
    o, lse = call()
    for _ in range(3):                                       # parts are summed in their order: the same bits every time
        o2, lse2 = call()
        assert torch.equal(o, o2) and torch.equal(lse, lse2)
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o3, lse3 = call()
    for _ in range(3):                                       # (a replay counts its parts in again)
        o3.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, o3) and torch.equal(lse, lse3)
        call()
    if N % 64 == 0:                                          # the library's own scratch memory: half as many parts
        from fa2_custom_mask import _ext
        lists = fm.block_mask_to_lists(mask)
        o4, lse4 = torch.empty_like(o), torch.empty_like(lse)
        code, st = _ext.dtype_code(dtype), _ext.strides4(q)
        rc = _ext.lib().bsattn_fwd_static(q.data_ptr(), k.data_ptr(), v.data_ptr(), o4.data_ptr(), lse4.data_ptr(), lists.row_ptr_ptr,
                                          lists.col_idx_ptr, 1, H, 1, H, N, 64, code, code, 0.125, st, st, st, st, _ext.current_stream(dev))
        torch.cuda.synchronize()
        assert rc == 0 and same_up_to_rounding(o4, o, rel=2.0 ** -6, abs_=2e-3)
        fin = torch.isfinite(lse)
        assert torch.equal(torch.isfinite(lse4), fin) and float((lse4 - lse)[fin].abs().max()) <= 2e-3
    for h in range(6 if N < 4000 else 3):
        keep = (mask[0, h] if elementwise else mask[0, h].repeat_interleave(64, 0)[:N].repeat_interleave(64, 1)[:, :N])
        s = (q[0, h].float() @ k[0, h].float().T * 0.125).masked_fill(~keep, float("-inf"))
        ref_lse = torch.logsumexp(s, -1)
        ref = torch.softmax(s, -1).nan_to_num(0.0) @ v[0, h].float()
        ma, rl = errors(o[0, h], ref)
        assert ma <= MAXABS[dtype] and rl <= RELL2[dtype], (h, ma, rl)
        fin = torch.isfinite(ref_lse)
        assert torch.equal(torch.isfinite(lse[0, h]), fin) and float((lse[0, h] - ref_lse)[fin].abs().max()) <= 2e-3


# Heads that are not a multiple of 8 share the XCDs unevenly (place.h); every head has a mask of its own, so that one taken
# for another shows.  D = 64: 24 row blocks (pairs of wavefronts), 390 (ranges of workgroups), 1690 (ranges of wavefronts), 3375
# (row blocks, heads in groups), 3250 (row blocks, all heads at once).
@pytest.mark.parametrize("H,N,D", [(3, 449, 64), (3, 8300, 64), (13, 8300, 64), (27, 8000, 64), (25, 8320, 64), (3, 1000, 128), (11, 3200, 128), (5, 700, 256)])
def test_uneven_heads(dev, H, N, D):
    import fa2_custom_mask as fm
    nb = -(-N // 64)
    q, k, v, do = [x.to(dev) for x in make_qkv(1, H, N, D, torch.float16, 900 + N, n=4)]
    block = uniform_block_mask(1, H, nb, 0.2, 901 + N).to(dev)
    sc = D ** -0.5
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, block, sc)
    for h in range(H):
        keep = block[0, h].repeat_interleave(64, 0)[:N].repeat_interleave(64, 1)[:, :N]
        s = (q[0, h].float() @ k[0, h].float().T * sc).masked_fill(~keep, float("-inf"))
        ma, rl = errors(o[0, h], torch.softmax(s, -1) @ v[0, h].float())
        assert ma <= MAXABS[torch.float16] and rl <= RELL2[torch.float16], (h, ma, rl)
        assert float((lse[0, h] - torch.logsumexp(s, -1)).abs().max()) <= 2e-3
    if N > 4000:
        return
    grads = fm.attention_forward_backward(q, k, v, block, sc, do)[2:]
    for h in range(H):
        sl = (slice(None), slice(h, h + 1))
        alone = fm.attention_forward_backward(q[sl], k[sl], v[sl], block[sl], sc, do[sl])[2:]
        for got, ref in zip(grads, alone):        # (another number of shares: another order of summation)
            assert errors(got[sl], ref)[1] <= 1e-3, h


# D = 128, block masks: two groups of wavefronts, up to four and two shares, single groups
@pytest.mark.parametrize("H,N", [(1, 832), (6, 1536), (6, 1500), (2, 4096), (4, 4096), (5, 4096), (7, 2048)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_shares_of_block_mask_lists(dev, H, N, dtype):
    import fa2_custom_mask as fm
    nb = -(-N // 64)
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, 128, dtype, 950 + N)]
    block = torch.cat([block_mask(nb, 0.3, 951 + N + h) for h in range(H)], 1)
    block[0, 0, 1] = False
    block[0, 0, 1, :2] = True                                # fewer tiles than shares
    sc = 128 ** -0.5
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, block.to(dev), sc)
    for h in range(H):
        keep = block[0, h].to(dev).repeat_interleave(64, 0)[:N].repeat_interleave(64, 1)[:, :N]
        s = (q[0, h].float() @ k[0, h].float().T * sc).masked_fill(~keep, float("-inf"))
        ma, rl = errors(o[0, h], torch.softmax(s, -1).nan_to_num(0.0) @ v[0, h].float())
        assert ma <= MAXABS[dtype] and rl <= RELL2[dtype], (h, ma, rl)
        ref = torch.logsumexp(s, -1)
        fin = torch.isfinite(ref)
        assert torch.equal(torch.isfinite(lse[0, h]), fin) and float((lse[0, h] - ref)[fin].abs().max()) <= 2e-3


# D = 64, few row blocks: 4 pairs of wavefronts per row block (1, 2 and 4 shares of its list), 2 pairs, the longest lists
# (128 tiles), the first length beyond; lists shorter than the pairs are many, empty ones, ragged lengths, queries without keys
@pytest.mark.parametrize("H,N", [(1, 64), (3, 130), (5, 512), (8, 2048), (9, 2048), (1, 3584), (1, 4090), (1, 5000), (2, 8192), (5, 6400), (1, 8193)])
@pytest.mark.parametrize("dtype,out_fp32", [(torch.float16, False), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("elementwise", [False, True])
def test_short_lists(dev, H, N, dtype, out_fp32, elementwise):
    import fa2_custom_mask as fm
    nb = -(-N // 64)
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, 64, dtype, 970 + N)]
    block = torch.cat([block_mask(nb, 0.3, 971 + N + h) for h in range(H)], 1) if nb > 2 else torch.ones(1, H, nb, nb, dtype=torch.bool)
    block[0, -1, nb - 1] = True                              # the last row block: all tiles
    mask = block.to(dev)
    if elementwise:
        i = torch.arange(N, device=dev)
        mask = mask.repeat_interleave(64, 2)[:, :, :N].repeat_interleave(64, 3)[..., :N] & ((i[:, None] - i[None, :]) % 7 != 0)
        mask[:, :, N // 2] = False                           # a query without keys
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, mask, 0.125, out_fp32=out_fp32)
    rel = 1e-3 if out_fp32 or dtype == torch.float16 else RELL2[dtype]
    for h in range(H):
        keep = mask[0, h] if elementwise else mask[0, h].repeat_interleave(64, 0)[:N].repeat_interleave(64, 1)[:, :N]
        s = (q[0, h].float() @ k[0, h].float().T * 0.125).masked_fill(~keep, float("-inf"))
        ma, rl = errors(o[0, h], torch.softmax(s, -1).nan_to_num(0.0) @ v[0, h].float())
        assert ma <= MAXABS[dtype] and rl <= rel, (h, ma, rl)
        ref = torch.logsumexp(s, -1)
        fin = torch.isfinite(ref)
        assert torch.equal(torch.isfinite(lse[0, h]), fin) and float((lse[0, h] - ref)[fin].abs().max()) <= 2e-3

# D = 256, block masks: a wavefront has half of a tile's keys, and the halves meet with references of their own (`skew`: scores
# of one half far above the other's, of the second or by turns).  One tile; shares (fewer tiles than shares); none; strided rows;
# ragged lengths with a key or none in the second half of the last tile.
@pytest.mark.parametrize("H,N,skew,strided", [(1, 64, 0, False), (2, 1024, 1, False), (4, 2048, 2, True), (24, 1344, 1, True), (9, 2048, 0, False),
                                                (2, 20, 0, False), (2, 33, 0, False), (4, 2000, 1, True), (24, 1313, 2, False)])
@pytest.mark.parametrize("dtype,out_fp32", [(torch.float16, False), (torch.bfloat16, False), (torch.bfloat16, True)])
def test_halves_of_keys(dev, H, N, skew, strided, dtype, out_fp32):
    import fa2_custom_mask as fm
    nb = -(-N // 64)
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, 256, dtype, 970 + N)]
    key = torch.arange(N, device=dev)
    if skew:
        k[:, :, (key % 64 >= 32) if skew == 1 else ((key // 32 + key // 64) % 2 == 1)] *= 5
    if strided:
        q, k, v = torch.stack([q, k, v], 3).unbind(3)
    block = torch.cat([uniform_block_mask(1, 1, nb, 0.3, 971 + N + h) for h in range(H)], 1)
    if nb > 1:
        block[0, 0, 1] = False
        block[0, 0, 0] = torch.arange(nb) == 1
    sc = 256 ** -0.5
    # fp16: the scale is folded into Q, whose rounding (rms 0.41 of 2^-11 per element) moves a score of rms 5 by 1.0e-3 rms; a
    # numerator moves by as much of itself, lse by at most 6 of these over all queries.  bf16 results: numerators are rounded to
    # bf16 and summed so, which moves the sum of a query with one dominant key by up to 2^-8.
    fold = 0.41 * 2.0 ** -11 * 5 if skew and dtype == torch.float16 else 0.0
    lse_max = 2.0 ** -8 if dtype == torch.bfloat16 and not out_fp32 else 2e-3 + 6 * fold
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, block.to(dev), sc, out_fp32=out_fp32)
    for h in sorted({0, 1 % H, H // 2, H - 1}):
        keep = block[0, h].to(dev).repeat_interleave(64, 0)[:N].repeat_interleave(64, 1)[:, :N]
        s = (q[0, h].float() @ k[0, h].float().T * sc).masked_fill(~keep, float("-inf"))
        ma, rl = errors(o[0, h], torch.softmax(s, -1).nan_to_num(0.0) @ v[0, h].float())
        assert ma <= MAXABS[dtype] and rl <= RELL2[torch.float16 if out_fp32 else dtype] + fold, (h, ma, rl)
        ref = torch.logsumexp(s, -1)
        fin = torch.isfinite(ref)
        assert torch.equal(torch.isfinite(lse[0, h]), fin) and float((lse[0, h] - ref)[fin].abs().max()) <= lse_max
