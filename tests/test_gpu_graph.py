"""The library calls under HIP graph capture: every entry point only enqueues kernels on the
given stream (no allocation, no synchronisation, no memset nodes), so a captured call can be
replayed.  Each graph is replayed several times, with new inputs written in place and eager work
and synchronisations between the replays, and every replay is checked against the eager result
on the same inputs (a replay repeats the launch parameters of the capture, including the number
that marks a launch's partial results in the forward workspace)."""
import numpy as np
import pytest
import torch

from helpers import make_qkv, uniform_block_mask, causal_block_mask, same_up_to_rounding, fwd_route_d64

pytestmark = pytest.mark.gpu


def replay_and_compare(dev, B, H, N, D, dtype, mask, seed, replays=4):
    import fa2_custom_mask as fm
    sc = 1.0 / np.sqrt(D)
    ins = [x.to(dev) for x in make_qkv(B, H, N, D, dtype, seed, n=4)]
    mask = mask.to(dev)
    eager = fm.attention_forward_backward(ins[0], ins[1], ins[2], mask, sc, ins[3])    # also fills the list cache
    torch.cuda.synchronize()
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        fm.attention_forward_backward(ins[0], ins[1], ins[2], mask, sc, ins[3])          # warm-up on the capture stream
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = fm.attention_forward_backward(ins[0], ins[1], ins[2], mask, sc, ins[3])
    for r in range(replays):
        if r > 0:     # new inputs, written in place into the tensors the graph reads
            fresh = make_qkv(B, H, N, D, dtype, seed + 100 * r, n=4)
            for dst, src in zip(ins, fresh):
                dst.copy_(src.to(dev))
            eager = fm.attention_forward_backward(ins[0], ins[1], ins[2], mask, sc, ins[3])
            torch.cuda.synchronize()
        for t in captured:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for name, got, ref in zip(("o", "lse", "dq", "dk", "dv"), captured, eager):
            fin = torch.isfinite(ref)
            assert torch.equal(torch.isfinite(got), fin), (r, name)      # lse = -inf for a query without keys
            # (forward nondeterminism: O may round differently, and the gradients see that O)
            assert same_up_to_rounding(got[fin], ref[fin], rel=2.0 ** -7, abs_=4e-3), (r, name)


def test_replay_d64_rows_shared_between_workgroups(dev):
    """One head, 64 row blocks: up to four shares of a row block's list, whose parts the last one in sums."""
    replay_and_compare(dev, 1, 1, 4096, 64, torch.float16, uniform_block_mask(1, 1, 64, 0.6, 3001), 3002)


# one head, 129 row blocks on 512 workgroups: every row block is finished from published parts; 3 heads (ranges that are not the
# same number on every XCD); ranges of wavefronts; row blocks, the long ones cut
@pytest.mark.parametrize("H,N,dtype,route", [(1, 8256, torch.float16, "workgroups"), (3, 8256, torch.bfloat16, "workgroups"),
                                             (12, 8192, torch.float16, "wavefronts"), (40, 5120, torch.bfloat16, "rows")])
def test_replay_d64_parts_counted_in(dev, H, N, dtype, route):
    """Row blocks that the workgroup counted in last finishes: a replay repeats the launch's mark, and the counters start from zero
    in every one."""
    assert fwd_route_d64(1, H, N) == route
    nb = N // 64
    m = uniform_block_mask(1, 1, nb, 0.1, 3011)
    m[0, 0, 5, :] = True                                     # (row blocks much longer than the others)
    m[0, 0, nb - 2, :] = True
    m[0, 0, 7, :] = False
    replay_and_compare(dev, 1, H, N, 64, dtype, m, 3012, replays=3)


def test_replay_d128_bf16_many_heads(dev):
    """The wavefront-pair forward, the backward without shared lists."""
    replay_and_compare(dev, 2, 8, 2048, 128, torch.bfloat16, causal_block_mask(1, 1, 32, 0.5, 3003), 3004)


def test_replay_d256_lists_shared(dev):
    """Head dimension 256 with few row blocks: the forward's shares summed by the last one in, the backward's parts by a second kernel."""
    replay_and_compare(dev, 1, 2, 2048, 256, torch.float16, uniform_block_mask(1, 2, 32, 0.5, 3005), 3006, replays=3)


@pytest.mark.parametrize("H,N", [(1, 2048), (3, 5120)])
def test_replay_d128_lists_shared(dev, H, N):
    """Head dimension 128 with few row blocks: up to four shares of every list, two of the long ones."""
    replay_and_compare(dev, 1, H, N, 128, torch.bfloat16, causal_block_mask(1, 1, N // 64, 1.0, 3007), 3008, replays=3)


def test_replay_elementwise_mask_ragged_length(dev):
    g = torch.Generator().manual_seed(3007)
    N = 1000
    m = (torch.rand(1, 1, N, N, generator=g) < 0.3) & torch.tril(torch.ones(N, N, dtype=torch.bool))
    m[0, 0, 17, :] = False
    replay_and_compare(dev, 1, 3, N, 64, torch.float16, m, 3008, replays=3)


def test_replay_mask_to_lists(dev):
    """The preprocessing kernels in a graph: the mask is rewritten in place between the replays."""
    import fa2_custom_mask as fm
    from oracle import bsattn_oracle as orc
    nb = 96
    mask = uniform_block_mask(2, 3, nb, 0.3, 3009).to(dev)
    fm.block_mask_to_lists(mask, want_groups=True)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        fm.block_mask_to_lists(mask, want_groups=True)
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        lists = fm.block_mask_to_lists(mask, want_groups=True)
    for r in range(4):
        new = uniform_block_mask(2, 3, nb, 0.1 + 0.2 * r, 3010 + r)
        if r == 3:
            new[:] = False
        mask.copy_(new.to(dev))
        graph.replay()
        torch.cuda.synchronize()
        g_ref, n_ref = orc.build_groups_from_block_mask(new.numpy())
        G, T = [int(x) for x in lists.counts.cpu()]
        if g_ref is None:
            assert G == 0 and T == 0
            continue
        assert G == len(g_ref) and T == len(n_ref)
        assert np.array_equal(lists.groups[:G].cpu().numpy(), g_ref)
        assert np.array_equal(lists.col_idx[:T].cpu().numpy(), n_ref)


@pytest.mark.parametrize("elementwise,N", [(False, 640), (True, 640), (False, 8256)])
def test_lists_made_under_capture_are_the_graphs(dev, elementwise, N):
    """A mask that is first seen while a graph is being captured: its lists (a block mask has some for N = 8256 only, with the other
    length the forward reads the mask itself) are made by the replays, also of what is written to the mask between them, and no
    eager call takes them for its own."""
    import fa2_custom_mask as fm
    from fa2_custom_mask import _ext
    from fa2_custom_mask.utils import lists_cache, grid_cache
    assert _ext.lib().bsattn_fwd_takes_mask(1, 2, N, 64) == (N == 640)
    q, k, v = [x.to(dev) for x in make_qkv(1, 2, N, 64, torch.float16, 81)]
    masks = [uniform_block_mask(1, 1, N // 64, 0.4, 82 + i).to(dev) for i in range(4)]
    if elementwise:
        masks = [m.repeat_interleave(64, 2).repeat_interleave(64, 3).tril().contiguous() for m in masks]
    call = lambda mask: fm.flash_attention_custom_mask(q, k, v, mask, 0.125)
    eager = [call(m.clone()) for m in masks]
    mask = masks[0].clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = call(mask)
    assert lists_cache.get(mask, N, False) is None and grid_cache.get(mask, N) is None
    assert same_up_to_rounding(call(mask), eager[0])                 # no replay has filled the graph's lists yet
    for i in (0, 1, 2, 3, 1):
        mask.copy_(masks[i])
        captured.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert same_up_to_rounding(captured, eager[i]), i
        assert same_up_to_rounding(call(mask), eager[i]), i


# D = 64 with a row block per workgroup (columns from the mask), 2 shares, ranges (lists); D = 128, 256
@pytest.mark.parametrize("H,N,D,takes_mask", [(2, 640, 64, 1), (1, 6400, 64, 1), (1, 8256, 64, 0), (2, 700, 128, 1), (1, 1024, 256, 1)])
@pytest.mark.parametrize("per_head", [False, True])
def test_mask_seen_before_the_capture_stays_as_it_was(dev, H, N, D, takes_mask, per_head):
    """A mask that one eager call has seen: a graph captured after it keeps seeing the mask as it was, whatever is written to the
    mask later, and eager calls see what is written."""
    import fa2_custom_mask as fm
    from fa2_custom_mask import _ext, utils
    assert _ext.lib().bsattn_fwd_takes_mask(1, H, N, D) == takes_mask
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, D, torch.float16, 91)]
    nb = -(-N // 64)
    masks = [uniform_block_mask(1, H if per_head else 1, nb, 0.3, 92 + i).to(dev) for i in range(3)]
    call = lambda mask: fm.flash_attention_custom_mask(q, k, v, mask, 0.125)
    eager = [call(m.clone()) for m in masks]
    utils.lists_cache.clear()
    mask = masks[0].clone()
    assert same_up_to_rounding(call(mask), eager[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = call(mask)
    for i in (0, 1, 2):
        mask.copy_(masks[i])
        captured.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert same_up_to_rounding(captured, eager[0]), i
    assert same_up_to_rounding(call(mask), eager[2])


@pytest.mark.parametrize("H,N,D", [(2, 640, 64), (1, 8256, 64), (2, 700, 128)])
@pytest.mark.parametrize("elementwise", [False, True])
def test_captured_lists_outlive_their_entries(dev, H, N, D, elementwise):
    """What a graph has captured of the caches is kept while the mask lives: its replays are right after eager calls with the mask
    written to, which replace the entries, and with many other masks, which push them out."""
    import fa2_custom_mask as fm
    from fa2_custom_mask import utils
    nb = -(-N // 64)
    if elementwise and N > 1000:
        N, nb = 1000, 16
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, D, torch.float16, 95)]
    masks = [uniform_block_mask(1, 1, nb, 0.3, 96 + i).to(dev) for i in range(12)]
    if elementwise:
        masks = [m.repeat_interleave(64, 2).repeat_interleave(64, 3)[:, :, :N, :N].tril().contiguous() for m in masks]
    call = lambda mask: fm.flash_attention_custom_mask(q, k, v, mask, 0.125)
    mask = masks[0].clone()
    eager = call(mask)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = call(mask)
    assert utils.captured._held[id(mask)][0]() is mask
    for i, other in enumerate(masks):
        if i % 2:
            mask.copy_(other)
        call(mask if i % 2 else other)
        captured.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert same_up_to_rounding(captured, eager), i
    held = id(mask)
    del mask
    assert held not in utils.captured._held
