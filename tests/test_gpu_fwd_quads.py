"""Launches with few row blocks at D = 128 and 256: key halves and groups of wavefronts merged in LDS, lists cut into shares that meet in the
workspace (fwd_quad_kernel, fwd_wide_kernel).  Sizes on both sides of the rules' lines, tiles left over, lists from empty to all tiles,
rows of K and V with and without gaps.

Against softmax attention in 64 bits.  P is rounded to the inputs' type (to fp16 with fp32 results) and the results to their own:
relative 2-norm 2^-11 each with fp16, 2^-9 each (uniform rounding of 2^-8 at most) with bf16, so 1e-3 and 4e-3 hold both."""
import pytest
import torch

from helpers import make_qkv

pytestmark = pytest.mark.gpu

D = 128
SIZES = [(1, 1), (1, 65), (2, 447), (7, 1000),       # two groups, whole lists
         (1, 1280), (1, 2047), (3, 1280),            # ... up to four shares
         (3, 2048), (2, 6016),                       # ... two (the second: only the long lists of a causal mask)
         (1, 8300),                                  # block masks: one group, three shares; words: two groups
         (4, 4096),                                  # two groups, one row block per compute unit
         (8, 2304), (4, 5121), (3, 5504)]            # one group; ... two shares; ... three of the longest lists, which fill the GPU
WIDE_SIZES = [(1, 450, True), (1, 512, False), (1, 700, True), (2, 1500, False),       # lists cut from six tiles on, at D = 256
              (3, 5504, True),                       # more than a workgroup per compute unit: three shares of the longest
              (8, 4000, True), (10, 4161, False)]    # nearly two; more than a round, whose last lists are cut


def reference(q, k, v, dense, sc):
    """O and lse in 64 bits, on the GPU head by head; a query without a key: 0 and -inf."""
    o, lse = torch.zeros(q.shape, dtype=torch.float64, device=q.device), torch.empty(q.shape[:3], dtype=torch.float64, device=q.device)
    for h in range(q.shape[1]):
        s = (q[0, h].double() @ k[0, h].double().T * sc).masked_fill(~dense, float("-inf"))
        lse[0, h] = torch.logsumexp(s, -1)
        o[0, h] = torch.nan_to_num(torch.softmax(s, -1)) @ v[0, h].double()
    return o, lse


def block_mask(nb, kind):
    g = torch.Generator().manual_seed(nb)
    m = torch.ones(nb, nb, dtype=torch.bool).tril() if kind == "causal" else torch.rand(nb, nb, generator=g) < 0.2
    if nb > 3:
        m[2] = False                                  # a row block that keeps nothing
        m[nb - 2] = True                              # ... and one that keeps everything
    return m


def check(dev, D, H, N, dtype, out_fp32, kind, strided):
    import fa2_custom_mask as fm
    nb = -(-N // 64)
    q, k, v = [x.to(dev) for x in make_qkv(1, H, N, D, dtype, N + H)]
    if strided:                                       # a packed projection's: [token][q, k, v][head]
        q, k, v = torch.stack([x.transpose(1, 2) for x in (q, k, v)], 2).transpose(1, 3).unbind(2)
        assert q.shape == (1, H, N, D) and k.stride(2) == 3 * H * D
    if kind.startswith("token"):
        mask = torch.ones(N, N, dtype=torch.bool, device=dev).tril() if kind.endswith("causal") else (
            torch.rand(N, N, generator=torch.Generator(dev).manual_seed(N), device=dev) < 0.3)
        mask[N // 2] = False                          # a query without a key
        dense = mask
    else:
        mask = block_mask(nb, kind).to(dev)
        dense = mask.repeat_interleave(64, 0).repeat_interleave(64, 1)[:N, :N]
    if mask.shape[0] == N and not kind.startswith("token"):
        pytest.skip("one token: a block mask cannot be told from an elementwise one")
    run = lambda: fm.flash_attention_custom_mask_lse(q, k, v, mask[None, None], D ** -0.5, out_fp32=out_fp32)
    o, lse = run()
    ref, ref_lse = reference(q, k, v, dense, D ** -0.5)
    none = torch.isinf(ref_lse)
    assert torch.equal(torch.isinf(lse), none) and bool((o[none] == 0).all())
    rel = float((o.double() - ref).norm() / ref.norm().clamp(min=1e-30))
    assert rel <= (4e-3 if dtype == torch.bfloat16 and not out_fp32 else 1e-3)
    assert float((lse.double() - ref_lse)[~none].abs().max()) <= 2e-3 if bool((~none).any()) else True
    again = run()
    assert torch.equal(again[0], o) and torch.equal(again[1], lse)      # whoever adds the shares up adds them in their order


@pytest.mark.parametrize("kind", ["causal", "uniform", "token causal", "token random"])
@pytest.mark.parametrize("dtype,out_fp32", [(torch.float16, False), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("H,N", SIZES)
def test_against_64_bits(dev, H, N, dtype, out_fp32, kind):
    check(dev, D, H, N, dtype, out_fp32, kind, False)


@pytest.mark.parametrize("kind", ["causal", "uniform", "token causal", "token random"])
@pytest.mark.parametrize("dtype,out_fp32", [(torch.float16, False), (torch.bfloat16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("D,H,N,strided", [(256,) + x for x in WIDE_SIZES] + [(128, 3, 1280, True), (128, 4, 5121, True)])
def test_other_rows(dev, D, H, N, strided, dtype, out_fp32, kind):
    check(dev, D, H, N, dtype, out_fp32, kind, strided)


# One head of long lists, sampled row blocks: a full round of single groups; a token window in one round of two groups and a little more,
# in less and in more than 256 row blocks of single groups.
@pytest.mark.parametrize("N,window", [(30720, 0), (16500, 1600), (16500, 8000), (18432, 9000)])
def test_long_lists(dev, N, window):
    import fa2_custom_mask as fm
    nb = -(-N // 64)
    q, k, v = [x.to(dev) for x in make_qkv(1, 1, N, D, torch.bfloat16, N)]
    if window:
        i = torch.arange(N, device=dev)
        dense = mask = (i[:, None] - i[None, :] >= 0) & (i[:, None] - i[None, :] < window)
    else:
        mask = block_mask(nb, "uniform").to(dev)
    o, lse = fm.flash_attention_custom_mask_lse(q, k, v, mask[None, None], D ** -0.5, out_fp32=True)
    for m in sorted({0, 2, 3, nb // 2, nb - 9, nb - 2, nb - 1}):
        rows = slice(64 * m, min(N, 64 * m + 64))
        keep = dense[rows] if window else mask[m].repeat_interleave(64)[None, :N].expand(64, -1)
        s = (q[0, 0, rows].double() @ k[0, 0].double().T * D ** -0.5).masked_fill(~keep, float("-inf"))
        ref, ref_lse = torch.nan_to_num(torch.softmax(s, -1)) @ v[0, 0].double(), torch.logsumexp(s, -1)
        assert float((o[0, 0, rows].double() - ref).norm()) <= 1e-3 * float(ref.norm()), m
        assert torch.equal(torch.isinf(lse[0, 0, rows]), torch.isinf(ref_lse)), m
        assert float(torch.nan_to_num(lse[0, 0, rows].double() - ref_lse, nan=0.0).abs().max()) <= 2e-3, m


def test_scratch_limit():
    """bsattn_fwd_static takes what it took: launches whose shares would not fit the library's scratch memory have fewer."""
    from fa2_custom_mask import _ext
    import fa2_custom_mask as fm
    q, k, v = [x.to("cuda") for x in make_qkv(1, 4, 8192, D, torch.float16, 3)]
    mask = torch.ones(1, 1, 128, 128, dtype=torch.bool, device="cuda").tril()
    lists = fm.block_mask_to_lists(mask)
    o = torch.empty_like(q)
    rc = _ext.lib().bsattn_fwd_static(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), None, lists.row_ptr_ptr, lists.col_idx_ptr, 1, 1,
                                      1, 4, 8192, D, 0, 0, D ** -0.5, _ext.strides4(q), _ext.strides4(k), _ext.strides4(v), _ext.strides4(o),
                                      _ext.current_stream(q.device))
    assert rc == 0
    ref = fm.flash_attention_custom_mask(q, k, v, mask, D ** -0.5)
    assert float((o.float() - ref.float()).norm() / ref.float().norm()) <= 1e-3
