"""Host boundary of the block-sparse attention operator.

Mirrors fa2_custom_mask/fa2_custom_mask.py of the reference: `build_groups_from_block_mask`
(:15-38) and the autograd function behind `flash_attention_custom_mask` (:40-157), with the
device work done by hand-written gfx950 kernels reached through the C ABI in include/bsattn.h.
"""
import ctypes

import torch

from . import _ext
from .utils import TILE, UNMADE, _host, block_mask_to_lists, lists_cache, grid_cache, mask_to_lists, num_tiles, is_block_form, _check_mask


def build_groups_from_block_mask(mask):
    """Same contract as the reference (fa2_custom_mask.py:15-38): bool [B,H,nb,nb] ->
    (groups int32 [G,5] = (b,h,m_block,start,length), n_list int32 [T]) on mask.device, rows
    without a kept tile omitted, (None, None) if nothing is kept.  The lists are produced by
    the GPU kernels; only the two sizes G and T are read back to shape the result."""
    assert mask.dtype == torch.bool                                   # :20
    _check_mask(mask)
    lists = block_mask_to_lists(mask, want_groups=True)
    G, T = lists.counts.tolist()
    if G == 0:                                                        # :34-35
        return None, None
    return lists.groups[:G].contiguous(), lists.col_idx[:T].contiguous()   # :36-38


def _prep(x):
    """Kernels need unit stride along the head dimension and 16-byte aligned rows."""
    if x.is_contiguous() and (x.shape[3] * x.element_size()) % 16 == 0 and x.data_ptr() % 16 == 0:
        return x                                                # (the usual case, decided without looking at strides)
    if x.stride(3) != 1 or any((s * x.element_size()) % 16 for s in x.stride()[:3]) or x.data_ptr() % 16:
        return x.contiguous()
    return x


def clear_workspaces():
    """Gives back the workspaces kept for reuse (one per device and stream, at most 8 and 256 MB each)."""
    _host.clear_workspaces()


def _like(x, dtype):
    """A result tensor laid out as the reference's torch.empty_like(x) lays it out (fa2_custom_mask.py:59,
    101-103): the dimension order of x by stride, without gaps.  For q, k, v sliced out of one packed
    [B, N, 3, H, D] tensor that is [B, N, H, D] order behind a [B, H, N, D] shape."""
    t = torch.empty_like(x, dtype=dtype)
    if x.is_contiguous() and x.shape[3] % 8 == 0:
        return t
    if t.stride(3) != 1 or any((s * t.element_size()) % 16 for s in t.stride()[:3]):
        t = torch.empty(x.shape, dtype=dtype, device=x.device)
    return t


_all_true = {}


def _dense_mask(device, nb):
    """mask=None means plain dense attention (the reference advertises the default but crashes on
    it: `groups` is unbound at fa2_custom_mask.py:69): one all-true block mask shared by all heads."""
    key = (device, nb)
    if key not in _all_true:
        with torch.inference_mode(False):    # an ordinary tensor also when first asked for in inference mode: its lists are cached
            _all_true[key] = torch.ones((1, 1, nb, nb), dtype=torch.bool, device=device)
    return _all_true[key]


def set_deterministic(on):
    """Process-wide switch (bsattn_set_deterministic), returns the previous setting.  On: two runs of the
    forward on the same inputs give the same bits; off (the default): the tiles of a row block go to
    the wavefronts as they become free, which is faster and changes the last bits from run to run.
    The backward is deterministic either way."""
    return bool(_ext.lib().bsattn_set_deterministic(1 if on else 0))


class ForwardPlan:
    """A forward call with every buffer allocated and every C argument marshalled once; run()
    only enqueues the kernels.  For loops that repeat the same shapes (serving, benchmarks)."""

    def __init__(self, q, k, v, lists, sm_scale, out_dtype=None, stream=None):
        B, H, N, D = q.shape
        if N % TILE or D not in (64, 128, 256):
            raise ValueError("a plan takes whole tiles only: N % 64 == 0 and D in {64, 128, 256}")
        self.q, self.k, self.v, self.lists = _prep(q), _prep(k), _prep(v), lists
        out_dtype = out_dtype or q.dtype
        self.o = _like(self.q, out_dtype)
        self.lse = torch.empty((B, H, N), dtype=torch.float32, device=q.device)
        wsb = _ext.fwd_workspace(B, H, N, D, q.device)
        self.ws = torch.empty(wsb, dtype=torch.uint8, device=q.device)
        self._keep = (_ext.strides4(self.q), _ext.strides4(self.k), _ext.strides4(self.v), _ext.strides4(self.o))
        stream = stream if stream is not None else torch.cuda.current_stream(q.device)
        tail = (lists.Bm, lists.Hm, B, H, N, D, _ext.dtype_code(q.dtype), _ext.dtype_code(out_dtype),
                float(sm_scale)) + self._keep + (self.ws.data_ptr(), wsb, ctypes.c_void_p(stream.cuda_stream))
        head = (self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(), self.o.data_ptr(), self.lse.data_ptr(),
                lists.row_ptr_ptr)
        if lists.bits is not None:
            raise ValueError("a plan takes block masks only")
        self._args = head + (lists.col_idx_ptr,) + tail
        self._fn = _ext.lib().bsattn_fwd

    def run(self):
        rc = self._fn(*self._args)
        if rc != 0:
            _ext.check(rc, "bsattn_fwd")
        return self.o, self.lse


class BackwardPlan:
    """The backward counterpart of ForwardPlan: dq, dk, dv and the workspace allocated once, the C
    arguments marshalled once; run() only enqueues the kernels.  o and lse are the forward's
    results for the same q, k, v; block masks only."""

    def __init__(self, q, k, v, o, do, lse, lists, lists_t, sm_scale, out_dtype=None, stream=None):
        B, H, N, D = q.shape
        if N % TILE or D not in (64, 128, 256) or lists.bits is not None:
            raise ValueError("a plan takes whole tiles and block masks only: N % 64 == 0 and D in {64, 128, 256}")
        self.q, self.k, self.v, self.o, self.do = _prep(q), _prep(k), _prep(v), _prep(o), _prep(do)
        self.lse, self.lists, self.lists_t = lse, lists, lists_t
        out_dtype = out_dtype or q.dtype
        self.dq, self.dk, self.dv = _like(self.q, out_dtype), _like(self.k, out_dtype), _like(self.v, out_dtype)
        wsb = _ext.bwd_workspace(B, H, N, D, q.device)
        self.ws = torch.empty(wsb, dtype=torch.uint8, device=q.device)
        self._keep = tuple(_ext.strides4(t) for t in (self.q, self.k, self.v, self.o, self.do, self.dq, self.dk, self.dv))
        stream = stream if stream is not None else torch.cuda.current_stream(q.device)
        self._args = (self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(), self.o.data_ptr(), self.do.data_ptr(),
                      lse.data_ptr(), self.dq.data_ptr(), self.dk.data_ptr(), self.dv.data_ptr(),
                      lists.row_ptr_ptr, lists.col_idx_ptr, lists_t.row_ptr_ptr,
                      lists_t.col_idx_ptr, lists.Bm, lists.Hm, B, H, N, D, _ext.dtype_code(q.dtype),
                      _ext.dtype_code(out_dtype), float(sm_scale)) + self._keep + (
                          self.ws.data_ptr(), wsb, ctypes.c_void_p(stream.cuda_stream))
        self._fn = _ext.lib().bsattn_bwd

    def run(self):
        rc = self._fn(*self._args)
        if rc != 0:
            _ext.check(rc, "bsattn_bwd")
        return self.dq, self.dk, self.dv


def _mask_of(q, k, v, mask):
    """(mask, N); mask=None is the dense mask."""
    N = _host.check_qkv(q, k, v)
    if mask is None:
        mask = _dense_mask(q.device, num_tiles(N))
    return mask, N


def _attend(q, k, v, mask, sm_scale, out_fp32, return_lse):
    mask, N = _mask_of(q, k, v, mask)
    seen = lists_cache.seen(mask, N)
    grad = torch.is_grad_enabled() and (q.requires_grad or k.requires_grad or v.requires_grad)
    if not grad and (seen is None or seen is UNMADE):
        # launches whose workgroups have a row block each take its columns from a block mask, new or not
        if seen is not None and (block := lists_cache.copy_of(mask, N)) is not None:
            made = _host.forward_mask(q, k, v, block, sm_scale, out_fp32, return_lse, False)
            if made is not None:
                return made[0]
        else:
            _check_mask(mask)
            if is_block_form(mask, N):
                kept = lists_cache.keeps(mask)
                made = _host.forward_mask(q, k, v, mask, sm_scale, out_fp32, return_lse, kept is not None)
                if made is not None:
                    if kept is not None:
                        lists_cache.put(mask, N, False, UNMADE, made[1], kept)
                    return made[0]
    lists = lists_cache.get(mask, N, False)
    if grad:
        if lists is None:
            lists = mask_to_lists(mask, N, both=True)                        # :48
        # The backward walks the column lists.  A block mask's are made here, where the GPU does not wait for them; those of
        # an elementwise mask, with a second set of its words, by the backward, which may never come.
        grid = None
        if lists.bits is None:
            lists_t = mask_to_lists(mask, N, transpose=True)
        else:
            lists_t = lists_cache.get(mask, N, True)
            if lists_t is None:
                grid = grid_cache.get(mask, N)
        return _host.attention(q, k, v, mask, lists, lists_t, grid, sm_scale, out_fp32, return_lse)
    if lists is None:
        if is_block_form(mask, N):
            # a block mask seen for the first time (or one that changes with every call): lists and forward in one call
            result, lists = _host.forward_block_mask(q, k, v, mask, sm_scale, out_fp32, return_lse)
            lists_cache.put(mask, N, False, lists)
            return result
        lists = mask_to_lists(mask, N)
    return _host.forward(q, k, v, lists, sm_scale, out_fp32, return_lse)


_host.set_python_lists(lambda mask, N: mask_to_lists(mask, N, transpose=True), lists_cache.put)


class _attention:
    """What the reference's autograd function offers (fa2_custom_mask.py:40-155): apply(q, k, v, mask, sm_scale); two extra
    trailing arguments select an fp32 output and the LSE as second result.  The function itself is Attention in
    csrc/host.cpp."""

    @staticmethod
    def apply(q, k, v, mask=None, sm_scale=1.3, out_fp32=False, return_lse=False):
        return _attend(q, k, v, mask, sm_scale, out_fp32, return_lse)


def flash_attention_custom_mask(q, k, v, mask=None, sm_scale=1.3):
    """Drop-in for the reference's `flash_attention_custom_mask = _attention.apply`
    (fa2_custom_mask.py:157): q,k,v [B,H,N,D] fp16/bf16 on the GPU, mask bool
    [B|1,H|1,nb,nb] with nb = ceil(N/64) (or elementwise [B|1,H|1,N,N]; None = dense attention),
    returns o like q.  D is 16, 32, 64, 128 or 256; N need not be a multiple of 64 (the last block of a
    block mask then covers the remaining tokens).  D = 16 and 32 cost one zero-padded copy of
    q, k, v per call.  The kept-tile lists of a mask tensor are cached
    until the tensor is modified.  When no gradient can be asked for (gradients disabled, or none of q, k, v
    requires one) nothing is kept for a backward."""
    return _attend(q, k, v, mask, sm_scale, False, False)


def flash_attention_custom_mask_lse(q, k, v, mask, sm_scale, out_fp32=False):
    """Same operator, also returning the natural-log logsumexp [B,H,N] fp32 of the kept scaled
    scores; out_fp32=True returns O in fp32.  (Not in the reference, whose second output M is
    only the running maximum: fa2_fwd.py:194-196.)"""
    return _attend(q, k, v, mask, sm_scale, out_fp32, True)


def attention_forward_backward(q, k, v, mask, sm_scale, do, out_fp32=False):
    """Non-autograd entry: (o, lse, dq, dk, dv) in one call; with out_fp32 all five results
    are fp32 (autograd itself can only hand back gradients in the dtype of q)."""
    mask, N = _mask_of(q, k, v, mask)
    lists = mask_to_lists(mask, N, both=True)
    return _host.forward_backward(q, k, v, lists, mask_to_lists(mask, N, transpose=True), sm_scale, do, out_fp32)
