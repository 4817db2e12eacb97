"""Head-wise token reorder wrappers, mirroring fa2_custom_mask/functional.py:5-84 of the
reference (same names, arguments, defaults and in-place write-back); the rows are moved by the HIP kernel behind
bsattn_reorder and bsattn_reorder_inplace."""
import ctypes

import numpy as np
import torch

from . import _ext
from .utils import _host

_PERMUTATIONS = [[0, 1, 2], [0, 2, 1], [1, 2, 0], [1, 0, 2], [2, 1, 0], [2, 0, 1]]       # functional.py:23-26
_PERMUTATIONS_INV = [[0, 1, 2], [0, 2, 1], [2, 0, 1], [1, 0, 2], [2, 1, 0], [1, 2, 0]]   # functional.py:69-76


def _launch(tensor, permute_orders, inv_permute_orders, F, H, W):
    if not tensor.is_cuda:
        raise RuntimeError("reorder needs a GPU tensor (there is no CPU path)")
    BS, N_head, N_token, D = tensor.shape
    assert N_token == F * H * W                                               # functional.py:7,48
    tensor = tensor.contiguous()
    orders = permute_orders.to(device=tensor.device, dtype=torch.int32).contiguous()
    inv = None
    if inv_permute_orders is not None:
        inv = inv_permute_orders.to(device=tensor.device, dtype=torch.int32).contiguous()
    output = torch.empty_like(tensor)                                         # functional.py:8,49
    rc = _ext.lib().bsattn_reorder(tensor.data_ptr(), output.data_ptr(), BS, N_head, F, H, W, D,
                                   tensor.element_size(), orders.data_ptr(),
                                   inv.data_ptr() if inv is not None else None,
                                   _ext.current_stream(tensor.device))
    _ext.check(rc, "bsattn_reorder")
    return output


def apply_head_wise_reorder(tensor, permute_orders, F, H, W):
    """functional.py:5-20: out[b,h,new_t,:] = tensor[b,h,t,:], new_t per head from permute_orders."""
    return _launch(tensor, permute_orders, None, F, H, W)


def apply_inv_reorder(tensor, permute_orders, inv_permute_orders, F, H, W):
    """functional.py:46-62: undo apply_head_wise_reorder."""
    return _launch(tensor, permute_orders, inv_permute_orders, F, H, W)


_tables = {}


def _table(device):
    """[permutations, permutations back, their numbers] as int32 tensors on `device`, copied there once."""
    if device not in _tables:
        with torch.inference_mode(False):
            _tables[device] = [torch.tensor(t, dtype=torch.int32, device=device)
                               for t in (_PERMUTATIONS, _PERMUTATIONS_INV, list(range(6)))]
    return _tables[device]


def _check_numbers(idx):
    """Permutation numbers that the host can read are checked before anything is moved.  Those in GPU memory are checked by
    the kernel, and the next reorder on the device raises (reading them here would wait for the GPU in every call)."""
    if isinstance(idx, torch.Tensor) and idx.is_cuda or not isinstance(idx, (torch.Tensor, np.ndarray, list, tuple)):
        return
    numbers = torch.as_tensor(idx)
    if numbers.dtype in (torch.int64, torch.int32, torch.int16, torch.int8) and numbers.numel() and (
            int(numbers.min()) < -len(_PERMUTATIONS) or int(numbers.max()) >= len(_PERMUTATIONS)):
        raise IndexError("permutation numbers %s: the table has %d rows" % (numbers.tolist(), len(_PERMUTATIONS)))


def _reorder_image_tokens(tensors, idx, inverse, F, H, W, n_text_tokens):
    """Reorders (inverse: brings back) the image tokens of every tensor where they are, head by head, by the
    permutation numbers idx [heads]."""
    if isinstance(idx, torch.Tensor) and idx.is_cuda and all(type(t) is torch.Tensor for t in tensors):
        rc = _host.reorder_inplace(tensors, idx, inverse, F, H, W, n_text_tokens)
        if rc is not None:
            _ext.check(rc, "bsattn_reorder_inplace")
            return
    _check_numbers(idx)
    x = tensors[0]
    image = [t[:, :, n_text_tokens:, :] for t in tensors]                     # functional.py:31-33, 81
    BS, NH, T, D = image[0].shape
    assert T == F * H * W                                                     # functional.py:7,48
    wsb = _inplace_workspace(tensors, image, F, H, W)
    if wsb is not None:
        numbers = idx
        if not (isinstance(idx, torch.Tensor) and idx.device == x.device and idx.dtype in (torch.int64, torch.int32)
                and idx.is_contiguous()):
            numbers = _table(x.device)[2][idx]
        if numbers.shape == (NH,):
            n = len(image)
            ws = _host.reorder_workspace(wsb, x)
            strides = (ctypes.c_int64 * (3 * n))(*[s for v in image for s in v.stride()[:3]])
            ptrs = (ctypes.c_void_p * n)(*[v.data_ptr() for v in image])
            rc = _ext.lib().bsattn_reorder_inplace(
                ptrs, strides, n, BS, NH, F, H, W, D, x.element_size(), numbers.data_ptr(), numbers.element_size(),
                1 if inverse else 0, ws.data_ptr(), wsb, _ext.current_stream(x.device))
            _ext.check(rc, "bsattn_reorder_inplace")
            for t in tensors:
                if not t.is_inference():
                    torch.autograd.graph.increment_version(t)
            return
    # layouts the kernel does not take, and tensors autograd watches: out of place, then copied back
    permutations, permutations_inv, _ = _table(x.device)
    orders = permutations[idx]                                                # :29, 79
    inv_orders = permutations_inv[idx] if inverse else None                   # :80
    outs = [_launch(v.contiguous(), orders, inv_orders, F, H, W) for v in image]
    for t, out in zip(tensors, outs):                                         # :39-41, 83
        t[:, :, n_text_tokens:, :] = out


def _inplace_workspace(tensors, image, F, H, W):
    """Bytes of workspace of bsattn_reorder_inplace on the views `image` of `tensors`, None if it does not take them."""
    x = tensors[0]
    BS, NH, _, D = image[0].shape
    size = x.element_size()
    for t, v in zip(tensors, image):
        if not t.is_cuda or t.device != x.device or t.shape != x.shape or t.dtype != x.dtype:
            return None
        if t.requires_grad and torch.is_grad_enabled():
            return None
        if v.stride(3) != 1 or v.data_ptr() % 16 or any(s * size % 16 for s in v.stride()[:3]):
            return None
    if not _disjoint(image):
        return None
    return _ext.reorder_inplace_workspace(len(image), BS, NH, F, H, W, D, size)


def _nested(dims, need):
    """Dimensions (stride, size) around stretches of `need` elements of which no two share an element."""
    for stride, size in sorted(dims):
        if size > 1:
            if stride < need:
                return False
            need += stride * (size - 1)
    return True


def _disjoint(views):
    """No row of the views shares memory with another: each view's rows, and those of views cut from one storage (the
    q, k, v of a packed projection)."""
    D = views[0].shape[3]
    dims = [list(zip(v.stride()[:3], v.shape[:3])) for v in views]
    if not all(_nested(d, D) for d in dims):
        return False
    for i, a in enumerate(views):
        for b in views[:i]:
            if a.untyped_storage().data_ptr() == b.untyped_storage().data_ptr():
                apart = abs(a.storage_offset() - b.storage_offset())
                if a.stride() != b.stride() or apart == 0 or not _nested(dims[i] + [(apart, 2)], D):
                    return False
    return True


def permute_qkv_triton(query, key, value, permute_plan, i_block, F=13, H=30, W=45, n_text_tokens=226):
    """functional.py:22-43 (the name is kept for drop-in use; nothing here uses Triton)."""
    idx = permute_plan['permute'][i_block]                                    # :28
    _reorder_image_tokens((query, key, value), idx, False, F, H, W, n_text_tokens)
    return query, key, value


def inv_permute_attn_triton(attn_out, permute_plan, i_block, F=13, H=30, W=45, n_text_tokens=226):
    """functional.py:64-84."""
    idx = permute_plan['permute'][i_block]                                    # :78
    _reorder_image_tokens((attn_out,), idx, True, F, H, W, n_text_tokens)
    return attn_out
