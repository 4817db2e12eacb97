"""The in-place token reorder (bsattn_reorder_inplace behind permute_qkv_triton / inv_permute_attn_triton) against the
CPU oracle, bit for bit, at the sizes where the split of a head over workgroups can go wrong, in other layouts, and
where the workgroups of a head cannot run together."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import bsattn_oracle as orc

pytestmark = pytest.mark.gpu


def reference(x, numbers, F, H, W, text, inverse=False):
    """x [1, heads, text + F H W, D] (any 2-byte dtype), as numpy int16."""
    ref = x.clone().view(torch.int16).numpy()
    orders = orc.PERMUTATIONS[numbers]
    image = x[:, :, text:].contiguous().view(torch.int16).numpy()
    ref[:, :, text:] = (orc.inv_reorder(image, orders, orc.PERMUTATIONS_INV[numbers], F, H, W) if inverse
                        else orc.reorder(image, orders, F, H, W))
    return ref


# one workgroup per head; exactly one full part; one piece more; several parts with a remainder; rows of 3 pieces
@pytest.mark.parametrize("F,H,W,D,text", [(1, 1, 1, 64, 0), (7, 16, 16, 64, 5), (3, 597, 1, 64, 0), (8, 7, 64, 32, 1),
                                          (5, 29, 41, 128, 3), (4, 37, 40, 24, 2)])
def test_parts_of_a_head(dev, F, H, W, D, text):
    import fa2_custom_mask as fm
    numbers = [0, 1, 2, 3, 4, 5, -1, -6]
    g = torch.Generator().manual_seed(F * H * W)
    q, k, v = [torch.randn(1, len(numbers), text + F * H * W, D, generator=g).half() for _ in range(3)]
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    plan = {"permute": [torch.tensor(numbers, device=dev)]}
    fm.permute_qkv_triton(qd, kd, vd, plan, 0, F=F, H=H, W=W, n_text_tokens=text)
    for got, x in ((qd, q), (kd, k), (vd, v)):
        assert np.array_equal(got.cpu().view(torch.int16).numpy(), reference(x, numbers, F, H, W, text))
    got = fm.inv_permute_attn_triton(q.to(dev), plan, 0, F=F, H=H, W=W, n_text_tokens=text)
    assert np.array_equal(got.cpu().view(torch.int16).numpy(), reference(q, numbers, F, H, W, text, inverse=True))
    fm.inv_permute_attn_triton(vd, plan, 0, F=F, H=H, W=W, n_text_tokens=text)
    assert torch.equal(vd.cpu(), v)


@pytest.mark.parametrize("layout", ["packed", "token_major", "same_tensor_twice", "list_of_numbers", "int32"])
def test_layouts_and_number_forms(dev, layout):
    import fa2_custom_mask as fm
    F, H, W, D, text, NH = 6, 21, 17, 64, 4, 3
    T = text + F * H * W
    numbers = [2, 4, 5]
    g = torch.Generator().manual_seed(7)
    src = torch.randn(1, T, 3, NH, D, generator=g).half()
    q, k, v = [src[:, :, i].permute(0, 2, 1, 3).contiguous() for i in range(3)]
    idx = torch.tensor(numbers, device=dev)
    if layout == "packed":
        qd, kd, vd = src.to(dev).permute(2, 0, 3, 1, 4).unbind(0)
    elif layout == "token_major":
        qd, kd, vd = [x.permute(0, 2, 1, 3).contiguous().to(dev).permute(0, 2, 1, 3) for x in (q, k, v)]
    else:
        qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    if layout == "same_tensor_twice":
        kd, k = qd, q
    if layout == "list_of_numbers":
        idx = numbers
    if layout == "int32":
        idx = idx.int()
    fm.permute_qkv_triton(qd, kd, vd, {"permute": [idx]}, 0, F=F, H=H, W=W, n_text_tokens=text)
    for got, x in ((qd, q), (kd, k), (vd, v)):
        assert np.array_equal(got.cpu().contiguous().view(torch.int16).numpy(), reference(x, numbers, F, H, W, text))


def test_group_that_cannot_run_together(dev):
    """Confined to 8 compute units (one per XCD) the workgroups of a head are never all resident: the waits run out and
    one workgroup moves each head."""
    import fa2_custom_mask as fm
    hip = ctypes.CDLL("libamdhip64.so")
    mask = (ctypes.c_uint32 * 8)(0xff, 0, 0, 0, 0, 0, 0, 0)
    handle = ctypes.c_void_p()
    if hip.hipExtStreamCreateWithCUMask(ctypes.byref(handle), 8, mask) != 0:
        pytest.skip("no CU-masked stream")
    F, H, W, D, text = 9, 30, 45, 64, 2
    numbers = [1, 2, 3, 4, 5, 0, 2, 4, 5]
    g = torch.Generator().manual_seed(11)
    x = torch.randn(1, len(numbers), text + F * H * W, D, generator=g).half()
    xd = x.to(dev)
    plan = {"permute": [torch.tensor(numbers, device=dev)]}
    torch.cuda.synchronize()
    try:
        with torch.cuda.stream(torch.cuda.ExternalStream(handle.value, device=dev)):
            for _ in range(2):
                fm.inv_permute_attn_triton(xd, plan, 0, F=F, H=H, W=W, n_text_tokens=text)
                back = xd.clone()
                fm.permute_qkv_triton(xd, xd.clone(), xd.clone(), plan, 0, F=F, H=H, W=W, n_text_tokens=text)
            assert hip.hipStreamSynchronize(handle) == 0
        torch.cuda.synchronize()
    finally:
        hip.hipStreamDestroy(handle)
    assert torch.equal(xd.cpu(), x)
    assert np.array_equal(back.cpu().view(torch.int16).numpy(), reference(x, numbers, F, H, W, text, inverse=True))


@pytest.mark.parametrize("number_type", [torch.int64, torch.int32])
@pytest.mark.parametrize("bad", [6, 100, -7])
def test_number_outside_the_table(dev, bad, number_type):
    """Numbers the host can read are refused before anything is moved; numbers in GPU memory are checked by the kernel:
    the head stays as it is and the next reorder raises, once."""
    import fa2_custom_mask as fm
    F, H, W, D, text = 5, 12, 17, 64, 3
    numbers = [3, bad, 1]
    size = dict(F=F, H=H, W=W, n_text_tokens=text)
    g = torch.Generator().manual_seed(13)
    x = torch.randn(1, 3, text + F * H * W, D, generator=g).half()
    for host_numbers in (numbers, torch.tensor(numbers, dtype=number_type), np.array(numbers)):
        xd = x.to(dev)
        with pytest.raises(IndexError):
            fm.inv_permute_attn_triton(xd, {"permute": [host_numbers]}, 0, **size)
        assert torch.equal(xd.cpu(), x)
    plan = {"permute": [torch.tensor(numbers, dtype=number_type, device=dev)]}
    good = {"permute": [torch.tensor([3, 0, 1], dtype=number_type, device=dev)]}
    moved = x.to(dev)
    fm.permute_qkv_triton(moved, moved.clone(), moved.clone(), plan, 0, **size)
    torch.cuda.synchronize()
    assert np.array_equal(moved.cpu().view(torch.int16).numpy(), reference(x, [3, 0, 1], F, H, W, text))
    xd = x.to(dev)
    with pytest.raises(RuntimeError, match="permutation number"):
        fm.permute_qkv_triton(xd, xd.clone(), xd.clone(), good, 0, **size)
    assert torch.equal(xd.cpu(), x)                          # nothing was enqueued
    fm.permute_qkv_triton(xd, xd.clone(), xd.clone(), good, 0, **size)
    assert torch.equal(xd.cpu(), moved.cpu())


FORMS = ["plain", "text of an odd width", "packed", "overlapping", "expanded heads", "requires grad", "other dtype", "numbers on the host", "strided numbers"]


@pytest.mark.parametrize("form", FORMS)
def test_native_call_takes_what_python_takes(dev, form):
    """The native path and the general one agree on which layouts are moved in place, and on the result."""
    import fa2_custom_mask as fm
    from fa2_custom_mask import functional
    from fa2_custom_mask.utils import _host
    F, H, W, NH = 3, 5, 7, 4
    D, text = (12, 1) if form == "text of an odd width" else (64, 2)
    T = text + F * H * W
    g = torch.Generator().manual_seed(17)
    make = lambda *shape: torch.randn(*shape, generator=g).half().to(dev)
    tensors = [make(1, NH, T, D) for _ in range(3)]
    numbers = torch.tensor([3, 1, 5, 2], device=dev)
    if form == "packed":
        tensors = list(make(1, T, 3, NH, D).permute(2, 0, 3, 1, 4).unbind(0))
    elif form == "overlapping":
        base = make(1, NH, T + 1, D)
        tensors = [base[:, :, :T], base[:, :, 1:], tensors[2]]
    elif form == "expanded heads":
        tensors[1] = make(1, 1, T, D).expand(1, NH, T, D)
    elif form == "requires grad":
        tensors[2].requires_grad_(True)
    elif form == "other dtype":
        tensors[1] = tensors[1].float()
    elif form == "numbers on the host":
        numbers = numbers.cpu()
    elif form == "strided numbers":
        numbers = torch.stack([numbers, numbers], 1)[:, 0]
    with torch.no_grad():
        want = [t.clone() for t in tensors]
    image = [t[:, :, text:] for t in tensors]
    size = dict(F=F, H=H, W=W, n_text_tokens=text)
    takes = functional._inplace_workspace(tensors, image, F, H, W) is not None and numbers.is_cuda and numbers.is_contiguous()
    assert takes == (form in ("plain", "packed"))
    versions = [t._version for t in tensors]
    rc = _host.reorder_inplace(tensors, numbers, False, F, H, W, text)
    assert (rc is not None) == takes and (rc in (None, 0))
    assert [t._version > v for t, v in zip(tensors, versions)] == [takes] * 3      # (views of one tensor count together)
    if takes:
        fm.permute_qkv_triton(*want, {"permute": [numbers.tolist()]}, 0, **size)      # (numbers the host holds: the general path)
        assert all(torch.equal(a, b) for a, b in zip(tensors, want))
    else:
        assert all(torch.equal(a, b) for a, b in zip(tensors, want))                     # nothing was moved
