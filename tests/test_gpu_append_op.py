"""The append operator behind HogwildCache against the ctypes entry it stands in for (attention.py:148-158, :313-315): the
forms it takes give the same bits, the others are declined with nothing written."""
import pytest
import torch

from inference_lib_amd import _lib
from inference_lib_amd import attention  # noqa: F401  (loads the operators)

pytestmark = pytest.mark.gpu


def _states(W, Hkv, S, D, dtype, form, g):
    k = torch.randn((W, S, Hkv, D), generator=g).to(dtype).cuda().transpose(1, 2)
    v = torch.randn((W, S, Hkv, D), generator=g).to(dtype).cuda().transpose(1, 2)
    if form == "packed":
        k, v = k.contiguous(), v.contiguous()
    if form == "strided_elements":
        k = k.transpose(2, 3).contiguous().transpose(2, 3)
    return k, v


@pytest.mark.parametrize("form", ["transposed", "packed", "strided_elements"])
@pytest.mark.parametrize("W,S,D,tables", [(2, 1, 128, "16"), (3, 5, 64, "32"), (65, 2, 64, "row"), (1, 1, 256, "none"), (2, 3, 128, "partial")])
def test_append_operator_equals_the_c_entry(form, W, S, D, tables):
    g = torch.Generator().manual_seed(W * 100 + S)
    Hkv, cap, dtype = 3, 11, torch.bfloat16
    k, v = _states(W, Hkv, S, D, dtype, form, g)
    cos = sin = None
    if tables != "none":
        rot = D // 2 if tables == "partial" else D
        shape = (W, 1 if tables == "row" else S, rot)
        cos, sin = (torch.rand(shape, generator=g).to(torch.float32 if tables == "32" else dtype).cuda() for _ in range(2))
    n_new = [max(0, S - w % 3) for w in range(W)]
    dst = [w % (cap - S + 1) for w in range(W)]

    def buffers():
        return [[torch.zeros((Hkv, cap, D), dtype=dtype, device="cuda") for _ in range(W)] for _ in range(2)]
    ka, va = buffers()
    kb, vb = buffers()
    took = torch.ops.libhogatt.rope_append(ka, va, dst, n_new, k, v, cos, sin, _lib.HW_ROPE_EAGER)
    assert took == (k.stride(3) == 1)          # (with one token the transposition leaves the elements adjacent)
    if not took:
        assert all(int(t.count_nonzero()) == 0 for t in ka + va)
        return
    _lib.rope_append(k, v, kb, vb, dst, cosines=cos, sines=sin, n_new=n_new, mode=_lib.HW_ROPE_EAGER)
    assert all(torch.equal(a, b) for a, b in zip(ka + va, kb + vb))


def test_append_operator_declines_what_does_not_fit():
    k = torch.randn((1, 2, 4, 64), device="cuda", dtype=torch.float16)
    buf = torch.zeros((2, 5, 64), device="cuda", dtype=torch.float16)
    for dst, n, kk in (([2], [4], k), ([-1], [4], k), ([0], [5], k), ([0], [4], k.float())):
        assert not torch.ops.libhogatt.rope_append([buf], [buf.clone()], dst, n, kk, k, None, None, _lib.HW_ROPE_EAGER)
    assert int(buf.count_nonzero()) == 0
    with pytest.raises(_lib.HogwildError):
        _lib.rope_append(k, k, [buf], [buf.clone()], [2], n_new=[4])


@pytest.mark.parametrize("what", ["wide_tables", "odd_tables", "mode"])
def test_refusals_of_the_library_reach_the_caller_as_hogwild_error(what):
    """What hw_rope_append refuses is declined by the operator too, so that the general path names it, status included."""
    from inference_lib_amd import cache
    rot = {"wide_tables": 66, "odd_tables": 33, "mode": 64}[what]
    mode = 7 if what == "mode" else _lib.HW_ROPE_EAGER
    k = torch.randn((1, 2, 1, 64), device="cuda", dtype=torch.float16)
    cos = torch.ones((1, 1, rot), device="cuda", dtype=torch.float16)
    seg = cache.SegmentCache(1, 2, 64, 8, dtype=torch.float16)
    c = cache.HogwildCache([[seg]], inv_freq=torch.ones(32, device="cuda"))
    with pytest.raises(_lib.HogwildError) as e:
        c.update_fused(k, k, cos, cos, 0, mode=mode)
    assert e.value.status == -3 and seg.lengths == [0]
    assert not torch.ops.libhogatt.rope_append(seg.k, seg.v, [0], [1], k, k, cos, cos, mode)


@pytest.mark.parametrize("n", [0, 1, 7])
def test_segment_views_are_slices(n):
    buf = torch.randn((3, 7, 64), device="cuda")
    got, = torch.ops.libhogatt.segment_views([buf], [n])
    want = buf[:, :n, :].unsqueeze(0)
    assert got.shape == want.shape and got.stride() == want.stride() and got.data_ptr() == want.data_ptr() and torch.equal(got, want)
