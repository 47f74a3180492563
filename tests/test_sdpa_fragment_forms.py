"""The fragments of hogwild_sdpa may come in any iterable (the reference's wrapper builds lists from them,
python/hogwild/attention.py:32-33): the operator gets lists, packed fragments as they are."""
import pytest
import torch

from inference_lib_amd.attention import _in_place_or_contiguous, hogwild_sdpa


@pytest.mark.parametrize("form", [list, tuple, iter, torch.stack, lambda ts: dict(enumerate(ts)).values()])
def test_fragments_in_any_iterable(form):
    frags = [torch.randn((2, 5, 64)) for _ in range(3)]
    ks, vs = _in_place_or_contiguous(form(frags), form([2 * t for t in frags]))
    assert type(ks) is list and type(vs) is list
    assert all(torch.equal(k, t) and torch.equal(v, 2 * t) for k, v, t in zip(ks, vs, frags)) and len(ks) == len(vs) == 3


@pytest.mark.gpu
def test_stacked_fragments_give_the_result_of_a_list():
    k, v = (torch.randn((2, 1, 40, 64), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    q = torch.randn((2, 1, 2, 1, 64), device="cuda", dtype=torch.bfloat16)
    loc = torch.full((2, 1, 1), 39, device="cuda", dtype=torch.int32)
    want = hogwild_sdpa(q, loc, list(k), list(v), 0.125)
    assert torch.equal(hogwild_sdpa(q, loc, k, v, 0.125), want)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [list, tuple])
def test_fragments_beyond_the_shorter_list_are_not_read(form):
    k, v = (list(torch.randn((3, 1, 40, 64), device="cuda", dtype=torch.bfloat16)) for _ in range(2))
    q = torch.randn((2, 1, 2, 1, 64), device="cuda", dtype=torch.bfloat16)
    loc = torch.full((2, 1, 1), 39, device="cuda", dtype=torch.int32)
    frag = torch.full((2,), 40, device="cuda", dtype=torch.int32)
    want = hogwild_sdpa(q, loc, k[:2], v[:2], 0.125, frag)
    assert torch.equal(hogwild_sdpa(q, loc, form(k[:2]), form(v), 0.125, frag), want)
    assert torch.equal(hogwild_sdpa(q, loc, form(k), form(v[:2]), 0.125, frag), want)
    with pytest.raises(RuntimeError, match="per row of locations"):
        hogwild_sdpa(q, loc, form(k), form(v), 0.125, frag)
