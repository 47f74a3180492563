"""step_inputs, the one native call behind layer 0 of a HogwildCache step, against build_inputs and the lengths themselves; what it
refuses comes back as False, a stream that is being captured as an error.  hogwild_sdpa on fragments that have to be copied."""
import pytest
import torch

from inference_lib_amd import _lib
from inference_lib_amd import attention as ops
from inference_lib_amd import cache as hc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,W,S,half,dtype", [(1, 1, 1, 32, torch.float32), (9, 4, 1, 64, torch.bfloat16), (5, 3, 7, 16, torch.float16),
                                              (500, 8, 2, 4, torch.bfloat16), (3, 2, 1, 0, torch.float32)])
def test_same_as_build_inputs(F, W, S, half, dtype):
    g = torch.Generator().manual_seed(F)
    pos = torch.randint(S, 70000, (F, W), generator=g).tolist()
    lens = torch.randint(0, 70000, (F,), generator=g).tolist()
    lens[0] = 0
    inv = torch.rand(half, generator=g).cuda()
    done, loc, cos, sin, frags = torch.ops.libhogatt.step_inputs([x for row in pos for x in row], lens, S, inv, 1.25, dtype)
    want = _lib.build_inputs(pos, S, inv, attention_scaling=1.25, table_dtype=None if dtype == torch.float32 else dtype)
    assert done and frags.dtype == torch.int32 and frags.tolist() == lens
    for got, ref in zip((loc, cos, sin), want):
        assert got.dtype == ref.dtype and torch.equal(got, ref)


def test_refused():
    inv = torch.ones(4, device="cuda")
    op = torch.ops.libhogatt.step_inputs
    assert op([1, 2, 3], [1, 2], 1, inv, 1.0, torch.float32)[0] is False               # not a full table
    assert op([1, 2], [1, -2], 1, inv, 1.0, torch.float32)[0] is False
    assert op([1, 2], [1, 2], 1, inv.double(), 1.0, torch.float32)[0] is False
    assert op([1, 2], [1, 2], 1, inv, 1.0, torch.float64)[0] is False
    assert op([7] * (1 << 13), [1], 1, inv, 1.0, torch.float32)[0] is False            # more workers than a launch's table holds


def test_sdpa_copies_what_it_cannot_read_in_place():
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn((2, 2, 8, 1, 64), generator=g, device="cuda").half()
    loc = torch.full((2, 2, 1), 60, dtype=torch.int32, device="cuda")
    frag = torch.tensor([40, 33], dtype=torch.int32, device="cuda")
    keys = [torch.randn((2, n, 64), generator=g, device="cuda").half() for n in (40, 33)]
    want = ops.hogwild_sdpa(q, loc, keys, keys, 0.125, frag)
    across = [k.transpose(0, 1).contiguous().transpose(0, 1) for k in keys]            # heads inside tokens
    assert not across[0].is_contiguous()
    assert torch.equal(ops.hogwild_sdpa(q, loc, across, across, 0.125, frag), want)
    assert torch.equal(ops.hogwild_sdpa(q, loc, tuple(across), tuple(across), 0.125), want)


@pytest.mark.parametrize("fused", [True, False])
def test_lengths_from_the_host_refuse_a_capture(fused):
    """Every replay of such a graph would append to the same rows.  With lengths on the device the same step is captured, and its
    replays append one behind the other."""
    Hkv, D = 2, 64
    segs = [hc.SegmentCache(1, Hkv, D, 64, dtype=torch.float16, device="cuda") for _ in range(2)]
    for seg in segs:
        seg.lengths = [5]
        for buf in (seg.k[0], seg.v[0]):
            buf.zero_()
    cache = hc.HogwildCache([segs, segs[::-1]], inv_freq=torch.ones(D // 2, device="cuda"))
    k, v = (torch.ones((2, Hkv, 1, D), dtype=torch.float16, device="cuda") for _ in range(2))
    cos, sin = torch.ones((2, 1, D), dtype=torch.float16, device="cuda"), torch.zeros((2, 1, D), dtype=torch.float16, device="cuda")
    step = (lambda: cache.update_fused(k, v, cos, sin, 0)) if fused else (lambda: cache.update(k, v, 0))
    step()                                                       # outside a capture: a token each
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError, match="use_device_lengths"):
        with torch.cuda.graph(graph):
            step()
    for seg in segs:
        seg.lengths = [6]
    cache.use_device_lengths(headroom=8)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(3):
        graph.replay()
    cache.sync_lengths()
    for seg in segs:
        assert seg.lengths == [10]
        assert bool((seg.v[0][:, 5:10] == 1).all()) and bool((seg.v[0][:, :5] == 0).all()) and bool((seg.v[0][:, 10:] == 0).all())
