"""K/V tiles that a CU's row groups of 128 rows read one after the other are kept in the L2 (keep_in_l2), others streamed past it:
calls on both sides of the line, in runs across row groups and in rounds, fused and pre-rotated, against float64."""
import pytest
import torch

from inference_lib_amd import attention as ops
from test_gpu_stream_runs import _inputs, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,S,Hq,Hkv,D,lens,dtype", [
    (1, 480, 16, 4, 128, (200, 480), torch.bfloat16),      # 15 row groups of 4 heads: streamed
    (1, 1100, 16, 4, 128, (40, 1100), torch.bfloat16),     # 35: kept
    (2, 230, 32, 8, 128, (300, 230, 230), torch.float16),  # 15 row groups of 8 heads: streamed
    (2, 250, 32, 8, 128, (300, 250, 250), torch.float16),  # 16: kept
    (1, 980, 16, 8, 64, (77, 980), torch.bfloat16),        # 16 row groups, rows without staged tables: kept
])
def test_both_sides_of_the_line(W, S, Hq, Hkv, D, lens, dtype):
    scale = D ** -0.5
    q, loc, cos, sin, keys, values = _inputs(W, S, Hq, Hkv, D, lens, dtype, D)
    frag = torch.tensor(lens, dtype=torch.int32, device="cuda")
    rq = torch.empty((len(lens),) + tuple(q.shape), dtype=dtype, device="cuda")
    out = torch.empty_like(q)
    ops.hogwild_fused(q, loc, keys, values, scale, frag, cos, sin, rotated_queries=rq, out=out)
    ref, _, bound = _reference(rq, loc, keys, values, scale, Hkv)
    assert bool(((out.double() - ref).abs() <= bound).all())
    again = ops.hogwild_sdpa(rq, loc, keys, values, scale, frag)
    assert bool(((again.double() - ref).abs() <= bound).all())
