"""Prompt chunks with at least a row group of 128 rows for every workgroup (whole_size): row groups dealt whole, whose workgroups
write the result themselves, and the remaining ones in runs -- one and several whole row groups a workgroup, no remainder, a last
row group of few rows, empty fragments, rows that see nothing -- against float64, with the rotated queries and the log-sum-exp."""
import pytest
import torch

from inference_lib_amd import _lib
from inference_lib_amd import attention as ops
from test_gpu_stream_runs import _inputs, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,S,Hq,Hkv,D,lens,dtype,hide", [
    (1, 1024, 32, 8, 128, (70, 1024), torch.bfloat16, False),        # 32 row groups of 8 heads: nothing left over
    (1, 1025, 32, 8, 128, (0, 33, 1025), torch.float16, False),      # a 33rd of one token's four rows, an empty fragment
    (1, 900, 64, 4, 64, (1, 0, 900, 0), torch.bfloat16, False),      # 113 of 4 heads: one whole, 49 in runs; an empty fragment last
    (2, 700, 32, 2, 64, (50, 700, 700), torch.float16, True),        # 175 of 2 heads (128 workgroups each)
    (1, 700, 20, 20, 64, (300, 700), torch.bfloat16, True),          # 6 of 20 heads (12 workgroups): all in runs, as before
    (1, 800, 80, 20, 64, (40, 800), torch.float16, False),           # 25 of 20 heads: two whole for each, one left over
])
def test_whole_row_groups_and_runs(W, S, Hq, Hkv, D, lens, dtype, hide):
    scale = D ** -0.5
    q, loc, cos, sin, keys, values = _inputs(W, S, Hq, Hkv, D, lens, dtype, D)
    if hide:                                       # some tokens see nothing of any fragment
        loc[:, :, 5::97] = -1
    F = len(lens)
    guard = 12345.0
    rq = torch.full((F, W, Hq, S, D), guard, dtype=dtype, device="cuda")
    out = torch.full_like(q, guard)
    lse = torch.full((W, Hq, S), guard, dtype=torch.float32, device="cuda")
    frag = torch.tensor(lens, dtype=torch.int32, device="cuda")
    ops.hogwild_fused(q, loc, keys, values, scale, frag, cos, sin, rotated_queries=rq, out=out, lse=lse)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    want_rq = ops.hogwild_rope(q, cos, sin)
    assert float((rq.float() - want_rq.float()).abs().max()) <= 4 * eps * float(want_rq.float().abs().max())
    ref, ref_lse, bound = _reference(rq, loc, keys, values, scale, Hkv)
    seen = ~torch.isneginf(ref_lse)
    assert bool(((out.double() - ref).abs() <= bound)[seen].all())
    assert float((lse.double() - ref_lse)[seen].abs().max()) <= 1e-4
    assert bool((out[~seen] == 0).all()) and bool(torch.isneginf(lse[~seen]).all())
    again = ops.hogwild_sdpa(rq, loc, keys, values, scale, frag)           # pre-rotated, no lse
    assert bool(((again.double() - ref).abs() <= bound)[seen].all())
    # the workspace as it is asked for holds everything
    pr = _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=again, cosines=cos, sines=sin)
    need = pr.workspace_bytes()
    space = torch.full((need + 4096,), 165, dtype=torch.uint8, device="cuda")
    pr.set_workspace(space[:need])
    pr.run()
    assert bool((space[need:] == 165).all()) and bool(((again.double() - ref).abs() <= bound)[seen].all())
