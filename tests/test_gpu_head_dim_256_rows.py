"""Head dimension 256 with many query rows per kv head: 128-row workgroups (the D = 256 form of the many-rows kernel), from the row
count where they begin up to several row groups for every workgroup -- row remainders, empty fragments, rows that see nothing, few
tiles, partial rotary width -- against float64."""
import ctypes as C

import pytest
import torch

from inference_lib_amd import _lib
from inference_lib_amd import attention as ops
from test_gpu_paged import build_paged
from test_gpu_paged import check as check_paged
from test_gpu_stream_runs import _inputs, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,S,Hq,Hkv,lens,dtype,rot,hide", [
    (3, 11, 2, 2, (70000, 33, 11, 7000), torch.bfloat16, 256, False),  # 33 rows of one row group
    (2, 32, 4, 2, (30000, 0, 64, 32), torch.float16, 256, False),      # 128 rows exactly, an empty fragment
    (1, 129, 8, 8, (6400, 129), torch.bfloat16, 256, False),           # a second row group of one row
    (1, 300, 16, 8, (1500, 300), torch.bfloat16, 256, True),           # five row groups in runs
    (1, 300, 16, 8, (1400, 300), torch.float16, 128, False),           # rotary width 128: rotated in front
    (1, 680, 96, 24, (90, 680, 0), torch.bfloat16, 256, False),        # 22 row groups of 24 heads: two whole for each, two in runs
    (1, 1000, 32, 16, (0, 1000), torch.float16, 256, True),            # 16 of 16 heads: nothing left over
    (1, 1500, 8, 1, (5, 1500), torch.bfloat16, 256, False),            # 94 of one head, fewer than workgroups
])
def test_many_rows_of_256(W, S, Hq, Hkv, lens, dtype, rot, hide):
    scale, D, F = 256 ** -0.5, 256, len(lens)
    q, loc, cos, sin, keys, values = _inputs(W, S, Hq, Hkv, D, lens, dtype, rot)
    if hide:
        loc[:, :, 5::97] = -1
    frag = torch.tensor(lens, dtype=torch.int32, device="cuda")
    guard = 12345.0
    rq = torch.full((F, W, Hq, S, D), guard, dtype=dtype, device="cuda")
    out = torch.full_like(q, guard)
    lse = torch.full((W, Hq, S), guard, dtype=torch.float32, device="cuda")
    ops.hogwild_fused(q, loc, keys, values, scale, frag, cos, sin, rotated_queries=rq, out=out, lse=lse)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    want_rq = ops.hogwild_rope(q, cos, sin)
    assert float((rq.float() - want_rq.float()).abs().max()) <= 4 * eps * float(want_rq.float().abs().max())
    ref, ref_lse, bound = _reference(rq, loc, keys, values, scale, Hkv)
    seen = ~torch.isneginf(ref_lse)
    assert bool(((out.double() - ref).abs() <= bound)[seen].all())
    assert float((lse.double() - ref_lse)[seen].abs().max()) <= 1e-4
    assert bool((out[~seen] == 0).all()) and bool(torch.isneginf(lse[~seen]).all())
    again = ops.hogwild_sdpa(rq, loc, keys, values, scale, frag)           # pre-rotated
    assert bool(((again.double() - ref).abs() <= bound)[seen].all())
    # segments inside larger buffers, and the workspace as it is asked for
    ks, vs = ([torch.cat([t, torch.full((Hkv, 3, D), float("nan"), dtype=dtype, device="cuda")], dim=1)[:, :t.size(1)] for t in x] for x in (keys, values))
    pr = _lib.Problem(q=q, locations=loc, keys=ks, values=vs, scale=scale, out=again, cosines=cos, sines=sin)
    need = pr.workspace_bytes()
    space = torch.full((need + 4096,), 165, dtype=torch.uint8, device="cuda")
    pr.set_workspace(space[:need])
    again.fill_(guard)
    pr.run()
    assert bool((space[need:] == 165).all()) and bool(((again.double() - ref).abs() <= bound)[seen].all())
    # a workspace sized for the 16-row kernel of hw_plan, and that kernel itself, give the same within the bound
    plan = _lib.HwPlan()
    _lib.check(_lib.lib.hw_plan_debug(C.byref(pr.p), _lib.lib.hw_device_cus(), C.byref(plan)), "hw_plan_debug")
    assert plan.row_blocks == 1
    pr.set_workspace(torch.empty(plan.workspace_bytes, dtype=torch.uint8, device="cuda"))
    again.fill_(guard)
    pr.run()
    assert bool(((again.double() - ref).abs() <= bound)[seen].all())
    narrow = torch.empty_like(q)
    _lib.Problem(q=q, locations=loc, keys=ks, values=vs, scale=scale, out=narrow, cosines=cos, sines=sin, row_blocks=1).run()
    assert bool(((narrow.double() - ref).abs() <= bound)[seen].all())
    assert not torch.equal(narrow, out), "not a call for 128-row workgroups"


@pytest.mark.parametrize("Hq,S,block", [(10, 4, 16), (14, 3, 16), (8, 8, 16), (22, 3, 16), (8, 40, 7), (2, 129, 64)])
def test_paged_rows_around_the_line_of_kept_tiles(Hq, S, block):
    """20, 21, 32 and 33 rows a sequence (the K/V tiles are kept in the L2 from 33 on), and many row groups of 16."""
    check_paged(build_paged("bf16", 1, 3, Hq, 2, 256, block, -(-900 // block), seq_lens=[900, S, 333], S=S, seed=S))


@pytest.mark.parametrize("q_lens", [(10, 1, 49), (10, 2, 49), (1, 64, 30)])
def test_packed_rows_around_the_line_of_kept_tiles(q_lens):
    """60 and 61 query rows of three packed sequences (kept from 61 on), and more."""
    check_paged(build_paged("bf16", 1, 3, 2, 2, 256, 16, 57, seq_lens=[900, 70, 333], q_lens=list(q_lens), seed=sum(q_lens)))
