"""128-row workgroups dealt in runs across row groups (KH_STREAM): prompt chunks whose row groups do not fill the CUs evenly,
at the places where a run can go wrong -- row remainders, few tiles, fragments that end inside a run, empty fragments, runs that
cut a row group in two and three, GQA ratios with and without staged rotation tables -- against float64 on the same inputs."""
import ctypes as C

import pytest
import torch

from inference_lib_amd import _lib
from inference_lib_amd import attention as ops
from inference_lib_amd.cases import locations_for, rope_tables

pytestmark = pytest.mark.gpu


def _orders(F, W):
    return [[f for f in range(F) if f != F - 1 - w % F] + [F - 1 - w % F] for w in range(W)]


def _reference(rq, loc, keys, values, scale, Hkv):
    """Softmax over the visible tokens of every fragment, in float64.  rq [F,W,Hq,S,D] as the kernels hold it (storage type).
    With out and lse comes a bound on the error of each result: with u the unit roundoff of the storage type (2^-8 for the 8
    significant bits of bf16, 2^-11 for the 11 of fp16), probabilities are rounded to it once (u sum p |v|; in fp16, where they
    may be subnormal, 2^-25 sum |v| more, the row sums being at least 1) and so is the result (u |out|); the fp32 sums of up to a
    few thousand terms are worth another 2^-16 sum p |v| at most."""
    F, W, Hq, S, D = rq.shape
    u = 2.0 ** -8 if rq.dtype == torch.bfloat16 else 2.0 ** -11
    tiny = 0.0 if rq.dtype == torch.bfloat16 else 2.0 ** -25
    out, bound = (torch.empty((W, Hq, S, D), dtype=torch.float64, device=rq.device) for _ in range(2))
    lse = torch.empty((W, Hq, S), dtype=torch.float64, device=rq.device)
    for h in range(Hq):
        for w in range(W):
            logits = []
            for f in range(F):
                k = keys[f][h // (Hq // Hkv)].double()
                x = rq[f, w, h].double() @ k.t().contiguous() * scale
                seen = torch.arange(k.size(0), device=rq.device)[None, :] <= loc[f, w][:, None]
                logits.append(x.masked_fill(~seen, float("-inf")))
            x = torch.cat(logits, dim=1)
            v = torch.cat([t[h // (Hq // Hkv)].double() for t in values], dim=0)
            lse[w, h] = torch.logsumexp(x, dim=1)
            p = torch.softmax(x, dim=1)
            out[w, h] = p @ v
            bound[w, h] = (u + 2.0 ** -16) * (p @ v.abs()) + u * out[w, h].abs() + tiny * v.abs().sum(dim=0)
    return out, lse, bound


def _inputs(W, S, Hq, Hkv, D, lens, dtype, rot):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    loc = locations_for(_orders(len(lens), W), list(lens), S)
    cos, sin = (t.cuda() for t in rope_tables(loc, rot, 1e6))
    q = torch.randn((W, Hq, S, D), generator=g, device="cuda").to(dtype)
    keys = [torch.randn((Hkv, n, D), generator=g, device="cuda").to(dtype) for n in lens]
    values = [torch.randn((Hkv, n, D), generator=g, device="cuda").to(dtype) for n in lens]
    return q, loc.cuda(), cos, sin, keys, values


def _rounds_plan(problem):
    """The launch in rounds of a call that is dealt in runs: its workspace is smaller (128-row slots, a row table)."""
    plan = _lib.HwPlan()
    _lib.check(_lib.lib.hw_plan_debug(C.byref(problem.p), _lib.lib.hw_device_cus(), C.byref(plan)), "hw_plan_debug")
    assert plan.row_blocks == 8 and problem.workspace_bytes() > plan.workspace_bytes, "not a call for runs"
    return plan


CASES = [
    # W, S, Hq, Hkv, D, lens, dtype
    (1, 830, 40, 8, 128, (100, 830), torch.bfloat16),            # 33 row groups, the last of 54 rows
    (1, 830, 40, 8, 64, (100, 0, 830), torch.float16),           # an empty fragment
    (1, 1400, 24, 3, 128, (33, 7, 1400), torch.bfloat16),        # 88 row groups of 3 heads: grid not a multiple of 8
    (2, 550, 16, 8, 64, (64, 550, 550), torch.bfloat16),         # GQA 2: every row loads its own table row; row groups in three
    (1, 1460, 28, 4, 128, (1, 1460), torch.float16),             # 80 row groups, one-token fragment
    (2, 1300, 8, 8, 64, (200, 1300, 1300), torch.float16),
]


@pytest.mark.parametrize("W,S,Hq,Hkv,D,lens,dtype", CASES)
def test_runs_across_row_groups(W, S, Hq, Hkv, D, lens, dtype):
    F = len(lens)
    scale = D ** -0.5
    q, loc, cos, sin, keys, values = _inputs(W, S, Hq, Hkv, D, lens, dtype, D)
    rq = torch.empty((F, W, Hq, S, D), dtype=dtype, device="cuda")
    out, lse = torch.empty_like(q), torch.empty((W, Hq, S), dtype=torch.float32, device="cuda")
    frag = torch.tensor(lens, dtype=torch.int32, device="cuda")

    problem = _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=out, cosines=cos, sines=sin, rq=rq)
    rounds = _rounds_plan(problem)

    ops.hogwild_fused(q, loc, keys, values, scale, frag, cos, sin, rotated_queries=rq, out=out, lse=lse)
    want_rq = ops.hogwild_rope(q, cos, sin)
    # (fused multiply-add or not: one rounding of the storage type)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert float((rq.float() - want_rq.float()).abs().max()) <= 4 * eps * float(want_rq.float().abs().max())
    ref, ref_lse, bound = _reference(rq, loc, keys, values, scale, Hkv)
    assert bool(((out.double() - ref).abs() <= bound).all())
    assert float((lse.double() - ref_lse).abs().max()) <= 1e-4

    # the same through pre-rotated queries, and a fixed split (workgroups per row group) on the same inputs
    out2 = ops.hogwild_sdpa(rq, loc, keys, values, scale, frag)
    assert bool(((out2.double() - ref).abs() <= bound).all())
    # (rotated anew in the kernel from the same inputs: the same rq)
    out3 = torch.empty_like(q)
    _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=out3, cosines=cos, sines=sin, splits=1).run()
    assert bool(((out3.double() - ref).abs() <= bound).all())
    # a workspace sized for the launch in rounds keeps to it
    out4 = torch.empty_like(q)
    small = _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=out4, cosines=cos, sines=sin)
    small.set_workspace(torch.empty(rounds.workspace_bytes, dtype=torch.uint8, device="cuda"))
    small.run()
    assert bool(((out4.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("W,S,Hq,Hkv,D,lens,dtype", [CASES[0], CASES[3]])
def test_partial_rotary_width_with_the_rotated_queries_in_the_workspace(W, S, Hq, Hkv, D, lens, dtype):
    """RotE < E without a buffer for the rotated queries: they lie in the workspace behind everything else, and the partial sums
    and the row table must not reach them."""
    scale = D ** -0.5
    q, loc, cos, sin, keys, values = _inputs(W, S, Hq, Hkv, D, lens, dtype, D // 2)
    rq = ops.hogwild_rope(q, cos, sin)
    ref, ref_lse, bound = _reference(rq, loc, keys, values, scale, Hkv)
    for in_rounds in (False, True):
        out, lse = torch.empty_like(q), torch.empty((W, Hq, S), dtype=torch.float32, device="cuda")
        pr = _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=out, cosines=cos, sines=sin, lse=lse)
        bytes_ = _rounds_plan(pr).workspace_bytes if in_rounds else pr.workspace_bytes()
        assert bytes_ > rq.numel() * rq.element_size()
        guard = torch.full((bytes_ + 4096,), 165, dtype=torch.uint8, device="cuda")
        pr.set_workspace(guard[:bytes_])
        pr.run()
        assert bool(((out.double() - ref).abs() <= bound).all()) and float((lse.double() - ref_lse).abs().max()) <= 1e-4
        assert bool((guard[bytes_:] == 165).all())


def test_the_attention_stage_alone_leaves_the_documented_partials():
    """hw_fused_attention_stages: a caller that reads or exchanges the partials finds [Hkv][workgroup][row][Ev] and behind it
    [Hkv][workgroup][row][2] (maximum in base-2 units, sum) with the workgroups of hw_plan_debug, also for a call that
    hw_fused_attention deals in runs."""
    W, S, Hq, Hkv, D, lens, dtype = CASES[3]
    scale = D ** -0.5
    q, loc, cos, sin, keys, values = _inputs(W, S, Hq, Hkv, D, lens, dtype, D)
    out = torch.empty_like(q)
    pr = _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=out, cosines=cos, sines=sin)
    plan = _rounds_plan(pr)
    ws = torch.zeros(pr.workspace_bytes(), dtype=torch.uint8, device="cuda")
    pr.set_workspace(ws)
    pr.run(stages=1)
    n = Hkv * plan.wgs_per_head * plan.rows
    part = ws.view(torch.float32)[: n * (D + 2)].double()
    o, ml = part[: n * D].view(Hkv, plan.wgs_per_head, plan.rows, D), part[n * D:].view(Hkv, plan.wgs_per_head, plan.rows, 2)
    weight = torch.exp2(ml[..., 0] - ml[..., 0].amax(dim=1, keepdim=True))
    got = (o * weight[..., None]).sum(1) / (ml[..., 1] * weight).sum(1)[..., None]            # [Hkv][(worker, token, head of group)]
    got = got.view(Hkv, W, S, Hq // Hkv, D).permute(1, 0, 3, 2, 4).reshape(W, Hq, S, D)
    ref, _, bound = _reference(ops.hogwild_rope(q, cos, sin), loc, keys, values, scale, Hkv)
    assert bool(((got - ref).abs() <= bound).all())
    pr.run(stages=2)
    assert bool(((out.double() - ref).abs() <= bound).all())
