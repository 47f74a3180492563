"""128-row workgroups dealt in runs across row groups (KH_STREAM): prompt chunks whose row groups do not fill the CUs evenly,
at the places where a run can go wrong -- row remainders, few tiles, fragments that end inside a run, empty fragments, runs that
cut a row group in two and three, GQA ratios with and without staged rotation tables -- against float64 on the same inputs."""
import pytest
import torch

from inference_lib_amd import _lib
from inference_lib_amd import attention as ops
from inference_lib_amd.cases import locations_for, rope_tables

pytestmark = pytest.mark.gpu


def _orders(F, W):
    return [[f for f in range(F) if f != F - 1 - w % F] + [F - 1 - w % F] for w in range(W)]


def _reference(rq, loc, keys, values, scale, Hkv):
    """Softmax over the visible tokens of every fragment, in float64.  rq [F,W,Hq,S,D] as the kernels hold it (storage type)."""
    F, W, Hq, S, D = rq.shape
    out = torch.empty((W, Hq, S, D), dtype=torch.float64, device=rq.device)
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
            out[w, h] = torch.softmax(x, dim=1) @ v
    return out, lse


CASES = [
    # W, S, Hq, Hkv, D, lens, dtype
    (1, 515, 40, 8, 128, (100, 515), torch.bfloat16),            # 21 row groups, the last of 15 rows
    (1, 515, 40, 8, 64, (100, 0, 515), torch.float16),           # an empty fragment
    (1, 1030, 12, 3, 128, (33, 7, 1030), torch.bfloat16),        # 33 row groups of 3 heads: grid not a multiple of 8
    (2, 640, 16, 8, 64, (64, 640, 640), torch.bfloat16),         # GQA 2: every row loads its own table row
    (1, 1460, 28, 4, 128, (1, 1460), torch.float16),             # 80 row groups, one-token fragment
    (2, 1300, 8, 8, 64, (200, 1300, 1300), torch.float16),
]


@pytest.mark.parametrize("W,S,Hq,Hkv,D,lens,dtype", CASES)
def test_runs_across_row_groups(W, S, Hq, Hkv, D, lens, dtype):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    F = len(lens)
    scale = D ** -0.5
    loc = locations_for(_orders(F, W), list(lens), S)
    cos, sin = (t.cuda() for t in rope_tables(loc, D, 1e6))
    loc = loc.cuda()
    q = torch.randn((W, Hq, S, D), generator=g, device="cuda").to(dtype)
    keys = [torch.randn((Hkv, n, D), generator=g, device="cuda").to(dtype) for n in lens]
    values = [torch.randn((Hkv, n, D), generator=g, device="cuda").to(dtype) for n in lens]
    rq = torch.empty((F, W, Hq, S, D), dtype=dtype, device="cuda")
    out, lse = torch.empty_like(q), torch.empty((W, Hq, S), dtype=torch.float32, device="cuda")
    frag = torch.tensor(lens, dtype=torch.int32, device="cuda")

    problem = _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=out, cosines=cos, sines=sin, rq=rq)
    rounds = _lib.plan(lens, W=W, S=S, Hq=Hq, Hkv=Hkv, Ev=D, num_cus=_lib.lib.hw_device_cus())
    assert rounds.row_blocks == 8 and problem.workspace_bytes() != rounds.workspace_bytes, "not a call for runs"

    ops.hogwild_fused(q, loc, keys, values, scale, frag, cos, sin, rotated_queries=rq, out=out, lse=lse)
    want_rq = ops.hogwild_rope(q, cos, sin)
    # (fused multiply-add or not: one rounding of the storage type)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert float((rq.float() - want_rq.float()).abs().max()) <= 4 * eps * float(want_rq.float().abs().max())
    ref, ref_lse = _reference(rq, loc, keys, values, scale, Hkv)
    # probabilities and results are rounded to the storage type once each: |error| <= 2 eps |v|max (softmax weights sum to 1)
    bound = 2 * eps * float(torch.cat([v.float().abs().flatten() for v in values]).max())
    assert float((out.double() - ref).abs().max()) <= bound
    assert float((lse.double() - ref_lse).abs().max()) <= 1e-4

    # the same through pre-rotated queries, and a fixed split (workgroups per row group) on the same inputs
    out2 = ops.hogwild_sdpa(rq, loc, keys, values, scale, frag)
    assert float((out2.double() - ref).abs().max()) <= bound
    out3 = torch.empty_like(q)
    _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=out3, cosines=cos, sines=sin, splits=1).run()
    assert float((out3.double() - out.double()).abs().max()) <= bound
    # a workspace sized for the launch in rounds keeps to it
    out4 = torch.empty_like(q)
    small = _lib.Problem(q=q, locations=loc, keys=keys, values=values, scale=scale, out=out4, cosines=cos, sines=sin)
    if rounds.workspace_bytes < problem.workspace_bytes():
        small.set_workspace(torch.empty(rounds.workspace_bytes, dtype=torch.uint8, device="cuda"))
        small.run()
        assert float((out4.double() - ref).abs().max()) <= bound
