"""128-row workgroups that bring what opening a fragment needs into LDS beside the tiles of the one before: fragments of one tile and of
none, many of them behind one another, fragments that some row groups or none see, GQA ratios without staged tables, whole row groups
and runs, pre-rotated queries with and without them -- against float64."""
import pytest
import torch

from inference_lib_amd import attention as ops
from test_gpu_stream_runs import _inputs, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,S,Hq,Hkv,D,lens,dtype", [
    (1, 1100, 28, 4, 128, (1, 40, 33, 0, 1100), torch.bfloat16),                  # one and two tiles, an empty one: whole row groups
    (1, 840, 40, 8, 128, (3, 31, 32, 65, 1, 1, 840, 17), torch.float16),          # eight fragments, the chunk not the last
    (1, 1879, 28, 4, 128, (208, 1879), torch.bfloat16),                           # a row group in five pieces, most in two: merged eight rows to a workgroup
    (1, 700, 20, 20, 128, (300, 20, 700), torch.bfloat16),                        # GQA 1: tables out of memory
    (2, 640, 16, 8, 128, (64, 640, 1, 640), torch.float16),                       # GQA 2, two workers
    (5, 7, 28, 4, 128, (1, 33, 7, 20, 64, 7, 200), torch.bfloat16),               # few rows: pre-rotated only
    (3, 30, 8, 2, 64, (500, 30, 1, 30, 30), torch.float16),
])
def test_openings(W, S, Hq, Hkv, D, lens, dtype):
    scale = D ** -0.5
    q, loc, cos, sin, keys, values = _inputs(W, S, Hq, Hkv, D, lens, dtype, D)
    F = len(lens)
    loc[F // 2, :, : S // 3] = -1                  # the first third of the tokens sees nothing of one fragment
    loc[F - 1, :, 3::50] = -1
    rq = torch.full((F, W, Hq, S, D), 12345.0, dtype=dtype, device="cuda")
    out, lse = torch.full_like(q, 12345.0), torch.full((W, Hq, S), 12345.0, dtype=torch.float32, device="cuda")
    frag = torch.tensor(lens, dtype=torch.int32, device="cuda")
    ops.hogwild_fused(q, loc, keys, values, scale, frag, cos, sin, rotated_queries=rq, out=out, lse=lse)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    want_rq = ops.hogwild_rope(q, cos, sin)
    assert float((rq.float() - want_rq.float()).abs().max()) <= 4 * eps * float(want_rq.float().abs().max())
    # and every element against float64: two fp32 roundings on the way, one to the storage type (2^-25: half the spacing of fp16's subnormals)
    h = D // 2
    x1, x2 = q.double()[None, ..., :h], q.double()[None, ..., h:]
    c, s = cos[:, :, None, :, :h].double(), sin[:, :, None, :, :h].double()
    rotated = torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], dim=-1)
    size = torch.cat([(x1 * c).abs() + (x2 * s).abs(), (x2 * c).abs() + (x1 * s).abs()], dim=-1)
    assert bool(((rq.double() - rotated).abs() <= eps * rotated.abs() + 2.0 ** -22 * size + (2.0 ** -25 if dtype == torch.float16 else 0.0)).all())
    ref, ref_lse, bound = _reference(rq, loc, keys, values, scale, Hkv)
    seen = ~torch.isneginf(ref_lse)
    assert bool(((out.double() - ref).abs() <= bound)[seen].all())
    assert float((lse.double() - ref_lse)[seen].abs().max()) <= 1e-4
    assert bool((out[~seen] == 0).all()) and bool(torch.isneginf(lse[~seen]).all())
    again = ops.hogwild_sdpa(rq, loc, keys, values, scale, frag)
    assert bool(((again.double() - ref).abs() <= bound)[seen].all())
