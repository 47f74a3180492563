"""hw_rope: rows in 16-byte chunks where the sizes and addresses allow it, element by element where they do not, against float64."""
import pytest
import torch

from inference_lib_amd import attention as ops

pytestmark = pytest.mark.gpu

CASES = [
    # F, W, Hq, S, E, RotE, elements by which the queries and the result are shifted
    (1, 1, 1, 1, 64, 64, 0),
    (3, 2, 5, 3, 128, 128, 0),
    (4, 3, 33, 9, 256, 256, 0),        # more than a workgroup per (fragment, worker) pair, the last one not full
    (2, 3, 7, 1, 128, 64, 0),          # a tail behind the rotary width
    (2, 1, 3, 2, 96, 32, 0),
    (2, 2, 3, 5, 80, 48, 0),           # a half of three chunks
    (1, 2, 3, 3, 64, 0, 0),            # nothing to rotate
    (2, 2, 3, 2, 60, 20, 0),           # odd widths
    (2, 2, 3, 2, 64, 24, 0),           # half the rotary width is no whole chunk
    (2, 2, 3, 2, 128, 128, 1),         # not aligned
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("F,W,Hq,S,E,RotE,shift", CASES)
def test_rope_against_float64(F, W, Hq, S, E, RotE, shift, dtype):
    g = torch.Generator(device="cuda").manual_seed(E + RotE + shift)
    n = W * Hq * S * E
    q = torch.randn(n + shift, generator=g, device="cuda").to(dtype)[shift:].view(W, Hq, S, E)
    cos, sin = (torch.rand((F, W, S, RotE), generator=g, device="cuda") * 2 - 1 for _ in range(2))
    room = torch.full((F * n + shift + 8,), 7.0, dtype=dtype, device="cuda")
    out = room[shift:shift + F * n].view(F, W, Hq, S, E)
    ops.hogwild_rope(q, cos, sin, out=out)
    h = RotE // 2
    x1, x2, tail = (t.double()[None] for t in (q[..., :h], q[..., h:RotE], q[..., RotE:]))
    c, s = (t[..., :h].double()[:, :, None] for t in (cos, sin))
    want = torch.cat([x1 * c - x2 * s, x2 * c + x1 * s, tail.expand(F, -1, -1, -1, -1)], dim=-1)
    size = torch.cat([(x1 * c).abs() + (x2 * s).abs(), (x2 * c).abs() + (x1 * s).abs(), torch.zeros_like(tail).expand(F, -1, -1, -1, -1)], dim=-1)
    # two fp32 roundings on the way (one with a fused multiply-add), one to the storage type (2^-25: half the spacing of fp16's subnormals)
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[dtype]
    bound = u * want.abs() + 2.0 ** -22 * size + (2.0 ** -25 if dtype == torch.float16 else 0.0)
    assert bool(((out.double() - want).abs() <= bound).all())
    assert torch.equal(out[..., RotE:], q[None, ..., RotE:].expand(F, -1, -1, -1, -1))
    assert bool((room[shift + F * n:] == 7.0).all())
