"""Paged decode steps of sequences of different length: the workgroups of a kv head are shared out by the visible tiles (paged_share) --
against the same call with the split fixed by the caller, which keeps equal shares, and in a workspace sized for those."""
import pytest
import torch

from inference_lib_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,lens,S,F,Hq,Hkv,D,bs", [
    (torch.bfloat16, (1, 5000), 1, 1, 8, 8, 128, 16),                            # one tile beside many
    (torch.float16, (300, 0, 7000, 33, 64, 1), 1, 1, 28, 4, 64, 32),             # a sequence that sees nothing
    (torch.bfloat16, (9000, 40, 40, 40, 40, 40, 40), 2, 1, 40, 8, 128, 16),      # several tokens; nearly all to the first
    (torch.float32, (700, 2900, 31), 1, 1, 8, 2, 64, 16),
    (torch.bfloat16, (100, 11000, 900, 2500), 1, 1, 16, 8, 256, 64),
    (torch.float16, (4000, 200, 1500), 1, 3, 16, 4, 128, 16),                    # three fragments of the same sequences
    (torch.bfloat16, tuple(64 + 97 * i for i in range(31)), 1, 1, 8, 2, 128, 16),
    (torch.bfloat16, (1000, 1190, 850), 1, 1, 40, 8, 128, 16),                   # within a fifth: equal shares
])
def test_shares_by_length(dtype, lens, S, F, Hq, Hkv, D, bs):
    g = torch.Generator(device="cuda").manual_seed(len(lens) + D)
    W, mb = len(lens), -(-max(lens) // bs) + 3
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)
    kc, vc = rnd(W * mb, Hkv, bs, D), rnd(W * mb, Hkv, bs, D)
    table = torch.randperm(W * mb, generator=g, device="cuda").to(torch.int32).reshape(W, mb)
    q = rnd(F, W, Hq, S, D)
    pos = torch.tensor([[n - S + s for s in range(S)] for n in lens], dtype=torch.int32, device="cuda").clamp(min=-1)
    loc = torch.stack([pos - 50 * f for f in range(F)]).clamp(min=-1).contiguous()
    frag = torch.full((F,), bs * mb, dtype=torch.int32, device="cuda")
    results = []
    for splits, sized_for_equal in ((0, False), (0, True), (3, False)):
        out, lse = torch.full((W, Hq, S, D), 7.0, dtype=dtype, device="cuda"), torch.full((W, Hq, S), 7.0, device="cuda")
        pr = _lib.PagedProblem(q=q, locations=loc, fragment_lengths=frag, key_cache=kc, value_cache=vc, block_table=table, scale=D ** -0.5, out=out, lse=lse,
                               splits=splits)
        need = pr.workspace_bytes()
        if sized_for_equal:                        # the row table does not fit: equal shares
            equal = _lib.paged_plan(W=W, Hq=Hq, Hkv=Hkv, Ev=D, block_size=bs, max_blocks=mb, num_cus=_lib.lib.hw_device_cus(), S=S, dtype=_lib._DTYPE_CODE[dtype])
            assert equal.splits > 1 and equal.workspace_bytes < need
            need = equal.workspace_bytes
        space = torch.full((need + 4096,), 165, dtype=torch.uint8, device="cuda")
        pr.set_workspace(space[:need])
        pr.run()
        assert bool((space[need:] == 165).all())
        results.append((out.double(), lse.double()))
    # float64, of the values as stored
    ref, ref_lse = torch.zeros((W, Hq, S, D), dtype=torch.float64, device="cuda"), torch.full((W, Hq, S), float("-inf"), dtype=torch.float64, device="cuda")
    bound = torch.zeros_like(ref)
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[dtype]
    for w in range(W):
        n = max(lens[w], 1)
        rows = table[w, : -(-n // bs)].long()
        k, v = (c[rows].transpose(1, 2).reshape(-1, Hkv, D)[:n].double() for c in (kc, vc))          # [n, Hkv, D]
        for h in range(Hq):
            kh, vh = k[:, h // (Hq // Hkv)], v[:, h // (Hq // Hkv)]
            x = torch.cat([(q[f, w, h].double() @ kh.t().contiguous() * D ** -0.5).masked_fill(torch.arange(n, device="cuda")[None] > loc[f, w][:, None], float("-inf"))
                           for f in range(F)], dim=1)
            ref_lse[w, h] = torch.logsumexp(x, dim=1)
            p = torch.nan_to_num(torch.softmax(x, dim=1))
            vv = vh.repeat(F, 1)
            ref[w, h] = p @ vv
            # probabilities and the result are rounded once (fp16: to 2^-25 where subnormal), the fp32 sums are worth another 2^-16
            bound[w, h] = (u + 2.0 ** -16) * (p @ vv.abs()) + u * ref[w, h].abs() + (2.0 ** -25 * vv.abs().sum(0) if dtype == torch.float16 else 0.0)
    seen = ~torch.isneginf(ref_lse)
    for out, lse in results:
        assert bool(((out - ref).abs() <= bound)[seen].all())
        assert bool((out[~seen] == 0).all()) and bool(torch.isneginf(lse[~seen]).all())
        assert float((lse - ref_lse)[seen].abs().max()) <= 1e-4


@pytest.mark.parametrize("dtype,lens,S,F,Hq,Hkv,D,bs,within", [
    # 64 sequences (a lane of a wave each) and F * S = 8; beyond them equal shares
    (torch.bfloat16, (6000,) + tuple(40 + 29 * i for i in range(62)) + (4500,), 1, 1, 8, 2, 64, 32, True),
    (torch.float16, (6000,) + tuple(40 + 29 * i for i in range(63)) + (4500,), 1, 1, 8, 2, 64, 32, False),
    (torch.bfloat16, (300, 7000, 1200, 8), 8, 1, 16, 8, 128, 32, True),
    (torch.float16, (300, 5000, 64), 4, 2, 28, 7, 128, 16, True),
    (torch.bfloat16, (300, 7000, 1200), 3, 3, 40, 8, 128, 16, False),
])
def test_limits_of_the_rule(dtype, lens, S, F, Hq, Hkv, D, bs, within):
    W, mb = len(lens), -(-max(lens) // bs) + 3
    g = torch.Generator(device="cuda").manual_seed(W)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)
    table = torch.randperm(W * mb, generator=g, device="cuda").to(torch.int32).reshape(W, mb)
    pos = torch.tensor([[n - S + s for s in range(S)] for n in lens], dtype=torch.int32, device="cuda")
    args = dict(q=rnd(F, W, Hq, S, D), locations=torch.stack([pos - 7 * f for f in range(F)]).clamp(min=-1).contiguous(), key_cache=rnd(W * mb, Hkv, bs, D),
                value_cache=rnd(W * mb, Hkv, bs, D), block_table=table, scale=D ** -0.5, fragment_lengths=torch.full((F,), bs * mb, dtype=torch.int32, device="cuda"))
    equal = _lib.paged_plan(W=W, Hq=Hq, Hkv=Hkv, Ev=D, block_size=bs, max_blocks=mb, num_cus=_lib.lib.hw_device_cus(), S=S, dtype=_lib._DTYPE_CODE[dtype])
    assert equal.splits > 1
    outs = []
    for splits in (0, equal.splits):
        outs.append(torch.full((W, Hq, S, D), 7.0, dtype=dtype, device="cuda"))
        pr = _lib.PagedProblem(out=outs[-1], splits=splits, **args)
        assert (pr.workspace_bytes() > equal.workspace_bytes) == (within and splits == 0)      # room for the row table of other shares
        pr.run()
    assert torch.equal(*outs) == (not within)
    if within:
        test_shares_by_length(dtype, lens, S, F, Hq, Hkv, D, bs)


def _step(lens, dtype, Hq, Hkv, D, bs, mb, seed, splits=0, change=None):
    """One decode step; sequence i has the data of its number in `lens`, a list of (number, length), wherever it is listed.
    change(q, keys, values, table) alters the data."""
    W, n = len(lens), len(lens) * mb
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)
    kc, vc, q = rnd(n, Hkv, bs, D), rnd(n, Hkv, bs, D), rnd(1, W, Hq, 1, D)
    table = torch.randperm(n, generator=g, device="cuda").to(torch.int32).reshape(W, mb)
    order = [i for i, _ in lens]
    if change is not None:
        change(q, kc, vc, table)
    loc = torch.tensor([[[m - 1] for _, m in lens]], dtype=torch.int32, device="cuda")
    out, lse = torch.empty((W, Hq, 1, D), dtype=dtype, device="cuda"), torch.empty((W, Hq, 1), device="cuda")
    frag = torch.tensor([bs * mb], dtype=torch.int32, device="cuda")
    _lib.PagedProblem(q=q[:, order].contiguous(), locations=loc, fragment_lengths=frag, key_cache=kc, value_cache=vc, block_table=table[order].contiguous(),
                      scale=D ** -0.5, out=out, lse=lse, splits=splits).run()
    back = torch.tensor(order).argsort().cuda()
    return out[back], lse[back]


@pytest.mark.parametrize("dtype,lens,Hq,Hkv,D", [
    (torch.bfloat16, (9600, 10880, 8160, 8160), 40, 8, 128),      # the first within a fifth of all others, the longest a fifth above the mean
    (torch.float16, (3000, 3550, 2550, 2550, 2550), 16, 8, 256),
    (torch.bfloat16, (400, 9000, 2000, 64, 5000, 33), 32, 8, 128),
    (torch.float32, (300, 4100, 900), 8, 8, 64),
    (torch.bfloat16, (7000,) + tuple(100 + 61 * i for i in range(23)), 40, 8, 128),      # more workgroups than CUs, and shares save many steps
])
def test_order_of_the_sequences_does_not_matter(dtype, lens, Hq, Hkv, D):
    """The same sequences listed in other orders: the same bits for each."""
    bs, mb = 32, -(-max(lens) // 32) + 1
    listed = list(enumerate(lens))
    first = _step(listed, dtype, Hq, Hkv, D, bs, mb, D)
    for order in (listed[::-1], listed[1:] + listed[:1], sorted(listed, key=lambda x: -x[1])):
        for a, b in zip(first, _step(order, dtype, Hq, Hkv, D, bs, mb, D)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,lens,Hq,Hkv,D", [
    (torch.bfloat16, (1318, 2139, 1454, 101, 419, 62, 2291, 197, 900), 8, 2, 64),      # two steps of a wave: nothing to gain by other shares
    (torch.bfloat16, (465, 191, 997, 358, 388, 1028, 84, 1466, 456, 213), 28, 4, 128),
    (torch.float16, (184, 101, 104, 74), 16, 8, 256),
    (torch.bfloat16, (886, 3433), 40, 8, 128),
    (torch.bfloat16, (4096, 4000, 4064, 3969), 40, 8, 128),                              # as many steps with even shares
    (torch.bfloat16, (2016,) + tuple(200 + 40 * i for i in range(47)), 28, 4, 128),      # more workgroups than CUs, and shares save few steps
    (torch.float16, tuple(60 + 50 * i for i in range(64)), 40, 8, 128),
])
def test_short_and_even_steps_keep_equal_shares(dtype, lens, Hq, Hkv, D):
    """The bits of the call whose split is fixed at that of equal shares, which is launched so whatever the lengths."""
    bs, mb = 32, -(-max(lens) // 32)
    equal = _lib.paged_plan(W=len(lens), Hq=Hq, Hkv=Hkv, Ev=D, block_size=bs, max_blocks=mb, num_cus=_lib.lib.hw_device_cus(), S=1, dtype=_lib._DTYPE_CODE[dtype])
    assert equal.splits > 1
    listed = list(enumerate(lens))
    for a, b in zip(_step(listed, dtype, Hq, Hkv, D, bs, mb, D), _step(listed, dtype, Hq, Hkv, D, bs, mb, D, splits=equal.splits)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,lens,Hq,Hkv,D", [
    (torch.bfloat16, (8989, 493, 7242, 1180, 231, 1815, 3425, 8850), 32, 8, 128),
    (torch.float16, (2194, 3461, 4600, 1232, 2019, 6230, 2042, 395), 16, 8, 256),
    (torch.bfloat16, (895, 7978, 64), 64, 8, 128),
    (torch.float16, (2852, 3640, 4675, 11537, 220, 2552, 4251, 578), 8, 2, 64),
])
def test_shares_cost_no_precision(dtype, lens, Hq, Hkv, D):
    """Short sequences get fewer workgroups than with equal shares, so fewer of their weights are the largest of a wave's first tile, which
    the storage type holds exactly; the reference follows the tiles instead, and every tile's largest is exact: no further from float64
    than equal shares, which hold a part of those."""
    bs, mb, kept = 32, -(-max(lens) // 32), []
    listed = list(enumerate(lens))
    equal = _lib.paged_plan(W=len(lens), Hq=Hq, Hkv=Hkv, Ev=D, block_size=bs, max_blocks=mb, num_cus=_lib.lib.hw_device_cus(), S=1, dtype=_lib._DTYPE_CODE[dtype])
    shared, _ = _step(listed, dtype, Hq, Hkv, D, bs, mb, D, change=lambda *data: kept.extend(data))
    fixed, _ = _step(listed, dtype, Hq, Hkv, D, bs, mb, D, splits=equal.splits)
    assert not torch.equal(shared, fixed)
    q, kc, vc, table = kept
    ref = torch.empty(shared.shape, dtype=torch.float64, device="cuda")
    for w, n in listed:
        rows = table[w, : -(-n // bs)].long()
        k, v = (c[rows].transpose(1, 2).reshape(-1, Hkv, D)[:n].double() for c in (kc, vc))
        for h in range(Hq):
            ref[w, h] = torch.softmax(q[0, w, h].double() @ k[:, h // (Hq // Hkv)].t().contiguous() * D ** -0.5, dim=1) @ v[:, h // (Hq // Hkv)]
    assert float((shared.double() - ref).norm()) <= float((fixed.double() - ref).norm())


@pytest.mark.parametrize("dtype,Hq,Hkv,D", [(torch.bfloat16, 40, 8, 128), (torch.float16, 16, 8, 256)])
def test_infinite_logits_and_values_under_shares(dtype, Hq, Hkv, D):
    """Logits of minus infinity (one, a whole tile, a sequence's first tiles) weigh nothing, and infinite values stay infinite, as with
    equal shares."""
    lens, bs = (700, 6000, 90, 2500), 32
    mb, listed = -(-max(lens) // bs), list(enumerate(lens))

    def change(q, kc, vc, table):
        q.abs_()
        for w, block, row in ((0, 3, 5), (3, 1, slice(None)), (1, 0, slice(None)), (1, 1, slice(None)), (2, 1, 3)):
            kc[int(table[w, block]), :, row] = float("-inf")
        vc[int(table[3, 40]), :, 7, : D // 2] = float("inf")
        vc[int(table[0, 2]), 0, 9] = float("-inf")

    equal = _lib.paged_plan(W=len(lens), Hq=Hq, Hkv=Hkv, Ev=D, block_size=bs, max_blocks=mb, num_cus=_lib.lib.hw_device_cus(), S=1, dtype=_lib._DTYPE_CODE[dtype])
    out, lse = _step(listed, dtype, Hq, Hkv, D, bs, mb, 3, change=change)
    want, want_lse = _step(listed, dtype, Hq, Hkv, D, bs, mb, 3, splits=equal.splits, change=change)
    finite = torch.isfinite(want)
    assert not torch.equal(out, want) and bool((~finite).any()) and not bool(torch.isnan(want).any()) and torch.equal(out[~finite], want[~finite])
    # the probabilities and the results of two launches, each rounded once; |values| < 6
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert float((out[finite].double() - want[finite].double()).abs().max()) <= 4 * u * 6.0
    assert float((lse - want_lse).abs().max()) <= 1e-4


@pytest.mark.parametrize("dtype,Hq,Hkv,D,S", [(torch.bfloat16, 40, 8, 128, 1), (torch.float16, 16, 8, 256, 3), (torch.float32, 8, 8, 128, 1), (torch.float16, 64, 8, 64, 4)])
def test_caches_of_4_gb_and_more(dtype, Hq, Hkv, D, S):
    """K rows are reached through one buffer descriptor below 4 GB and through 64-bit addresses from there on: the same blocks at the end of
    a cache of 4.3 GB and in a small one give the same bits."""
    bs, lens = 32, (700, 90, 2500)
    W, mb = len(lens), -(-max(lens) // bs)
    g = torch.Generator(device="cuda").manual_seed(D)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)
    k, v, q = rnd(W * mb, Hkv, bs, D), rnd(W * mb, Hkv, bs, D), rnd(1, W, Hq, S, D)
    table = torch.randperm(W * mb, generator=g, device="cuda").to(torch.int32).reshape(W, mb)
    loc = torch.tensor([[[n - S + s for s in range(S)] for n in lens]], dtype=torch.int32, device="cuda")
    frag = torch.tensor([max(lens)], dtype=torch.int32, device="cuda")
    many = -(-(2 ** 32 + 2 ** 20) // (Hkv * bs * D * k.element_size()))
    results = []
    for blocks in (W * mb, many):
        kc, vc = (torch.empty((blocks, Hkv, bs, D), dtype=dtype, device="cuda") for _ in range(2))
        kc[blocks - W * mb:], vc[blocks - W * mb:] = k, v
        out = torch.empty((W, Hq, S, D), dtype=dtype, device="cuda")
        _lib.PagedProblem(q=q, locations=loc, fragment_lengths=frag, key_cache=kc, value_cache=vc, block_table=table + (blocks - W * mb), scale=D ** -0.5, out=out).run()
        results.append(out)
    assert torch.equal(*results) and bool(torch.isfinite(results[0].float()).all())


@pytest.mark.parametrize("dtype,tokens,lens,Hq,Hkv,D", [
    (torch.bfloat16, (120, 100, 60, 40, 20), (1200, 5200, 800, 3000, 9000), 40, 8, 128),     # 16 row groups of 32 slots, 51 provided
    (torch.float16, (30, 90, 5, 128, 60, 2, 17), (1300, 3200, 700, 5100, 400, 2000, 6000), 64, 8, 128),      # 24: two rounds
    (torch.bfloat16, (128,) * 5, (1300, 3200, 700, 5100, 400), 64, 8, 128),                  # 40: more than the CUs of a head
    (torch.float16, (30, 0, 60), (3000, 700, 64), 8, 2, 64),                                 # 128 slots a head, a sequence without tokens
    (torch.bfloat16, (40,) + (1,) * 40, (4000,) + tuple(60 + 31 * i for i in range(40)), 40, 8, 128),
])
def test_packed_rounds(dtype, tokens, lens, Hq, Hkv, D):
    g = torch.Generator(device="cuda").manual_seed(sum(tokens))
    bs, W, T = 32, len(lens), sum(tokens)
    mb = -(-max(lens) // bs)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)
    kc, vc, q = rnd(W * mb, Hkv, bs, D), rnd(W * mb, Hkv, bs, D), rnd(1, T, Hq, D)
    table = torch.randperm(W * mb, generator=g, device="cuda").to(torch.int32).reshape(W, mb)
    cu = torch.tensor([sum(tokens[:w]) for w in range(W + 1)], dtype=torch.int32, device="cuda")
    pos = torch.cat([torch.arange(n - t, n, dtype=torch.int32) for t, n in zip(tokens, lens)]).cuda()
    frag = torch.tensor([lens], dtype=torch.int32, device="cuda")
    out, lse = torch.full((T, Hq, D), 7.0, dtype=dtype, device="cuda"), torch.full((T, Hq), 7.0, device="cuda")
    pr = _lib.PagedProblem(q=q, locations=pos[None].contiguous(), fragment_lengths=frag, key_cache=kc, value_cache=vc, block_table=table, scale=D ** -0.5,
                           out=out, lse=lse, cu_seqlens_q=cu)
    need = pr.workspace_bytes()
    space = torch.full((need + 4096,), 165, dtype=torch.uint8, device="cuda")
    pr.set_workspace(space[:need])
    pr.run()
    assert bool((space[need:] == 165).all())
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for w in range(W):
        n, rows = lens[w], slice(int(cu[w]), int(cu[w + 1]))
        blocks = table[w, : -(-n // bs)].long()
        k, v = (c[blocks].transpose(1, 2).reshape(-1, Hkv, D)[:n].double() for c in (kc, vc))
        hidden = torch.arange(n, device="cuda")[None] > pos[rows][:, None]
        for h in range(Hq):
            kh, vh = k[:, h // (Hq // Hkv)], v[:, h // (Hq // Hkv)]
            x = (q[0, rows, h].double() @ kh.t().contiguous() * D ** -0.5).masked_fill(hidden, float("-inf"))
            p = torch.softmax(x, dim=1)
            ref = p @ vh
            bound = (u + 2.0 ** -16) * (p @ vh.abs()) + u * ref.abs() + (2.0 ** -25 * vh.abs().sum(0) if dtype == torch.float16 else 0.0)
            assert bool(((out[rows, h].double() - ref).abs() <= bound).all())
            assert bool(((lse[rows, h].double() - torch.logsumexp(x, dim=1)).abs() <= 1e-4).all())
