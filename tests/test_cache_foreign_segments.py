"""Segments that are only read may be any object with the members the reference uses of its caches (get_seq_length,
key_cache[layer], value_cache[layer]; python/hogwild/attention.py:160-181), and a SegmentCache's key_cache / value_cache may be
replaced by another object: HogwildCache hands out what those members give."""
import pytest
import torch

from inference_lib_amd import _lib, cache


class Prompt:
    """Keys and values of a finished prompt, kept by somebody else."""

    def __init__(self, keys, values):
        self.key_cache, self.value_cache = keys, values          # per layer [1, Hkv, n, D]

    def get_seq_length(self, layer_idx=0):
        return self.key_cache[layer_idx or 0].size(2)


class Doubled:
    """A key_cache that computes what it hands out."""

    def __init__(self, inner):
        self.inner = inner

    def __getitem__(self, layer):
        return 2 * self.inner[layer]


def _segment(layers, n, dtype, device, g):
    seg = cache.SegmentCache(layers, 2, 64, 16, dtype=dtype, device=device)
    for b in seg.k + seg.v:
        b.copy_(torch.randn(b.shape, generator=g).to(dtype))
    seg.lengths = [n] * layers
    return seg


def _cache(dtype, device):
    g = torch.Generator().manual_seed(3)
    kv = [[torch.randn((1, 2, 9, 64), generator=g).to(dtype).to(device) for _ in range(2)] for _ in range(2)]
    prompt = Prompt(*kv)
    shared = _segment(2, 5, dtype, device, g)
    own = [_segment(2, 3, dtype, device, g) for _ in range(2)]
    shared.key_cache = Doubled(shared.key_cache)
    inv = (1e4 ** (-torch.arange(32, dtype=torch.float64) / 32)).to(torch.float32).to(device)
    c = cache.HogwildCache([[prompt, shared, own[1], own[0]], [prompt, shared, own[0], own[1]]], inv_freq=inv)
    new = [torch.randn((2, 2, 1, 64), generator=g).to(dtype).to(device) for _ in range(2)]
    return c, prompt, shared, own, new


def _check(c, prompt, shared, own, new):
    for layer in range(2):
        cs = c.update(new[0], new[1], layer)
        for got, of in ((cs.keys, lambda s: s.key_cache[layer]), (cs.values, lambda s: s.value_cache[layer])):
            for t, seg in zip(got, (prompt, shared, own[1], own[0])):
                assert torch.equal(t, of(seg)) and t.dim() == 4
        assert cs.keys[0] is prompt.key_cache[layer] and torch.equal(cs.keys[1], 2 * shared.k[layer][None, :, :5])
        assert [t.size(2) for t in cs.keys] == [9, 5, 4, 4]


def test_read_only_segments_of_another_kind(monkeypatch):
    def append(ks, vs, k_dst, v_dst, dst_len, *, n_new, **kw):
        for w, (k, v, n) in enumerate(zip(k_dst, v_dst, dst_len)):
            k[:, n:n + n_new[w]], v[:, n:n + n_new[w]] = ks[w], vs[w]
    monkeypatch.setattr(_lib, "rope_append", append)
    monkeypatch.setattr(_lib, "build_inputs", lambda *a, **kw: (None, None, None))
    _check(*_cache(torch.float32, "cpu"))


@pytest.mark.gpu
def test_read_only_segments_of_another_kind_on_the_gpu():
    _check(*_cache(torch.bfloat16, "cuda"))
