"""merge_caches in one launch for all layers (hw_merge_segments) against the layer-by-layer path it replaces
(hw_build_inputs + hw_rope_append, themselves compared with the oracle in test_gpu_cache.py): the same arithmetic in the
same order, so keys and values must be equal bit for bit."""
import pytest
import torch

from inference_lib_amd import attention  # noqa: F401  (loads the operators)

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TDT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def segment(layers, Hkv, E, Ev, cap, lens, tdt, seed):
    from inference_lib_amd import cache
    g = torch.Generator().manual_seed(seed)
    seg = cache.SegmentCache(layers, Hkv, E, cap, dtype=tdt, device=DEV, value_head_dim=Ev)
    for b in (seg.k, seg.v):
        for i in range(layers):
            b[i].copy_(torch.randn(tuple(b[i].shape), generator=g).to(tdt))
    seg.lengths = list(lens)
    return seg


def layer_by_layer(target, source, inv, scaling, tdt, mode):
    from inference_lib_amd import _lib
    _, cos, sin = _lib.build_inputs([[target.get_seq_length() + 1]], 1, inv, attention_scaling=scaling,
                                    table_dtype=None if tdt == torch.float32 else tdt)
    cos, sin = cos.reshape(1, 1, -1).to(tdt), sin.reshape(1, 1, -1).to(tdt)
    for layer in range(len(target.k)):
        m = source.lengths[layer]
        target.reserve(layer, m)
        _lib.rope_append(source.k[layer][:, :m].unsqueeze(0), source.v[layer][:, :m].unsqueeze(0), [target.k[layer]], [target.v[layer]],
                         [target.lengths[layer]], cosines=cos, sines=sin, mode=mode)
        target.lengths[layer] += m


@pytest.fixture
def taken(monkeypatch):
    """What the one-launch operator answers: merge_caches falls back silently when it declines."""
    op, answers = torch.ops.libhogatt.merge_segments, []

    def record(*args):
        answers.append(op(*args))
        return answers[-1]
    monkeypatch.setattr(torch.ops.libhogatt, "merge_segments", record)
    return answers


@pytest.mark.parametrize("dtype,E,Ev,rot,table,mode", [
    ("bf16", 128, 128, 128, None, 0), ("bf16", 128, 128, 128, "f32", 0), ("f16", 64, 64, 64, None, 1), ("f32", 64, 64, 64, None, 0),
    ("bf16", 256, 256, 256, None, 1), ("f16", 128, 64, 96, None, 0), ("bf16", 80, 72, 36, None, 0), ("f32", 7, 5, 6, None, 1),
    ("bf16", 33, 33, 0, None, 0)])
def test_all_layers_at_once_equal_layer_by_layer(taken, dtype, E, Ev, rot, table, mode):
    """Layers of different length (0, 1, the edges of a 64-row block, many blocks), more layers than one launch takes, a
    target that has to grow in some layers; chunked and element-wise forms, partial rotary widths."""
    from inference_lib_amd import cache
    tdt = TDT[dtype]
    layers, Hkv = 50, 3
    src_lens = [200] + [(0, 1, 63, 64, 65, 130, 257)[i % 7] for i in range(layers - 1)]
    dst_lens = [41] + [7 * (i % 11) for i in range(layers - 1)]
    inv = (10000.0 ** (-torch.arange(rot // 2, dtype=torch.float64) / max(rot // 2, 1))).to(torch.float32).to(DEV)
    got, want = (segment(layers, Hkv, E, Ev, 256, dst_lens, tdt, 5) for _ in range(2))
    source = segment(layers, Hkv, E, Ev, 300, src_lens, tdt, 6)
    cache.merge_caches(got, source, inv_freq=inv, attention_scaling=1.25, table_dtype=None if table is None else TDT[table], mode=mode)
    layer_by_layer(want, source, inv, 1.25, tdt if table is None else TDT[table], mode)
    torch.cuda.synchronize()
    assert taken == [True]
    assert got.lengths == want.lengths == [a + b for a, b in zip(dst_lens, src_lens)]
    for i in range(layers):
        n = got.lengths[i] if got.k[i].size(1) != 256 else 256        # rows behind the appended ones keep what they held
        assert got.k[i].shape == want.k[i].shape
        assert torch.equal(got.k[i][:, :n], want.k[i][:, :n]) and torch.equal(got.v[i][:, :n], want.v[i][:, :n]), i


def test_layers_of_several_forms_and_a_segment_merged_into_itself(taken):
    """Buffers that are not all of one form go layer by layer; a segment may be appended to itself."""
    from inference_lib_amd import cache
    inv = (10000.0 ** (-torch.arange(32, dtype=torch.float64) / 32)).to(torch.float32).to(DEV)
    segs = []
    for _ in range(2):
        target, source = (segment(2, 2, 64, 64, 100, (20, 20), torch.bfloat16, s) for s in (1, 2))
        for seg, s in ((target, 3), (source, 4)):       # layer 1 has more heads than layer 0
            extra = segment(1, 5, 64, 64, 100, (20,), torch.bfloat16, s)
            seg.k[1], seg.v[1] = extra.k[0], extra.v[0]
        segs.append((target, source))
    cache.merge_caches(segs[0][0], segs[0][1], inv_freq=inv)
    layer_by_layer(segs[1][0], segs[1][1], inv, 1.0, torch.bfloat16, 0)
    one, two = (segment(3, 2, 64, 64, 90, (30, 30, 30), torch.float16, 9) for _ in range(2))
    cache.merge_caches(one, one, inv_freq=inv)
    layer_by_layer(two, two, inv, 1.0, torch.float16, 0)
    torch.cuda.synchronize()
    assert taken == [False, True]
    for a, b in ((segs[0][0], segs[1][0]), (one, two)):
        assert a.lengths == b.lengths
        for i in range(len(a.k)):
            assert torch.equal(a.k[i][:, : a.lengths[i]], b.k[i][:, : b.lengths[i]])
            assert torch.equal(a.v[i][:, : a.lengths[i]], b.v[i][:, : b.lengths[i]])


@pytest.mark.parametrize("Hkv,E,Ev,rot", [(1, 8224, 8, 8200), (65537, 2, 1, 2)])
def test_what_one_launch_does_not_take_goes_layer_by_layer(taken, Hkv, E, Ev, rot):
    """A table row that does not fit the LDS, more kv heads than a grid dimension."""
    from inference_lib_amd import cache
    inv = (10000.0 ** (-torch.arange(rot // 2, dtype=torch.float64) / (rot // 2))).to(torch.float32).to(DEV)
    got, want = (segment(2, Hkv, E, Ev, 8, (3, 1), torch.bfloat16, 5) for _ in range(2))
    source = segment(2, Hkv, E, Ev, 4, (2, 4), torch.bfloat16, 6)
    cache.merge_caches(got, source, inv_freq=inv)
    layer_by_layer(want, source, inv, 1.0, torch.bfloat16, 0)
    assert taken == [False] and got.lengths == want.lengths == [5, 5]
    for i in range(2):
        assert torch.equal(got.k[i], want.k[i]) and torch.equal(got.v[i], want.v[i])


def test_an_unknown_mode_is_refused_as_hogwild_error():
    from inference_lib_amd import _lib, cache
    target, source = (segment(2, 2, 64, 64, 8, (2, 2), torch.bfloat16, s) for s in (1, 2))
    before = [t.clone() for t in target.k + target.v]
    with pytest.raises(_lib.HogwildError) as e:
        cache.merge_caches(target, source, inv_freq=torch.ones(32, device=DEV), mode=7)
    assert e.value.status == -3 and target.lengths == [2, 2] and all(torch.equal(a, b) for a, b in zip(before, target.k + target.v))


def test_layers_in_one_tensor():
    """Anything that yields a layer's buffer by index holds the layers of a segment."""
    from inference_lib_amd import cache
    inv = (10000.0 ** (-torch.arange(32, dtype=torch.float64) / 32)).to(torch.float32).to(DEV)
    got, want = (segment(2, 2, 64, 64, 40, (3, 3), torch.bfloat16, 5) for _ in range(2))
    source = segment(2, 2, 64, 64, 16, (16, 16), torch.bfloat16, 6)
    layer_by_layer(want, source, inv, 1.0, torch.bfloat16, 0)
    source.k, source.v = torch.stack(source.k), torch.stack(source.v)
    cache.merge_caches(got, source, inv_freq=inv)
    assert all(torch.equal(a, b) for a, b in zip(got.k + got.v, want.k + want.v))
