"""GPU: several tokens appended to a KIVI cache in one launch, and the fp16 view,
bit for bit against the general path (the separate writers, and torch's
unpacking and concatenation for the view), through the cache classes."""
from __future__ import annotations

import types

import pytest
import torch

from llmik_cuda import kv_cache as kvc

pytestmark = pytest.mark.gpu


def _general(monkeypatch):
    monkeypatch.setattr(kvc, "_C", types.SimpleNamespace(kivi_append_int4=lambda *a: None))


@pytest.fixture
def launches(monkeypatch):
    """Whether the one-launch path took each call that the cache classes made of it."""
    taken, real = [], kvc._C.kivi_append_int4

    def count(*args):
        out = real(*args)
        taken.append(out is not None)
        return out

    monkeypatch.setattr(kvc, "_C", types.SimpleNamespace(kivi_append_int4=count))
    return taken


def _tokens(cuda, B, H, n, seed, special=False):
    g = torch.Generator(device=cuda).manual_seed(seed)
    x = torch.randn((B, H, n, 128), generator=g, device=cuda, dtype=torch.float16)
    if special:
        x[0, 0, 0, 3] = float("nan")
        x[-1, -1, n // 2, 7] = float("inf")
        x[0, -1, n - 1] = 0.0
        x[-1, 0, n // 3, 64] = -float("inf")
    return x


def _bits(t):
    return t.contiguous().view(torch.int16) if t.dtype == torch.float16 else t


def _equal(a, b, nan_payload=True):
    if not nan_payload:
        both = a.isnan() & b.isnan()
        a, b = a.masked_fill(both, 0), b.masked_fill(both, 0)
    return torch.equal(_bits(a), _bits(b))


# group size and appends; a group is left open, filled exactly, filled and
# another opened (two launches), skipped over, and grown token by token.
SEQUENCES = [
    (32, [100, 1, 1, 30, 64, 3, 61]),
    (32, [32, 31, 33, 2, 95]),
    (16, [5, 11, 5, 12, 200]),
    (48, [47, 2, 48, 96, 5]),
    (64, [1, 62, 2, 130, 61, 64]),
    (128, [127, 2, 300, 83, 129]),
    (1, [3, 7]),
    (20, [19, 2, 60, 38, 3]),
]


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("g,appends", SEQUENCES, ids=[f"g{s[0]}" for s in SEQUENCES])
def test_appends_and_views_equal_the_general_path(llmik, cuda, monkeypatch, launches, g, appends, special):
    from llmik_cuda.hf import KIVILayer
    B, H, max_len = 2, 3, sum(appends) + 5

    def run():
        layer, plain = KIVILayer(max_len, g), kvc.Int4KIVICache(B, H, max_len, g, device=cuda)
        views = []
        for i, n in enumerate(appends):
            k, v = _tokens(cuda, B, H, n, 2 * i, special), _tokens(cuda, B, H, n, 2 * i + 1, special)
            views.append(layer.update(k, v) if n > 1 else (layer.update(k, v), layer.fp16_view())[1])
            views.append(layer.fp16_view())
            # a token slice of a longer buffer
            long_k, long_v = _tokens(cuda, B, H, n + 9, 90), _tokens(cuda, B, H, n + 4, 91)
            long_k[:, :, 2:2 + n], long_v[:, :, 1:1 + n] = k, v
            plain.append(long_k[:, :, 2:2 + n], long_v[:, :, 1:1 + n])
        torch.cuda.synchronize()
        return layer, plain, views

    layer, plain, views = run()
    # layer updates and plain appends of several tokens, and the other views
    assert launches == [True] * (2 * len(appends) + sum(n > 1 for n in appends))
    _general(monkeypatch)
    layer0, plain0, views0 = run()
    for a, b in ((layer.cache, layer0.cache), (plain, plain0)):
        r = a.length % g
        assert a.length == b.length == sum(appends)
        for name in ("k_q", "k_scale", "v_q", "v_scale"):
            assert _equal(getattr(a, name), getattr(b, name)), name
        assert _equal(a.k_open[:, :, :r], b.k_open[:, :, :r])
    assert _equal(layer.v_open[:, :, :layer.cache.length % g], layer0.v_open[:, :, :layer.cache.length % g])
    for (k, v), (k0, v0) in zip(views, views0):
        assert k.shape == k0.shape and k.is_contiguous() and v.is_contiguous()
        assert _equal(k, k0, nan_payload=False) and _equal(v, v0, nan_payload=False)


@pytest.mark.parametrize("g,n", [(128, 700), (100, 301), (64, 513), (33, 100)])
def test_many_rows(llmik, cuda, monkeypatch, launches, g, n):
    """More workgroups than CUs: the other workgroup size of groups above 64."""
    k, v = _tokens(cuda, 8, 9, n, 5), _tokens(cuda, 8, 9, n, 6)
    caches = []
    for general in (False, True):
        if general:
            _general(monkeypatch)
        c = kvc.Int4KIVICache(8, 9, n + 1, g, device=cuda)
        c.append(k, v)
        caches.append(c)
    assert launches == [True]
    a, b = caches
    for name in ("k_q", "k_scale", "v_q", "v_scale"):
        assert torch.equal(getattr(a, name), getattr(b, name)), name
    assert torch.equal(a.k_open[:, :, :n % g], b.k_open[:, :, :n % g])


def test_nothing_past_the_live_length_is_written(llmik, cuda, launches):
    cache = kvc.Int4KIVICache(2, 2, 200, 32, device=cuda)
    for t in (cache.k_q, cache.v_q):
        t.fill_(77)
    for t in (cache.k_scale, cache.v_scale):
        t.fill_(7.0)
    cache.append(_tokens(cuda, 2, 2, 70, 1), _tokens(cuda, 2, 2, 70, 2))
    assert launches == [True]
    assert bool((cache.k_q[:, :, 70:] == 77).all()) and bool((cache.v_q[:, :, 70:] == 77).all())
    assert bool((cache.k_scale[:, :, 3:] == 7).all()) and bool((cache.v_scale[:, :, 70:] == 7).all())


def test_rows_the_launch_does_not_take(llmik, cuda, launches):
    """Odd strides and addresses keep the general path's answer: K tokens that
    only fill the open group may have any strides; V may not, nor may either
    be misaligned where a writer reads it."""
    k, v = _tokens(cuda, 2, 2, 5, 1), _tokens(cuda, 2, 2, 5, 2)
    want = kvc.Int4KIVICache(2, 2, 64, 32, device=cuda)
    want.append(k, v)
    kt = k.transpose(2, 3).contiguous().transpose(2, 3)
    got = kvc.Int4KIVICache(2, 2, 64, 32, device=cuda)
    got.append(kt, v)
    assert torch.equal(got.k_q, want.k_q) and torch.equal(got.k_scale, want.k_scale)
    with pytest.raises(RuntimeError):
        got.append(k, v.transpose(2, 3).contiguous().transpose(2, 3))
    flat = torch.zeros(v.numel() + 4, dtype=torch.float16, device=cuda)
    odd = flat[4:].view(v.shape)   # 8 bytes past a 16-byte boundary
    with pytest.raises(RuntimeError):
        kvc.Int4KIVICache(2, 2, 64, 32, device=cuda).append(k, odd)
    assert launches == [True, False, False, False]


def _layer_run(cuda, record):
    """Two prefill chunks through a layer; the views and what autograd says of them."""
    from llmik_cuda.hf import KIVILayer
    layer = KIVILayer(128, 32)
    ks, vs = [], []
    for i, n in enumerate((45, 40)):   # 13 tokens open, then 21
        ks.append(_tokens(cuda, 2, 2, n, 2 * i))
        vs.append(_tokens(cuda, 2, 2, n, 2 * i + 1))
    return layer, ks, vs, record(layer, ks, vs)


def test_gradients_of_the_open_group(llmik, cuda, launches):
    """The views hold the open group's tokens themselves: their gradient is the
    view's, the quantised tokens' is zero, as through the general path."""
    def record(layer, ks, vs):
        for t in ks + vs:
            t.requires_grad_(True)
        for k, v in zip(ks, vs):
            view_k, view_v = layer.update(k, v)
        assert view_k.requires_grad and view_v.requires_grad
        w = torch.arange(1, 86, device=cuda, dtype=torch.float16)[:, None] / 64
        ((view_k * w).sum() + 2 * (view_v * w).sum()).backward()
        return w, layer.fp16_view()

    layer, ks, vs, (w, later) = _layer_run(cuda, record)
    for t, f in ((ks[1], 1), (vs[1], 2)):
        want = torch.zeros_like(t)
        want[:, :, -21:] = f * w[-21:]
        assert torch.equal(t.grad, want)
    assert all(t.grad is None or not t.grad.any() for t in (ks[0], vs[0]))
    with torch.no_grad():
        a, b = layer.fp16_view()
    assert launches and not any(launches[:-1]) and launches[-1]   # the launch again without gradients
    assert not a.requires_grad and torch.equal(a, later[0]) and torch.equal(b, later[1])


def test_forward_mode_tangents_of_the_open_group(llmik, cuda):
    import torch.autograd.forward_ad as fw

    def record(layer, ks, vs):
        with fw.dual_level():
            for k, v in zip(ks, vs):
                views = layer.update(fw.make_dual(k, torch.ones_like(k)), fw.make_dual(v, 2 * torch.ones_like(v)))
            return [fw.unpack_dual(t).tangent for t in views]

    *_, tangents = _layer_run(cuda, record)
    for t, f in zip(tangents, (1, 2)):
        assert bool((t[:, :, -21:] == f).all()) and not bool(t[:, :, :-21].any())


def test_capture_and_replay(llmik, cuda, launches):
    k, v = _tokens(cuda, 2, 4, 90, 1), _tokens(cuda, 2, 4, 90, 2)
    eager = kvc.Int4KIVICache(2, 4, 128, 32, device=cuda)
    eager.append(k, v)
    cache = kvc.Int4KIVICache(2, 4, 128, 32, device=cuda)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        cache.append(k, v)
    assert launches == [True, True]
    for _ in range(3):
        cache.k_q.zero_()
        cache.v_scale.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(cache.k_q, eager.k_q) and torch.equal(cache.v_scale, eager.v_scale)
