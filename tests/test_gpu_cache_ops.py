"""cab_kv_append and cab_key_sums: the appended rows bit for bit whatever the
strides, alignment and element size, and the sums against torch in float64."""

import ctypes

import pytest
import torch

from cab_attention import _native as nat

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,n,D,layout", [
    (1, 8, 1, 128, "plain"),        # a decode step: 16-byte units
    (2, 3, 300, 64, "plain"),
    (1, 2, 5, 20, "plain"),         # rows of no whole 16 bytes (bf16), padded buffer
    (2, 4, 33, 128, "transposed"),  # [B, n, H, D] as a projection leaves it
    (1, 2, 7, 64, "strided"),       # last-dim stride 2
    (1, 2, 9, 64, "offset"),        # rows one element past a 16-byte boundary
    (1, 1, 1, 1, "plain"),
    (1, 8, 1100, 128, "offset"),    # off 16-byte boundaries and long: torch's copies
])
def test_append_matches_copy(cuda, dt, B, H, n, D, layout):
    from cab_attention.cache.store import LayeredKV
    g = torch.Generator().manual_seed(n + D)

    def make():
        if layout == "transposed":
            return torch.randn((B, n, H, D), generator=g).to(dt).to(cuda).transpose(1, 2)
        if layout == "strided":
            return torch.randn((B, H, n, 2 * D), generator=g).to(dt).to(cuda)[..., ::2]
        if layout == "offset":
            flat = torch.randn(B * H * n * D + 1, generator=g).to(dt).to(cuda)
            return flat[1:].view(B, H, n, D)
        return torch.randn((B, H, n, D), generator=g).to(dt).to(cuda)

    store, want_k, want_v = LayeredKV(initial_capacity=4), [], []
    for _ in range(3):  # the later ones grow the buffers
        k, v = make(), make().contiguous()  # (K and V strides differ)
        store.append(0, k, v)
        want_k.append(k)
        want_v.append(v)
    got_k, got_v = store.view(0)
    assert torch.equal(got_k, torch.cat(want_k, 2)) and torch.equal(got_v, torch.cat(want_v, 2))


@gpu
def test_append_keeps_gradients_to_torch(cuda):
    from cab_attention.cache.store import LayeredKV
    store = LayeredKV()
    k = torch.randn((1, 2, 3, 64), device=cuda, requires_grad=True)
    store.append(0, k, k.detach())
    store.view(0)[0].sum().backward()
    assert torch.equal(k.grad, torch.ones_like(k))


@gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Nq,Nk,n_old", [(1, 32, 1, 2000, 1999), (1, 32, 16, 4500, 0),
                                             (2, 3, 7, 63, 63), (1, 1, 1, 1, 0), (2, 8, 9, 65, 200)])
def test_importance_update(cuda, dt, B, H, Nq, Nk, n_old):
    from cab_attention.scoring import ImportanceTracker
    g = torch.Generator(device=cuda).manual_seed(Nk)
    full = torch.softmax(torch.randn((B, H, Nq, Nk + 3), generator=g, device=cuda), -1).to(dt)
    w = full[..., :Nk]  # rows of a longer buffer
    t = ImportanceTracker(device="cuda")
    base = torch.zeros(max(n_old, Nk), dtype=torch.float64, device=cuda)
    if n_old:
        t.cumulative_scores = torch.rand(n_old, generator=g, device=cuda)
        base[:n_old] = t.cumulative_scores.double()
    before = t.cumulative_scores
    t.update(w)
    got = t.get_scores()
    assert (got is before) == (n_old >= Nk) and t.total_queries == Nq
    base[:Nk] += w.double().sum((0, 1, 2))
    # fp32 sums of non-negative terms; 16-bit sums end rounded to their type
    ulp = {torch.float32: 2e-6, torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}[dt]
    torch.testing.assert_close(got.double(), base, rtol=ulp, atol=1e-7)


@gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,Nq,Nk", [(32, 1, 4500), (7, 5, 3000), (32, 16, 4500), (3, 171, 130),
                                     (32, 500, 500), (8, 2000, 130),
                                     (32, 128, 12000), (32, 129, 12000),
                                     (8, 32, 32768), (8, 32, 32769)])
def test_importance_sums_are_as_exact_as_torch(cuda, H, Nq, Nk, dt):
    """Where the kernel sums (few rows, or up to 4096 of 12000 to 24000 keys), the
    fp32 sums' rms relative error against float64 is that of a tree of additions: a rounding
    is uniform within half an ulp, rms 0.4 * 2^-24 of the sum (over mantissas),
    and a tree's levels add their variances halved each time, 2 in all: 3.4e-8;
    the eight-row steps of a wave in sequence (32 at most, in each of 16 waves: 2/3
    more) make it 3.9e-8, and 5.2e-8 is allowed. 16 terms in sequence alone would
    give sqrt(16 / 3) * 0.4 * 2^-24 = 5.5e-8. The rest is torch's sum."""
    from cab_attention.scoring import ImportanceTracker
    g = torch.Generator(device=cuda).manual_seed(Nk)
    w = torch.softmax(torch.randn((1, H, Nq, Nk), generator=g, device=cuda), -1).to(dt)
    t = ImportanceTracker(device="cuda")
    t.update(w)
    if (H, Nq, Nk) in [(32, 500, 500), (8, 2000, 130), (32, 129, 12000), (8, 32, 32769)]:
        assert torch.equal(t.get_scores(), w.sum((0, 1, 2)).float())
        return
    want = w.double().sum((0, 1, 2))
    if dt == torch.float32:
        rel = (t.get_scores().double() - want) / want
        assert float(rel.pow(2).mean().sqrt()) <= 5.2e-8
    else:  # rounded to 8 significant bits: at most 2^-8 of it, plus the fp32 sum's error
        assert bool(((t.get_scores().double() - want).abs() <= want * (2.0 ** -8 + 1e-6)).all())


def _negated(shape, dtype, cuda, g):
    """A tensor that stands for the negated values of its memory."""
    z = torch.randn((*shape, 2), generator=g).to(dtype).to(cuda)
    x = torch._neg_view(z[..., 0].contiguous())
    assert x.is_neg() and type(x) is torch.Tensor
    return x


@gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_negated_views_keep_their_sign(cuda, dt):
    from cab_attention.cache.store import LayeredKV
    from cab_attention.scoring import ImportanceTracker
    g = torch.Generator().manual_seed(3)
    k, v, w = (_negated((1, 2, 5, 64), dt, cuda, g) for _ in range(3))
    store = LayeredKV()
    store.append(0, k, v)
    assert torch.equal(store.view(0)[0], k.resolve_neg())
    assert torch.equal(store.view(0)[1], v.resolve_neg())
    t = ImportanceTracker(device="cuda")
    t.update(w)
    torch.testing.assert_close(t.get_scores(), w.resolve_neg().sum((0, 1, 2)).float())


@gpu
def test_dispatch_modes_see_the_ops(cuda):
    from torch.utils._python_dispatch import TorchDispatchMode
    from cab_attention.cache.store import LayeredKV
    from cab_attention.scoring import ImportanceTracker

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(func.overloadpacket.__name__)
            return func(*args, **(kwargs or {}))

    names = []
    k, w = torch.rand((1, 2, 3, 64), device=cuda), torch.rand((1, 2, 3, 7), device=cuda)
    with Names():
        LayeredKV().append(0, k, k)
        ImportanceTracker(device="cuda").update(w)
    assert names.count("copy_") == 2 and "sum" in names


@gpu
def test_in_place_writes_are_seen_by_autograd(cuda):
    """What a backward pass has saved and an update then writes over raises, as for
    torch's own in-place ops."""
    from cab_attention.cache.store import LayeredKV
    from cab_attention.scoring import ImportanceTracker
    t = ImportanceTracker(device="cuda")
    w = torch.rand((1, 2, 3, 7), device=cuda)
    t.update(w)
    x = torch.ones(7, device=cuda, requires_grad=True)
    y = (x * t.get_scores()).sum()
    before = t.get_scores()._version
    t.update(w)
    assert t.get_scores()._version > before
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()
    store, k = LayeredKV(), torch.rand((1, 2, 3, 64), device=cuda)
    store.append(0, k, k)
    kept = store.view(0)
    before = [s._version for s in kept]
    store.append(0, k, k)
    assert all(s._version > b for s, b in zip(kept, before))


@gpu
def test_inference_tensors_stay_closed_outside_inference_mode(cuda):
    from cab_attention.cache.store import LayeredKV
    from cab_attention.scoring import ImportanceTracker
    t, store = ImportanceTracker(device="cuda"), LayeredKV()
    w, k = torch.rand((1, 2, 3, 7), device=cuda), torch.rand((1, 2, 3, 64), device=cuda)
    with torch.inference_mode():
        for _ in range(2):
            t.update(w)
            store.append(0, k, k)
    torch.testing.assert_close(t.get_scores(), 2 * w.sum((0, 1, 2)))
    assert store.length(0) == 6
    with pytest.raises(RuntimeError, match="[Ii]nference"):
        t.update(w)
    with pytest.raises(RuntimeError, match="[Ii]nference"):
        store.append(0, k, k)


@gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_importance_update_under_autocast(cuda, dt):
    """Autocast sums in fp32: 16-bit weights' sums are not rounded to their type."""
    from cab_attention.scoring import ImportanceTracker
    g = torch.Generator(device=cuda).manual_seed(4)
    w = torch.softmax(torch.randn((1, 8, 16, 300), generator=g, device=cuda), -1).to(dt)
    t = ImportanceTracker(device="cuda")
    with torch.autocast("cuda", dtype=dt):
        t.update(w)
    want = w.double().sum((0, 1, 2))
    torch.testing.assert_close(t.get_scores().double(), want, rtol=1e-6, atol=0.0)


def test_cache_ops_validation():
    lib = nat.load()
    s = (ctypes.c_int64 * 4)(64, 64, 64, 1)
    bad = (ctypes.c_int64 * 4)(64, 64, 64, 2)
    fake = 0x7f0000000000
    app = lambda **kw: lib.cab_kv_append(  # noqa: E731
        kw.get("k", fake), fake, kw.get("kd", fake), fake, kw.get("es", 2), kw.get("B", 1), 1,
        kw.get("n", 1), 64, s, s, kw.get("ds", s), kw.get("row", 0), None)
    assert app(es=8) == nat.CAB_EDTYPE
    assert app(n=-1) == nat.CAB_ESHAPE and app(row=-1) == nat.CAB_ESHAPE
    assert app(k=None) == nat.CAB_EINVAL
    assert app(ds=bad) == nat.CAB_ESHAPE
    assert app(k=fake + 1) == nat.CAB_ESHAPE
    assert app(B=1 << 40) == nat.CAB_ESHAPE
    assert app(n=0) == nat.CAB_OK
    sums = lambda **kw: lib.cab_key_sums(  # noqa: E731
        kw.get("a", fake), kw.get("dt", nat.CAB_F32), 1, 1, kw.get("Nq", 1), 64, s,
        kw.get("old", None), kw.get("n_old", 0), fake, None)
    assert sums(dt=9) == nat.CAB_EDTYPE
    assert sums(Nq=0) == nat.CAB_ESHAPE
    assert sums(a=None) == nat.CAB_EINVAL
    assert sums(n_old=3) == nat.CAB_EINVAL
