"""Host-side generation plumbing on the CPU: the trimmable sliding-window cache
(``tests/test_spec_cache.py:18-38`` of the reference), the rotating window cache under chunked
updates, and the greedy loop over plain bf16 caches. The HIP paths are in test_gpu_model.py."""
import numpy as np
import pytest
import torch

from lagunalab_amd.cache import (KVCache, RotatingKVCache, TrimmableWindowCache,
                                 make_quantized_cache, make_trimmable_cache)
from lagunalab_amd.generate import generate_greedy
from tiny_model import TinyLM


@pytest.fixture(scope="module")
def model():
    return TinyLM(lm_head_scale=1.0, attn_dtype=torch.float32)


def _ids(n, seed=4, vocab=1024):
    return torch.tensor(np.random.default_rng(seed).integers(0, vocab, size=(1, n)))


def _cache(model):
    # slack 4 with window 8, so truncation happens constantly in a 30-token run
    return [TrimmableWindowCache(8, slack=4) if isinstance(c, TrimmableWindowCache) else c
            for c in make_trimmable_cache(model)]


def _chunks(n0=13, n=30):
    return [(0, 5), (5, 12), (12, n0)] + [(i, i + 1) for i in range(n0, n)]


@torch.no_grad()
def test_decode_matches_full_forward_with_truncation(model):
    ids = _ids(30)
    full = model(ids)
    cache = _cache(model)
    outs = [model(ids[:, a:b], cache=cache) for a, b in _chunks()]
    torch.testing.assert_close(torch.cat(outs, dim=1), full, atol=1e-4, rtol=1e-3)
    assert cache[1].keys.shape[2] <= 8 + 4 + 1 and cache[1].offset == 30


@torch.no_grad()
def test_trim_after_window_wrap_forgets_rejected_tokens(model):
    ids = _ids(30)
    full = model(ids)
    cache = _cache(model)
    model(ids[:, :20], cache=cache)
    model(_ids(5, seed=99), cache=cache)  # a rejected draft block
    for c in cache:
        assert c.trim(5) == 5
    out = model(ids[:, 20:], cache=cache)
    torch.testing.assert_close(out, full[:, 20:], atol=1e-4, rtol=1e-3)


def test_trim_is_clamped_to_stored_rows():
    c = TrimmableWindowCache(4, slack=2)
    k = torch.randn(1, 2, 3, 16)
    c.update_and_fetch(k, k)
    assert c.trim(10) == 3 and c.offset == 0 and c.keys.shape[2] == 0
    assert c.trim(1) == 0


@torch.no_grad()
def test_rotating_window_cache_matches_full_forward(model):
    """Sliding layers of the quantized cache keep only the window; chunked prefill followed by
    single-token steps equals the full forward pass."""
    ids = _ids(30, seed=7)
    full = model(ids)
    cache = [RotatingKVCache(8) if lt == "sliding_attention" else KVCache()
             for lt in model.args.layer_types]
    outs = [model(ids[:, a:b], cache=cache) for a, b in [(0, 11), (11, 20), (20, 23)] +
            [(i, i + 1) for i in range(23, 30)]]
    torch.testing.assert_close(torch.cat(outs, dim=1), full, atol=1e-4, rtol=1e-3)


def test_quantized_cache_factory_layout(model):
    cache = make_quantized_cache(model, 8, fused_decode=True)
    kinds = [type(c).__name__ for c in cache]
    assert kinds == ["DequantKVCache", "RotatingKVCache", "DequantKVCache"]
    assert all(c.fused_decode for c in cache if hasattr(c, "fused_decode"))
    cache = make_quantized_cache(model, 8, fused_decode=True, trim_slack=8)
    assert isinstance(cache[1], TrimmableWindowCache) and cache[1].slack == 8
    assert all(c.is_trimmable() for c in cache)


@torch.no_grad()
def test_greedy_plain_cache_equals_recompute(model):
    """The cached greedy loop equals re-running the whole sequence every step."""
    prompt = [int(t) for t in _ids(9, seed=3)[0]]
    got = generate_greedy(model, prompt, 6)
    ids = list(prompt)
    for _ in range(6):
        ids.append(int(torch.argmax(model(torch.tensor([ids]))[0, -1])))
    assert got == ids[len(prompt):]


@torch.no_grad()
def test_greedy_stops_at_eos(model):
    prompt = [int(t) for t in _ids(9, seed=3)[0]]
    free = generate_greedy(model, prompt, 6)
    got = generate_greedy(model, prompt, 6, eos=(free[2],))
    assert got == free[:free.index(free[2]) + 1]


def test_pending_rows_behave_as_the_tuple_of_views():
    """The tuple of a fused step makes its views on first use: every Python-level way of reading it
    completes the append first and gives the views of the step's own buffers and length, also after the cache has
    grown or been trimmed."""
    import copy
    from lagunalab_amd.cache import _PendingRows

    class Cache:
        flushed = 0

        def _flush(self):
            self.flushed += 1

    bufs = tuple(torch.arange(24.).reshape(1, 2, 4, 3) + i for i in range(3))
    want = tuple(t[:, :, :3] for t in bufs)
    same = lambda a, b: len(a) == len(b) and all(torch.equal(x, y) for x, y in zip(a, b))  # noqa: E731
    reads = [tuple, list, lambda p: [p[0], p[1], p[-1]], lambda p: [*p], lambda p: p[:],
             lambda p: (lambda *a: a)(*p), lambda p: list(reversed(p))[::-1], lambda p: p + (),
             lambda p: () + p, lambda p: p * 1, copy.copy, lambda p: (lambda a, b, c: (a, b, c))(*p)]
    for read in reads:
        c = Cache()
        p = _PendingRows(bufs, 3, c)
        assert isinstance(p, tuple) and len(p) == 3 and c.flushed == 0
        assert same(read(p), want) and c.flushed > 0
    p = _PendingRows(bufs, 3, Cache())
    assert p == p and p[0] is p[0] and p[0] in p and p.index(p[0]) == 0 and hash(p) == hash(tuple(p))
    assert "tensor" in repr(p)
    # ordering compares the views (here the first ones, of one value each), on either side
    ones = tuple(torch.full((1, 1, 4, 1), float(i)) for i in range(3))
    more = (ones[0][:, :, :1] + 1,) + ones[1:]
    for cmp in (lambda a: a < more, lambda a: a <= more, lambda a: more > a, lambda a: more >= a):
        c = Cache()
        assert cmp(_PendingRows(ones, 1, c)) and c.flushed > 0
    for cmp in (lambda a: a > more, lambda a: a >= more, lambda a: more < a, lambda a: more <= a):
        c = Cache()
        assert not cmp(_PendingRows(ones, 1, c)) and c.flushed > 0
    # what a tuple's C readers need
    c = Cache()
    assert torch.cat(tuple(_PendingRows(bufs, 3, c)), -1).shape == (1, 2, 3, 9) and c.flushed > 0
