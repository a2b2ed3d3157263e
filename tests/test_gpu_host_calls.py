"""The native host path of the ops (csrc/host_calls.cpp) against the Python code it stands in for: the same results bit for bit for every
form of call it takes, and the same answers for the calls it leaves alone."""
import pytest
import torch

import paraattention_amd  # noqa: F401
from oracle import inputs
from paraattention_amd import _lib, ops

pytestmark = pytest.mark.gpu
NS = torch.ops.para_attn


def _flat(x):
    if isinstance(x, torch.Tensor):
        return [x]
    return [t for y in x for t in _flat(y)]


def _both(monkeypatch, call):
    taken = []

    def watched(name, device, *args):
        res = native(name, device, *args)
        taken.append(res is not None)
        return res

    native = ops._native
    monkeypatch.setattr(ops, "_native", watched)
    a = _flat(call())
    monkeypatch.setattr(ops, "_native", lambda *args: None)
    b = _flat(call())
    monkeypatch.undo()
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride() and torch.equal(x, y)
    return all(taken) and bool(taken)


def _heads(B, H, S, D, dtype, layout):
    t = torch.randn((B, S, H, D) if layout == "bshd" else (B, H, S, D), generator=torch.Generator().manual_seed(S + D)).to(dtype).cuda()
    return t.transpose(1, 2) if layout == "bshd" else t


@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("D", [64, 128, 72, 40])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_attention_calls(cuda, monkeypatch, dtype, D, layout):
    B, H, Sq, Skv = 2, 3, 200, 333
    q, k, v = _heads(B, H, Sq, D, dtype, layout), _heads(B, H, Skv, D, dtype, layout), _heads(B, H, Skv, D, dtype, layout)
    for kw in ({}, {"is_causal": True}, {"scale": 0.25}):
        assert _both(monkeypatch, lambda: NS.attention_forward_with_lse(q, k, v, **kw))
        assert _both(monkeypatch, lambda: NS.attention_forward(q, k, v, **kw))
    g = torch.Generator().manual_seed(1)
    keep = torch.rand(B, 1, 1, Skv, generator=g).cuda() < 0.7
    masks = [keep, keep[0, 0, 0], torch.rand(Sq, Skv, generator=g).cuda() < 0.7, torch.randn(H, 1, Skv, generator=g).cuda(),
             torch.randn(1, H, Sq, Skv, generator=g).to(dtype).cuda(), torch.randn(B, 1, Skv, Sq, generator=g).cuda().transpose(2, 3)]
    for m in masks:
        assert _both(monkeypatch, lambda: NS.attention_forward_with_lse(q, k, v, m)) == (D in (64, 128))
    assert _both(monkeypatch, lambda: NS.attention_forward_sparse_kv(q, k, v, keep)) == (D in (64, 128))
    assert _both(monkeypatch, lambda: NS.attention_forward_sparse_kv(q, k, v))


def test_attention_calls_it_leaves_alone(cuda, monkeypatch):
    q, k, v = (t.cuda() for t in inputs.qkv(1, 2, 64, 96, 128, seed=1))
    odd = torch.randn(1, 2, 64, 129, device=cuda).bfloat16()[..., 1:]  # rows that start off 16 bytes: copied first
    cut = torch.randn(1, 2, 64, 256, device=cuda).bfloat16()[..., ::2]
    for x in (odd, cut):
        assert not _both(monkeypatch, lambda: NS.attention_forward_with_lse(x, k, v))
    assert not _both(monkeypatch, lambda: NS.attention_forward(q, k, v[..., :80]))  # values narrower than the keys
    assert not _both(monkeypatch, lambda: NS.attention_forward(q, k, v, torch.zeros(64, 96, dtype=torch.float64, device=cuda)))
    assert not _both(monkeypatch, lambda: NS.attention_forward(q[:, :, :0], k, v))
    assert not _both(monkeypatch, lambda: NS.attention_forward_with_lse(q, k[:, :, :0], v[:, :, :0]))
    for bad in (lambda: NS.attention_forward(q, k.half(), v), lambda: NS.attention_forward(q.float(), k.float(), v.float()),
                lambda: NS.attention_forward(q, k, v, dropout_p=0.1), lambda: NS.attention_forward(q, k, v, torch.ones(64, 96, device=cuda), is_causal=True),
                lambda: NS.attention_forward(q, k, v, torch.ones(63, 96, dtype=torch.bool, device=cuda)),
                lambda: NS.attention_forward(q, k, v, torch.ones(64, 96, dtype=torch.int32, device=cuda)),
                lambda: NS.attention_forward(q, k, v, scale=-1.0), lambda: NS.attention_forward(q[0], k[0], v[0]),
                lambda: NS.attention_forward(q, k[:, :1], v[:, :1])):
        with pytest.raises((ValueError, NotImplementedError)):
            bad()


def test_block_sparse_cache_and_taylorseer_calls(cuda, monkeypatch):
    q, k, v = (t.cuda() for t in inputs.qkv(1, 2, 256, 384, 128, seed=2))
    for bm in (torch.tensor([[True, False, True], [False, True, True]]), torch.rand(2, 2, 3) < 0.5):
        assert _both(monkeypatch, lambda: NS.attention_forward_block_sparse(q, k, v, bm.cuda()))
    assert not _both(monkeypatch, lambda: NS.attention_forward_block_sparse(q, k, v, torch.ones(2, 2, dtype=torch.bool, device=cuda), 0, 200, 0, 300))
    for dtype in (torch.bfloat16, torch.float16, torch.float32):
        a, b, c, d = (torch.randn(2, 50, 64, device=cuda).to(dtype) for _ in range(4))
        t, r = torch.randn(2, 7, 64, device=cuda).to(dtype), torch.randn(2, 7, 64, device=cuda).to(dtype)
        assert _both(monkeypatch, lambda: NS.fbcache_first_residual_diff(a, b, None))
        assert _both(monkeypatch, lambda: NS.fbcache_first_residual_diff(a, b, c))
        assert _both(monkeypatch, lambda: NS.fbcache_first_residual_diff_strided(a, b, c[..., ::2].contiguous(), 2))
        assert _both(monkeypatch, lambda: NS.fbcache_apply_residual(a, b))
        assert _both(monkeypatch, lambda: NS.fbcache_apply_residual_pair(a, b, t, r))
        assert _both(monkeypatch, lambda: NS.taylorseer_derivatives(a, [b, c], 3.0))
        for elapsed in (0, 1, 7, -3):
            assert _both(monkeypatch, lambda: NS.taylorseer_value([a, b, c], elapsed, d))
        assert _both(monkeypatch, lambda: NS.taylorseer_value([a], 2))
        # what is not contiguous is copied by the general path
        assert not _both(monkeypatch, lambda: NS.fbcache_apply_residual(a.transpose(0, 1), b.transpose(0, 1)))
        assert not _both(monkeypatch, lambda: NS.taylorseer_value([a.transpose(0, 1), b.transpose(0, 1)], 2))
        with pytest.raises(ValueError):
            NS.fbcache_apply_residual(a, t)


def test_a_library_error_becomes_the_ops_exception(cuda):
    q, k, v = (t.cuda() for t in inputs.qkv(1, 1, 16, 16, 64, seed=3))
    with pytest.raises(NotImplementedError, match="scale"):
        NS.attention_forward(q, k, v, scale=0.0)
    assert _lib.host_calls().attention(q.cpu(), k, v, None, None, False, False, 0) is None


def test_the_ops_run_without_the_module(cuda, monkeypatch):
    q, k, v = (t.cuda() for t in inputs.qkv(1, 2, 64, 96, 128, seed=4))
    want = NS.attention_forward_with_lse(q, k, v)
    monkeypatch.setattr(_lib, "_host", False)  # what host_calls() leaves where the module cannot be used
    got = NS.attention_forward_with_lse(q, k, v)
    assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])
