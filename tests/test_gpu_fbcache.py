"""FBCache reduction: the ratio and the hit/miss decision must be bit-exact against the oracle."""
import numpy as np
import pytest
import torch

import paraattention_amd
from paraattention_amd import fbcache
from oracle import fbcache as ofb
from oracle import inputs

pytestmark = pytest.mark.gpu

NAMES = {torch.bfloat16: "bf16", torch.float16: "f16", torch.float32: "f32"}


@pytest.mark.parametrize("shape", [(1,), (7,), (1, 33, 40), (2, 257, 129), (1, 3276, 5120)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("noise", [0.05, 0.2])
def test_ratio_bit_exact(cuda, shape, dtype, noise):
    prev, cur = inputs.fbcache_pair(shape, seed=sum(shape), noise=noise, dtype=dtype)
    want, _, _ = ofb.residual_diff_ratio(prev.float().numpy(), cur.float().numpy(), NAMES[dtype])
    got = torch.ops.para_attn.fbcache_residual_diff(prev.to(cuda), cur.to(cuda))
    assert got.dtype == dtype and got.ndim == 0
    if dtype == torch.float32:
        assert abs(got.item() - want) <= 2e-6 * abs(want)  # fp32 means: summation order differs in the last bits
    else:
        assert got.item() == want
    # called again on the same stream: the workspace must have been left clean
    assert torch.ops.para_attn.fbcache_residual_diff(prev.to(cuda), cur.to(cuda)).item() == got.item()


def test_wan_shape_decision(cuda):
    # the Wan 2.1 shape: bf16 [1,32760,5120] pair, threshold 0.12 -> hit; 0.2 noise -> miss
    prev, cur = inputs.fbcache_pair((1, 32760, 5120), seed=1234, noise=0.05)
    want, md, mt = ofb.residual_diff_ratio(prev.float().numpy(), cur.float().numpy())
    got = torch.ops.para_attn.fbcache_residual_diff(prev.to(cuda), cur.to(cuda)).item()
    assert got == want == 0.050048828125 and (md, mt) == (0.039794921875, 0.796875)
    assert fbcache.are_two_tensors_similar(prev.to(cuda), cur.to(cuda), threshold=0.12) is True
    prev, cur = inputs.fbcache_pair((1, 32760, 5120), seed=1234, noise=0.2)
    want, _, _ = ofb.residual_diff_ratio(prev.float().numpy(), cur.float().numpy())
    assert torch.ops.para_attn.fbcache_residual_diff(prev.to(cuda), cur.to(cuda)).item() == want
    assert fbcache.are_two_tensors_similar(prev.to(cuda), cur.to(cuda), threshold=0.12) is False


def test_known_answers(cuda):
    prev, cur = inputs.fbcache_pair((2, 100, 64), seed=3)
    p = prev.to(cuda)
    assert torch.ops.para_attn.fbcache_residual_diff(p, p).item() == 0.0  # identical -> 0 -> similar
    assert fbcache.are_two_tensors_similar(p, p, threshold=1e-9) is True
    z = torch.zeros_like(p)
    assert torch.ops.para_attn.fbcache_residual_diff(p, z).item() == 1.0  # cur = 0 -> ratio 1
    assert fbcache.are_two_tensors_similar(p, z, threshold=0.12) is False
    assert fbcache.are_two_tensors_similar(p, p, threshold=0.0) is False  # utils.py:222-223
    assert fbcache.are_two_tensors_similar(p, p[:, :50], threshold=0.5) is False  # utils.py:225-226


def test_near_threshold_decisions(cuda):
    # thresholds one bf16 step either side of the computed ratio: strict "<" must flip exactly there
    prev, cur = inputs.fbcache_pair((1, 999, 320), seed=8, noise=0.1)
    ratio, _, _ = ofb.residual_diff_ratio(prev.float().numpy(), cur.float().numpy())
    p, c = prev.to(cuda), cur.to(cuda)
    assert fbcache.are_two_tensors_similar(p, c, threshold=ratio) is False
    assert fbcache.are_two_tensors_similar(p, c, threshold=float(np.nextafter(np.float32(ratio), np.float32(1)))) is True
    assert fbcache.are_two_tensors_similar(p, c, threshold=float(np.nextafter(np.float32(ratio), np.float32(0)))) is False


@pytest.mark.parametrize("k", [2, 3, 4])
def test_downsample_and_gates(cuda, k):
    shape = (1, 300, 512)
    prev_full, cur = inputs.fbcache_pair(shape, seed=k, noise=0.08)
    ctx = fbcache.create_cache_context(residual_diff_threshold=0.12, downsample_factor=k, warmup_steps=1)
    with fbcache.cache_context(ctx):
        ctx.mark_step_begin()  # step 0 = warm-up
        assert fbcache.get_can_use_cache(cur.to(cuda)) is False  # warm-up gate, utils.py:271
        fbcache.set_first_hidden_states_residual(prev_full.to(cuda))
        stored = fbcache.get_first_hidden_states_residual()
        assert stored.shape[-1] == len(range(0, 512, k)) and stored.is_contiguous()
        ctx.mark_step_begin()
        want = ofb.get_can_use_cache(prev_full.float().numpy()[..., ::k], cur.float().numpy(), 0.12, downsample_factor=k)
        assert fbcache.get_can_use_cache(cur.to(cuda)) is want
        # ratio itself on the strided view
        r, _, _ = ofb.residual_diff_ratio(prev_full.float().numpy()[..., ::k], cur.float().numpy()[..., ::k])
        assert torch.ops.para_attn.fbcache_residual_diff(stored, cur.to(cuda)[..., ::k]).item() == r
    ctx2 = fbcache.create_cache_context(residual_diff_threshold=0.12)
    with fbcache.cache_context(ctx2):
        ctx2.mark_step_begin()
        assert fbcache.get_can_use_cache(cur.to(cuda)) is False  # no previous residual, utils.py:280


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_first_block_step(cuda, dtype):
    # residual = hidden - hidden0 fused with the reduction; must equal the two-step form bit for bit
    shape = (1, 777, 520)
    g = torch.Generator().manual_seed(5)
    h0 = torch.randn(shape, generator=g).to(dtype)
    prev = torch.randn(shape, generator=g).to(dtype)
    h = (h0.float() + prev.float() + 0.07 * torch.randn(shape, generator=g)).to(dtype)
    resid_ref = (h - h0)  # torch CPU: rounded to dtype
    want, _, _ = ofb.residual_diff_ratio(prev.float().numpy(), resid_ref.float().numpy(), NAMES[dtype])
    resid, ratio = torch.ops.para_attn.fbcache_first_residual_diff(h.to(cuda), h0.to(cuda), prev.to(cuda))
    assert torch.equal(resid.cpu(), resid_ref) and ratio.item() == want
    resid2, ratio2 = torch.ops.para_attn.fbcache_first_residual_diff(h.to(cuda), h0.to(cuda), None)
    assert torch.equal(resid2.cpu(), resid_ref) and ratio2.item() == float("inf")
    applied = torch.ops.para_attn.fbcache_apply_residual(resid, h.to(cuda))
    assert torch.equal(applied.cpu(), resid_ref + h)
    ctx = fbcache.create_cache_context(residual_diff_threshold=0.12)
    with fbcache.cache_context(ctx):
        r1, hit1 = fbcache.first_block_step(h.to(cuda), h0.to(cuda))
        assert hit1 is False and torch.equal(r1.cpu(), resid_ref)
        fbcache.set_first_hidden_states_residual(prev.to(cuda))
        r2, hit2 = fbcache.first_block_step(h.to(cuda), h0.to(cuda))
        assert hit2 is (want < 0.12)


@pytest.mark.parametrize("n", [4 * 65536 * 8 - 1, 4 * 65536 * 8, 5 * 65536 * 8 + 13, (64 << 20), (64 << 20) + 1])
def test_residual_and_apply_at_the_edges_of_their_loops(cuda, n):
    """Four vectors per thread and step on a full grid (256 workgroups of 256 threads), the step that ends early, a remainder that
    fills no vector, and 128 MiB with and without one: bit for bit what torch gives."""
    g = torch.Generator(device=cuda).manual_seed(n % 1000)
    h, h0, prev = (torch.randn(1, n, generator=g, device=cuda, dtype=torch.bfloat16) for _ in range(3))
    resid, ratio = torch.ops.para_attn.fbcache_first_residual_diff(h, h0, prev)
    assert torch.equal(resid, h - h0)
    assert torch.equal(torch.ops.para_attn.fbcache_apply_residual(resid, h), resid + h)
    if n < 1 << 22:
        want, _, _ = ofb.residual_diff_ratio(prev.float().cpu().numpy(), resid.float().cpu().numpy())
        assert ratio.item() == want


@pytest.mark.parametrize("step", [2, 4, 8])
@pytest.mark.parametrize("shape", [(1, 3, 8), (2, 257, 136), (1, 1500, 1920)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_down_sampled_comparison_in_the_residual_pass(cuda, dtype, shape, step):
    """The residual compared with every step-th column of the previous one in the pass that writes it: residual bit for bit, ratio
    bit for bit in 16 bits (fp32 means differ in the last bits with the order of the sums); 256 threads x 4 vectors x 256 workgroups and less."""
    a, b = inputs.fbcache_pair(shape, seed=sum(shape) + step, noise=0.1, dtype=dtype)
    hidden, prev = a + b, (b + 0.05 * a)[..., ::step].contiguous()
    takes = paraattention_amd.ops.strided_residual_takes(hidden, prev, step)
    assert takes == (shape[-1] % step == 0 and not (step == 8 and dtype == torch.float32))
    if not takes:
        with pytest.raises(NotImplementedError):
            torch.ops.para_attn.fbcache_first_residual_diff_strided(hidden.to(cuda), a.to(cuda), prev.to(cuda), step)
        return
    resid, ratio = torch.ops.para_attn.fbcache_first_residual_diff_strided(hidden.to(cuda), a.to(cuda), prev.to(cuda), step)
    want = hidden - a
    assert torch.equal(resid.cpu(), want)
    want_ratio, _, _ = ofb.residual_diff_ratio(prev.float().numpy(), want[..., ::step].contiguous().float().numpy(), NAMES[dtype])
    if dtype == torch.float32:
        assert abs(ratio.item() - want_ratio) <= 2e-6 * abs(want_ratio)
    else:
        assert ratio.item() == want_ratio
    again = torch.ops.para_attn.fbcache_first_residual_diff_strided(hidden.to(cuda), a.to(cuda), prev.to(cuda), step)
    assert again[1].item() == ratio.item()  # the workspace was left clean


@pytest.mark.parametrize("sizes", [((1, 1, 1), (1, 1, 3)), ((1, 2000, 1920), (1, 7, 1920)), ((1, 5, 64), (2, 900, 520)), ((1, 333, 77), (1, 512, 77))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_both_streams_in_one_launch(cuda, dtype, sizes):
    """fbcache_apply_residual_pair against two eager additions: sizes that leave one workgroup to either tensor, ragged ends."""
    g = torch.Generator().manual_seed(5)
    ts = [torch.randn(s, generator=g).to(dtype).to(cuda) for s in (sizes[0], sizes[0], sizes[1], sizes[1])]
    out, out2 = torch.ops.para_attn.fbcache_apply_residual_pair(*ts)
    assert torch.equal(out, ts[0] + ts[1]) and torch.equal(out2, ts[2] + ts[3])


def test_residual_without_a_previous_one(cuda):
    a, b = (t.to(cuda) for t in inputs.fbcache_pair((2, 100, 61), seed=9))
    resid, ratio = torch.ops.para_attn.fbcache_first_residual_diff(a, b, None)
    assert torch.equal(resid, a - b) and ratio.item() == float("inf")
