"""The 256-query-row prefill attention (eight waves of two query tiles, direct-to-LDS K / V ring) forced onto
every shape class: causal with and without an offset into a longer key range, non-causal, grouped KV
heads, ragged tails, a device-side key count, strided (packed-QKV) inputs; against the fp32 reference,
repeated (its ring is ordered by counted waits and barriers), and its log-sum-exp feeding the backward."""
import pytest
import torch

from eventgpt_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _rand(*shape, dev, scale=1.0, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed + sum(shape))
    return (torch.randn(*shape, device=dev, generator=g) * scale).to(torch.bfloat16)


@pytest.fixture()
def wide():
    from eventgpt_amd.ops import hip
    hip.raw.attn_enable_wide(2)
    yield hip
    hip.raw.attn_enable_wide(1)


@pytest.mark.parametrize("D,H,Hkv,Sq,Sk,causal", [
    (128, 4, 4, 641, 641, True), (128, 8, 2, 300, 300, True), (128, 2, 2, 129, 700, True), (128, 2, 2, 128, 128, True),
    (64, 16, 16, 577, 577, False), (64, 4, 4, 250, 250, False), (128, 2, 2, 1, 130, True), (64, 2, 2, 130, 259, True),
    (128, 4, 4, 1500, 1500, True), (128, 2, 1, 257, 1000, False), (128, 2, 2, 700, 2300, True),
    (128, 16, 4, 2100, 2100, True), (64, 32, 32, 1100, 1100, False)])    # several blocks a sequence
def test_wide_attention_matches_reference(dev, wide, D, H, Hkv, Sq, Sk, causal):
    B = 2
    q, k, v = _rand(B, Sq, H, D, dev=dev), _rand(B, Sk, Hkv, D, dev=dev, seed=1), _rand(B, Sk, Hkv, D, dev=dev, seed=2)
    rep = H // Hkv
    want = ref.attention(q, k.repeat_interleave(rep, 2), v.repeat_interleave(rep, 2), causal, q_offset=Sk - Sq)
    first = None
    for i in range(3):
        o = wide.attention(q, k, v, causal, None, Sk - Sq)
        assert torch.allclose(o.float(), want.float(), atol=2e-2, rtol=2e-2), (i, float((o.float() - want.float()).abs().max()))
        first = o if first is None else first
        assert torch.equal(o, first)
    wide.raw.attn_enable_wide(0)
    narrow = wide.attention(q, k, v, causal, None, Sk - Sq)
    wide.raw.attn_enable_wide(2)
    assert torch.allclose(first.float(), narrow.float(), atol=1e-2, rtol=1e-2)


def test_wide_attention_packed_qkv_and_spike(dev, wide):
    """q / k / v as strided views of one packed projection output; a late key with a huge score forces
    the online-softmax rescale."""
    B, S, H, D = 1, 400, 4, 128
    qkv = _rand(B, S, 3, H, D, dev=dev)
    q, k, v = qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2]
    k[0, 333] = q[0, 399] * 4.0
    o = wide.attention(q, k, v, True, None, 0)
    want = ref.attention(q.contiguous(), k.contiguous(), v.contiguous(), True)
    assert torch.allclose(o.float(), want.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("mode", [0, 2])                      # 64-row blocks, ring-staged blocks
@pytest.mark.parametrize("D,H,S,causal,step", [(128, 4, 700, True, 5.0), (64, 4, 577, False, 9.0), (128, 16, 2100, True, 0.5), (128, 4, 300, True, -5.0)])
def test_attention_whose_maximum_creeps(dev, wide, mode, D, H, S, causal, step):
    """Scores that rise (or fall) by ``step`` in base 2 from one tile of 64 keys to the next, the largest of a tile in every column of
    its 16 x 4 in turn: the maximum over a lane's keys and over the lanes that share a query."""
    g = torch.Generator(device=dev).manual_seed(S)
    unit = torch.zeros(D, device=dev)
    unit[0] = 1.0
    at = torch.arange(S, device=dev)
    level = ((at // 64).float() * step + 4.0 * (at % 64 == (at // 64 * 7) % 64)) * 0.6931472
    q = (torch.randn(1, S, H, D, device=dev, generator=g) * 0.5 * (1 - unit) + 16.0 * unit).bfloat16()
    k = (torch.randn(1, S, H, D, device=dev, generator=g) * (1 - unit) + (level * D ** 0.5 / 16.0)[None, :, None, None] * unit).bfloat16()
    v = _rand(1, S, H, D, dev=dev)
    wide.raw.attn_enable_wide(mode)
    o, lse = wide.raw.attention_fwd_lse(q, k, v, causal, D ** -0.5, 0)
    s = torch.matmul(q.double().transpose(1, 2), k.double().permute(0, 2, 3, 1).contiguous()) * D ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(S, S, device=dev, dtype=torch.bool).triu(1), float("-inf"))
    want = torch.matmul(torch.softmax(s, -1), v.double().transpose(1, 2).contiguous()).transpose(1, 2)
    # weights and outputs are rounded to bf16 once each: 2^-9 of values up to 4, twice
    assert torch.allclose(o.double(), want, atol=2e-2, rtol=2e-2), float((o.double() - want).abs().max())
    assert torch.allclose(lse.double(), torch.logsumexp(s, -1) * 1.4426950408889634, atol=1e-3, rtol=1e-5)


def test_wide_attention_against_cache_with_device_length(dev, wide):
    from eventgpt_amd.ops import hip, reference
    D, Hq, Hkv, Sq, kv, Lmax = 128, 4, 2, 300, 900, 1024
    g = torch.Generator(device=dev).manual_seed(1)
    q = torch.randn(1, Sq, Hq, D, device=dev, generator=g).to(torch.bfloat16)
    kc = torch.randn(1, Hkv, Lmax, D, device=dev, generator=g).to(torch.bfloat16)
    vc = torch.randn(1, Hkv, Lmax, D, device=dev, generator=g).to(torch.bfloat16)
    out = torch.empty_like(q)
    hip.raw.attention_cache(q, kc, vc, out, torch.tensor([kv], dtype=torch.int32, device=dev), D ** -0.5)
    k = kc[:, :, :kv].transpose(1, 2).float().repeat_interleave(2, dim=2)
    v = vc[:, :, :kv].transpose(1, 2).float().repeat_interleave(2, dim=2)
    want = reference.attention(q.float(), k, v, causal=True, q_offset=kv - Sq)
    assert torch.allclose(out.float(), want, atol=2e-2, rtol=2e-2)


def test_wide_forward_feeds_backward(dev, wide):
    """attention through the autograd Function: the wide forward's log-sum-exp drives the backward kernels."""
    from eventgpt_amd import ops
    B, S, H, D = 1, 384, 4, 128
    q, k, v = (_rand(B, S, H, D, dev=dev, seed=i, scale=0.5).requires_grad_(True) for i in range(3))
    go = _rand(B, S, H, D, dev=dev, seed=7)
    o = ops.attention(q, k, v, True)
    assert type(o.grad_fn).__name__ == "_AttentionBackward"
    o.backward(go)
    qf, kf, vf = (t.detach().float().requires_grad_(True) for t in (q, k, v))
    ref.attention(qf, kf, vf, True).backward(go.float())
    for got, want in ((q.grad, qf.grad), (k.grad, kf.grad), (v.grad, vf.grad)):
        assert torch.allclose(got.float(), want, atol=3e-2, rtol=3e-2), float((got.float() - want).abs().max())


# a round of 256-row blocks whose rows are mostly padding, and next to the lines (seven tenths with a mask and more than one block, half without)
@pytest.mark.parametrize("B,S,H,D,causal,wide", [
    (8, 20, 32, 128, True, False), (8, 100, 32, 128, True, False), (8, 256, 32, 128, True, False), (4, 358, 32, 128, True, False), (4, 359, 32, 128, True, True),
    (5, 520, 16, 128, True, False), (2, 836, 32, 128, True, True), (8, 128, 32, 128, False, False), (8, 129, 32, 128, False, True),
    (8, 64, 32, 64, False, False), (5, 577, 16, 64, False, True), (8, 200, 32, 64, True, False)])
def test_blocks_of_256_rows_where_they_are_filled(dev, B, S, H, D, causal, wide):
    from eventgpt_amd.ops import hip
    q, k, v = (torch.randn(B, S, H, D, device=dev).bfloat16() for _ in range(3))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        o, _ = hip.raw.attention_fwd_lse(q, k, v, causal, D ** -0.5, 0)
        torch.cuda.synchronize()
    names = [e.key for e in p.key_averages() if "attn_prefill" in e.key]
    assert len(names) == 1 and ("attn_prefill_wide_kernel" in names[0]) == wide, names
    want = torch.nn.functional.scaled_dot_product_attention(*(t.transpose(1, 2).float() for t in (q, k, v)), is_causal=causal).transpose(1, 2)
    assert torch.allclose(o.float(), want, atol=2e-2, rtol=2e-2)
