"""Training kernels of the hidden-state adapters (``csrc/kernels/adapter_train.hip``) against plain
fp32 PyTorch references: head_dim-512 attention forward + backward (masks, dropout), LayerNorm
backward, GELU forward / backward, counter-based dropout; and whole L4 / L5F training steps under
the profiler (no library GEMM, attention, normalisation, activation or dropout kernel)."""
import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _rand(*shape, dev, scale=1.0, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed + sum(shape))
    return (torch.randn(*shape, device=dev, generator=g) * scale).to(torch.bfloat16)


def _attn_ref(qkv, heads, causal, kpm, keep, drop_p):
    """fp32 attention over a packed projection; ``keep`` [B,H,64,64] is the kernel's own dropout mask."""
    b, s, _ = qkv.shape
    q, k, v = qkv.float().view(b, s, 3, heads, 512).permute(2, 0, 3, 1, 4)      # [B,H,S,512]
    sc = q @ k.transpose(-1, -2) / math.sqrt(512)
    dead = torch.zeros(b, 1, s, s, dtype=torch.bool, device=qkv.device)
    if causal:
        dead = dead | ~torch.ones(s, s, dtype=torch.bool, device=qkv.device).tril()
    if kpm is not None:
        dead = dead | kpm[:, None, None, :]
    p = torch.softmax(sc.masked_fill(dead, float("-inf")), -1)
    if drop_p > 0:
        p = p * keep[:, :, :s, :s].float() / (1 - drop_p)
    return (p @ v).transpose(1, 2).reshape(b, s, heads * 512)


@pytest.mark.parametrize("B,S,H,causal,masked,drop_p", [
    (2, 1, 2, False, False, 0.0), (3, 17, 8, True, False, 0.0), (2, 50, 8, False, True, 0.0),
    (2, 64, 4, True, True, 0.0), (4, 33, 8, True, True, 0.1), (2, 50, 8, False, False, 0.25)])
def test_attention_d512_forward_backward(dev, B, S, H, causal, masked, drop_p):
    from eventgpt_amd.ops import hip
    from eventgpt_amd.ops import differentiable as diff
    qkv = _rand(B, S, 3 * H * 512, dev=dev, scale=0.7, seed=S).requires_grad_(True)
    kpm = None
    if masked:
        lens = torch.tensor([max(1, S - 3 * i) for i in range(B)], device=dev)
        kpm = torch.arange(S, device=dev)[None, :] >= lens[:, None]
    seed = 12345
    out, probs = hip.raw.attn512_fwd(qkv.detach(), H, causal, kpm, 1 / math.sqrt(512), drop_p, seed, True)
    keep = hip.raw.attn512_mask(B, H, drop_p, seed, qkv.detach()).bool()
    if drop_p > 0:
        frac = keep.float().mean().item()
        assert abs(frac - (1 - drop_p)) < 0.01, frac                 # the hash is uniform
    ref_in = qkv.detach().clone().requires_grad_(True)
    want = _attn_ref(ref_in, H, causal, kpm, keep, drop_p)
    assert torch.allclose(out.float(), want, rtol=2e-2, atol=2e-2), (out.float() - want).abs().max()
    # probabilities: rows sum to one over the live keys, zero elsewhere
    ps = probs.float()[:, :, :S, :S].sum(-1)
    assert torch.allclose(ps, torch.ones_like(ps), atol=2e-2)
    assert float(probs.float()[:, :, S:, :].abs().max()) == 0.0 if S < 64 else True
    # backward against autograd through the fp32 reference, same upstream gradient
    g = _rand(B, S, H * 512, dev=dev, scale=0.5, seed=7)
    want.backward(g.float())
    dqkv = hip.raw.attn512_bwd(qkv.detach(), g, probs, H, 1 / math.sqrt(512), drop_p, seed)
    err = (dqkv.float() - ref_in.grad).abs().max().item()
    assert err < 3e-2 * ref_in.grad.abs().max().item() + 2e-3, err
    # the autograd Function returns the same (eval-style call: no dropout, so seeds do not matter)
    if drop_p == 0:
        o2 = diff.attention_d512(qkv, H, causal, kpm, 0.0)
        o2.backward(g)
        assert torch.equal(o2, out) and torch.equal(qkv.grad, dqkv)


def test_attention_d512_is_deterministic_and_seeded(dev):
    from eventgpt_amd.ops import hip
    qkv = _rand(2, 40, 3 * 8 * 512, dev=dev, scale=0.5)
    a, _ = hip.raw.attn512_fwd(qkv, 8, True, None, 1 / math.sqrt(512), 0.2, 99, False)
    b, _ = hip.raw.attn512_fwd(qkv, 8, True, None, 1 / math.sqrt(512), 0.2, 99, False)
    c, _ = hip.raw.attn512_fwd(qkv, 8, True, None, 1 / math.sqrt(512), 0.2, 100, False)
    assert torch.equal(a, b) and not torch.equal(a, c)


@pytest.mark.parametrize("rows,H,bias", [(3200, 4096, True), (37, 1024, True), (130, 512, False), (5, 8192, True)])
def test_layernorm_forward_backward(dev, rows, H, bias):
    from eventgpt_amd.ops import differentiable as diff
    x = _rand(rows, H, dev=dev, seed=1).requires_grad_(True)
    w = (1 + 0.1 * torch.randn(H, device=dev)).requires_grad_(True)          # fp32 parameters, as under autocast
    b = (0.1 * torch.randn(H, device=dev)).requires_grad_(True) if bias else None
    g = _rand(rows, H, dev=dev, seed=2)
    y = diff.layernorm(x, w, b, 1e-5)
    assert y.dtype == torch.bfloat16
    y.backward(g)
    xr = x.detach().float().requires_grad_(True)
    wr = w.detach().to(torch.bfloat16).float().requires_grad_(True)
    br = None if b is None else b.detach().to(torch.bfloat16).float().requires_grad_(True)
    yr = F.layer_norm(xr, (H,), wr, br, 1e-5)
    yr.backward(g.float())
    assert torch.allclose(y.float(), yr, rtol=2e-2, atol=2e-2)
    assert (x.grad.float() - xr.grad).abs().max() < 2e-2 * xr.grad.abs().max() + 1e-3
    assert w.grad.dtype == torch.float32
    assert (w.grad - wr.grad).abs().max() < 1e-2 * wr.grad.abs().max() + 1e-3
    if bias:
        assert (b.grad - br.grad).abs().max() < 1e-2 * br.grad.abs().max() + 1e-3


def test_gelu_and_dropout(dev):
    from eventgpt_amd.ops import differentiable as diff
    x = _rand(640, 2048, dev=dev, scale=2.0).requires_grad_(True)
    g = _rand(640, 2048, dev=dev, seed=3)
    y = diff.gelu(x)
    y.backward(g)
    xr = x.detach().float().requires_grad_(True)
    yr = F.gelu(xr)
    yr.backward(g.float())
    assert torch.allclose(y.float(), yr, rtol=1e-2, atol=1e-2)
    assert torch.allclose(x.grad.float(), xr.grad, rtol=2e-2, atol=1e-2)
    # dropout: inverted scaling, the expected keep rate, and a backward that uses the forward's mask
    torch.manual_seed(5)
    z = torch.ones(512, 4096, device=dev, dtype=torch.bfloat16, requires_grad=True)
    d = diff.dropout(z, 0.1, True)
    kept = d != 0
    assert abs(kept.float().mean().item() - 0.9) < 0.005
    assert torch.allclose(d[kept].float(), torch.full_like(d[kept].float(), 1 / 0.9), rtol=1e-2)
    d.backward(torch.ones_like(d))
    assert torch.equal(z.grad != 0, kept)
    assert diff.dropout(z, 0.1, False) is z and diff.dropout(z, 0.0, True) is z
    torch.manual_seed(5)
    d2 = diff.dropout(z, 0.1, True)
    assert torch.equal(d2, d)                   # seeds come from torch's generator: repeatable
    assert not torch.equal(diff.dropout(z, 0.1, True), d)


@pytest.mark.parametrize("level", [4, 6])
def test_attention_adapter_training_step_matches_library(dev, level):
    """Loss and parameter gradients of an L4 / L5F step (eval mode: no dropout, so the functions are
    equal) on the in-tree kernels against the library path (fp32 LayerNorm / GELU, library attention)."""
    from eventgpt_amd.align.adapters import create_adapter
    from eventgpt_amd.ops.intree_mode import InTreeLinear
    torch.manual_seed(0)
    a = create_adapter(level, 1024, num_heads=2, ffn_dim=256).to(dev)
    b = create_adapter(level, 1024, num_heads=2, ffn_dim=256).to(dev)
    b.load_state_dict(a.state_dict())
    a.eval(), b.eval()
    h = torch.randn(6, 40, 1024, device=dev)
    t = h + 0.1 * torch.randn_like(h)
    mask = torch.ones(6, 40, device=dev)
    mask[1, 30:] = 0
    mask[4, 12:] = 0
    la = a.float().compute_loss(h, t, mask)["total_loss"]          # fp32, library kernels throughout
    with torch.autocast("cuda", dtype=torch.bfloat16), InTreeLinear() as mode:
        lb = b.compute_loss(h, t, mask)["total_loss"]
    assert mode.routed >= 8, (mode.routed, mode.passed)
    la.backward()
    lb.backward()
    assert abs(float(la) - float(lb)) < 3e-2 * abs(float(la)) + 1e-3, (float(la), float(lb))
    for (n, pa), (_, pb) in zip(a.named_parameters(), b.named_parameters()):
        if pa.grad is None:
            assert pb.grad is None, n
            continue
        assert pb.grad is not None and pb.grad.dtype == torch.float32, n
        err = (pa.grad - pb.grad).abs().max().item()
        assert err < 6e-2 * pa.grad.abs().max().item() + 1e-5, (n, err, pa.grad.abs().max().item())


@pytest.mark.parametrize("level", [4, 6])
def test_attention_adapter_training_step_uses_only_intree_kernels(dev, level):
    """An L4 / L5F training step (train mode: dropout everywhere, 4096 wide, 8 heads of 512) under the
    profiler: no Tensile GEMM, no library attention, no ATen LayerNorm / GELU / dropout / softmax kernel."""
    from eventgpt_amd.align.adapters import create_adapter
    from eventgpt_amd.ops.intree_mode import InTreeLinear
    torch.manual_seed(1)
    m = create_adapter(level, 4096).to(dev).train()
    h = torch.randn(16, 48, 4096, device=dev)
    t = h + 0.1 * torch.randn_like(h)
    mask = torch.ones(16, 48, device=dev)
    mask[3, 20:] = 0
    for _ in range(2):                      # first pass: module loads, outside the profile
        m.zero_grad()
        with torch.autocast("cuda", dtype=torch.bfloat16), InTreeLinear():
            m.compute_loss(h, t, mask)["total_loss"].backward()
    m.zero_grad()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        with torch.autocast("cuda", dtype=torch.bfloat16), InTreeLinear():
            loss = m.compute_loss(h, t, mask)["total_loss"]
        loss.backward()
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    for need in ("attn512_fwd_kernel", "attn512_bwd_kernel", "layernorm_bwd_kernel", "adapter_elementwise_kernel",
                 "gemm"):
        assert any(need in n for n in names), (need, names)
    bad = [n for n in names if n.startswith("Cijk_") or "attn_fwd" in n or "bwd_kernel_dk_dv" in n
           or "layer_norm" in n.lower() or "GammaBeta" in n or "gelu" in n.lower().replace("adapter_elementwise", "")
           or "fused_dropout" in n or "softmax" in n.lower()]
    assert not bad, bad
    assert torch.isfinite(loss) and all(torch.isfinite(p.grad).all() for p in m.parameters() if p.grad is not None)


@pytest.mark.parametrize("M,V,K,n_ignored", [(48, 32003, 4096, 0), (840, 1003, 512, 800), (130, 2048, 512, 64),
                                             (17, 32003, 4096, 5)])
def test_linear_cross_entropy_matches_fp32(dev, M, V, K, n_ignored):
    """Loss and both gradients of the fused LM-head cross-entropy against F.cross_entropy over fp32
    logits of the same bf16 operands; unsupervised rows take no part (and get zero gradient)."""
    from eventgpt_amd.ops import differentiable as diff
    x = _rand(M, K, dev=dev, scale=1.0, seed=1).requires_grad_(True)
    w = _rand(V, K, dev=dev, scale=0.05, seed=2).requires_grad_(True)
    g = torch.Generator(device=dev).manual_seed(3)
    labels = torch.randint(0, V, (M,), device=dev, generator=g)
    if n_ignored:
        labels[torch.randperm(M, device=dev, generator=g)[:n_ignored]] = -100
    loss = diff.linear_cross_entropy(x, w, labels)
    (loss * 0.5).backward()                       # an upstream factor, as gradient accumulation applies
    xr = x.detach().float().requires_grad_(True)
    wr = w.detach().float().requires_grad_(True)
    want = F.cross_entropy(xr @ wr.t(), labels, ignore_index=-100)
    (want * 0.5).backward()
    assert abs(float(loss) - float(want)) < 2e-2 * abs(float(want)) + 1e-3, (float(loss), float(want))
    assert x.grad.shape == x.shape and w.grad.shape == w.shape
    assert (x.grad.float() - xr.grad).abs().max() < 3e-2 * xr.grad.abs().max() + 1e-5
    assert (w.grad.float() - wr.grad).abs().max() < 3e-2 * wr.grad.abs().max() + 1e-5
    if n_ignored:
        assert float(x.grad[labels == -100].abs().max()) == 0.0


def test_model_training_loss_uses_the_fused_head(dev):
    """EventChatModel.forward with labels in a training step: same loss and gradients as the full-logits
    path, no fp32 softmax kernel, and ``logits`` is not materialised."""
    from eventgpt_amd.models import EventChatConfig, EventChatModel
    cfg = EventChatConfig(vocab_size=1003, hidden_size=512, intermediate_size=1408, num_hidden_layers=2,
                          num_attention_heads=4, max_position_embeddings=512)
    a = EventChatModel.from_config(cfg, torch.bfloat16, dev, seed=0)
    b = EventChatModel.from_config(cfg, torch.bfloat16, dev, seed=0)
    for m in (a, b):
        for p in m.parameters():
            p.requires_grad_(True)
    ids = torch.randint(3, 1000, (1, 90), device=dev)
    labels = ids.clone()
    labels[:, :70] = -100
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out = a(input_ids=ids, labels=labels)
        out.loss.backward()
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    assert out.logits is None and any("ce_fwd_kernel" in n for n in names), names
    assert not [n for n in names if "softmax" in n.lower() or "nll_loss" in n.lower()], names
    # reference: all logits in fp32
    h = b.model(input_ids=ids, use_cache=False).last_hidden_state
    logits = b.lm_head(h).float()
    want = F.cross_entropy(logits[:, :-1].reshape(-1, 1003), labels[:, 1:].reshape(-1), ignore_index=-100)
    want.backward()
    assert abs(float(out.loss) - float(want)) < 2e-2 * abs(float(want)) + 1e-3
    ga, gb = a.lm_head.weight.grad.float(), b.lm_head.weight.grad.float()
    assert (ga - gb).abs().max() < 5e-2 * gb.abs().max() + 1e-4
    ga, gb = a.model.layers[0].mlp.down_proj.weight.grad.float(), b.model.layers[0].mlp.down_proj.weight.grad.float()
    assert (ga - gb).abs().max() < 8e-2 * gb.abs().max() + 1e-4


def test_padded_batch_step_equals_single_sample_steps(dev):
    """Three samples of different lengths in ONE right-padded forward / backward (fused attention, no mask,
    ``loss_reduction="sequence_mean"``) against the three single-sample passes averaged: same loss, same
    gradients, and the attention launches are the in-tree kernels."""
    from eventgpt_amd.constants import EVENT_TOKEN_INDEX
    from eventgpt_amd.models import EventChatConfig, EventChatModel
    cfg = EventChatConfig(vocab_size=1003, hidden_size=512, intermediate_size=1408, num_hidden_layers=2,
                          num_attention_heads=4, max_position_embeddings=1024)
    a = EventChatModel.from_config(cfg, torch.bfloat16, dev, seed=0)
    b = EventChatModel.from_config(cfg, torch.bfloat16, dev, seed=0)
    for m in (a, b):
        m.train()
        for p in m.parameters():
            p.requires_grad_(True)
    g = torch.Generator().manual_seed(0)
    lens, n_ev = [70, 96, 83], 40
    ids, labels, feats = [], [], []
    for n in lens:
        t = torch.randint(3, 1000, (n,), generator=g)
        t[5] = EVENT_TOKEN_INDEX
        lab = t.clone()
        lab[: n - 12] = -100
        ids.append(t), labels.append(lab)
        feats.append((torch.randn(n_ev, 512, generator=g) * 0.1).to(torch.bfloat16).to(dev))
    width = max(lens)
    pid = torch.zeros(3, width, dtype=torch.long)
    plab = torch.full((3, width), -100, dtype=torch.long)
    pmask = torch.zeros(3, width, dtype=torch.long)
    for i, n in enumerate(lens):
        pid[i, :n], plab[i, :n], pmask[i, :n] = ids[i], labels[i], 1
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out = a(input_ids=pid.to(dev), attention_mask=pmask.to(dev), labels=plab.to(dev),
                event_features=torch.stack(feats), already_adapted=True, loss_reduction="sequence_mean")
        out.loss.backward()
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    assert any("attn_bwd_dkv_kernel" in n for n in names) and not [n for n in names if "attn_fwd" in n], names
    total = 0.0
    for i in range(3):
        o = b(input_ids=ids[i][None].to(dev), labels=labels[i][None].to(dev), event_features=feats[i][None],
              already_adapted=True)
        (o.loss / 3).backward()
        total += float(o.loss) / 3
    assert abs(float(out.loss) - total) < 1e-2 * abs(total) + 1e-3, (float(out.loss), total)
    for (n, pa), (_, pb) in zip(a.named_parameters(), b.named_parameters()):
        if pb.grad is None:
            continue
        ga, gb = pa.grad.float(), pb.grad.float()
        assert (ga - gb).abs().max() < 6e-2 * gb.abs().max() + 1e-4, (n, float((ga - gb).abs().max()), float(gb.abs().max()))


# one row, a slab's remainder, columns past a block of 512 and short of a wave, many rows over few columns
@pytest.mark.parametrize("m,n", [(1, 8), (15, 520), (17, 4096), (3200, 4096), (203, 1000), (70001, 16)])
def test_column_sum_at_its_edges(dev, m, n):
    from eventgpt_amd.ops import hip
    g = torch.randn(m, n, generator=torch.Generator().manual_seed(m)).to(torch.bfloat16)
    want = g.double().sum(0)
    got = hip.raw.column_sum(g.to(dev)).cpu()
    # float32 chains of at most the row count: m 2^-24 of the sum of magnitudes, then half a step of bfloat16
    bound = m * 2.0 ** -24 * g.double().abs().sum(0) + 2.0 ** -8 * want.abs()
    assert bool(((got.double() - want).abs() <= bound).all())
    g[m // 2, n - 1] = float("inf")
    got = hip.raw.column_sum(g.to(dev)).cpu()
    assert got[-1] == float("inf") and bool(torch.isfinite(got[:-1]).all())


@pytest.mark.parametrize("rows,H", [(1, 8), (60, 72), (64, 8), (65, 136), (508, 64), (513, 1000), (2049, 8)])
def test_layernorm_parameter_gradients_of_few_columns(dev, rows, H):
    """Partial sums of 1 to 512 blocks of rows: fewer than the waves that add them, either side of what those hold in
    flight, columns short of a wave."""
    from eventgpt_amd.ops import hip
    x, g, w = _rand(rows, H, dev=dev, seed=1), _rand(rows, H, dev=dev, seed=2), _rand(H, dev=dev, seed=3)
    _, dw, db = hip.raw.layernorm_bwd(x, w, g, 1e-5)
    xd, gd = x.double(), g.double()
    xh = (xd - xd.mean(1, keepdim=True)) / torch.sqrt(xd.var(1, unbiased=False, keepdim=True) + 1e-5)
    # float32 chains of at most the row count, and of the eight or fewer operations that make a row's term
    for got, term in ((dw, gd * xh), (db, gd)):
        assert bool(((got.double() - term.sum(0)).abs() <= (rows + H + 8) * 2.0 ** -23 * (term.abs().sum(0) + gd.abs().sum(0))).all())


@pytest.mark.parametrize("rows,k,n,uses,passes", [(16, 8, 8, 1, 1), (65, 128, 520, 1, 2), (200, 512, 1024, 2, 1), (333, 1024, 512, 2, 2)])
def test_fp32_parameters_get_the_sums_of_the_weight_gradient(dev, rows, k, n, uses, passes):
    """Gradients of fp32 parameters of in-tree linears are fp32 sums of bf16 products, written into the optimizer's slot: used once or
    twice in a graph, over one or two backward passes.  An fp32 sum of ``rows`` products in any order is within ``rows * 2^-24`` of the sum of
    their absolute values; a second use or pass adds one rounding of the total."""
    from eventgpt_amd.ops.intree_mode import InTreeLinear
    from eventgpt_amd.parallel.dp import ShardedAdamW
    g = torch.Generator().manual_seed(rows)
    lin = torch.nn.Linear(k, n).to(dev)
    xs = [torch.randn(rows, k, generator=g).to(dev) for _ in range(uses)]
    gys = [torch.randn(rows, n, generator=g).to(dev).bfloat16() for _ in range(uses)]
    opt = ShardedAdamW(lin.parameters(), lr=1e-3)
    opt.zero_grad()
    for _ in range(passes):
        with torch.autocast("cuda", dtype=torch.bfloat16), InTreeLinear() as mode:
            ys = [torch.nn.functional.linear(x, lin.weight, lin.bias) for x in xs]
        assert mode.routed == uses
        torch.autograd.backward(ys, gys)
    opt.global_grad_norm()                                  # settles every gradient into its slot
    want = passes * sum(gy.double().T @ x.bfloat16().double() for x, gy in zip(xs, gys))
    size = passes * sum(gy.double().abs().T @ x.bfloat16().double().abs() for x, gy in zip(xs, gys))
    flat = opt.buckets[0].flat_grad
    for p, w, s in ((lin.weight, want, size), (lin.bias, passes * sum(gy.double().sum(0) for gy in gys),
                                               passes * sum(gy.double().abs().sum(0) for gy in gys))):
        assert p.grad.dtype == torch.float32 and flat.data_ptr() <= p.grad.data_ptr() < flat.data_ptr() + 4 * flat.numel()
        assert bool(((p.grad.double() - w).abs() <= (rows + 4) * 2.0 ** -24 * s + 1e-30).all())


def _in_tree_loss(net, x):
    """A loss of ``net`` with its linears on the in-tree products; their weight gradients are the same bits from call to call."""
    from eventgpt_amd.ops.intree_mode import InTreeLinear
    with torch.autocast("cuda", dtype=torch.bfloat16), InTreeLinear() as mode:
        y = net(x)
    assert mode.routed > 0
    return y.float().square().mean()


def test_gradients_after_zero_grad_are_zeros_that_count(dev):
    """``zero_grad`` leaves every fp32 gradient as zeros in its slot: what a program adds to it before the backward counts, and a
    parameter that takes no part has a gradient of zeros."""
    from eventgpt_amd.parallel.dp import ShardedAdamW
    torch.manual_seed(0)
    net = torch.nn.Sequential(torch.nn.Linear(64, 128), torch.nn.LayerNorm(128), torch.nn.Linear(128, 64)).to(dev)
    unused = torch.nn.Linear(64, 64).to(dev)
    x = torch.randn(48, 64, generator=torch.Generator().manual_seed(1)).to(dev)
    want = torch.autograd.grad(_in_tree_loss(net, x), list(net.parameters()))
    opt = ShardedAdamW([*net.parameters(), *unused.parameters()], lr=1e-3)
    flat = opt.buckets[0].flat_grad
    for plus in (0.0, 0.5, 0.0):
        flat.fill_(7.0)
        opt.zero_grad()
        for p in (*net.parameters(), *unused.parameters()):
            assert p.grad is not None and flat.data_ptr() <= p.grad.data_ptr() < flat.data_ptr() + 4 * flat.numel()
            assert not bool(p.grad.any())
        if plus:
            net[0].weight.grad.add_(plus)
            net[1].weight.grad.add_(plus)
        _in_tree_loss(net, x).backward()
        for p, w in zip(net.parameters(), want):
            assert torch.equal(p.grad, w + plus if plus and (p is net[0].weight or p is net[1].weight) else w)
        assert all(not bool(p.grad.any()) for p in unused.parameters())
        assert (net[2].weight.grad.data_ptr() == net[2].weight._grad_sink.data_ptr()) and net[2].weight._grad_sink_used
        opt.global_grad_norm()
        assert all(flat.data_ptr() <= p.grad.data_ptr() < flat.data_ptr() + 4 * flat.numel() for p in net.parameters())


@pytest.mark.parametrize("kind", ["fp32", "bf16", "lora"])
def test_gradients_handed_out_are_not_the_optimizers_memory(dev, kind):
    """What ``torch.autograd.grad`` returns and what a hook keeps is theirs: later passes, ``zero_grad`` and steps leave it alone, and
    a backward after it still counts in full."""
    from eventgpt_amd.ops import differentiable as diff
    from eventgpt_amd.parallel.dp import ShardedAdamW
    g = torch.Generator().manual_seed(3)
    x = torch.randn(96, 128, generator=g).to(dev).bfloat16()
    w0 = (torch.randn(64, 128, generator=g) / 8).to(dev)
    a, b = (torch.nn.Parameter((torch.randn(*s, generator=g) / 8).to(dev).bfloat16()) for s in ((8, 128), (64, 8)))
    w = torch.nn.Parameter(w0 if kind == "fp32" else w0.bfloat16())
    frozen = w0.bfloat16()
    params = [a, b] if kind == "lora" else [w]

    def loss():
        if kind == "lora":
            return diff.lora_projection(x, frozen, [(0, a, b)], 2.0).float().square().mean()
        if kind == "bf16":
            return diff.linear(x, w).float().square().mean()
        return _in_tree_loss(lambda t: F.linear(t, w), x)
    want = [t.clone() for t in torch.autograd.grad(loss(), params)]
    opt = ShardedAdamW(params, lr=1e-3)
    flat = opt.buckets[0].flat_grad
    inside = lambda t: flat.data_ptr() <= t.data_ptr() < flat.data_ptr() + flat.numel() * flat.element_size()
    opt.zero_grad()
    got = torch.autograd.grad(loss(), params)
    loss().backward()                                    # the first gradient that is accumulated
    assert all(inside(p.grad) and torch.equal(p.grad, t) for p, t in zip(params, want))
    opt.zero_grad()
    kept = []
    hooks = [p.register_hook(kept.append) for p in params]
    loss().backward()
    for h in hooks:
        h.remove()
    assert len(kept) == len(params) and all(torch.equal(p.grad, t) for p, t in zip(params, want))
    opt.global_grad_norm()
    assert all(inside(p.grad) and torch.equal(p.grad, t) for p, t in zip(params, want))
    opt.zero_grad()
    opt.global_grad_norm()                               # settles gradients of zeros
    flat.fill_(7.0)
    kept.sort(key=lambda t: [p.shape for p in params].index(t.shape))
    for t, k, w_ in zip(got, kept, want):
        assert torch.equal(t, w_) and torch.equal(k, w_)


def _misaligned_slots(params):
    return [p for p in params if p.dim() == 2 and p._grad_sink.data_ptr() % 16]


@pytest.mark.parametrize("level", [2, 3])
def test_fp32_gradients_behind_scalar_parameters(dev, level):
    """Adapters whose scalars shift the slots of the matrices behind them off 16 bytes: the gradients are what the same products give
    without an optimizer, and no kernel stores its four floats at once into such a slot."""
    from eventgpt_amd.align.adapters import create_adapter
    from eventgpt_amd.parallel.dp import ShardedAdamW
    torch.manual_seed(level)
    net = create_adapter(level, 64, bottleneck_dim=64, num_blocks=3, dropout=0.0).to(dev).train()
    with torch.no_grad():
        for p in net.parameters():
            p.add_(torch.randn_like(p) * 0.05)           # (the up-projections start at zero)
    x = torch.randn(40, 64, generator=torch.Generator().manual_seed(level)).to(dev)
    names, params = zip(*net.named_parameters())
    want = torch.autograd.grad(_in_tree_loss(net, x), params)
    opt = ShardedAdamW(params, lr=1e-3)
    odd = _misaligned_slots(params)
    assert odd
    opt.zero_grad()
    _in_tree_loss(net, x).backward()
    assert not any(p._grad_sink_used for p in odd)
    for name, p, w in zip(names, params, want):
        assert torch.equal(p.grad, w), name
    opt.global_grad_norm()
    for name, p, w in zip(names, params, want):
        assert torch.equal(p.grad, w), name


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("M,N,K", [(64, 64, 40), (264, 520, 96), (1032, 1304, 128)])
def test_weight_gradients_into_memory_off_16_bytes(dev, f32, M, N, K):
    """``linear_wgrad`` into an ``out`` at every element of a 16-byte line: the same bits as into a tensor of its own, and nothing beside it."""
    from eventgpt_amd.ops import differentiable as diff
    gy, x = _rand(K, M, dev=dev), _rand(K, N, dev=dev, seed=1)
    want = diff.linear_wgrad(gy, x, None, f32)
    for off in range(1, 16 // want.element_size()):
        buf = torch.full((M * N + 32,), 3.0, device=dev, dtype=want.dtype)
        out = buf[off:off + M * N].view(M, N)
        assert out.data_ptr() % 16
        got = diff.linear_wgrad(gy, x, out, f32)
        assert got.data_ptr() == out.data_ptr() and torch.equal(out, want)
        assert bool((buf[:off] == 3).all()) and bool((buf[off + M * N:] == 3).all())


def test_computed_fp32_weights_are_not_kept_for_the_backward(dev):
    """A weight that is itself the result of an operation is freed with its last reference, as the backward needs its bf16 copy only."""
    import weakref
    from eventgpt_amd.ops.intree_mode import InTreeLinear
    p, s = torch.nn.Parameter(torch.randn(64, 128, device=dev)), torch.nn.Parameter(torch.randn(64, 1, device=dev))
    x = torch.randn(32, 128, device=dev)
    w = p * s
    with torch.autocast("cuda", dtype=torch.bfloat16), InTreeLinear() as mode:
        y = F.linear(x, w)
    assert mode.routed == 1
    ref = weakref.ref(w)
    want = y.detach().float().T @ x.bfloat16().float()            # dW of y^2 / 2, up to the products' roundings
    del w
    assert ref() is None
    (y.float().square().sum() / 2).backward()
    assert float((p.grad - want * s.detach()).norm() / p.grad.norm()) < 1e-4


# columns about a thread's chunks (2 048 a chunk, two or four of them), rows about a block's share
@pytest.mark.parametrize("rows,H", [(16, 8), (17, 520), (33, 2048), (2049, 2056), (65, 4096), (40, 4104), (19, 8192)])
@pytest.mark.parametrize("residual", [True, False])
def test_residual_step_and_norm_in_one_launch(dev, rows, H, residual):
    """``add_norm`` inside the mode against float64 of the same expression (the norm of the sum rounded to bf16): values and all gradients, with
    and without a gradient that reaches the sum beside the norm.  bf16 results are off by 2^-8 of their row's largest term, the parameters' sums by
    that of every row's."""
    from eventgpt_amd.ops.intree_mode import InTreeLinear, add_norm
    g = torch.Generator(device=dev).manual_seed(rows + H)
    def rnd(*shape):
        return torch.randn(*shape, device=dev, generator=g)
    norm = torch.nn.LayerNorm(H).to(dev)
    with torch.no_grad():
        norm.weight.copy_(1 + 0.1 * rnd(H)), norm.bias.copy_(0.1 * rnd(H))
    x, d = rnd(1, rows, H).requires_grad_(), rnd(1, rows, H).bfloat16().requires_grad_()
    gs, gh = rnd(1, rows, H), rnd(1, rows, H).bfloat16()
    with InTreeLinear() as mode:
        s, h = add_norm(x, d, norm)
    assert mode.routed == 1 and type(h.grad_fn).__name__ == "_AddLayerNormBackward"
    torch.autograd.backward([s, h] if residual else [h], [gs, gh] if residual else [gh])
    assert torch.equal(s, x + d)
    x64, w, b = s.detach().bfloat16().double().requires_grad_(), norm.weight.detach().bfloat16().double(), norm.bias.detach().bfloat16().double()
    w.requires_grad_(), b.requires_grad_()
    want = F.layer_norm(x64, (H,), w, b, norm.eps)
    want.backward(gh.double())
    def close(got, ref, size):
        assert bool(((got.double() - ref).abs() <= 2.0 ** -8 * size + 1e-6).all()), float(((got.double() - ref).abs() / (size + 1e-9)).max())
    close(h, want.detach(), want.detach().abs())
    ref = x64.grad + (gs.double() if residual else 0)
    close(x.grad, ref, x64.grad.abs().amax(-1, keepdim=True) * 2.0 ** -8)
    close(d.grad, ref, ref.abs() + x64.grad.abs().amax(-1, keepdim=True) * 2.0 ** -8)
    close(norm.weight.grad, w.grad, 2.0 ** -8 * (gh.double().abs() * 5).sum((0, 1)))
    close(norm.bias.grad, b.grad, 2.0 ** -8 * gh.double().abs().sum((0, 1)))


@pytest.mark.parametrize("n", [8, 2048, 2056, 2048 * 2048 + 8])
def test_step_toward_the_output_in_one_launch(dev, n):
    from eventgpt_amd.ops.intree_mode import InTreeLinear, toward
    g = torch.Generator(device=dev).manual_seed(n)
    base, y = torch.randn(n, device=dev, generator=g), torch.randn(n, device=dev, generator=g).bfloat16().requires_grad_()
    alpha = torch.nn.Parameter(torch.tensor(0.3, device=dev))
    with InTreeLinear() as mode:
        out = toward(base, y, alpha)
        plain = toward(base.requires_grad_(), y, alpha)              # rows that need a gradient stay with the expression
    assert mode.routed == 1 and type(out.grad_fn).__name__ == "_TowardBackward" and type(plain.grad_fn).__name__ == "AddBackward0"
    gy = torch.randn(n, device=dev, generator=g)
    out.backward(gy)
    b, t = base.detach().double(), y.detach().double()
    want, terms = b + alpha.detach().double() * (t - b), gy.double() * (t - b)
    assert bool(((out.double() - want).abs() <= 2.0 ** -22 * (b.abs() + t.abs())).all())
    assert torch.equal(y.grad, (gy * alpha.detach()).bfloat16())
    assert abs(float(alpha.grad) - float(terms.sum())) <= 64 * 2.0 ** -24 * float(terms.abs().sum()) + 1e-6      # (sums of up to 64 in a row)


def test_parts_of_a_block_that_is_listened_to_are_called_whole(dev):
    """Hooks on a norm or on the output projection see their calls inside the mode; the loss is the same but for roundings."""
    from eventgpt_amd.align.adapters import create_adapter
    from eventgpt_amd.ops.intree_mode import InTreeLinear
    torch.manual_seed(3)
    m, h = create_adapter(4, 512, num_heads=1, ffn_dim=256).to(dev).eval(), torch.randn(4, 16, 512, device=dev)
    def loss():
        with torch.autocast("cuda", dtype=torch.bfloat16), InTreeLinear():
            return float(m.compute_loss(h, h + 0.1 * h.roll(1, 0))["total_loss"].detach())
    seen, quiet = [], loss()
    hooks = [part.register_forward_hook(lambda part, *a: seen.append(type(part).__name__)) for part in (m.output_proj, m.layers[0]["ffn_norm"])]
    assert abs(loss() - quiet) < 1e-2 * quiet and seen == ["LayerNorm", "Sequential"]
    for hook in hooks:
        hook.remove()
    assert loss() == quiet and len(seen) == 2
    norm = m.layers[0]["ffn_norm"]
    norm.forward = lambda x: seen.append("own") or torch.nn.LayerNorm.forward(norm, x)      # a forward put on the module itself
    assert abs(loss() - quiet) < 1e-2 * quiet and seen[2:] == ["own"]
