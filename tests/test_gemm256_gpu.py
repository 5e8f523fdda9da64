"""The 256 x 256 GEMMs forced onto shapes that exercise their edges: rows / columns that do not fill a tile, one K-tile, odd
and even K-tile counts, every epilogue, the K-strided operand layouts of the backward products; each against an fp32 matmul.
A forced product runs on the four waves of ``gemm_quad.hip`` where those take it (K-contiguous operands, two K-tiles or more in every
split, bf16 output in whole 16-byte chunks, fp32 sums or slabs) and on the eight phase-staggered ones of ``gemm256_kernel`` otherwise.  Then the
tiles of ``gemm_ring.hip``.  Every case runs several times: the synchronisation is counted waits and barriers, so a race would show as
a difference between repeats."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(*shape, dev, scale=1.0, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed + sum(shape))
    return (torch.randn(*shape, device=dev, generator=g) * scale).to(torch.bfloat16)


@pytest.fixture()
def force256():
    from eventgpt_amd.ops import hip
    hip.raw.gemm_force_config(5)
    yield hip.raw
    hip.raw.gemm_force_config(-1)


def _check(y, want, K):
    err = (y.float() - want).abs()
    tol = 2e-2 * math.sqrt(K / 64) * float(want.abs().max()) / 8 + 2e-2 * want.abs()
    assert bool((err <= tol).all()), (float(err.max()), float(want.abs().max()))


@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (256, 256, 128), (256, 256, 192), (512, 768, 4096), (1000, 520, 1024),
                                   (37, 4096, 4096), (2115, 4096, 11008), (4643, 1000, 1024), (300, 264, 320)])
def test_forced_256_matches_fp32(dev, force256, M, N, K):
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    want = x.float() @ w.float().t()
    first = None
    for rep in range(4):
        y = force256.linear(x, w, None, None, 0, False)
        _check(y, want, K)
        first = y if first is None else first
        assert torch.equal(y, first), rep            # deterministic: same schedule, same bits


def test_forced_256_epilogues(dev, force256):
    M, N, K = 700, 1032, 512
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    lin = x.float() @ w.float().t() + bias.float()
    y = force256.linear(x, w, bias, res, 1, False)                      # bias + GELU + residual
    want = torch.nn.functional.gelu(lin).to(torch.bfloat16).float() + res.float()
    _check(y, want, K)
    yf = force256.linear(x, w, bias, None, 0, True)                      # fp32 output
    assert yf.dtype == torch.float32
    _check(yf, lin, K)
    pv, pi = force256.linear_argmax_partials(x, w, bias)
    got = pi.gather(1, pv.argmax(1, keepdim=True))[:, 0].long()
    assert torch.equal(lin.gather(1, got[:, None]).to(torch.bfloat16), lin.max(1, keepdim=True).values.to(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", [(1024, 512, 4096), (836, 4096, 1000), (2115, 1024, 264), (264, 11008, 2120)])
def test_forced_256_kstrided_operands(dev, force256, M, N, K):
    """dX = dY W (weight K-strided) and dW = dY^T X (both K-strided) on the 8-wave kernel."""
    from eventgpt_amd.ops import differentiable as diff
    gy, w, x = _rand(M, N, dev=dev, scale=0.5), _rand(N, K, dev=dev, seed=1, scale=0.05), _rand(M, K, dev=dev, seed=2)
    for rep in range(3):
        dx = diff.linear_dgrad(gy, w)
        _check(dx, gy.float() @ w.float(), N)
        dw = diff.linear_wgrad(gy, x)
        _check(dw, gy.float().t() @ x.float(), M)


def test_forced_256_identity_exact(dev, force256):
    """A = I against an asymmetric operand: a wrong row / column / k map gives exact mismatches."""
    n = 512
    eye = torch.eye(n, device=dev, dtype=torch.bfloat16)
    w = (torch.arange(n * 320, device=dev).reshape(320, n) % 251).to(torch.bfloat16)     # [N=320][K=n]
    assert torch.equal(force256.linear(eye, w, None, None, 0, False), w.t())
    wt = (torch.arange(n * 264, device=dev).reshape(n, 264) % 241).to(torch.bfloat16)    # [K=n][N=264]
    assert torch.equal(force256.linear_t(eye, wt, False, True, None, None, 0, False, n), wt)
    a = (torch.arange(n * 328, device=dev).reshape(n, 328) % 239).to(torch.bfloat16)     # [K=n][M=328]
    assert torch.equal(force256.linear_t(a, wt, True, True, None, None, 0, True, n), a.float().t() @ wt.float())
    assert torch.equal(force256.linear_t(a, eye, True, False, None, None, 0, False, n), a.t())


def test_auto_dispatch_uses_256_for_large_shapes(dev):
    from eventgpt_amd.ops import hip
    x, w = _rand(4643, 4096, dev=dev), _rand(12288, 4096, dev=dev, seed=1, scale=0.05)
    y_auto = hip.raw.linear(x, w, None, None, 0, False)
    hip.raw.gemm_enable_256(False)
    try:
        y_old = hip.raw.linear(x, w, None, None, 0, False)
    finally:
        hip.raw.gemm_enable_256(True)
    want = x.float() @ w.float().t()
    _check(y_auto, want, 4096)
    _check(y_old, want, 4096)


@pytest.mark.parametrize("M,N,K", [(4643, 4608, 4096), (4643, 4096 + 264, 4096), (4643, 4096, 512), (2600, 6400, 128)])
def test_auto_dispatch_column_split_for_partial_rounds(dev, M, N, K):
    """Tile counts just over whole rounds of CUs (342 = 256 + 86, 323 = 256 + 67) run as two launches over
    disjoint column ranges -- the tail on the 4-wave kernel or K-split on the 8-wave one; every epilogue operand is
    offset with them.  (Contractions under 2048 take the 4-wave tiles throughout.)"""
    from eventgpt_amd.ops import hip
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    lin = x.float() @ w.float().t() + bias.float()
    y = hip.raw.linear(x, w, bias, res, 1, False)
    want = torch.nn.functional.gelu(lin).to(torch.bfloat16).float() + res.float()
    _check(y, want, K)
    yf = hip.raw.linear(x, w, bias, None, 0, True)
    _check(yf, lin, K)
    r2 = res.clone()
    y2 = hip.raw.linear(x, w, None, r2, 0, False)          # plain residual
    _check(y2, (x.float() @ w.float().t()).to(torch.bfloat16).float() + res.float(), K)


@pytest.mark.parametrize("M,I,K,cfg", [(636, 11008, 4096, -1), (4643, 1408, 512, -1), (100, 96, 64, -1), (300, 2816, 1024, 0),
                                       (300, 2816, 1024, 1), (300, 2816, 1024, 2), (1030, 704, 256, 5), (257, 32, 128, 5)])
def test_linear_swiglu_epilogue(dev, M, I, K, cfg):
    """Gate/up projection with the activation in the GEMM epilogue == GEMM, then the activation kernel
    (bitwise: both round the two factors to bf16 before multiplying), on every tile config."""
    from eventgpt_amd.ops import hip
    x, w = _rand(M, K, dev=dev), _rand(2 * I, K, dev=dev, seed=1, scale=0.05)
    hip.raw.gemm_force_config(cfg)
    try:
        fused = hip.raw.linear_swiglu(x, w)
        again = hip.raw.linear_swiglu(x, w)
    finally:
        hip.raw.gemm_force_config(-1)
    plain = hip.raw.swiglu(hip.raw.linear(x, w, None, None, 0, False))
    assert fused.shape == (M, I) and torch.equal(fused, again)
    gu = x.float() @ w.float().t()
    want = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
    _check(fused, want, K)
    assert torch.allclose(fused.float(), plain.float(), atol=2e-2 * float(want.abs().max()), rtol=2e-2)


@pytest.mark.parametrize("M,N,K", [(4643, 4096, 4096), (4643, 4096, 11008), (4000, 4608, 4160),
                                   (2115, 4096, 11008), (1500, 4096, 8192)])   # the last two: one partial round, all tiles split
def test_last_round_tiles_with_k_split(dev, M, N, K):
    """Default dispatch of a shape whose 256 x 256 tiles are one full round plus a few: the few run the
    8-wave kernel with K split over the idle CUs (fp32 slabs + reduce, bias / activation / residual applied
    by the reduce).  Same result as with the split switched off (those columns on the 4-wave kernel) up to
    the summation order, repeatable, and right against fp32."""
    from eventgpt_amd.ops import hip
    raw = hip.raw
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    want = torch.nn.functional.gelu(x.float() @ w.float().t() + bias.float()).to(torch.bfloat16).float() + res.float()
    try:
        raw.gemm_enable_tail_splitk(True)
        first = None
        for _ in range(3):
            y = raw.linear(x, w, bias, res, 1, False)
            first = y if first is None else first
            assert torch.equal(y, first)
        raw.gemm_enable_tail_splitk(False)
        off = raw.linear(x, w, bias, res, 1, False)
    finally:
        raw.gemm_enable_tail_splitk(True)
    _check(first, want, K)
    assert torch.allclose(first.float(), off.float(), atol=3e-2, rtol=2e-2)
    # fp32 output path as well
    yf = raw.linear(x, w, None, None, 0, True)
    _check(yf, x.float() @ w.float().t(), K)


# two to four row tiles: the fewest and most rows, one round, a few tiles past it, two rounds of them against three of the others
@pytest.mark.parametrize("M,N,K", [(257, 22016, 2048), (400, 16640, 2112), (767, 11008, 2048), (636, 22016, 2048), (520, 28672, 2048), (700, 12288, 4096), (900, 9216, 2048)])
def test_two_to_four_row_tiles(dev, M, N, K):
    from eventgpt_amd.ops import hip
    raw = hip.raw
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    y = x.float() @ w.float().t()
    _check(raw.linear(x, w, None, None, 0, False), y, K)
    _check(raw.linear(x, w, bias, res, 1, False), torch.nn.functional.gelu(y + bias.float()).to(torch.bfloat16).float() + res.float(), K)
    _check(raw.linear_partial(x, w).sum(0), y, K)
    _check(raw.linear_swiglu(x, w), torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:], K)


# columns and epilogues that the four-wave kernel does not take: (plain, with a residual, an fp32 output with a bias) on the eight-wave kernel
@pytest.mark.parametrize("M,N,K,eight", [(300, 32003, 4096, (1, 1, 1)), (636, 32003, 4096, (1, 1, 1)), (500, 20483, 2048, (1, 0, 1)),
                                         (548, 13159, 2048, (0, 0, 0)), (548, 13160, 2048, (0, 0, 0)), (640, 5002, 8192, (0, 0, 0))])
def test_two_to_four_row_tiles_of_other_columns(dev, M, N, K, eight):
    from eventgpt_amd.ops import hip
    from torch.profiler import ProfilerActivity, profile
    raw = hip.raw
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    y = x.float() @ w.float().t()
    calls = [(lambda: raw.linear(x, w, None, None, 0, False), y), (lambda: raw.linear(x, w, None, res, 0, False), y.to(torch.bfloat16).float() + res.float()),
             (lambda: raw.linear(x, w, bias, None, 0, True), y + bias.float())]
    for (call, want), on in zip(calls, eight):
        with profile(activities=[ProfilerActivity.CUDA]) as p:
            got = call()
            torch.cuda.synchronize()
        _check(got, want, K)
        ran = [e.key for e in p.key_averages() if "gemm" in e.key]
        served = N % 8 == 0 and got.dtype == torch.bfloat16
        assert any(("gemm_quad_kernel" if served else "gemm256_kernel" if on else "gemm_bf16_kernel") in k for k in ran), ran


# slabs of three row tiles in K splits: the lines at 513 rows and at 170 tiles of 128 x 128
@pytest.mark.parametrize("M,N,K", [(513, 4480, 8192), (641, 4096, 8192), (640, 4096, 8192), (767, 5120, 8256)])
def test_slabs_of_three_row_tiles(dev, M, N, K):
    from eventgpt_amd.ops import hip
    raw = hip.raw
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    res, want = _rand(M, N, dev=dev, seed=3), x.float() @ w.float().t()
    _check(raw.linear_partial(x, w).sum(0), want, K)
    _check(raw.linear(x, w, None, res, 0, False), want.to(torch.bfloat16).float() + res.float(), K)


@pytest.mark.parametrize("M,I,K", [(2115, 4096, 1024), (1500, 11008, 512), (2115, 11008, 4096)])
def test_swiglu_gemm_last_tiles_on_small_tiles(dev, M, I, K):
    """The gate/up GEMM with the SwiGLU epilogue when its 256 x 128 output tiles are whole rounds plus a
    handful: those columns run 64 x 64 tiles (a second launch over a column range of the packed
    [gate | up] matrix).  Same result as the single launch, right against fp32."""
    from eventgpt_amd.ops import hip
    raw = hip.raw
    x, w = _rand(M, K, dev=dev), _rand(2 * I, K, dev=dev, seed=1, scale=0.05)
    gu = x.float() @ w.float().t()
    want = torch.nn.functional.silu(gu[:, :I].to(torch.bfloat16).float()) * gu[:, I:].to(torch.bfloat16).float()
    try:
        raw.gemm_enable_tail_splitk(True)
        y = raw.linear_swiglu(x, w)
        assert torch.equal(y, raw.linear_swiglu(x, w))
        raw.gemm_enable_tail_splitk(False)
        one = raw.linear_swiglu(x, w)
    finally:
        raw.gemm_enable_tail_splitk(True)
    _check(y, want, K)
    assert torch.allclose(y.float(), one.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("M,N,K", [(128, 256, 64), (128, 256, 192), (636, 4096, 4096), (636, 12288, 4096), (300, 264, 320),
                                   (1000, 520, 1024), (37, 4096, 512)])
def test_forced_128_row_variant_matches_fp32(dev, M, N, K):
    """The 8-phase schedule on a 128 x 256 tile (config 6): values, determinism, bias / activation / residual
    epilogue, an identity operand against an asymmetric one, and K split over its slabs."""
    from eventgpt_amd.ops import hip
    raw = hip.raw
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    want = x.float() @ w.float().t()
    raw.gemm_force_config(6)
    try:
        first = None
        for rep in range(3):
            y = raw.linear(x, w, None, None, 0, False)
            _check(y, want, K)
            first = y if first is None else first
            assert torch.equal(y, first), rep
        bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
        y = raw.linear(x, w, bias, res, 1, False)
        _check(y, torch.nn.functional.gelu(want + bias.float()).to(torch.bfloat16).float() + res.float(), K)
        if K >= 1024:
            raw.gemm_force_splitk(2)
            _check(raw.linear(x, w, None, None, 0, False), want, K)
            raw.gemm_force_splitk(0)
        n = 256
        eye = torch.eye(n, device=dev, dtype=torch.bfloat16)
        wa = (torch.arange(n * 520, device=dev).reshape(520, n) % 251).to(torch.bfloat16)
        assert torch.equal(raw.linear(eye, wa, None, None, 0, False), wa.t())
    finally:
        raw.gemm_force_splitk(0)
        raw.gemm_force_config(-1)


@pytest.mark.parametrize("M,N,K", [(4643, 4608, 192), (4643, 4608, 64), (5000, 5000, 1024), (4643, 12288, 512),
                                   (23080, 1024, 320)])
def test_forced_256_walks_several_tiles_per_workgroup(dev, force256, M, N, K):
    """More tiles than CUs: a workgroup runs its tiles one after the other and stages the next tile's first
    K-tile under the epilogue of the current one.  Values, determinism, bias + residual, and equality with the
    one-workgroup-per-tile launch."""
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    want = x.float() @ w.float().t()
    y = force256.linear(x, w, None, None, 0, False)
    _check(y, want, K)
    for rep in range(3):
        assert torch.equal(force256.linear(x, w, None, None, 0, False), y), rep
    yb = force256.linear(x, w, bias, res, 0, False)
    _check(yb, (want + bias.float()).to(torch.bfloat16).float() + res.float(), K)
    force256.gemm_persist_256(False)
    try:
        assert torch.equal(force256.linear(x, w, None, None, 0, False), y)
        assert torch.equal(force256.linear(x, w, bias, res, 0, False), yb)
    finally:
        force256.gemm_persist_256(True)


def test_persistent_256_with_k_split_glu_and_kstrided_operands(dev, force256):
    from eventgpt_amd.ops import differentiable as diff
    # K split: tile x split pairs beyond the CU count
    x, w = _rand(2600, 2048, dev=dev), _rand(2560, 2048, dev=dev, seed=1, scale=0.05)
    force256.gemm_force_splitk(4)
    try:
        _check(force256.linear(x, w, None, None, 0, False), x.float() @ w.float().t(), 2048)
    finally:
        force256.gemm_force_splitk(0)
    # SwiGLU epilogue, 19 x 22 = 418 tiles
    x, wg = _rand(4643, 512, dev=dev), _rand(2 * 2816, 512, dev=dev, seed=2, scale=0.05)
    h = force256.linear_swiglu(x, wg)
    g, u = (x.float() @ wg.float().t()).to(torch.bfloat16).float().chunk(2, -1)
    _check(h, torch.nn.functional.silu(g) * u, 512)
    # K-strided operands: dgrad and wgrad of a 5000-row batch
    gy, w2, x2 = _rand(5000, 4608, dev=dev, scale=0.5), _rand(4608, 4352, dev=dev, seed=1, scale=0.05), _rand(5000, 4352, dev=dev, seed=2)
    _check(diff.linear_dgrad(gy, w2), gy.float() @ w2.float(), 4608)
    _check(diff.linear_wgrad(gy, x2), gy.float().t() @ x2.float(), 5000)


@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (65, 136, 128), (577, 4096, 1024), (700, 2056, 320), (64, 128, 1024),
                                   (1154, 4096, 1024), (1155, 3080, 320), (1700, 2056, 64), (1601, 2048, 192)])
def test_eight_waves_on_the_64_row_tile(dev, M, N, K):
    """The 64 x 128 tile of eight waves, forced: under 400 tiles with three stages, the last four with two; row and column
    remainders, one K-tile and contractions that are no multiple of the stages, bias, activation and residual, argmax partials;
    and as the rule takes it.  Repeats are equal."""
    from eventgpt_amd.ops import hip
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    lin = x.float() @ w.float().t() + bias.float()
    want = torch.nn.functional.gelu(lin).to(torch.bfloat16).float() + res.float()
    try:
        hip.raw.gemm_force_config(7)
        y = hip.raw.linear(x, w, bias, res, 1, False)
        _check(y, want, K)
        for _ in range(3):
            assert torch.equal(hip.raw.linear(x, w, bias, res, 1, False), y)
        _check(hip.raw.linear(x, w, bias, None, 0, True), lin, K)
        pv, pi = hip.raw.linear_argmax_partials(x, w, bias)
        got = pi.gather(1, pv.argmax(1, keepdim=True))[:, 0].long()
        assert torch.equal(lin.gather(1, got[:, None]).to(torch.bfloat16), lin.max(1, keepdim=True).values.to(torch.bfloat16))
    finally:
        hip.raw.gemm_force_config(-1)
    _check(hip.raw.linear(x, w, bias, res, 1, False), want, K)


# either side of the lines between the tiles for short contractions: one and two rounds of 128 x 128 tiles, of 256 x 256 tiles; and
# of the line at 336 tiles of 128 x 128 where rows leave some half empty
@pytest.mark.parametrize("M,N,K", [(256, 32000, 1024), (836, 8192, 640), (836, 8192, 704), (2308, 3072, 320), (2308, 4096, 384), (3300, 2560, 1024),
                                   (2885, 3072, 1024), (2885, 4096, 960), (156, 21504, 2048), (156, 22016, 2048), (156, 21376, 2048)])
def test_short_contractions_beside_the_lines_of_the_tile_choice(dev, M, N, K):
    from eventgpt_amd.ops import hip
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    lin = x.float() @ w.float().t() + bias.float()
    _check(hip.raw.linear(x, w, bias, None, 0, True), lin, K)
    _check(hip.raw.linear(x, w, bias, res, 0, False), lin.to(torch.bfloat16).float() + res.float(), K)
    _check(hip.raw.linear(x, w, bias, None, 1, False), torch.nn.functional.gelu(lin), K)


@pytest.mark.parametrize("M,N,K,slabs", [(1154, 1024, 4096, 3), (2885, 1024, 4096, 2), (900, 4096, 4096, 2), (1025, 1024, 4160, 3)])
def test_slabs_of_about_a_round_of_tiles(dev, M, N, K, slabs):
    """Products whose caller sums the slabs, split where 128 x 128 tiles are at most one a CU: the slabs add up."""
    from eventgpt_amd.ops import hip
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    part = hip.raw.linear_partial(x, w)
    assert part.shape == (slabs, M, N)
    _check(part.sum(0), x.float() @ w.float().t(), K)


def _kernels(fn):
    """What ``fn`` returns and the names of the kernels it launches."""
    fn()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out = fn()
        torch.cuda.synchronize()
    return out, [e.key for e in prof.key_averages() if "evgpt" in e.key]


def _act(h, act):
    return (h, torch.nn.functional.gelu(h), h * torch.sigmoid(1.702 * h))[act]


@pytest.mark.parametrize("M,N,K,act", [(33, 8, 128, 0), (257, 264, 128, 2), (300, 520, 192, 1), (5000, 4104, 128, 0), (5000, 4104, 192, 2),
                                       (9000, 2056, 320, 0)])
def test_four_waves_on_the_256_tile(dev, force256, M, N, K, act):
    """``gemm_quad.hip``: two and odd numbers of K-tiles, one and several output tiles a workgroup, ragged rows and columns, every
    epilogue it has, against fp32 (``_check``'s bound: bf16 operands and outputs); the same bits from run to run."""
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    lin = x.float() @ w.float().t() + bias.float()
    want = _act(lin, act).to(torch.bfloat16).float() + res.float()
    first, ran = _kernels(lambda: force256.linear(x, w, bias, res, act, False))
    assert len(ran) == 1 and "gemm_quad_kernel" in ran[0], ran
    _check(first, want, K)
    for _ in range(3):
        assert torch.equal(force256.linear(x, w, bias, res, act, False), first)
    if N % 16 == 0 or act:
        return
    half = N // 2 // 32 * 32                              # gated: gate rows, then up rows
    gu = x.float() @ w[:2 * half].float().t()
    if half >= 16:
        g, u = gu[:, :half].to(torch.bfloat16).float(), gu[:, half:].to(torch.bfloat16).float()
        gated, ran = _kernels(lambda: force256.linear_swiglu(x, w[:2 * half].contiguous()))
        assert len(ran) == 1 and "gemm_quad_kernel" in ran[0], ran
        _check(gated, torch.nn.functional.silu(g) * u, K)


@pytest.mark.parametrize("M,N,K,kind,quad", [
    (2600, 5120, 576, "plain", False), (2600, 5120, 640, "plain", True), (2600, 9216, 192, "plain", False), (2600, 9216, 256, "plain", True),
    (2600, 5120, 1024, "slabs", False), (2600, 5120, 1088, "slabs", True), (2600, 9216, 192, "slabs", False), (2600, 9216, 256, "slabs", True),
    (2600, 5120, 1024, "gated", False), (2600, 5120, 1088, "gated", True), (2600, 9216, 768, "gated", False), (2600, 9216, 832, "gated", True),
    (2600, 5120, 128, "residual", True), (2600, 5120, 128, "bias", True), (2600, 5120, 128, "gelu", True), (2600, 5120, 64, "bias", False)])
def test_which_kernel_takes_256_tiles(dev, M, N, K, kind, quad):
    """Both sides of every line of ``gemm_quad_ahead``: the kernel it names runs, and its result is right and what the tiles forced onto the
    other kernel's shapes give (``_check``'s bound; plain, bias and residual bit for bit what the general tiles make of the product)."""
    from eventgpt_amd.ops import hip
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    fn = dict(plain=lambda: hip.raw.linear(x, w, None, None, 0, False), slabs=lambda: hip.raw.linear_partial(x, w),
              gated=lambda: hip.raw.linear_swiglu(x, w), residual=lambda: hip.raw.linear(x, w, None, res, 0, False),
              bias=lambda: hip.raw.linear(x, w, bias, None, 0, False), gelu=lambda: hip.raw.linear(x, w, bias, None, 1, False))[kind]
    got, ran = _kernels(fn)
    assert len(ran) == 1 and ("gemm_quad_kernel" if quad else "gemm256_kernel") in ran[0], ran
    lin = x.float() @ w.float().t()
    half = N // 2
    want = dict(plain=lambda: lin, slabs=lambda: lin, residual=lambda: lin.to(torch.bfloat16).float() + res.float(),
                bias=lambda: lin + bias.float(), gelu=lambda: _act(lin + bias.float(), 1),
                gated=lambda: torch.nn.functional.silu(lin[:, :half].to(torch.bfloat16).float()) * lin[:, half:].to(torch.bfloat16).float())[kind]()
    _check(got.sum(0) if kind == "slabs" else got, want, K)
    if kind in ("plain", "bias", "residual"):
        hip.raw.gemm_force_config(0)
        other, ran = _kernels(fn)
        hip.raw.gemm_force_config(-1)
        assert "gemm_bf16_kernel" in ran[0] and torch.equal(got, other)


RING = {"64x64": "<2, 1, 2, 4, 4,", "128x64": "<2, 2, 4, 2, 5,", "64x128": "<2, 2, 2, 4, 5,", "64x192": "<2, 3, 2, 4, 4,",
        "128x128": "<4, 2, 2, 4, 4,"}


def _ring_tile(ran):
    """The tile of ``gemm_ring.hip`` that ran, None: another kernel's."""
    assert len(ran) == 1, ran
    return next((t for t, args in RING.items() if "gemm_ring_kernel" + args in ran[0]), None)


@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("M,N,K,tile", [(577, 1000, 576, "64x64"), (577, 3080, 1024, "128x64"), (4039, 500, 1088, "128x64"), (576, 3400, 384, "64x128"),
                                        (577, 4104, 64, "64x192"), (577, 4096, 1024, "64x192"), (1154, 3064, 1088, "128x128"), (257, 9800, 1088, "128x128")])
def test_one_round_of_tiles_on_the_deep_ring(dev, M, N, K, act, tile):
    """``gemm_ring.hip`` by the rule that chooses it: all five tiles with bias, every activation and a residual, ragged rows and columns, rows
    walked along either side of the output, fewer K-tiles than the ring, bf16 and fp32 out, against fp32 (``_check``'s bound); the same bits from
    run to run."""
    from eventgpt_amd.ops import hip
    if (tile, K, act) == ("64x192", 64, 2):
        pytest.skip("eight waves on 64 x 128 take quick-gelu over so short a contraction")
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    lin = x.float() @ w.float().t()
    h = _act(lin + bias.float(), act).to(torch.bfloat16).float()
    first, ran = _kernels(lambda: hip.raw.linear(x, w, bias, res, act, False))
    assert _ring_tile(ran) == tile, ran
    _check(first, h + res.float(), K)
    for _ in range(3):
        assert torch.equal(hip.raw.linear(x, w, bias, res, act, False), first)
    y, ran = _kernels(lambda: hip.raw.linear(x, w, bias, None, act, False))
    assert _ring_tile(ran) == tile, ran
    _check(y, h, K)
    if act == 0:
        y, ran = _kernels(lambda: hip.raw.linear(x, w, None, None, 0, True))
        assert _ring_tile(ran) == tile, ran
        _check(y, lin, K)


@pytest.mark.parametrize("M,N,K,tile", [(577, 1000, 64, "64x64"), (577, 3080, 64, "128x64"), (576, 3400, 64, "64x128"), (300, 4096, 128, "128x64")])
def test_activations_over_fewer_k_tiles_than_the_ring(dev, M, N, K, tile):
    from eventgpt_amd.ops import hip
    x, w, bias = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05), _rand(N, dev=dev, seed=2)
    for act in (1, 2):
        y, ran = _kernels(lambda: hip.raw.linear(x, w, bias, None, act, False))
        assert _ring_tile(ran) == tile, ran
        _check(y, _act(x.float() @ w.float().t() + bias.float(), act), K)


@pytest.mark.parametrize("M,N,K,tile", [(577, 1024, 4096, "128x64"), (1154, 1024, 4096, "128x128")])
def test_split_contractions_on_the_deep_ring(dev, M, N, K, tile):
    """K in splits, as fp32 slabs and (with the sum's launch) as a finished product."""
    from eventgpt_amd.ops import hip
    x, w, bias = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05), _rand(N, dev=dev, seed=2)
    lin = x.float() @ w.float().t()
    slabs, ran = _kernels(lambda: hip.raw.linear_partial(x, w))
    assert slabs.shape[0] > 1 and _ring_tile(ran) == tile, (slabs.shape, ran)
    _check(slabs.sum(0), lin, K)
    assert torch.equal(hip.raw.linear_partial(x, w), slabs)
    _check(hip.raw.linear(x, w, bias, None, 2, False), _act(lin + bias.float(), 2), K)


@pytest.mark.parametrize("M,half,K,tile", [(33, 4640, 576, "128x64"), (577, 1536, 64, "128x64"), (4039, 192, 128, "128x64"), (192, 4160, 1024, "64x128"),
                                           (1154, 1536, 192, "128x128"), (3000, 480, 256, "128x128"), (300, 5056, 1024, "128x128")])
def test_gated_products_on_the_deep_ring(dev, M, half, K, tile):
    from eventgpt_amd.ops import hip
    x, w = _rand(M, K, dev=dev), _rand(2 * half, K, dev=dev, seed=1, scale=0.05)
    lin = x.float() @ w.float().t()
    g, u = lin[:, :half].to(torch.bfloat16).float(), lin[:, half:].to(torch.bfloat16).float()
    first, ran = _kernels(lambda: hip.raw.linear_swiglu(x, w))
    assert _ring_tile(ran) == tile, ran
    _check(first, torch.nn.functional.silu(g) * u, K)
    for _ in range(3):
        assert torch.equal(hip.raw.linear_swiglu(x, w), first)


@pytest.mark.parametrize("M,N,K,kind,tile", [
    (577, 3080, 192, "plain", None), (577, 3080, 256, "plain", "128x64"), (577, 3080, 320, "f32", None), (577, 3080, 384, "f32", "128x64"),
    (577, 3080, 320, "residual", None), (577, 3080, 384, "residual", "128x64"), (577, 3080, 64, "bias", "128x64"),
    (577, 1664, 512, "bias", None), (577, 1664, 576, "bias", "128x64"), (577, 1664, 2048, "residual", None), (577, 1664, 2112, "residual", "128x64"),
    (577, 1664, 512, "quick-gelu", None), (577, 1664, 576, "quick-gelu", "128x64"), (577, 1664, 1024, "gelu", None), (577, 1664, 1088, "gelu", "128x64"),
    (577, 1000, 128, "plain", None), (577, 1000, 192, "plain", "64x64"), (700, 1000, 64, "plain", "64x64"), (577, 1000, 192, "residual", None),
    (577, 900, 512, "residual", None), (577, 900, 576, "residual", "64x64"), (1154, 3064, 320, "plain", None), (1154, 3064, 384, "plain", "128x128"),
    (1154, 3064, 1024, "bias", None), (577, 4104, 192, "quick-gelu", None), (577, 4104, 256, "quick-gelu", "64x192")])
def test_which_products_go_on_the_deep_ring(dev, M, N, K, kind, tile):
    """Both sides of the lines of ``gemm_ring_tile``: the tile it names runs (None: a kernel of ``gemm.hip``), and the result is bit for bit what a
    general tile makes of the product."""
    from eventgpt_amd.ops import hip
    x, w = _rand(M, K, dev=dev), _rand(N, K, dev=dev, seed=1, scale=0.05)
    bias, res = _rand(N, dev=dev, seed=2), _rand(M, N, dev=dev, seed=3)
    fn = dict(plain=lambda: hip.raw.linear(x, w, None, None, 0, False), f32=lambda: hip.raw.linear(x, w, None, None, 0, True),
              residual=lambda: hip.raw.linear(x, w, None, res, 0, False), bias=lambda: hip.raw.linear(x, w, bias, None, 0, False),
              gelu=lambda: hip.raw.linear(x, w, bias, None, 1, False))
    fn["quick-gelu"] = lambda: hip.raw.linear(x, w, bias, None, 2, False)
    got, ran = _kernels(fn[kind])
    assert _ring_tile(ran) == tile, ran
    hip.raw.gemm_force_config(1)
    other, ran = _kernels(fn[kind])
    hip.raw.gemm_force_config(-1)
    assert "gemm_bf16_kernel" in ran[0] and torch.equal(got, other)


@pytest.mark.parametrize("m,n,k", [(1027, 8192, 1088), (1027, 8196, 1088), (1027, 8195, 1088), (2060, 4096, 1024), (1100, 14336, 1152),
                                   (1100, 14340, 4096), (200, 1028, 640), (70, 131, 192)])
def test_fp32_outputs(m, n, k):
    """Sums stored as they are: whole and ragged columns, contractions on both sides of the lines between the kernels, columns in two launches
    (280 tiles), and the same product with an addend, which the general epilogue keeps."""
    from eventgpt_amd.ops import hip
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, bias = (torch.randn(s, generator=g, device="cuda").bfloat16() for s in ((m, k), (n, k), (n,)))
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    # an element is K / 32 additions to a register and the sums of 32 inside the matrix instruction, 2^-24 of the sum so far each
    bound = (k / 32 + 32) * 2.0 ** -24 * size
    assert bool(((hip.raw.linear(a, w, None, None, 0, True).double() - want).abs() <= bound).all())
    y = hip.raw.linear(a, w, bias, None, 0, True).double() - bias.double()
    assert bool(((y - want).abs() <= bound + 2.0 ** -23 * (want + bias.double()).abs()).all())


@pytest.mark.parametrize("m,n,t", [(1032, 8192, 1100), (1032, 8192, 70), (264, 1032, 130), (72, 8, 64)])
def test_fp32_weight_gradients(m, n, t):
    """dY^T X into a new tensor and into a slice of a flat buffer whose neighbours stay."""
    from eventgpt_amd.ops import hip
    g = torch.Generator(device="cuda").manual_seed(m + n + t)
    a, w = (torch.randn(s, generator=g, device="cuda").bfloat16() for s in ((t, m), (t, n)))
    want, size = a.double().T @ w.double(), a.double().abs().T @ w.double().abs()
    bound = (t / 32 + 32) * 2.0 ** -24 * size
    kk = (t + 63) // 64 * 64
    assert bool(((hip.raw.linear_t(a, w, True, True, None, None, 0, True, kk).double() - want).abs() <= bound).all())
    for at in (4, 3):                                 # aligned and not
        flat = torch.full((m * n + 8,), 7.0, device="cuda")
        hip.raw.linear_t(a, w, True, True, None, None, 0, True, kk, flat[at:at + m * n].view(m, n))
        assert bool(((flat[at:at + m * n].view(m, n).double() - want).abs() <= bound).all())
        assert bool((flat[:at] == 7).all()) and bool((flat[at + m * n:] == 7).all())


@pytest.mark.parametrize("m,n,k", [(40, 516, 320), (40, 514, 320), (300, 260, 192), (577, 1024, 1024), (577, 1028, 256), (1154, 3076, 128),
                                   (130, 4100, 640), (836, 4096, 576)])
def test_bias_and_residual(m, n, k):
    """Whole and broken quads of columns, edges of tiles, with a bias, a residual and both."""
    from eventgpt_amd.ops import hip
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, b, r = (torch.randn(s, generator=g, device="cuda").bfloat16() for s in ((m, k), (n, k), (n,), (m, n)))
    sums, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    exact = (k / 32 + 32) * 2.0 ** -24 * size                # (as in test_fp32_outputs)
    for bias, res in ((b, None), (None, r), (b, r)):
        mid = sums + (bias.double() if bias is not None else 0)
        want = mid + (res.double() if res is not None else 0)
        y = hip.raw.linear(a, w, bias, res, 0, False).double()
        # bf16 rounds by up to 2^-8 of the value (8 significant bits): the sum with the bias, then the total with the residual
        bound = exact + 2.0 ** -8 * 1.01 * (want.abs() + (mid.abs() + exact if res is not None else 0)) + 1e-30
        assert bool(((y - want).abs() <= bound).all()), (bias is None, res is None)


@pytest.mark.parametrize("m,n,k", [(33, 16, 4096), (300, 22, 4096), (40, 4100, 2048), (577, 1024, 4096), (836, 4096, 8192), (1800, 4096, 8192)])
def test_sums_of_split_products(m, n, k):
    """Two to sixteen slabs, whole and broken quads of columns: bias, activation, residual and fp32 outputs of the pass that adds them."""
    from eventgpt_amd.ops import hip
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, b, r = (torch.randn(s, generator=g, device="cuda").bfloat16() for s in ((m, k), (n, k), (n,), (m, n)))
    w = (w * 0.03125).contiguous()
    sums, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    exact = (k / 32 + 32) * 2.0 ** -24 * size                # (as in test_fp32_outputs; the slabs' sum is a few additions of these)
    for bias, res, act in ((None, None, 0), (b, None, 0), (None, r, 0), (b, r, 0), (b, r, 1)):
        mid = sums + (bias.double() if bias is not None else 0)
        if act:
            mid = torch.nn.functional.gelu(mid)              # (slope at most 1.13; its value in fp32 to 2^-20)
        want = mid + (res.double() if res is not None else 0)
        near = 1.13 * exact + 2.0 ** -20 * (mid.abs() + 1)
        for f32 in (False, True):
            y = hip.raw.linear(a, w, bias, res, act, f32).double()
            # 2^-8 of the value where bf16 holds it: the sum before a residual is added, and a bf16 result
            bound = near + 2.0 ** -8 * 1.01 * ((mid.abs() + near if res is not None else 0) + (0 if f32 else want.abs() + near))
            assert bool(((y - want).abs() <= bound).all()), (bias is None, res is None, act, f32)
