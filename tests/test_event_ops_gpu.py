"""GPU event front end vs the numpy implementation."""
import numpy as np
import pytest
import torch

from eventgpt_amd.data import clip_preprocess as cp
from eventgpt_amd.data.events import (polarity_histogram, rasterize, slice_bounds_by_count,
                                      synthetic_events, voxel_grid)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("conflict", ["last", "negative"])
def test_raster_matches_numpy(dev, conflict):
    from eventgpt_amd.ops import event_ops as eo
    ev = synthetic_events(50_000, 160, 120, seed=4)
    d = eo.events_to_device(ev, dev)
    img = eo.rasterize_gpu(d, 5, (120, 160), conflict).cpu().numpy()
    for i, (a, b) in enumerate(slice_bounds_by_count(50_000, 5)):
        want = rasterize(ev["x"][a:b], ev["y"][a:b], ev["p"][a:b], size=(120, 160), conflict=conflict)
        assert np.array_equal(img[i], want), i


def test_voxel_and_histogram_match_numpy(dev):
    from eventgpt_amd.ops import event_ops as eo
    ev = synthetic_events(30_000, 64, 48, seed=2)
    d = eo.events_to_device(ev, dev)
    hist, vox = eo.voxel_grid_gpu(d, 5, (48, 64))
    assert np.array_equal(hist.cpu().numpy(), polarity_histogram(ev, 5, (48, 64)))
    assert np.allclose(vox.cpu().numpy(), voxel_grid(ev, 5, (48, 64)))
    _, voxc = eo.voxel_grid_gpu(d, 5, (48, 64), signed=False, by="count")
    assert np.allclose(voxc.cpu().numpy(), voxel_grid(ev, 5, (48, 64), signed=False, by="count"))


@pytest.mark.parametrize("n,hw,bins", [(200_000, (480, 640), 5), (70_001, (97, 130), 3), (5000, (48, 64), 7)])
@pytest.mark.parametrize("by", ["time", "count"])
@pytest.mark.parametrize("chunks", [0, 1, 37])
def test_voxel_lds_bands_equal_atomic_kernel_and_numpy(dev, n, hw, bins, by, chunks):
    """The kernel that orders events in LDS (``chunks`` 0), the per-band LDS histogram (one chunk and several) and the
    one-atomic-per-event kernel give identical counts; all match the host implementation, with out-of-canvas events dropped."""
    from eventgpt_amd.ops import event_ops as eo
    ev = synthetic_events(n, hw[1] + 6, hw[0] + 4, seed=n % 97)      # some events fall outside the canvas
    d = eo.events_to_device(ev, dev)
    h_lds, v_lds = eo.voxel_grid_gpu(d, bins, hw, by=by, privatised=True, chunks=chunks)
    h_at, v_at = eo.voxel_grid_gpu(d, bins, hw, by=by, privatised=False)
    assert torch.equal(h_lds, h_at) and torch.equal(v_lds, v_at)
    inside = (ev["x"] < hw[1]) & (ev["y"] < hw[0])
    assert int(h_lds.sum()) == int(inside.sum())
    if by == "time":
        keep = {k: v[inside] for k, v in ev.items()}
        t0, t1 = int(ev["t"].min()), int(ev["t"].max())
        b = np.clip(((keep["t"] - t0).astype(np.float64) / max(t1 - t0, 1) * bins).astype(np.int64), 0, bins - 1)
        want = np.zeros((bins, 2) + hw, np.int64)
        np.add.at(want, (b, (keep["p"] != 0).astype(np.int64), keep["y"], keep["x"]), 1)
        assert np.array_equal(h_lds.cpu().numpy(), want)


@pytest.mark.parametrize("chunks", [0, 1])
def test_voxel_unsorted_stream(dev, chunks):
    """Ordered in LDS, or, where index ranges are asked for (``chunks``) that it does not have, by the atomic kernel."""
    from eventgpt_amd.ops import event_ops as eo
    ev = synthetic_events(20_000, 64, 48, seed=5)
    perm = np.random.default_rng(0).permutation(20_000)
    shuffled = {k: v[perm] for k, v in ev.items()}
    d = eo.events_to_device(shuffled, dev)
    assert eo._bin_bounds(d, 5, "time", int(ev["t"].min()), int(ev["t"].max() - ev["t"].min())) is None
    hist, _ = eo.voxel_grid_gpu(d, 5, (48, 64), privatised=True, chunks=chunks)
    assert np.array_equal(hist.cpu().numpy(), polarity_histogram(ev, 5, (48, 64)))


@pytest.mark.parametrize("order", ["sorted", "shuffled", "constant", "one bin late"])
@pytest.mark.parametrize("n,hw,bins", [(1, (3, 5), 2), (8192, (48, 64), 5), (8193, (1, 700), 9), (40_001, (97, 130), 3),
                                       (30_000, (2, 19200), 2), (20_000, (480, 64), 8)])
@pytest.mark.parametrize("by", ["time", "count"])
def test_voxel_sorting_kernels_equal_the_atomic_kernel(dev, n, hw, bins, by, order):
    """Events ordered by (bin, band) in LDS: chunk remainders, chunks of several bins, streams in any order, widths of
    one-row bands, events outside the image.  Whole numbers: equal."""
    from eventgpt_amd.ops import event_ops as eo, hip
    g = torch.Generator().manual_seed(n + bins)
    t = {"sorted": torch.sort(torch.randint(0, 1000, (n,), generator=g)).values, "shuffled": torch.randint(-50, 1000, (n,), generator=g),
         "constant": torch.full((n,), 7), "one bin late": (torch.arange(n) >= n - 1).long() * 100}[order]
    d = {"x": torch.randint(-2, hw[1] + 2, (n,), generator=g, dtype=torch.int32), "t": t,
         "y": torch.randint(-1, hw[0] + 2, (n,), generator=g, dtype=torch.int32),
         "p": torch.randint(-1, 2, (n,), generator=g, dtype=torch.int32)}
    d = {k: v.to(dev) for k, v in d.items()}
    assert hip.raw.event_voxel_sorted_ok(bins, *hw)
    for signed in (True, False):
        h, v = eo.voxel_grid_gpu(d, bins, hw, signed=signed, by=by, privatised=True)
        h_at, v_at = eo.voxel_grid_gpu(d, bins, hw, signed=signed, by=by, privatised=False)
        assert torch.equal(h, h_at) and torch.equal(v, v_at)
    if order == "sorted" and hw[1] < 19200:      # the band kernel that serves other timestamp types
        h, v = eo.voxel_grid_gpu({**d, "t": d["t"].int()}, bins, hw, signed=False, by="time", privatised=True)
        h_at, v_at = eo.voxel_grid_gpu(d, bins, hw, signed=False, by="time", privatised=False)
        assert torch.equal(h, h_at) and torch.equal(v, v_at)


@pytest.mark.parametrize("order", ["sorted", "shuffled"])
def test_voxel_counts_over_more_chunks_than_one_pass_lists(dev, order):
    """8 192 events a chunk, 1 024 chunks a pass of the counting kernel: its list of runs is filled twice."""
    from eventgpt_amd.ops import event_ops as eo
    n, hw, bins = 1024 * 8192 + 3, (97, 130), 3
    g = torch.Generator().manual_seed(5)
    t = torch.randint(0, 100_000, (n,), generator=g)
    d = {"x": torch.randint(0, hw[1], (n,), generator=g, dtype=torch.int32), "y": torch.randint(0, hw[0], (n,), generator=g, dtype=torch.int32),
         "p": torch.randint(0, 2, (n,), generator=g, dtype=torch.int32), "t": torch.sort(t).values if order == "sorted" else t}
    d = {k: v.to(dev) for k, v in d.items()}
    (h, v), (h_at, v_at) = (eo.voxel_grid_gpu(d, bins, hw, privatised=private) for private in (True, False))
    assert int(h.sum()) == n and torch.equal(h, h_at) and torch.equal(v, v_at)


# events per chunk of the busiest band from under one load of a wave to a whole chunk; blocks of 1 024 threads (fewer than 512 blocks, or 5 000
# events each) and of 512; one pass over the chunks (4 096 and 2 048 of them) and a second one
@pytest.mark.parametrize("bins,n,spread", [(3, 20_000, 97), (3, 300_000, 40), (3, 300_000, 1), (6, 300_000, 12), (6, 300_000, 1),
                                           (6, 3_000_000, 97), (900, 2048 * 8192 + 3, 97), (3, 4096 * 8192 + 3, 97)])
def test_voxel_counts_runs_of_any_length(dev, bins, n, spread):
    from eventgpt_amd.ops import event_ops as eo
    hw, g = (97, 130), torch.Generator(device=dev).manual_seed(n + spread)
    def ints(hi):
        return torch.randint(0, hi, (n,), generator=g, device=dev, dtype=torch.int32)
    d = {"x": ints(hw[1]), "y": ints(spread) + (hw[0] - spread) // 2, "p": ints(2), "t": torch.arange(n, device=dev)}
    (h, v), (h_at, v_at) = (eo.voxel_grid_gpu(d, bins, hw, privatised=private) for private in (True, False))
    assert int(h.sum()) == n and torch.equal(h, h_at) and torch.equal(v, v_at)


@pytest.mark.parametrize("hw", [(480, 640), (120, 160), (336, 336), (400, 300)])
def test_clip_preprocess_matches_host(dev, hw):
    from eventgpt_amd.ops import event_ops as eo
    rng = np.random.default_rng(0)
    frames = rng.integers(0, 256, (2, hw[0], hw[1], 3), dtype=np.uint8)
    got = eo.clip_preprocess_gpu(torch.from_numpy(frames).to(dev)).float().cpu()
    want = torch.stack([torch.from_numpy(cp.preprocess_image(f)) for f in frames])
    assert got.shape == (2, 3, 336, 336)
    # bf16 output: compare after the same rounding
    assert torch.equal(got, want.to(torch.bfloat16).float())


def test_event_frames_gpu_end_to_end(dev):
    from eventgpt_amd.ops import event_ops as eo
    from eventgpt_amd.data.events import event_frames
    ev = synthetic_events(60_000, 640, 480, seed=9)
    size, px = eo.event_frames_gpu(ev, dev, 5)
    assert size == [480, 640] and px.shape == (5, 3, 336, 336) and px.dtype == torch.bfloat16
    host = event_frames(ev, 5)
    same_canvas = [f for f in host if f.shape[:2] == (480, 640)]
    if len(same_canvas) == 5:
        want = torch.stack([torch.from_numpy(cp.preprocess_image(f)) for f in host])
        assert torch.equal(px.float().cpu(), want.to(torch.bfloat16).float())


# pixels one by one, tiles of four and of eight rows: either side of both lines, remainders of a tile's columns and rows
@pytest.mark.parametrize("T,S", [(1, 267), (1, 268), (5, 113), (6, 113), (3, 276), (3, 277), (35, 81), (2, 32), (2, 33)])
def test_clip_preprocess_beside_the_lines_of_the_kernel_choice(dev, T, S):
    from eventgpt_amd.ops import event_ops as eo
    img = np.random.default_rng(S).integers(0, 256, (T, 200, 150, 3)).astype(np.uint8)
    got = eo.clip_preprocess_gpu(torch.from_numpy(img).to(dev), S).float().cpu().numpy()
    # as for the packed frames below: the same bytes, normalised in another order
    np.testing.assert_allclose(got, np.stack([cp.preprocess_image(f, S) for f in img]), rtol=2.0 ** -8, atol=1e-5)


@pytest.mark.parametrize("order", ["reversed", "scattered"])
def test_clip_preprocess_with_tables_of_any_order(dev, order):
    """Rows that reach further over the source than a tile holds: what a host resize by the same tables gives."""
    from eventgpt_amd.ops import hip
    rng = np.random.default_rng(4)
    H, S, taps = 300, 224, 3
    img = rng.integers(0, 256, (2, H, S, 3)).astype(np.uint8)
    start = np.linspace(0, H - taps, S).astype(np.int64)
    start = start[::-1].copy() if order == "reversed" else rng.permutation(start)
    weight = rng.dirichlet(np.ones(taps), S)
    weight = np.round(weight * (1 << 22)).astype(np.int64)
    rows = sum(weight[:, k][None, :, None, None] * img[:, start + k].astype(np.int64) for k in range(taps))
    resized = np.ascontiguousarray(np.clip((rows + (1 << 21)) >> 22, 0, 255).astype(np.uint8))
    table = [torch.from_numpy(a.astype(np.int32)).to(dev) for a in (start, np.full(S, taps), weight)]
    none = [torch.zeros(1, dtype=torch.int32, device=dev)] * 2 + [torch.zeros(1, 1, dtype=torch.int32, device=dev)]
    tail = (S, S, S, 0, 0, [0.48, 0.46, 0.41], [0.27, 0.26, 0.28])
    got = hip.raw.clip_preprocess(torch.from_numpy(img).to(dev), *none, *table, *tail)
    want = hip.raw.clip_preprocess(torch.from_numpy(resized).to(dev), *none, *none, *tail)
    assert torch.equal(got, want)


def test_preprocess_frames_device_dispatch(dev):
    """The frame preprocessing entry point gives the same pixels from the GPU kernel
    and from the host path, and the verifier's processor uses it when given a device."""
    from eventgpt_amd.ops import event_ops as eo
    rng = np.random.default_rng(3)
    frames = [rng.integers(0, 256, (120, 160, 3), dtype=np.uint8) for _ in range(4)]
    g = eo.preprocess_frames(frames, dev, 56)
    c = eo.preprocess_frames(frames, "cpu", 56)
    assert g.is_cuda and g.shape == (4, 3, 56, 56) and g.dtype == torch.bfloat16
    assert torch.equal(g.cpu(), c)
    # unequal sizes (per-slice canvases) run the kernel frame by frame: same pixels as the host path
    mixed = frames[:2] + [rng.integers(0, 256, (100, 90, 3), dtype=np.uint8)]
    m = eo.preprocess_frames(mixed, dev, 56)
    assert m.is_cuda and m.shape == (3, 3, 56, 56)
    assert torch.equal(m.cpu(), eo.preprocess_frames(mixed, "cpu", 56))
    from eventgpt_amd.data.tokenizer import ByteTokenizer
    from eventgpt_amd.models.video_llava import VideoLlavaConfig, VideoProcessor
    cfg = VideoLlavaConfig.tiny()
    proc = VideoProcessor(cfg, ByteTokenizer())
    S = cfg.vision_config.image_size
    out = proc("USER: <video>\nwhat? ASSISTANT:", frames, device=dev)
    host = proc("USER: <video>\nwhat? ASSISTANT:", frames)
    assert out["pixel_values_videos"].shape == (1, 4, 3, S, S) and out["pixel_values_videos"].is_cuda
    assert torch.equal(out["pixel_values_videos"].float().cpu(), host["pixel_values_videos"].to(torch.bfloat16).float())


def _host_stream(n, h, w, dtype, p_dtype, seed=3):
    rng = np.random.default_rng(seed)
    x, y = rng.integers(0, w, n), rng.integers(0, h, n)
    x[0], y[0] = w - 1, h - 1
    return {"x": x.astype(dtype), "y": y.astype(dtype), "p": rng.integers(0, 2, n).astype(p_dtype),
            "t": np.sort(rng.integers(0, 50_000, n))}


# bands with a short last one, rows that need no resize, a resize near the tiles' limit and one past it, one slice (short tiles),
# slices with a remainder, as many events as slices and fewer; every integer type that is packed and some that are not
@pytest.mark.parametrize("n,h,w,slices,dtype,p_dtype", [
    (20_003, 120, 160, 5, np.int16, np.int8), (7_001, 481, 640, 3, np.uint16, np.uint8), (5_000, 336, 336, 5, np.int32, np.bool_),
    (4_099, 97, 53, 7, np.int64, np.int64), (3_000, 1300, 1281, 2, np.int32, np.int32), (3_000, 1700, 1501, 2, np.int32, np.int32), (901, 60, 80, 1, np.int16, np.int8),
    (5, 40, 40, 5, np.uint8, np.uint8),
    (3, 40, 40, 5, np.int32, np.int16), (901, 60, 80, 1, np.float32, np.int8), (901, 60, 80, 4, ">i4", np.int8)])
@pytest.mark.parametrize("conflict", ["last", "negative"])
def test_packed_frames_equal_the_general_ops(dev, n, h, w, slices, dtype, p_dtype, conflict):
    from eventgpt_amd.ops import event_ops as eo
    ev = _host_stream(n, h, w, dtype, p_dtype)
    size, px = eo.event_frames_gpu(ev, dev, slices, conflict=conflict)
    img = eo.rasterize_gpu(eo.events_to_device(ev, dev), slices, (h, w), conflict)
    want = np.stack([cp.preprocess_image(f) for f in img.cpu().numpy()])
    assert size == [h, w] and torch.equal(px, eo.clip_preprocess_gpu(img))
    # the same bytes, normalised in another order: rounding to 8 significant bits is off by half of 2^(e-7), at most 2^-8 of a
    # value of 2^e or more; the float32 forms differ by a few 2^-24 of terms below 4
    np.testing.assert_allclose(px.float().cpu().numpy(), want, rtol=2.0 ** -8, atol=1e-5)


@pytest.mark.parametrize("n,h,w,slices,packs", [(4, 40, 40, 5, False), (5, 40, 40, 5, True), (500_001, 40, 40, 1, False), (500_000, 40, 40, 1, True),
                                                (1_000_001, 40, 40, 2, True), (200_000, 1500, 1700, 5, False), (199_999, 1500, 1700, 5, True)])
def test_streams_whose_words_would_not_be_used_are_not_packed(dev, n, h, w, slices, packs, monkeypatch):
    """By length, and for a long stream by its first events; the frames are the general ops' either way."""
    from eventgpt_amd.ops import event_ops as eo
    ev, seen = _host_stream(n, h, w, np.int32, np.int8), []
    monkeypatch.setattr(eo, "_packed", lambda e, pack=eo._packed: seen.append(1) or pack(e))
    size, px = eo.event_frames_gpu(ev, dev, slices)
    assert size == [h, w] and bool(seen) == packs
    assert torch.equal(px, eo.clip_preprocess_gpu(eo.rasterize_gpu(eo.events_to_device(ev, dev), slices, (h, w))))


def test_streams_that_do_not_pack_stay_on_the_general_ops(dev):
    from eventgpt_amd.ops import event_ops as eo
    good = _host_stream(50, 40, 40, np.int64, np.int8)
    assert eo._packed(good) is not None
    for key, value in (("x", np.where(np.arange(50) == 9, 1 << 33, good["x"])), ("y", np.where(np.arange(50) == 9, -1, good["y"])),
                       ("x", np.where(np.arange(50) == 9, 32768, good["x"])), ("p", good["p"][:-1]), ("p", good["p"].astype(np.float32))):
        assert eo._packed({**good, key: value}) is None
    assert eo._packed({k: v[:0] for k, v in good.items()}) is None
    locked = {k: v.copy() for k, v in good.items()}
    for v in locked.values():
        v.flags.writeable = False
    assert torch.equal(eo._packed(locked)[0], eo._packed(good)[0])


def test_words_in_flight_and_words_that_are_held_are_not_written_over(dev):
    """Clips one after another without a wait, of growing and shrinking length, on two streams and from two threads: each is what its
    events give.  Packed words that a caller still holds stay as they are while others are packed."""
    import threading
    from eventgpt_amd.ops import event_ops as eo
    clips = [_host_stream(n, 97 + i, 130, np.int32, np.int8, seed=i) for i, n in enumerate((20_000, 70_000, 5_000, 200_000, 20_001, 7))]
    want = [eo.clip_preprocess_gpu(eo.rasterize_gpu(eo.events_to_device(ev, dev), 5, (97 + i, 130))) for i, ev in enumerate(clips)]
    torch.cuda.synchronize()
    bad = []
    def go():
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        got = []
        for turn in range(3):
            for i, ev in enumerate(clips):
                with torch.cuda.stream(streams[(i + turn) % 2]):
                    got.append((i, eo.event_frames_gpu(ev, dev)[1]))
        torch.cuda.synchronize()
        bad.extend(i for i, px in got if not torch.equal(px, want[i]))
    threads = [threading.Thread(target=go) for _ in range(2)]
    [t.start() for t in threads], [t.join() for t in threads], go()
    assert not bad
    held = [eo._packed(ev)[0] for ev in clips]
    for words, ev in zip(held, clips):
        assert np.array_equal(words.numpy(), ev["x"] | ev["y"] << 15 | (ev["p"] != 0).astype(np.int32) << 30)
