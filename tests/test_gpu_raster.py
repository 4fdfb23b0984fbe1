"""The HIP rasteriser against the oracle on the same packed splats: counts,
projected records, sorted (tile, splat) pairs and tile ranges bit-exact; images
within tolerance of the oracle's restatement of the reference blend and of the
brute force, on the reference's own scenes and cameras
(tests/render/test_splat_render.cpp:70-121) and on the benchmark scenes."""
import numpy as np
import pytest

import fixtures as F
import harness as H
import oracle_lib as O
from lucabrtrender_amd import _abi, raster, scenes

pytestmark = pytest.mark.gpu

W, HGT = 250, 190


@pytest.fixture(scope="module")
def rast():
    return raster.TileRasterizer()


@pytest.fixture(scope="module")
def cloud():
    return F.random_cloud(3000, 7).decode(3)


def _cam(eye, target, **lens):
    c = raster.Camera.looking_at(eye, target)
    c.lens = raster.Lens(**lens)
    return c


CAMERAS = {
    "perspective": (_cam((1.5, 1.0, 6.0), (0, 0, 0), focal=30.0), dict()),
    "frustum-edge": (_cam((0.3, -0.2, 2.2), (0, 0, 0), focal=18.0), dict()),
    "orthographic": (_cam((0.0, 3.0, 5.0), (0, 0, 0), orthographic=True, focal=5.0), dict()),
    "no-aa-window": (_cam((-2.0, 0.5, 5.0), (0, 0, 0), window_translate=(0.2, 0.0), window_scale=(1.0, 1.3),
                          window_roll=25.0), dict(antialias=False)),
}


def _image_checks(gpu, ora, truth=None, tol_max=1e-2):
    d = np.abs(gpu["colour"].astype(np.float64) - ora["colour"])
    assert d.max() <= tol_max and np.quantile(d, 0.99) <= 1e-4, (d.max(), np.quantile(d, 0.99))
    dd = np.abs(gpu["depth"].astype(np.float64) - ora["depth"])
    assert np.quantile(dd, 0.99) <= 1e-4 * max(1.0, float(np.abs(ora["depth"]).max()))
    if truth is not None:
        p99, mx, _ = O.compare_images(gpu["colour"], truth)
        assert p99 <= 2, (p99, mx)


@pytest.mark.parametrize("name", list(CAMERAS))
def test_reference_scene_and_cameras(rast, cloud, name):
    cam, extra = CAMERAS[name]
    s = raster.RenderSettings(width=W, height=HGT, **extra)
    inst = [(cloud, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    H.assert_bit_exact(gpu, ora)
    truth, _ = O.reference(ora["frames"], ora["clouds"], ora["n"])
    _image_checks(gpu, ora, truth)
    # The walk's end agrees wherever no alpha or transmittance sits on a threshold
    # within the hardware exp2's last bits.
    assert np.mean(gpu["last_count"] == ora["last_count"]) >= 0.999


def test_two_instances_one_turned_scaled_and_moved(rast, cloud):
    o2w = np.eye(4)
    a = np.radians(40.0)
    o2w[:3, :3] = np.array([[np.cos(a), 0, np.sin(a)], [0, 1, 0], [-np.sin(a), 0, np.cos(a)]]) @ np.diag([1, 0.7, 1.3])
    o2w[:3, 3] = [0.5, 0.0, -1.5]
    inst = [(cloud, np.eye(4), raster.SplatEdit()), (cloud, o2w, raster.SplatEdit())]
    cam = _cam((2.0, 1.5, 7.0), (0.0, 0.0, -0.5))
    s = raster.RenderSettings(width=W, height=HGT)
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


@pytest.mark.parametrize("edit", [
    raster.SplatEdit(active=True, shape=0, mode=0, size=(1.0, 0.8, 1.2)),
    raster.SplatEdit(active=True, shape=1, mode=1, size=(0.9, 0, 0), centre=(0.3, 0.0, 0.2)),
    raster.SplatEdit(active=True, mode=2, tint=(1.2, 0.8, 0.6), saturation=0.3, brightness=1.4, opacity=0.7,
                     size=(1.5, 1.5, 1.5)),
    raster.SplatEdit(active=True, mode=2, min_opacity=0.5, max_scale=0.3, invert=True),
])
def test_splat_edits(rast, cloud, edit):
    cam, _ = CAMERAS["perspective"]
    s = raster.RenderSettings(width=W, height=HGT)
    inst = [(cloud, np.eye(4), edit)]
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


@pytest.mark.parametrize("settings", [
    dict(depth_mode=1, depth_threshold=0.3, background=(0.2, 0.3, 0.4, 1.0)),
    dict(linearise=False, max_sh_degree=1),
    dict(max_sh_degree=0, dilation=0.1),
])
def test_settings_variants(rast, cloud, settings):
    cam, _ = CAMERAS["frustum-edge"]
    s = raster.RenderSettings(width=W, height=HGT, **settings)
    inst = [(cloud, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


def test_plain_65k_full_size(rast):
    cfg = scenes.workload("plain-fwd-65k-640x480")
    s = raster.RenderSettings(width=cfg.width, height=cfg.height)
    inst = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cfg.camera, s, inst, rast)
    ora = H.run_oracle(cfg.camera, s, inst)
    print("plain 65k: pairs", ora["pairs"], "visible", ora["visible"])
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)
    # brute force on a pixel subset, exact view-z order and the rasteriser's key order
    rng = np.random.default_rng(0)
    xs, ys = rng.integers(0, cfg.width, 400), rng.integers(0, cfg.height, 400)
    exact, _ = O.reference(ora["frames"], ora["clouds"], ora["n"], pixels=(xs, ys))
    keyed, _ = O.reference(ora["frames"], ora["clouds"], ora["n"], pixels=(xs, ys), keyed=True)
    ours = gpu["colour"][ys, xs]
    e99, emax = O.linear_error(ours, exact)
    k99, kmax = O.linear_error(ours, keyed)
    print(f"plain 65k vs brute force: exact order p99 {e99:.2e} max {emax:.2e}; key order p99 {k99:.2e} "
          f"max {kmax:.2e}")
    assert e99 <= 1e-3 and k99 <= 1e-3 and kmax <= 1e-2


@pytest.mark.parametrize("count", [200_000])
def test_clustered_scene_scaled(rast, count):
    cfg = scenes.workload("scene-fwd-3M-1080p", count=count)
    s = raster.RenderSettings(width=cfg.width, height=cfg.height, dilation=cfg.dilation, filter3d=cfg.filter3d)
    inst = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cfg.camera, s, inst, rast)
    ora = H.run_oracle(cfg.camera, s, inst)
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


def test_sort_stress_large_footprints_scaled(rast):
    cfg = scenes.workload("sort-stress-6M-2160p", count=60_000)
    s = raster.RenderSettings(width=cfg.width, height=cfg.height)
    inst = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cfg.camera, s, inst, rast)
    ora = H.run_oracle(cfg.camera, s, inst)
    t = ora["touched"]
    print("sort stress scaled: pairs", ora["pairs"], "max tiles a splat", int(t.max()))
    assert int(t.max()) > 256
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


def test_clustered_3m_full_size_bit_exact_and_deterministic(rast):
    cfg = scenes.workload("scene-fwd-3M-1080p")
    s = raster.RenderSettings(width=cfg.width, height=cfg.height, dilation=cfg.dilation, filter3d=cfg.filter3d)
    inst = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cfg.camera, s, inst, rast)
    ora = H.run_oracle(cfg.camera, s, inst)
    print("scene 3M: pairs", ora["pairs"], "visible", ora["visible"])
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)
    again = H.run_gpu(cfg.camera, s, inst, rast)
    assert np.array_equal(again["colour"].view(np.uint32), gpu["colour"].view(np.uint32))
    assert np.array_equal(again["keys"], gpu["keys"])


def test_empty_and_degenerate_frames(rast, cloud):
    s = raster.RenderSettings(width=37, height=21, background=(0.1, 0.2, 0.3, 0.4))
    behind = _cam((0.0, 0.0, 50.0), (0.0, 0.0, 100.0))      # looking away: everything culled
    gpu = H.run_gpu(behind, s, [(cloud, np.eye(4), raster.SplatEdit())], rast)
    assert gpu["counts"][2] == 0
    assert np.allclose(gpu["colour"], np.array([0.1, 0.2, 0.3, 0.4], np.float32))
    one = F.CloudBuilder()
    one.add(0.0, 0.0, -3.0, 0.8, 0.1, 0.1, 0.1, (1, 0, 0, 0), (0.3, 0.6, 0.9))
    sc = one.decode(3)
    s1 = raster.RenderSettings(width=64, height=48)
    gpu = H.run_gpu(raster.Camera(), s1, [(sc, np.eye(4), raster.SplatEdit())], rast)
    ora = H.run_oracle(raster.Camera(), s1, [(sc, np.eye(4), raster.SplatEdit())])
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


def test_errors_carry_the_reference_codes(rast, cloud):
    import torch
    dev = cloud.to_device()
    t = raster.RenderTargets(10, 10)
    with pytest.raises(raster.LrtError) as e:
        rast.render(raster.Camera(), [raster.SplatInstance(dev)], raster.RenderSettings(width=0, height=10), t)
    assert e.value.name == "InvalidArgument"
    with pytest.raises(raster.LrtError) as e:
        rast.render(raster.Camera(), [raster.SplatInstance(dev)], raster.RenderSettings(width=12, height=10), t)
    assert e.value.name == "InvalidArgument"
    with pytest.raises(raster.LrtError) as e:
        rast.render(raster.Camera(), [raster.SplatInstance(dev)],
                    raster.RenderSettings(width=10, height=10, filter3d=True), t)
    assert e.value.name == "InvalidArgument"
    bad = raster.GpuSplats(dev.positions, dev.shape, dev.sh, 3)
    bad._c.rest_per_colour = 5
    with pytest.raises(raster.LrtError) as e:
        rast.render(raster.Camera(), [raster.SplatInstance(bad)], raster.RenderSettings(width=10, height=10), t)
    assert e.value.name == "InvalidArgument"
    with pytest.raises(raster.LrtError) as e:
        rast.radix_sort(torch.zeros(4, dtype=torch.int64, device="cuda"), torch.zeros(4, dtype=torch.int32,
                        device="cuda"), torch.zeros(4, dtype=torch.int64, device="cuda"),
                        torch.zeros(4, dtype=torch.int32, device="cuda"), 65)
    assert e.value.name == "InvalidArgument"
    # still renders after the failures
    s = raster.RenderSettings(width=W, height=HGT)
    gpu = H.run_gpu(CAMERAS["perspective"][0], s, [(cloud, np.eye(4), raster.SplatEdit())], rast)
    assert gpu["counts"][2] > 0
    assert rast.debug(_abi.DEBUG_COUNTS)[2] == gpu["counts"][2]


@pytest.mark.parametrize("batch,order", [(256, 0), (256, 1), (64, 1)])
def test_every_tile_order_draws_the_same_frame(rast, cloud, batch, order):
    """The launch order is a performance parameter only; blend_batch is accepted
    at values other than its default and changes nothing."""
    cam, _ = CAMERAS["perspective"]
    s = raster.RenderSettings(width=W, height=HGT, blend_batch=batch, tile_order=order)
    inst = [(cloud, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)
    cfg = scenes.workload("plain-fwd-65k-640x480", count=20000)
    s1 = raster.RenderSettings(width=cfg.width, height=cfg.height, blend_batch=batch, tile_order=order, depth_mode=1)
    inst1 = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cfg.camera, s1, inst1, rast)
    ora = H.run_oracle(cfg.camera, s1, inst1)
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


@pytest.mark.parametrize("tile", [8, 32])
@pytest.mark.parametrize("name", ["perspective", "frustum-edge", "no-aa-window"])
def test_tile_sizes_bin_as_the_oracle_and_draw_the_16_pixel_frame(rast, cloud, name, tile):
    """At 8- and 32-pixel tiles the counts, records, pairs and ranges are the
    oracle's at that tile size, bit for bit, and the images are the 16-pixel
    frame's: the quadrants are the same 8x8 blocks and each walks the splats
    that reach it in the same (depth key, index) order."""
    print(f"tile size {tile} camera {name}", flush=True)
    cam, extra = CAMERAS[name]
    inst = [(cloud, np.eye(4), raster.SplatEdit())]
    base = H.run_gpu(cam, raster.RenderSettings(width=W, height=HGT, **extra), inst, rast)
    s = raster.RenderSettings(width=W, height=HGT, tile_size=tile, **extra)
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    assert len(ora["ranges"]) == (-(-W // tile)) * (-(-HGT // tile))
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)
    np.testing.assert_array_equal(gpu["colour"].view(np.uint32), base["colour"].view(np.uint32))
    np.testing.assert_array_equal(gpu["depth"].view(np.uint32), base["depth"].view(np.uint32))
    np.testing.assert_array_equal(gpu["final_t"].view(np.uint32), base["final_t"].view(np.uint32))
    # The 1080p benchmark camera over a clustered scene, heavy tiles split.
    cfg = scenes.workload("plain-fwd-65k-640x480", count=20000)
    inst1 = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    for segment in (0, 64):
        s1 = raster.RenderSettings(width=cfg.width, height=cfg.height, tile_size=tile, blend_segment=segment,
                                   depth_mode=1)
        gpu = H.run_gpu(cfg.camera, s1, inst1, rast)
        ora = H.run_oracle(cfg.camera, s1, inst1)
        H.assert_bit_exact(gpu, ora)
        _image_checks(gpu, ora)


@pytest.mark.parametrize("radix", [8, 9, 10])
@pytest.mark.parametrize("tile", [8, 16])
def test_sort_digit_widths_give_the_oracle_s_pairs(rast, radix, tile):
    """The frame's sort at digits of up to 8, 9 and 10 bits: the same pairs and
    ranges as the oracle's, bit for bit, in the passes the widths make."""
    print(f"radix {radix} tile {tile}", flush=True)
    cfg = scenes.workload("plain-fwd-65k-640x480", count=20000)
    inst = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    s = raster.RenderSettings(width=cfg.width, height=cfg.height, tile_size=tile, radix_bits=radix)
    gpu = H.run_gpu(cfg.camera, s, inst, rast)
    ora = H.run_oracle(cfg.camera, s, inst)
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


def _heaviest_first(ranges):
    """Tiles by the bit length of their pair count, descending, index order within one length."""
    counts = (ranges[:, 1].astype(np.int64) - ranges[:, 0].astype(np.int64))
    lengths = np.array([int(c).bit_length() for c in counts])
    return np.array(sorted(range(len(counts)), key=lambda t: (-lengths[t], t)), dtype=np.uint32)


@pytest.mark.gpu
@pytest.mark.parametrize("size", [(W, HGT), (640, 480), (1920, 1080)])
def test_tile_order_is_a_stable_heaviest_first_permutation(rast, cloud, size):
    """Every tile exactly once, buckets by pair-count bit length descending, stable inside a bucket."""
    cam, _ = CAMERAS["perspective"]
    s = raster.RenderSettings(width=size[0], height=size[1], tile_order=1)
    inst = [(cloud, np.eye(4), raster.SplatEdit())]
    H.run_gpu(cam, s, inst, rast)
    ranges = rast.debug(_abi.DEBUG_RANGES).reshape(-1, 2)
    order = rast.debug(_abi.DEBUG_TILE_ORDER)
    assert len(order) == len(ranges)
    np.testing.assert_array_equal(order, _heaviest_first(ranges))
    s.tile_order = 0
    H.run_gpu(cam, s, inst, rast)
    assert len(rast.debug(_abi.DEBUG_TILE_ORDER)) == 0


@pytest.mark.parametrize("segment", [16, 64, 300])
@pytest.mark.parametrize("depth_mode", [0, 1])
def test_split_tiles_draw_the_frame_the_one_walk_draws(rast, segment, depth_mode):
    """Tiles of more than `segment` pairs walked in segments by waves of their
    own and composited: the same images (to float association), the same last
    contributor and final transmittance, as the one walk; and the oracle's frame."""
    print(f"split blend segment {segment} depth mode {depth_mode}", flush=True)
    cfg = scenes.workload("plain-fwd-65k-640x480", count=20000)
    inst = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    whole = H.run_gpu(cfg.camera, raster.RenderSettings(width=cfg.width, height=cfg.height, depth_mode=depth_mode,
                                                        blend_segment=0), inst, rast)
    s = raster.RenderSettings(width=cfg.width, height=cfg.height, depth_mode=depth_mode, blend_segment=segment)
    gpu = H.run_gpu(cfg.camera, s, inst, rast)
    split = int(np.sum(np.diff(gpu["ranges"], axis=1) > segment))
    assert split > 0
    np.testing.assert_allclose(gpu["colour"], whole["colour"], rtol=0, atol=3e-5)
    np.testing.assert_allclose(gpu["depth"], whole["depth"], rtol=1e-4, atol=1e-4)
    np.testing.assert_allclose(gpu["final_t"], whole["final_t"], rtol=1e-4, atol=1e-7)
    assert np.mean(gpu["last_count"] == whole["last_count"]) >= 0.9999
    ora = H.run_oracle(cfg.camera, s, inst)
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


def test_a_frame_that_outgrows_the_pair_buffers_is_the_oracle_s():
    """The duplication runs behind the pair-count readback at the buffers'
    present size; a frame with more pairs runs it again after they grow."""
    print("pair buffers grown between frames", flush=True)
    r = raster.TileRasterizer()
    cfg = scenes.workload("plain-fwd-65k-640x480")
    s = raster.RenderSettings(width=cfg.width, height=cfg.height)
    small = scenes.workload("plain-fwd-65k-640x480", count=500)
    H.run_gpu(small.camera, s, [(small.scene, np.eye(4), raster.SplatEdit())], r)
    inst = [(cfg.scene, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cfg.camera, s, inst, r)
    ora = H.run_oracle(cfg.camera, s, inst)
    assert ora["pairs"] > 20 * 500
    H.assert_bit_exact(gpu, ora)
    _image_checks(gpu, ora)


def test_walk_steps_are_counted_by_the_same_blend(rast):
    """LRT_DEBUG_WALK_STEPS runs the last frame's blend again and counts its
    quadrant waves' list steps: positive, no more than every quadrant walking its
    whole tile (each list fill padded to a group of four), the same on each call, and
    leaving the frame's images as they were."""
    cfg = scenes.workload("scene-fwd-3M-1080p", count=100_000)
    s = raster.RenderSettings(width=640, height=360, dilation=cfg.dilation, filter3d=cfg.filter3d)
    inst = [raster.SplatInstance(cfg.scene.to_device())]
    t = raster.RenderTargets(640, 360)
    rast.render(cfg.camera, inst, s, t)
    before = t.colour.clone()
    steps = rast.debug(_abi.DEBUG_WALK_STEPS)
    assert steps.size == 1
    ranges = rast.debug(_abi.DEBUG_RANGES).reshape(-1, 2).astype(np.int64)
    pairs = ranges[:, 1] - ranges[:, 0]
    bound = int((4 * (pairs + 4 * (pairs // 128 + 1))).sum())   # each list fill padded to a group of 4
    print(f"walk steps {int(steps[0])}, bound {bound}")
    assert 0 < int(steps[0]) <= bound
    assert int(rast.debug(_abi.DEBUG_WALK_STEPS)[0]) == int(steps[0])
    assert bool((t.colour == before).all())


def test_every_half_pattern_decodes_as_the_oracle_does(rast):
    """All 65,536 fp16 patterns (zeros, subnormals, infinities, quiet and
    signalling NaNs among them) as the 3,000-splat scene's harmonic
    coefficients, and a cycle of special halves as its base colours: the
    records, counts, pairs and ranges agree bit for bit with the oracle, whose
    decode is the exact bit-level one (the GPU converts in hardware and puts a
    NaN's quiet bit back from its payload)."""
    import dataclasses
    cloud = F.random_cloud(3000, 7).decode(15)   # degree 3: 23 words a splat, 138,000 halves
    halves = np.resize(np.arange(65536, dtype=np.uint32), cloud.sh.size * 2)
    sh = (halves[0::2] | (halves[1::2] << np.uint32(16))).reshape(cloud.sh.shape).astype(np.uint32)
    special = np.array([0x0000, 0x8000, 0x0001, 0x03FF, 0x8001, 0x7BFF, 0x7C00, 0xFC00, 0x7C01, 0x7E00, 0xFDFF,
                        0x3C00, 0x3555], np.uint32)
    shape = cloud.shape.copy()
    n = shape.shape[0]
    pick = special[np.arange(3 * n) % special.size].reshape(n, 3)
    shape[:, 2] = (shape[:, 2] & np.uint32(0xFFFF)) | (pick[:, 0] << np.uint32(16))   # z log-scale kept
    shape[:, 3] = pick[:, 1] | (pick[:, 2] << np.uint32(16))
    scene = dataclasses.replace(cloud, shape=shape, sh=sh)
    cam, _ = CAMERAS["perspective"]
    s = raster.RenderSettings(width=W, height=HGT)
    inst = [(scene, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    H.assert_bit_exact(gpu, ora)


@pytest.mark.parametrize("tile", [8, 16, 32])
def test_a_frame_of_one_pair_draws_it(rast, tile):
    """One splat inside one tile: the sort has nothing to order, but its key is
    still the narrowed one the ranges read."""
    fields = np.zeros((1, 14), np.float32)
    fields[0, :4] = (0.2, 0.2, 0.0, 0.9)
    fields[0, 4:7] = -3.3
    fields[0, 10] = 1.0
    fields[0, 11:14] = (0.9, 0.5, 0.2)
    cam = _cam((0.0, 0.0, 4.0), (0.0, 0.0, 0.0), focal=60.0)
    s = raster.RenderSettings(width=32, height=32, tile_size=tile)
    inst = [(scenes.pack_splats(fields, 0), np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    assert ora["pairs"] == 1
    H.assert_bit_exact(gpu, ora)
    assert ora["colour"].max() > 0.1
    np.testing.assert_allclose(gpu["colour"], ora["colour"], rtol=0, atol=2e-5)


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("count", [1, 3, 15, 17, 63, 65, 255, 257, 769])
@pytest.mark.parametrize("opacity,depth_mode", [(0.02, 0), (0.6, 0), (0.6, 1)])
def test_lists_of_every_length_blend_as_the_oracle(rast, count, tile, opacity, depth_mode):
    """The ends of the blend's groups of four records, sixteens, chunks of 64 and
    rounds of a pair a lane, on a frame whose last blocks have pixels past both
    edges; faint splats (no pixel stops) and strong ones (pixels stop at every
    place of a group). Colours and depths are sums of at most `count` 32-bit
    terms whose exponents are off by a few ulps of |q| <= 16 (2e-6 of a weight):
    2e-5 of their size, and a pixel whose pair lies at its cutoff, its floor or
    its last place may differ by that pair (1/255 of a weight at the floor)."""
    rng = np.random.default_rng(count)
    fields = np.zeros((count, 14), np.float32)
    fields[:, 0] = rng.uniform(-0.35, 0.35, count)
    fields[:, 1] = rng.uniform(-0.25, 0.25, count)
    fields[:, 2] = rng.uniform(-1.0, 1.0, count)
    fields[:, 3] = opacity
    fields[:, 4:7] = rng.uniform(-4.0, -1.5, (count, 3))
    fields[:, 7:11] = rng.normal(0.0, 1.0, (count, 4))
    fields[:, 11:14] = rng.uniform(0.0, 1.0, (count, 3))
    scene = scenes.pack_splats(fields, 0)
    cam = _cam((0.0, 0.0, 4.0), (0.0, 0.0, 0.0), focal=60.0)
    s = raster.RenderSettings(width=37, height=27, tile_size=tile, depth_mode=depth_mode)
    inst = [(scene, np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    H.assert_bit_exact(gpu, ora)
    for name, scale in (("colour", 1.0), ("depth", 5.0)):
        d = np.abs(gpu[name].astype(np.float64) - ora[name])
        assert np.quantile(d, 0.97) <= 2e-5 * scale, (name, np.quantile(d, 0.97))
        assert d.max() <= (1.0 if (name, depth_mode) == ("depth", 1) else scale / 255.0 * 2.0), (name, d.max())


def _fma(a, b, c):
    """float32 fused multiply-add (the product is exact in float64; a second
    rounding at a midpoint is a 2^-29 chance a step)."""
    return (np.asarray(a, np.float64) * np.asarray(b, np.float64) + np.asarray(c, np.float64)).astype(np.float32)


def test_pairs_at_their_bound_fall_as_the_nested_form_says(rast):
    """Which pixels a pair is drawn on, in float32 and step by step as the walk
    takes it: q = u (A u + (B v + D)) + (v (C v + E) + F) about the quadrant's
    centre, drawn where q >= the bound. Another order of the same sum takes about
    one such decision in ten million otherwise (it is asserted that these splats
    hold one at least); each is worth 1/255 of a pixel's transmittance. The
    opacity is a power of two, so its logarithm is exact on both sides; what is
    left is the product of a few hundred float32 factors, 6e-8 each."""
    count, width, height = 6000, 384, 288
    rng = np.random.default_rng(1)
    fields = np.zeros((count, 14), np.float32)
    fields[:, 0] = rng.uniform(-1.0, 1.0, count)
    fields[:, 1] = rng.uniform(-0.8, 0.8, count)
    fields[:, 2] = rng.uniform(-1.0, 1.0, count)
    fields[:, 3] = 2.0 ** -6
    fields[:, 4:7] = rng.normal(-3.0, 2.0, (count, 3))
    fields[:, 7:11] = rng.normal(0.0, 1.0, (count, 4))
    fields[:, 11:14] = 0.5
    cam = _cam((0.0, 0.0, 4.0), (0.0, 0.0, 0.0), focal=50.0)
    s = raster.RenderSettings(width=width, height=height, antialias=False)
    inst = [(scenes.pack_splats(fields, 0), np.eye(4), raster.SplatEdit())]
    gpu = H.run_gpu(cam, s, inst, rast)
    ora = H.run_oracle(cam, s, inst)
    H.assert_bit_exact(gpu, ora)

    f = np.float32
    scale, floor = f(-0.72134752044448170368), f(-7.99435343685885793775)
    tiles_x = (width + 15) // 16
    y, x = np.mgrid[0:16, 0:16]
    u, v = ((x & 7) - 3.5).astype(f), ((y & 7) - 3.5).astype(f)
    t = np.ones((tiles_x * 16, (height + 15) // 16 * 16)).T.copy()
    otherwise = 0
    for i in range(0, len(ora["pair_splats"]), 4096):
        tile = ora["pair_tiles"][i:i + 4096].astype(np.int64)
        r = ora["proj"][ora["pair_splats"][i:i + 4096]][:, :, None, None]
        px, py = (tile % tiles_x * 16)[:, None, None] + x, (tile // tiles_x * 16)[:, None, None] + y
        cx, cy, cutoff, opacity = r[:, 0], r[:, 1], r[:, 3], r[:, 7]
        a, b, c = scale * r[:, 4], scale * (r[:, 5] + r[:, 5]), scale * r[:, 6]
        ux, vy = cx - ((px & ~7) + 4).astype(f), cy - ((py & ~7) + 4).astype(f)
        d, e = -(f(2) * a * ux + b * vy), -(f(2) * c * vy + b * ux)
        log = np.log2(opacity).astype(f)
        at = ux * (a * ux + b * vy) + c * vy * vy + log
        bound = np.maximum(log + scale * cutoff, floor)
        q = _fma(u, _fma(a, u, _fma(b, v, d)), _fma(v, _fma(c, v, e), at))
        drawn = (q >= bound) & (px < width) & (py < height)
        flat = _fma(a, u * u, _fma(b, u * v, _fma(c, v * v, _fma(d, u, _fma(e, v, at)))))
        otherwise += int((((flat >= bound) != drawn) & (px < width) & (py < height)).sum())
        np.multiply.at(t, (py, px), np.where(drawn, 1.0 - np.exp2(q.astype(np.float64)), 1.0))
    assert otherwise > 0
    t = t[:height, :width]
    assert t.min() > 2e-4   # no pixel's walk ends early
    np.testing.assert_allclose(gpu["final_t"], t, rtol=2e-4)


def _broad_splats(count, seed, log_scale):
    """Splats wide enough to reach hundreds of tiles each, their depths spread
    with some equal (ties that the slot order breaks)."""
    rng = np.random.default_rng(seed)
    fields = np.zeros((count, 14), np.float32)
    fields[:, :2] = rng.uniform(-1.2, 1.2, (count, 2))
    fields[:, 2] = np.round(rng.uniform(-1.0, 1.0, count) * 300.0) / 300.0
    fields[:, 3] = rng.uniform(0.02, 0.9, count)
    fields[:, 4:7] = rng.normal(log_scale, 0.3, (count, 3))
    fields[:, 7:11] = rng.normal(0.0, 1.0, (count, 4))
    fields[:, 11:14] = rng.uniform(0.0, 1.0, (count, 3))
    return scenes.pack_splats(fields, 0)


@pytest.mark.parametrize("size,tile,count,log_scale,discs", [((1920, 1080), 16, 60_011, -2.7, 0),
                                                            ((1923, 1077), 32, 250_001, -2.7, 0),
                                                            ((3840, 2160), 8, 2_003, -2.4, 0),
                                                            ((1920, 1080), 16, 60_011, -2.7, 3_000)])
def test_frames_of_many_pairs_a_splat_bin_as_the_oracle(size, tile, count, log_scale, discs):
    """Past the pair count where the slots are sorted by depth first and the pairs
    by tile alone: u16 tiles, u32 tiles (more than 65,536), discs among the
    splats. Pairs, ranges and images are the one sort's; the first frame, the
    same again (whose duplication waits for the counts) and one of few pairs
    after it (whose duplication does not)."""
    rast = raster.TileRasterizer()
    cam = _cam((0.0, 0.0, 4.0), (0.0, 0.0, 0.0), focal=30.0)
    s = raster.RenderSettings(width=size[0], height=size[1], tile_size=tile)
    inst = [(_broad_splats(count, 3, log_scale), np.eye(4), raster.SplatEdit())]
    points = []
    if discs:
        pos, col = F.random_points(discs, 5)
        points = [(pos, col, np.eye(4), raster.PointStyle(size=0.05))]
        ora = H.run_oracle_composite(cam, s, inst, points)
    else:
        ora = H.run_oracle(cam, s, inst)
    assert ora["pairs"] > 6_000_000 + 1.25 * ora["visible"]
    for _ in range(2):
        if discs:
            gpu = H.run_gpu_composite(cam, s, inst, points, rast=rast)
        else:
            gpu = H.run_gpu(cam, s, inst, rast)
        assert gpu["stats"].pairs == ora["pairs"] and gpu["stats"].key_bits == H.expected_key_bits(ora)
        depth_bits = gpu["stats"].key_bits - H.bits_for(len(ora["ranges"]))
        assert gpu["stats"].sort_passes == (H.expected_passes(depth_bits)
                                            + H.expected_passes(H.bits_for(len(ora["ranges"]))))
        H.assert_bit_exact(dict(gpu, stats=None), ora)
        d = np.abs(gpu["colour"].astype(np.float64) - ora["colour"])
        assert np.quantile(d, 0.99) <= 1e-3 and d.max() <= 1e-2   # the image targets of every frame test
    few = raster.RenderSettings(width=250, height=190, tile_size=tile)
    small = [(_broad_splats(500, 4, -3.5), np.eye(4), raster.SplatEdit())]
    for _ in range(2):
        H.assert_bit_exact(H.run_gpu(cam, few, small, rast), H.run_oracle(cam, few, small))


def test_a_large_and_a_small_view_in_turn_keep_their_own_order():
    """Two views on one rasteriser, one of many pairs a splat: from its second
    frame on the large one sorts by depth first, whatever was drawn in between,
    and the small one never does; the images are the same either way."""
    import dataclasses

    import torch
    rast = raster.TileRasterizer()
    cam = _cam((0.0, 0.0, 4.0), (0.0, 0.0, 0.0), focal=30.0)
    large = raster.RenderSettings(width=1920, height=1080, time_stages=True)
    small = dataclasses.replace(large, width=250, height=190)
    broad, few = _broad_splats(60_011, 3, -2.7).to_device(), _broad_splats(500, 4, -3.5).to_device()
    images = []
    for turn in range(3):
        for s, cloud, settings in (("small", few, small), ("large", broad, large)):
            targets = raster.RenderTargets(settings.width, settings.height)
            st = rast.render(cam, [raster.SplatInstance(cloud)], settings, targets)
            torch.cuda.synchronize()
            if s == "small":
                assert st.depth_sort_ms == 0.0
                continue
            assert st.pairs > 6_000_000 + 1.25 * st.visible
            assert turn == 0 or st.depth_sort_ms > 0.0, turn
            images.append(targets.colour.view(torch.int32))
    assert torch.equal(images[0], images[1]) and torch.equal(images[0], images[2])


def test_a_frame_duplicated_in_vain_bins_as_the_oracle():
    """A large frame of a shape not drawn before, on a rasteriser whose buffers
    hold its pairs: they are duplicated before the counts are known, and so many
    that sorting by depth first still gains. Pairs and ranges are the oracle's,
    the images and walk state a fresh rasteriser's."""
    rast = raster.TileRasterizer()
    cam = _cam((0.0, 0.0, 4.0), (0.0, 0.0, 0.0), focal=30.0)
    inst = [(_broad_splats(60_011, 3, -2.7), np.eye(4), raster.SplatEdit())]
    wide = raster.RenderSettings(width=2400, height=1350, time_stages=True)
    new = raster.RenderSettings(width=2160, height=1215, time_stages=True)
    assert H.run_gpu(cam, wide, inst, rast)["stats"].depth_sort_ms > 0.0
    gpu = H.run_gpu(cam, new, inst, rast)
    ora = H.run_oracle(cam, new, inst)
    assert 3 * ora["pairs"] > 30_000_000 + 10 * ora["visible"]
    assert gpu["stats"].depth_sort_ms > 0.0
    H.assert_bit_exact(dict(gpu, stats=None), ora)
    fresh = H.run_gpu(cam, new, inst, raster.TileRasterizer())
    for name in ("colour", "depth", "final_t", "last_count"):
        np.testing.assert_array_equal(gpu[name].view(np.uint32), fresh[name].view(np.uint32))


def test_one_splat_over_millions_of_tiles_draws_as_at_larger_tiles():
    """A single drawn splat past the pair count where slots are sorted by depth
    first: there is nothing to sort, and its pairs are its own. 6.25M 8-pixel
    tiles against the same frame in 16-pixel tiles, whose 1.6M pairs take the
    one sort: bit for bit, with another splat's frame drawn before."""
    import torch
    side = 20_000
    fields = np.zeros((3, 14), np.float32)
    fields[:, 3] = 0.6
    fields[:, 4:7] = (3.0, 2.5, 2.0)
    fields[:, 10] = 1.0
    fields[:, 11:14] = (0.9, 0.5, 0.2)
    fields[1:, :3] = ((0.3, 0.2, 0.5), (0.0, 0.0, 9.0))   # the last behind the camera
    cam = _cam((0.0, 0.0, 4.0), (0.0, 0.0, 0.0), focal=30.0)
    rast = raster.TileRasterizer()

    def draw(rows, tile):
        scene = scenes.pack_splats(np.ascontiguousarray(fields[rows]), 0).to_device()
        targets = raster.RenderTargets(side, side)
        st = rast.render(cam, [raster.SplatInstance(scene)],
                         raster.RenderSettings(width=side, height=side, tile_size=tile), targets)
        torch.cuda.synchronize()
        return st, targets

    draw([1, 0], 8)
    st, one = draw([2, 0], 8)
    assert st.visible == 1 and st.pairs == (side // 8) ** 2
    st, want = draw([2, 0], 16)
    assert st.visible == 1 and st.pairs == (side // 16) ** 2
    assert float(want.colour[::999, ::999].min()) > 0.0
    assert torch.equal(one.colour.view(torch.int32), want.colour.view(torch.int32))
    assert torch.equal(one.depth.view(torch.int32), want.depth.view(torch.int32))
