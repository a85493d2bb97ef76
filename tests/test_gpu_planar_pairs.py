"""The 2D projections through the pair copy of the images and the 2D backprojections through the
bordered copy of the projections: the dispatch's edges (lanes per ray, remainders of the ray
groups, rows of the copies, spacings of each division, the largest copy) against the oracle."""
import math

import numpy as np
import pytest
import torch

import gpu_helpers as gh
import oracle as orc
from pyronn_layers import geometry as geo
from pyronn_layers import native as nat

pytestmark = pytest.mark.gpu


def _run(fan, img, sp, n, det, ds, step, sid, storage=torch.float32, arc=2 * math.pi, off=(0.0, 0.0)):
    import pyronn_layers as pl
    H, W = img.shape[-2:]
    org = (geo.centred_origin((H, W), sp) + np.asarray(off)).astype(np.float32)
    sp = np.asarray(sp, np.float32)
    rays = geo.parallel_ray_vectors(n, arc).astype(np.float32)
    do = np.float32(-(det - 1) / 2 * ds)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    x = dev(img)[None].to(storage)
    geom = [dev(org)[None], dev([[do]]), dev(sp)[None], dev([[ds]])]
    if fan:
        out = pl.fan_projection2d(x, [n, det], *geom, dev([[sid]]), dev([[1.4 * sid]]), dev(rays)[None], step)
        ref = orc.fan_forward(x[0].float().cpu().numpy(), rays, det, org, sp, do, np.float32(ds),
                              sid=np.float32(sid), sdd=np.float32(1.4 * sid), step_factor=step)[0]
    else:
        out = pl.parallel_projection2d(x, [n, det], *geom, dev(rays)[None], step)
        ref = orc.parallel_forward(x[0].float().cpu().numpy(), rays, det, org, sp, do, np.float32(ds),
                                   step_factor=step)[0]
    # both entries, whichever of them the operator took
    both = gh.forward2d(fan, x.float().cpu().numpy(), rays, det, org, sp, do, np.float32(ds), sid, 1.4 * sid, step,
                        {torch.float32: "f32", torch.bfloat16: "bf16", torch.float16: "f16"}[storage])
    assert np.array_equal(both[0], out[0].cpu().numpy(), equal_nan=True)
    return out[0].cpu().numpy(), ref


@pytest.mark.parametrize("fan", [False, True])
@pytest.mark.parametrize("storage", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H, W, sp, n, det", [
    (1, 1, (1.0, 1.0), 5, 3),            # one pixel; 16 lanes per ray, a partly filled wave
    (3, 70, (0.5, 0.5), 9, 65),          # power-of-two spacing below the box's 0.5 mm edge
    (70, 3, (0.7, 1.3), 9, 66),          # refined division, two spacings
    (33, 31, (0.3, 0.3), 7, 61),         # coordinates below -1: the copy's second border cell
    (40, 44, (0.9, 1.0), 300, 110),      # 33000 rays: 8 lanes per ray, det no multiple of 8
    (21, 26, (0.8, 0.8), 550, 121),      # 66550 rays: 4 lanes per ray, det no multiple of 16
    (24, 24, (1e-19, 1e-19), 3, 17),     # a spacing the refined division does not serve
])
def test_pairs_match_the_oracle(fan, storage, H, W, sp, n, det):
    img = np.random.default_rng(H * 100 + W).normal(size=(H, W)).astype(np.float32)
    ext = max(H * sp[0], W * sp[1])
    got, ref = _run(fan, img, sp, n, det, 1.3 * ext / det, 0.2 if sp[0] > 0.1 else 0.5, 1.5 * ext, storage)
    assert np.array_equal(got, ref, equal_nan=True), int((got != ref).sum())


@pytest.mark.parametrize("fan", [False, True])
def test_pairs_far_box_and_capped_march(fan):
    # alpha of about 3e6 spacings at a step of 0.2: the additions are rounded (the capped march)
    img = np.random.default_rng(5).normal(size=(20, 18)).astype(np.float32)
    got, ref = _run(fan, img, (1.0, 1.0), 5, 33, 1.0, 0.2, 60.0, arc=0.3, off=(4.0e6, 3.0e6))
    assert np.array_equal(got, ref, equal_nan=True)
    got, ref = _run(fan, img, (1.0, 1.0), 5, 33, 1.0, 1e-3, 3.0e5 if fan else 60.0)
    assert np.array_equal(got, ref, equal_nan=True)


@pytest.mark.parametrize("H, W", [(2049, 4084), (2050, 4084)])
def test_pairs_largest_copy_and_the_first_image_past_it(H, W):
    size = nat.lib().pyronn_projection2d_workspace_size(1, H, W, nat.F32)
    assert (size > 0) == ((W + 4) * (H + 3) < 2 ** 23)
    img = np.random.default_rng(H).normal(size=(H, W)).astype(np.float32)
    got, ref = _run(False, img, (1.0, 1.0), 3, 400, 12.0, 0.5, 0.0)
    assert np.array_equal(got, ref)


def test_pairs_infinite_and_nan_pixels_reach_the_same_rays():
    img = np.random.default_rng(8).normal(size=(16, 18)).astype(np.float32)
    img[0, 3], img[15, 0], img[7, 17] = np.inf, np.nan, -np.inf
    for sp in ((0.25, 0.25), (1.0, 1.0), (0.3, 0.6)):
        got, ref = _run(False, img, sp, 40, 41, 0.5, 0.2, 0.0)
        assert np.array_equal(got, ref, equal_nan=True)


def _back(fan, sino, shape, sp, ds, sid, storage=torch.float32, off=(0.0, 0.0)):
    import pyronn_layers as pl
    n, det = sino.shape[-2:]
    org = (geo.centred_origin(shape, sp) + np.asarray(off)).astype(np.float32)
    sp = np.asarray(sp, np.float32)
    rays = geo.parallel_ray_vectors(n, 2 * math.pi).astype(np.float32)
    do = np.float32(-(det - 1) / 2 * ds)
    dev = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")
    x = dev(sino)[None].to(storage)
    geom = [dev(org)[None], dev([[do]]), dev(sp)[None], dev([[ds]])]
    s = x[0].float().cpu().numpy()
    if fan:
        out = pl.fan_backprojection2d(x, list(shape), *geom, dev([[sid]]), dev([[1.4 * sid]]), dev(rays)[None])
        ref = orc.fan_backward(s, rays, shape, org, sp, do, np.float32(ds), sid=np.float32(sid),
                               sdd=np.float32(1.4 * sid))
    else:
        out = pl.parallel_backprojection2d(x, list(shape), *geom, dev(rays)[None])
        ref = orc.parallel_backward(s, rays, shape, org, sp, do, np.float32(ds))
    both = gh.backward2d(fan, s[None], rays, shape, org, sp, do, np.float32(ds), sid, 1.4 * sid,
                         {torch.float32: "f32", torch.bfloat16: "bf16", torch.float16: "f16"}[storage])
    assert np.array_equal(both[0], out[0].cpu().numpy(), equal_nan=True)
    return out[0].cpu().numpy(), ref[0] if isinstance(ref, tuple) else ref


@pytest.mark.parametrize("fan", [False, True])
@pytest.mark.parametrize("storage", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape, sp, n, det, ds", [
    ((1, 1), (1.0, 1.0), 1, 1, 1.0),          # one pixel, one view, one detector pixel
    ((17, 15), (0.7, 1.3), 7, 2, 9.0),        # a detector of one cell; refined division
    ((33, 47), (1.0, 1.0), 129, 65, 0.5),     # one view past a block's table of 128
    ((30, 31), (0.3, 0.3), 256, 40, 0.25),    # a detector smaller than the shadow
    ((728, 730), (1.0, 1.0), 6, 911, 1.7),    # 2116 blocks, ragged rows
    ((20, 20), (1.0, 1.0), 5, 30, 1e-12),     # a spacing outside the refined division's range
])
def test_rows_match_the_oracle(fan, storage, shape, sp, n, det, ds):
    sino = np.random.default_rng(n + det).normal(size=(n, det)).astype(np.float32)
    got, ref = _back(fan, sino, shape, sp, ds, 1.5 * max(shape[0] * sp[0], shape[1] * sp[1]), storage)
    assert np.array_equal(got, ref, equal_nan=True), int((got != ref).sum())


def test_rows_source_inside_the_image_and_far_lengths():
    sino = np.random.default_rng(3).normal(size=(24, 50)).astype(np.float32)
    # the source on pixels of the image: infinite weights and degenerate intersections
    got, ref = _back(True, sino, (31, 31), (1.0, 1.0), 1.0, 10.0)
    assert np.array_equal(got, ref, equal_nan=True)
    # lengths of 2^20 mm and more take the IEEE sequences
    got, ref = _back(True, sino, (31, 29), (1.0, 1.0), 1.0, 3.0e6, off=(1.1e6, 0.0))
    assert np.array_equal(got, ref, equal_nan=True)


@pytest.mark.parametrize("back", [False, True])
def test_no_room_for_the_copy(back):
    # 67 MB of data, copies of 136 and 69 MB, an allocator that may take 16 MB more and whose free
    # blocks of 60 MB and more (other tests leave some) are taken first
    import pyronn_layers as pl
    x = torch.randn(64, 512, 512, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    dev = lambda *a: torch.tensor(a, dtype=torch.float32, device="cuda")
    if back:
        geom = [dev(-7.5, -7.5), dev(-255.5), dev(1.0, 1.0), dev(1.0)]
        rays = torch.tensor(geo.parallel_ray_vectors(512, math.pi), dtype=torch.float32, device="cuda")
        run = lambda: pl.parallel_backprojection2d(x, [16, 16], *geom, rays)
    else:
        geom = [dev(-255.5, -255.5), dev(-120.0), dev(1.0, 1.0), dev(8.0)]
        rays = torch.tensor(geo.parallel_ray_vectors(4, math.pi), dtype=torch.float32, device="cuda")
        run = lambda: pl.parallel_projection2d(x, [4, 31], *geom, rays)
    want = run()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (16 << 20)) / total)
        taken = []
        with pytest.raises(torch.cuda.OutOfMemoryError):
            for _ in range(total // (60 << 20)):
                taken.append(torch.empty(60 << 20, dtype=torch.uint8, device="cuda"))
        got = run()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, want)


def _mixed(B, H, W, n, det):
    """Geometries of B items that differ in everything: spacings of every division, offsets, rays, radii."""
    rng = np.random.default_rng(B * 1000 + H)
    sp = np.array([(1.0, 1.0), (0.7, 1.3), (0.5, 0.25), (1e-19, 1e-19), (0.3, 0.3)], np.float32)
    vs = sp[np.arange(B) % len(sp)]
    ext = (np.array([H, W]) * vs).max(1)
    vo = np.array([geo.centred_origin((H, W), v) for v in vs]) + rng.normal(size=(B, 2)) * ext[:, None] * 0.05
    ds = np.where(np.arange(B) % 4 == 1, 2.0 ** np.round(np.log2(1.3 * ext / det)), 1.3 * ext / det)
    do = -(det - 1) / 2 * ds + rng.normal(size=B) * ds
    rays = np.stack([geo.parallel_ray_vectors(n, 1.0 + b) for b in range(B)])
    f = lambda a: np.asarray(a, np.float32)
    return f(vo), f(do), f(vs), f(ds), f(rays), f(1.6 * ext), f(2.1 * ext)


@pytest.mark.parametrize("fan", [False, True])
@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("B, H, W, n, det", [
    (5, 19, 23, 7, 31),        # 16 lanes per ray
    (6, 33, 31, 50, 90),       # 8
    (6, 17, 12, 110, 101),     # 4
    (41, 5, 6, 3, 9),          # several rows and items per layout block
])
def test_batches_of_different_items(fan, storage, B, H, W, n, det):
    vo, do, vs, ds, rays, sid, sdd = _mixed(B, H, W, n, det)
    rng = np.random.default_rng(B)
    img = gh.quantise(rng.normal(size=(B, H, W)), storage)
    sino = gh.quantise(rng.normal(size=(B, n, det)), storage)
    # one step for the launch: a step of half a spacing
    fwd = gh.forward2d(fan, img, rays, det, vo, vs, do, ds, sid, sdd, 0.5, storage)
    back = gh.backward2d(fan, sino, rays, (H, W), vo, vs, do, ds, sid, sdd, storage)
    for b in range(B):
        if fan:
            ref = orc.fan_forward(img[b], rays[b], det, vo[b], vs[b], do[b], ds[b], sid=sid[b], sdd=sdd[b], step_factor=0.5)[0]
            rb = orc.fan_backward(sino[b], rays[b], (H, W), vo[b], vs[b], do[b], ds[b], sid=sid[b], sdd=sdd[b])
        else:
            ref = orc.parallel_forward(img[b], rays[b], det, vo[b], vs[b], do[b], ds[b], step_factor=0.5)[0]
            rb = orc.parallel_backward(sino[b], rays[b], (H, W), vo[b], vs[b], do[b], ds[b])
        rb = rb[0] if isinstance(rb, tuple) else rb
        assert np.array_equal(fwd[b], ref, equal_nan=True), f"forward, item {b}"
        assert np.array_equal(back[b], rb, equal_nan=True), f"backward, item {b}"


@pytest.mark.parametrize("n, det", [
    (1, 1), (70, 4),               # 8 lanes a row of the copy: one row and blocks partly filled
    (33, 12), (17, 13),            # 16, all of them used, and 32
    (9, 124), (9, 125),            # 128 and 256
    (5, 252), (5, 253),            # one and two blocks a row
    (9000, 2), (700, 600),         # more row blocks than are launched at once: several steps each
])
def test_rows_of_every_length(n, det):
    H, W = 5, 7
    vo, do, vs, ds, rays, sid, sdd = _mixed(2, H, W, n, det)
    sino = gh.quantise(np.random.default_rng(det).normal(size=(2, n, det)), "bf16")
    back = gh.backward2d(False, sino, rays, (H, W), vo, vs, do, ds, storage="bf16")
    for b in range(2):
        ref = orc.parallel_backward(sino[b], rays[b], (H, W), vo[b], vs[b], do[b], ds[b])
        assert np.array_equal(back[b], ref[0] if isinstance(ref, tuple) else ref, equal_nan=True)


@pytest.mark.parametrize("H, W", [(1, 4), (30, 4), (61, 12), (29, 28), (13, 252), (14, 253), (65532, 1)])
def test_pairs_of_every_width(H, W):
    vo, do, vs, ds, rays, sid, sdd = _mixed(2, H, W, 3, 40)
    img = gh.quantise(np.random.default_rng(W).normal(size=(2, H, W)), "f16")
    vs[:], ds[:] = 1.0, 1.3 * max(H, W) / 40
    fwd = gh.forward2d(False, img, rays, 40, vo, vs, do, ds, step_factor=0.5, storage="f16")
    for b in range(2):
        ref = orc.parallel_forward(img[b], rays[b], 40, vo[b], vs[b], do[b], ds[b], step_factor=0.5)[0]
        assert np.array_equal(fwd[b], ref)


def test_more_pixels_than_a_round_of_blocks_in_a_batch():
    B, H, W, n, det = 40, 112, 117, 6, 160      # 2240 blocks
    vo, do, vs, ds, rays, sid, sdd = _mixed(B, H, W, n, det)
    sino = np.random.default_rng(2).normal(size=(B, n, det)).astype(np.float32)
    back = gh.backward2d(True, sino, rays, (H, W), vo, vs, do, ds, sid, sdd)
    for b in (0, 1, 2, 3, 17, 39):
        rb = orc.fan_backward(sino[b], rays[b], (H, W), vo[b], vs[b], do[b], ds[b], sid=sid[b], sdd=sdd[b])
        assert np.array_equal(back[b], rb[0] if isinstance(rb, tuple) else rb, equal_nan=True), f"item {b}"


@pytest.mark.parametrize("fan", [False, True])
@pytest.mark.parametrize("name", ["vo", "do", "ds", "rays"])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_geometry_that_is_not_finite(fan, name, value):
    # one item of a batch of two: same values from the copy and in place, the other item untouched by it
    H, W, n, det = 12, 14, 6, 20
    vo, do, vs, ds, rays, sid, sdd = _mixed(2, H, W, n, det)
    bad = {"vo": vo, "do": do, "ds": ds, "rays": rays}[name]
    bad.reshape(2, -1)[1, 0] = value
    rng = np.random.default_rng(1)
    img, sino = rng.normal(size=(2, H, W)).astype(np.float32), rng.normal(size=(2, n, det)).astype(np.float32)
    fwd = gh.forward2d(fan, img, rays, det, vo, vs, do, ds, sid, sdd, 0.5)
    back = gh.backward2d(fan, sino, rays, (H, W), vo, vs, do, ds, sid, sdd)
    assert np.isfinite(fwd[0]).all() and np.isfinite(back[0]).all()


@pytest.mark.parametrize("det, copied", [(2 ** 22 - 1, True), (2 ** 22, False)])
@pytest.mark.parametrize("fan", [False, True])
def test_rows_longest_detector_and_the_first_past_it(fan, det, copied):
    assert (nat.lib().pyronn_backprojection2d_workspace_size(1, 3, det, nat.F32) > 0) == copied
    rng = np.random.default_rng(det)
    sino = rng.normal(size=(3, det)).astype(np.float32)
    H, W = 9, 2100
    vs, vo = np.ones(2, np.float32), geo.centred_origin((H, W), (1.0, 1.0)).astype(np.float32)
    ds = np.float32(2.0 ** -11)                     # the pixels reach both ends of the detector
    do = np.float32(-(det - 1) / 2 * float(ds))
    rays = geo.parallel_ray_vectors(3, math.pi).astype(np.float32)
    kw = dict(sid=np.float32(9000.0), sdd=np.float32(9500.0)) if fan else {}
    back = gh.backward2d(fan, sino, rays, (H, W), vo, vs, do, ds, **kw)
    ref = (orc.fan_backward if fan else orc.parallel_backward)(sino, rays, (H, W), vo, vs, do, ds, **kw)
    assert np.array_equal(back[0], ref[0] if isinstance(ref, tuple) else ref)


@pytest.mark.parametrize("size, views", [(30, 28), (31, 27), (31, 17), (20, 16)])
@pytest.mark.parametrize("fan", [False, True])
def test_operators_on_both_sides_of_where_a_copy_pays(fan, size, views):
    rng = np.random.default_rng(size)
    got, ref = _run(fan, rng.normal(size=(size, size)).astype(np.float32), (1.0, 1.0), views, 40, 1.3 * size / 40, 1.0,
                    1.6 * size)
    assert np.array_equal(got, ref)
    got, ref = _back(fan, rng.normal(size=(views, 40)).astype(np.float32), (size, size), (1.0, 1.0), 1.3 * size / 40,
                     1.6 * size)
    assert np.array_equal(got, ref)
