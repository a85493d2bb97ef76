"""The 2D projections through the pair copy of the images and the 2D backprojections through the
bordered copy of the projections: the dispatch's edges (lanes per ray, remainders of the ray
groups, pixels per lane, spacings of each division, the largest copy) against the oracle."""
import math

import numpy as np
import pytest
import torch

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
    return out[0].cpu().numpy(), ref[0] if isinstance(ref, tuple) else ref


@pytest.mark.parametrize("fan", [False, True])
@pytest.mark.parametrize("storage", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape, sp, n, det, ds", [
    ((1, 1), (1.0, 1.0), 1, 1, 1.0),          # one pixel, one view, one detector pixel
    ((17, 15), (0.7, 1.3), 7, 2, 9.0),        # a detector of one cell; refined division
    ((33, 47), (1.0, 1.0), 129, 65, 0.5),     # one view past a block's table of 128
    ((30, 31), (0.3, 0.3), 256, 40, 0.25),    # a detector smaller than the shadow
    ((728, 730), (1.0, 1.0), 6, 911, 1.7),    # 2116 blocks: two pixels per lane, ragged rows
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
