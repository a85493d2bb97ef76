"""How the cone kernels deal their tiles to the XCDs, at tile counts around the 8 XCDs and the
four strips, the backprojection's voxels per lane, and the f32 forward's cell indexes at the
limit of its 32-bit byte offsets, all against the oracle."""
import numpy as np
import pytest
import torch

import gpu_helpers as gh
import oracle as orc
from pyronn_layers import batched
from pyronn_layers import geometry as geo
from test_gpu_limits import _check_views, _orbit, _rand_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("det", [(16, 16), (17, 113), (129, 16), (15, 128), (40, 152), (100, 50)])
@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_forward_tiles_one_to_forty(det, storage):
    shape = (20, 24, 18)
    sp, og, P = _orbit(shape, 5, 100.0, 160.0, det, (60.0 / det[0], 60.0 / det[1]))
    vol = _rand_volume(shape, det[0], gh.DT[storage][1])
    _check_views(vol, P, sp, og, det, 0.5, False, views=range(5))


@pytest.mark.parametrize("det, n", [
    ((16, 16), 1), ((20, 33), 8), ((33, 100), 32),     # ranges of neighbouring tiles: 1, 6, 21 of them
    ((20, 33), 33), ((40, 16), 40), ((33, 100), 33),   # dealt, with a partial last turn
    ((40, 120), 41), ((20, 250), 57), ((64, 60), 67),  # 8, 16 and 4 tile columns; partial groups of views
    ((320, 512), 2), ((320, 513), 2),                  # 640 and 660 tiles
])
@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_forward_tile_orders(det, n, storage):
    shape = (20, 24, 18)
    sp, og, P = _orbit(shape, n, 100.0, 160.0, det, (60.0 / det[0], 60.0 / det[1]))
    vol = _rand_volume(shape, det[0], gh.DT[storage][1])
    _check_views(vol, P, sp, og, det, 0.5, False, views=range(n))


@pytest.mark.parametrize("blocks_per_cu", [0, 2])
@pytest.mark.parametrize("views", [(4, 30), (40, 9), (33, 50)])   # all in ranges; too many views; too many blocks
def test_batched_forward_tile_orders(views, blocks_per_cu):
    det = [(40, 120), (100, 130)]
    geoms = [geo.ConeGeometry((20, 24, 18), (1.0, 1.0, 1.0), d, (60.0 / d[0], 60.0 / d[1]), n, 100.0, 160.0, step_size=0.5)
             for d, n in zip(det, views)]
    vols = [_rand_volume((20, 24, 18), n) for n in views]
    for tile in range(4):
        got = batched.cone_projection3d_batched(vols, geoms, blocks_per_cu=blocks_per_cu, forward_tile=tile)
        for x, v, g in zip(got, vols, geoms):
            P = g.projection_matrices().astype(np.float32)
            sp, og = np.asarray(g.volume_spacing, np.float32), np.asarray(g.volume_origin, np.float32)
            assert np.array_equal(x.cpu().numpy(), gh.cone_forward(v.cpu().numpy(), P, sp, og, g.detector_shape, 0.5)[0])


@pytest.mark.parametrize("det", [(512, 33), (497, 16), (528, 17), (496, 20), (640, 18)])
@pytest.mark.parametrize("storage", ["bf16", "f16"])
def test_forward_tile_rows_around_thirty_two(det, storage):
    # 31, 32, 33 and 40 tile rows of one to three tiles: rows that fill the XCDs evenly and rows that do not
    shape = (20, 24, 18)
    sp, og, P = _orbit(shape, 3, 100.0, 160.0, det, (60.0 / det[0], 60.0 / det[1]))
    vol = _rand_volume(shape, det[0], gh.DT[storage][1])
    _check_views(vol, P, sp, og, det, 0.5, False, views=range(3))


@pytest.mark.parametrize("plane", [(16, 16), (1, 80), (112, 33), (40, 150), (129, 65), (64, 64)])
@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_backprojection_tiles_one_to_forty(plane, storage):
    shape = (11,) + plane
    det = (24, 40)
    sp = np.ones(3, np.float32)
    og = geo.centred_origin(shape, sp).astype(np.float32)
    P = geo.circular_projection_matrices(6, 300.0, 480.0, det, (1.5, 6.0)).astype(np.float32)
    s = np.random.default_rng(plane[0]).normal(size=(6,) + det).astype(np.float32)
    s = torch.tensor(s).to(gh.DT[storage][1]).float().numpy()
    got = gh.cone_backward(s, P, sp, og, shape, storage=storage)[0]
    ref, _ = orc.cone_backward(s, P, shape, sp, og)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("tilt", [0.0, 1e-4])
@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape, n", [
    ((13, 30, 20), 3),       # 8 blocks of 8 voxels per lane: one voxel per lane, fewer views than four at a time
    ((80, 77, 75), 9),       # 250 blocks: one voxel per lane, two groups of views and one more
    ((61, 120, 131), 5),     # 576 blocks: four voxels per lane
    ((43, 200, 170), 5),     # 858 blocks of 8, a tenth of them padding: four
    ((47, 200, 170), 5),     # 858 blocks: eight
    ((5, 520, 410), 3),      # one slab of 8 for five slices: eight (four per lane pad as much)
    ((4, 520, 410), 3),      # and for four: four
    ((76, 160, 170), 2),     # the deepest range that four serve for its padding
    ((84, 160, 170), 2),     # the first beyond
])
def test_backprojection_voxels_per_lane(shape, n, storage, tilt):
    det = (90, 150)
    sp = np.ones(3, np.float32)
    og = geo.centred_origin(shape, sp).astype(np.float32)
    P = geo.circular_projection_matrices(n, 400.0, 640.0, det, (1.5, 2.2)).astype(np.float32)
    P[:, 2, 2] += np.float32(tilt)   # depth varies along z: no column shares its reciprocal
    s = np.random.default_rng(n).normal(size=(n,) + det).astype(np.float32)
    s = torch.tensor(s).to(gh.DT[storage][1]).float().numpy()
    got = gh.cone_backward(s, P, sp, og, shape, storage=storage)[0]
    ref, _ = orc.cone_backward(s, P, shape, sp, og)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("shapes", [
    ((3, 36, 40), (12, 45, 40)),        # few blocks: four voxels per lane by default
    ((5, 300, 320), (16, 250, 340)),    # 380 + 704 blocks and no padding that four would save: eight
    ((4, 500, 400), (12, 300, 310)),    # 800 + 760 blocks, padded: four
])
def test_batched_backprojection_default_voxels_per_lane(shapes, storage):
    det, n = (20, 60), 3
    geoms = [geo.ConeGeometry(s, (1.0, 1.0, 1.0), det, (1.5, 12.0), n, 600.0, 960.0) for s in shapes]
    rng = np.random.default_rng(len(shapes))
    sinos = [torch.tensor(rng.normal(size=(n,) + det)).to("cuda", gh.DT[storage][1]) for _ in shapes]
    for x, g, got in zip(sinos, geoms, batched.cone_backprojection3d_batched(sinos, geoms)):
        ref, _ = orc.cone_backward(x.float().cpu().numpy(), g.projection_matrices().astype(np.float32),
                                   g.volume_shape, np.asarray(g.volume_spacing, np.float32),
                                   np.asarray(g.volume_origin, np.float32), mult=np.float32(g.projection_multiplier))
        assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("shape, fits", [
    ((1000, 1019, 368), True),    # 3.034e9 bytes of x pairs, the last size within the byte offsets
    ((1000, 1020, 368), False),   # one row more: the 32-bit cell index
    ((1021, 1021, 2), False),     # 8 (H + 3)(D + 3) = 2^23
])
def test_forward_f32_cell_index_at_the_byte_offsets_limit(shape, fits):
    plane = (shape[1] + 3) * (shape[0] + 3)
    assert (8 * plane < 2 ** 23 and 8 * (shape[2] + 2) * plane <= 0xB5000000) == fits
    det = (32, 48)
    sp, og, P = _orbit(shape, 4, 3000.0, 5000.0, det, (30.0, 12.0 if shape[2] > 2 else 0.5))
    print(f"f32 cells {shape}", flush=True)
    _check_views(_rand_volume(shape, 7), P, sp, og, det, 0.5, False, views=(0, 1))
