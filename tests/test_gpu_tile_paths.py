"""Back projections by image tiles, with the kernels that run on either side
named by the library: tiles (MI_TUNE_BP_IMAGE_TILES 2: wherever the geometry
allows them) against the column kernels or stored TOF records
(MI_TUNE_BP_IMAGE_TILES 0), GPU; and which of them the default takes.

The geometries and tolerances are those of test_gpu_tile.py, test_gpu_tile_short.py
and test_gpu_tile_tof.py. An infinite bin at the centre of a direct sinogram
reaches voxels on both sides, the same ones, and leaves no NaN.
"""
import numpy as np
import pytest

import test_gpu_tile
import test_gpu_tile_short
import test_gpu_tile_tof
from stir_amd import _native
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid
from stir_amd.projectors import ProjectorByBinPairMI355X, ProjMatrixByBinUsingRayTracing

pytestmark = pytest.mark.gpu

NAMES = ([("tall", n) for n in sorted(test_gpu_tile.CASES)] + [("short", n) for n in sorted(test_gpu_tile_short.CASES)] +
         [("tof", n) for n in sorted(test_gpu_tile_tof.CASES)])


def geometry(kind, name):
    """(projection data, image, parameters, kernel of the tiles, of the other side, the same bits)"""
    if kind == "tall":
        rings, crystals, span, mrd, views, tang, nz, ny, nx, vz, pm = test_gpu_tile.CASES[name]
        sc = Scanner.cylindrical(rings, crystals, 100.0, 4.0, name=name)
        pdi = ProjDataInfoCylindrical.construct(sc, span=span, max_delta=mrd, num_views=views, num_tangential_poss=tang)
        return (pdi, VoxelsOnCartesianGrid(nz, ny, nx, vz, 2.5, 2.5), RayTracingMatrixParameters(**pm),
                _native.MI_BACK_TILES, _native.MI_BACK_COLUMNS, True)
    if kind == "short":
        rings, span, mrd, views, nz, ny, nx, vz, ntof, same = test_gpu_tile_short.CASES[name]
        sc = Scanner(name, rings, 2 * views, 100.0, 0.0, 4.0, 4.0, 0.0, 44, 44, 400.0 if ntof else 0.0,
                     2500.0 / ntof if ntof else 0.0, ntof)
        tiles = _native.MI_BACK_SHORT_TILES
    else:
        rings, span, mrd, nz, ny, nx, ntof, ps = test_gpu_tile_tof.CASES[name]
        views, vz, same = 32, 2.0, False
        sc = Scanner(name, rings, 64, 100.0, 0.0, 4.0, 4.0, 0.0, 44, 44, 400.0, ps, ntof)
        tiles = _native.MI_BACK_TILES
    pdi = ProjDataInfoCylindrical.construct(sc, span, mrd, views, 44, False)
    if ntof:
        pdi = pdi.with_tof(1)
    return (pdi, VoxelsOnCartesianGrid(nz, ny, nx, vz, 2.5, 2.5), RayTracingMatrixParameters(), tiles,
            _native.MI_BACK_TOF_ROWS if ntof else _native.MI_BACK_COLUMNS, same)


def make(pdi, img, pm, tiles, num_subsets=4):
    P = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(pm))
    P.context.set_tuning(_native.MI_TUNE_BP_IMAGE_TILES, tiles)
    P.set_up(pdi, img, num_subsets=num_subsets)
    return P


@pytest.mark.parametrize("kind,name", NAMES)
def test_tiles_against_columns(kind, name):
    pdi, img, pm, tiles, other, same = geometry(kind, name)
    print(f"[tile paths] {kind} {name}: {pdi.num_bins} bins, image {img.shape}", flush=True)
    T, C = make(pdi, img, pm, 2), make(pdi, img, pm, 0)
    for subset in (-1, 3):
        assert T.context.projection_kernels(subset)[1] == tiles
        assert C.context.projection_kernels(subset)[1] == other
    rng = np.random.default_rng(91)
    terms = pdi.num_views * (2 * pdi.max_segment_num + 1) * 3 * max(T.info().tof_live_span, 1)
    mean = terms / 100.0
    for subset in (-1, 0, 3):
        y = rng.uniform(0.5, 2.0, pdi.num_bins).astype(np.float32)
        y[rng.uniform(size=pdi.num_bins) > 0.01] = 0.0
        a, b = T.back_project(y, subset=subset), C.back_project(y, subset=subset)
        assert b.max() > 0
        assert test_gpu_tile_short.same_or_close(a, b, same, mean + 16.0 * np.sqrt(mean) + 16.0), subset
    y = rng.uniform(0.5, 2.0, pdi.num_bins).astype(np.float32)
    block = pdi.num_bins // max(pdi.num_tof_bins, 1)
    y[pdi.num_tof_bins // 2 * block + pdi.bin_index(0, 5, pdi.num_axial_poss_of(0) // 2, 1)] = np.inf
    a, b = T.back_project(y), C.back_project(y)
    assert np.isinf(b).any()
    assert not np.isnan(a).any() and np.array_equal(np.isinf(a), np.isinf(b))
    T.close()
    C.close()


# rings, span, maximum ring difference, ny, nx, TOF bins, whether the default takes tiles: sides whose tiles in the
# field of view lie on either side of the line for one plane per axial position (350), two (150 of several slots, 260
# of one), mixed ones (95, 135), TOF (92, 45 and 55 a mean live bin), and never too few of short images
DEFAULTS = [
    (40, 5, 20, 96, 96, 0, False), (40, 5, 20, 160, 160, 0, False), (40, 5, 20, 176, 176, 0, True),
    (40, 5, 20, 60, 600, 0, False), (24, 5, 12, 130, 130, 0, False), (24, 5, 12, 200, 200, 0, True),
    (40, 1, 4, 96, 96, 0, False), (40, 1, 4, 120, 120, 0, True), (18, 1, 4, 128, 128, 0, False),
    (18, 1, 4, 150, 150, 0, True), (40, 3, 11, 60, 60, 0, False), (20, 3, 17, 96, 96, 0, False),
    (20, 3, 17, 112, 112, 0, True), (12, 1, 4, 24, 24, 0, True), (24, 3, 8, 100, 100, 9, False),
    (24, 3, 8, 260, 260, 9, True),
]


@pytest.mark.parametrize("rings,span,mrd,ny,nx,ntof,tiles", DEFAULTS)
def test_default_takes_tiles_only_where_they_are_faster(rings, span, mrd, ny, nx, ntof, tiles):
    sc = Scanner("default", rings, 64, 150.0, 0.0, 4.0, 4.0, 0.0, 30, 30, 400.0 if ntof else 0.0,
                 200.0 if ntof else 0.0, ntof)
    pdi = ProjDataInfoCylindrical.construct(sc, span, mrd, 32, 30, False)
    if ntof:
        pdi = pdi.with_tof(1)
    vox = 200.0 / max(nx, ny)
    img = VoxelsOnCartesianGrid(2 * rings - 1, ny, nx, 2.0, vox, vox)
    print(f"[tile paths] {rings} rings, span {span}, {ny} x {nx}, {ntof} TOF bins", flush=True)
    kernels = {True: (_native.MI_BACK_TILES, _native.MI_BACK_SHORT_TILES),
               False: (_native.MI_BACK_TOF_ROWS if ntof else _native.MI_BACK_COLUMNS,)}
    y = np.random.default_rng(92).uniform(0.5, 2.0, pdi.num_bins).astype(np.float32)
    default, other = make(pdi, img, RayTracingMatrixParameters(), 1), make(pdi, img, RayTracingMatrixParameters(),
                                                                           0 if tiles else 2)
    assert default.context.projection_kernels()[1] in kernels[tiles]
    assert other.context.projection_kernels()[1] in kernels[not tiles]
    a, b = default.back_project(y), other.back_project(y)
    assert np.abs(a - b).max() <= 1e-5 * b.max()
    default.close()
    other.close()


@pytest.mark.parametrize("kind,name", [("tall", "127planes_span11"), ("short", "31planes_many_phases"),
                                       ("tof", "64planes_9bins")])
def test_memory_limit_falls_back_to_the_other_table(kind, name):
    """The table does not fit at any of its allocations: the set-up succeeds with the other one."""
    pdi, img, pm, tiles, other, same = geometry(kind, name)
    y = np.random.default_rng(93).uniform(0.5, 2.0, pdi.num_bins).astype(np.float32)
    ref = make(pdi, img, pm, 0)
    b = ref.back_project(y)
    ref.close()
    P = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(pm))
    P.context.set_tuning(_native.MI_TUNE_BP_IMAGE_TILES, 2)
    kernels = []
    for mb in (1, 2, 4, 8, 16, 32, 64, 128, 256, 512, 0, 1):  # one context: a refused table leaves nothing behind
        P.context.set_tuning(_native.MI_TUNE_BP_TILE_MEMORY_MB, mb)
        P.set_up(pdi, img, num_subsets=4)
        kernels.append(P.context.projection_kernels()[1])
        assert np.abs(P.back_project(y) - b).max() <= 1e-5 * b.max(), mb
    print(f"[tile paths] {kind} {name}: kernels by limit {kernels}", flush=True)
    n = kernels.index(tiles)
    assert n >= 2 and kernels == [other] * n + [tiles] * (11 - n) + [other]
    P.close()


@pytest.mark.parametrize("name", ["64planes", "127planes_span11"])
def test_one_launch_per_subset_on_columns_and_blocks(name):
    """MI_TUNE_BP_SPLIT_SUBSETS acts on the column and block kernels: the sums of tiles, bit for bit."""
    pdi, img, pm, tiles, other, same = geometry("tall", name)
    y = np.random.default_rng(94).uniform(0.0, 2.0, pdi.num_bins).astype(np.float32)
    T = make(pdi, img, pm, 2)
    assert T.context.projection_kernels()[1] == _native.MI_BACK_TILES
    ref = T.back_project(y)
    T.close()
    Q = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(pm))
    Q.context.set_tuning(_native.MI_TUNE_BP_QUAD, 1)
    Q.set_up(pdi, img, num_subsets=4)
    for quad, kernel in ((0, _native.MI_BACK_COLUMNS), (1, _native.MI_BACK_BLOCKS)):
        Q.context.set_tuning(_native.MI_TUNE_BP_QUAD, quad)
        for split in (0, 1):
            Q.context.set_tuning(_native.MI_TUNE_BP_SPLIT_SUBSETS, split)
            assert Q.context.projection_kernels()[1] == kernel
            got = Q.back_project(y)
            assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (quad, split)
    Q.close()
