"""Back projection by image tiles of short images (up to 32 planes) against the
column kernels, GPU.

The column kernels run on a context set up with the 2 x 2 block table asked
for. With one plane per axial position, or mixed ones, both sides add the same
terms to a voxel in the same order and agree bit for bit. With two planes per
axial position (span 1) and with TOF the grouping differs. Tolerances there,
per voxel and relative (all terms are >= 0): a float32 sum of n terms by any
grouping is within n 2^-24 of the exact one to first order, so two of them are
within 2 n 2^-24. With one bin in 100 set, a voxel has a few tens of non-zero
terms, so that a term that is lost or misplaced shows.

Sizes at the edges: 1, 15, 16, 17, 31 and 32 planes (8, 16 and 32 lanes per
line), image sides that are not multiples of the 8 x 4 or 4 x 4 tile, fewer and
no fewer than 512 tiles (one or two sets of lines per wave), four planes per axial position, more than 64 phases per tile and fewer rows than one copy.
"""
import numpy as np
import pytest

from stir_amd import _native
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid
from stir_amd.projectors import (OSMAPOSLReconstruction, PoissonLogLikelihoodWithLinearModelForMeanAndProjData,
                                 ProjectorByBinPairMI355X, ProjMatrixByBinUsingRayTracing)

pytestmark = pytest.mark.gpu

# rings, span, maximum ring difference, views, planes, ny, nx, voxel z, TOF bins, the same bits
CASES = {
    "1plane": (1, 1, 0, 32, 1, 41, 39, 2.0, 0, False),
    "15planes_span1": (8, 1, 7, 32, 15, 41, 47, 2.0, 0, False),
    "15planes_span3": (8, 3, 7, 32, 15, 41, 47, 2.0, 0, True),
    "16planes_span1": (8, 1, 3, 32, 16, 32, 32, 2.0, 0, False),
    "17planes_span1": (9, 1, 8, 32, 17, 33, 35, 2.0, 0, False),
    "31planes_span3": (16, 3, 10, 32, 31, 40, 41, 2.0, 0, True),
    "32planes_mixed": (16, 3, 15, 32, 32, 40, 40, 2.0, 0, True),
    "31planes_many_phases": (16, 1, 15, 96, 31, 30, 30, 2.0, 0, False),
    "31planes_span1_512tiles": (16, 1, 3, 32, 31, 130, 132, 2.0, 0, False),
    "32planes_span3_512tiles": (16, 3, 7, 32, 32, 128, 128, 2.0, 0, True),
    "31planes_tof_512tiles": (16, 1, 3, 32, 31, 130, 132, 2.0, 5, False),
    "31planes_span3_tof_512tiles": (16, 3, 7, 32, 31, 128, 128, 2.0, 5, False),
    "14planes_zoom2": (4, 1, 3, 32, 14, 40, 40, 1.0, 0, True),
    "15planes_tof": (8, 1, 7, 32, 15, 41, 47, 2.0, 5, False),
    "31planes_span3_tof": (16, 3, 10, 32, 31, 40, 41, 2.0, 9, False),
}


@pytest.fixture(scope="module", params=sorted(CASES))
def case(request):
    rings, span, mrd, views, nz, ny, nx, vz, ntof, same = CASES[request.param]
    sc = Scanner(request.param, rings, 2 * views, 100.0, 0.0, 4.0, 4.0, 0.0, 44, 44, 400.0 if ntof else 0.0,
                 2500.0 / ntof if ntof else 0.0, ntof)
    pdi = ProjDataInfoCylindrical.construct(sc, span, mrd, views, 44, False)
    if ntof:
        pdi = pdi.with_tof(1)
    img = VoxelsOnCartesianGrid(nz, ny, nx, vz, 2.5, 2.5)
    out = []
    for quad in (0, 1):
        P = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(RayTracingMatrixParameters()))
        P.context.set_tuning(_native.MI_TUNE_BP_QUAD, quad)
        P.set_up(pdi, img, num_subsets=4)
        P.context.set_tuning(_native.MI_TUNE_BP_QUAD, 0)
        out.append(P)
    print(f"[tile short] {request.param}: {pdi.num_bins} bins, image {img.shape}", flush=True)
    yield pdi, img, out[0], out[1], same
    for P in out:
        P.close()


def same_or_close(a, b, same, n):
    if same:
        return np.array_equal(a.view(np.uint32), b.view(np.uint32))
    a, b = a.astype(np.float64), b.astype(np.float64)
    return np.array_equal(a == 0, b == 0) and (np.abs(a - b) <= 2.0 * n * 2.0 ** -24 * b).all()


def test_back_projection(case):
    pdi, img, T, C, same = case
    rng = np.random.default_rng(71)
    # a (view, segment) has at most 3 rays through a voxel, each with the live
    # span's TOF bins; of sparse data 16 standard deviations above the mean
    terms = pdi.num_views * (2 * pdi.max_segment_num + 1) * 3 * max(T.info().tof_live_span, 1)
    for subset in (-1, 0, 3):
        y = rng.uniform(0.5, 2.0, pdi.num_bins).astype(np.float32)
        a, b = T.back_project(y, subset=subset), C.back_project(y, subset=subset)
        assert b.max() > 0
        assert same_or_close(a, b, same, terms), subset
        y[rng.uniform(size=pdi.num_bins) > 0.01] = 0.0
        mean = terms / 100.0
        a, b = T.back_project(y, subset=subset), C.back_project(y, subset=subset)
        assert same_or_close(a, b, same, mean + 16.0 * np.sqrt(mean) + 16.0), subset


def test_infinite_value_stays_in_its_voxels(case):
    pdi, img, T, C, same = case
    y = np.random.default_rng(72).uniform(0.5, 2.0, pdi.num_bins).astype(np.float32)
    y[pdi.num_bins // 2 + 22] = np.inf
    a, b = T.back_project(y), C.back_project(y)
    assert not np.isnan(a).any() and np.array_equal(np.isinf(a), np.isinf(b))


def test_osem_update(case):
    pdi, img, T, C, same = case
    y = np.random.default_rng(73).poisson(3.0, pdi.num_bins).astype(np.float32)
    x = np.random.default_rng(74).uniform(0.5, 1.5, img.shape).astype(np.float32)
    out = []
    for P in (T, C):
        obj = PoissonLogLikelihoodWithLinearModelForMeanAndProjData(P)
        obj.set_up(y, 0.1)
        obj.set_estimate(x)
        recon = OSMAPOSLReconstruction(obj, 2)
        recon.update_estimate(1, 1)
        recon.update_estimate(2, 2)
        out.append(obj.get_estimate())
    mask = out[1] > 1e-3 * out[1].max()
    assert (np.abs(out[0] - out[1])[mask] <= 1e-4 * out[1][mask]).all()
    if same:
        assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
