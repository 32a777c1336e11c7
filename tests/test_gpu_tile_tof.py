"""TOF back projection by image tiles (the default for TOF matrices of more
than 32 planes) against the stored back records, GPU.

The records run on a context that is set up with the 2 x 2 block table asked
for, which keeps the tile table from being made. Both kernels add
weight x bin with the same float32 weights, in another order and grouping.

Tolerances, per voxel and relative (all terms are >= 0): a float32 sum of n
terms by any grouping is within n 2^-24 of the exact one to first order, so two
of them are within 2 n 2^-24. With one bin in 400 set, a voxel has a few tens
of non-zero terms, so that a term that is lost or misplaced shows.
"""
import numpy as np
import pytest

from stir_amd import _native
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid
from stir_amd.projectors import (OSMAPOSLReconstruction, PoissonLogLikelihoodWithLinearModelForMeanAndProjData,
                                 ProjectorByBinPairMI355X, ProjMatrixByBinUsingRayTracing)

pytestmark = pytest.mark.gpu

# rings, span, maximum ring difference, planes, ny, nx, TOF bins, ps per bin
CASES = {
    "33planes_span1_5bins": (17, 1, 6, 33, 40, 40, 5, 500.0),
    "64planes_9bins": (32, 3, 7, 64, 41, 47, 9, 250.0),
    "65planes_mixed_11bins": (33, 3, 32, 65, 48, 48, 11, 130.0),
    "139planes_7bins": (60, 5, 40, 139, 35, 37, 7, 300.0),
    "255planes_5bins": (64, 11, 40, 255, 24, 24, 5, 500.0),
}


@pytest.fixture(scope="module", params=sorted(CASES))
def case(request):
    rings, span, mrd, nz, ny, nx, ntof, ps = CASES[request.param]
    sc = Scanner(request.param, rings, 64, 100.0, 0.0, 4.0, 4.0, 0.0, 44, 44, 400.0, ps, ntof)
    pdi = ProjDataInfoCylindrical.construct(sc, span, mrd, 32, 44, False).with_tof(1)
    img = VoxelsOnCartesianGrid(nz, ny, nx, 2.0, 2.5, 2.5)
    out = []
    for quad in (0, 1):
        P = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(RayTracingMatrixParameters()))
        P.context.set_tuning(_native.MI_TUNE_BP_QUAD, quad)
        P.set_up(pdi, img, num_subsets=4)
        out.append(P)
    info = out[0].info()
    print(f"[tile tof] {request.param}: {pdi.num_bins} bins, image {img.shape}, live span {info.tof_live_span}", flush=True)
    yield pdi, img, out[0], out[1]
    for P in out:
        P.close()


def test_sparse_data(case):
    pdi, img, T, R = case
    rng = np.random.default_rng(61)
    for subset in (-1, 0, 3, -1):
        y = np.zeros(pdi.num_bins, np.float32)
        at = rng.choice(pdi.num_bins, pdi.num_bins // 400, replace=False)
        y[at] = rng.uniform(0.5, 2.0, at.size).astype(np.float32)
        a, b = T.back_project(y, subset=subset).astype(np.float64), R.back_project(y, subset=subset).astype(np.float64)
        assert b.max() > 0
        # terms of a voxel: a (view, segment) has at most 3 rays through it and
        # each has live_span bins; 16 standard deviations above the mean number set
        mean = pdi.num_views * (2 * pdi.max_segment_num + 1) * 3 * T.info().tof_live_span / 400.0
        n = mean + 16.0 * np.sqrt(mean) + 16.0
        assert np.array_equal(a == 0, b == 0)
        assert (np.abs(a - b) <= 2.0 * n * 2.0 ** -24 * b).all(), (subset, (np.abs(a - b) / np.maximum(b, 1e-30)).max())


def test_dense_data_and_infinity(case):
    pdi, img, T, R = case
    y = np.random.default_rng(62).uniform(0.0, 2.0, pdi.num_bins).astype(np.float32)
    for subset in (-1, 2):
        a, b = T.back_project(y, subset=subset), R.back_project(y, subset=subset)
        assert np.abs(a - b).max() <= 1e-5 * b.max()
    y[pdi.num_bins // 2] = np.inf  # the middle TOF bin's block
    a, b = T.back_project(y), R.back_project(y)
    assert not np.isnan(a).any() and np.array_equal(np.isinf(a), np.isinf(b))


@pytest.mark.parametrize("tof_sens", [False, True])
def test_osem(case, tof_sens):
    pdi, img, T, R = case
    y = np.random.default_rng(63).poisson(3.0, pdi.num_bins).astype(np.float32)
    x = np.random.default_rng(64).uniform(0.5, 1.5, img.shape).astype(np.float32)
    out = []
    for P in (T, R):
        obj = PoissonLogLikelihoodWithLinearModelForMeanAndProjData(P)
        obj.set_up(y, 0.1, use_tof_sensitivities=tof_sens)
        obj.set_estimate(x)
        recon = OSMAPOSLReconstruction(obj, 2)
        recon.update_estimate(1, 1)
        recon.update_estimate(2, 2)
        out.append(obj.get_estimate())
    mask = out[1] > 1e-3 * out[1].max()
    assert (np.abs(out[0] - out[1])[mask] <= 1e-4 * out[1][mask]).all()
