"""Forward projection by row groups (the families of small scanners) against
the task kernel, GPU.

The projection of given view-segments runs the task kernel; both sum every bin
over its row in row order, so the projections agree bit for bit, and so do the
log-likelihood's values within FP64 rounding of another summation order (1e-12).

Geometries at the edges: one ring (families of one bin), families whose groups
fill whole waves (8 x 8 bins) or leave one bin over, images with fewer planes
than the scanner covers (rows that reach past the padding zeros), 16 planes (no
padding at all), a square field of view, no symmetries (groups of one family).
"""
import numpy as np
import pytest

from stir_amd import _native
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid
from stir_amd.projectors import (ForwardProjectorByBinMI355X, PoissonLogLikelihoodWithLinearModelForMeanAndProjData,
                                 ProjectorByBinPairMI355X, ProjMatrixByBinUsingRayTracing)

pytestmark = pytest.mark.gpu

# rings, span, maximum ring difference, planes, image side, parameters
CASES = {
    "one_ring": (1, 1, 0, 1, 40, {}),
    "8rings": (8, 1, 3, 15, 40, {}),
    "9rings_16planes": (9, 1, 8, 16, 41, {}),
    "13rings_few_planes": (13, 3, 12, 11, 40, {}),
    "12rings_square": (12, 1, 5, 23, 40, dict(restrict_to_cylindrical_FOV=False)),
    "10rings_no_symmetries": (10, 1, 4, 19, 39, dict(do_symmetry_90degrees_min_phi=False,
                                                     do_symmetry_180degrees_min_phi=False,
                                                     do_symmetry_swap_segment=False, do_symmetry_swap_s=False)),
    "16rings_2lors": (16, 1, 6, 31, 40, dict(num_tangential_LORs=2)),
}


@pytest.fixture(scope="module", params=sorted(CASES))
def case(request):
    rings, span, mrd, nz, n, pm = CASES[request.param]
    sc = Scanner.cylindrical(rings, 64, 100.0, 4.0, name=request.param)
    pdi = ProjDataInfoCylindrical.construct(sc, span=span, max_delta=mrd, num_views=32, num_tangential_poss=43)
    img = VoxelsOnCartesianGrid(nz, n, n, 2.0, 2.5, 2.5)
    print(f"[rows] {request.param}: {pdi.num_bins} bins, image {img.shape}", flush=True)
    P = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(RayTracingMatrixParameters(**pm)))
    P.set_up(pdi, img, num_subsets=4)
    yield pdi, img, P
    P.close()


def test_forward_projection_bit_identical(case):
    pdi, img, P = case
    x = np.random.default_rng(61).uniform(0.0, 2.0, img.shape).astype(np.float32)
    F = ForwardProjectorByBinMI355X(P)
    F.set_input(x)
    for subset in (0, 3):
        ref = F.forward_project(subset_num=subset, num_subsets=4)
        got = P.forward_project(x, subset=subset)
        assert ref.max() > 0
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), subset
    ref = F.forward_project()
    assert np.array_equal(P.forward_project(x).view(np.uint32), ref.view(np.uint32))


def test_log_likelihood_value(case):
    pdi, img, P = case
    x = np.random.default_rng(62).uniform(0.5, 2.0, img.shape).astype(np.float32)
    y = np.random.default_rng(63).poisson(3.0, pdi.num_bins).astype(np.float32)
    obj = PoissonLogLikelihoodWithLinearModelForMeanAndProjData(P)
    obj.set_up(y, 0.25, compute_sensitivities=False)
    ybar = P.forward_project(x) + np.float32(0.25)
    est = np.maximum(ybar, y / np.float32(10000)).astype(np.float64)
    terms = np.where(y > 0, y * np.log(est), 0.0) - est
    value = obj.compute_objective_function_without_penalty(x)
    # FP64 rounding of 2^k terms in two orders, the device's logarithm within an ulp or two
    assert abs(value - terms.sum()) <= 1e-12 * np.abs(terms).sum()
