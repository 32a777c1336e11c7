"""Back projection by image tiles (the default for non-TOF matrices of more
than 32 planes) against the column kernel, GPU.

The column kernel runs on a context set up with the 2 x 2 block table and that
table switched off again; both kernels add the same terms to every voxel in
the same order with the same multiply and add, so they agree bit for bit, and
an infinite projection value reaches the same voxels.

Geometries at the edges: 33 planes (the fewest), 63, 64 and 65 (one or two
64-plane slots), 127, 139 and 255 planes (three and four slots), one plane per
axial position, two (span 1), both mixed, four (z zoom 2), image sides that are
not multiples of the 8 x 8 tile, two tangential LORs, no symmetries.
"""
import numpy as np
import pytest

from stir_amd import _native
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid
from stir_amd.projectors import (OSMAPOSLReconstruction, PoissonLogLikelihoodWithLinearModelForMeanAndProjData,
                                 ProjectorByBinPairMI355X, ProjMatrixByBinUsingRayTracing)

pytestmark = pytest.mark.gpu

# rings, crystals, span, maximum ring difference, views, tangential positions, planes, ny, nx, voxel z, parameters
CASES = {
    "33planes_span1": (17, 64, 1, 9, 32, 41, 33, 40, 40, 2.0, {}),
    "63planes_span3": (32, 64, 3, 4, 32, 48, 63, 41, 47, 2.0, {}),
    "64planes": (32, 64, 3, 7, 32, 48, 64, 48, 48, 2.0, {}),
    "65planes_mixed": (33, 64, 3, 32, 32, 48, 65, 48, 48, 2.0, {}),
    "127planes_span11": (64, 64, 11, 60, 32, 48, 127, 33, 33, 2.0, {}),
    "139planes_2lors": (70, 64, 5, 40, 32, 40, 139, 35, 37, 2.0, dict(num_tangential_LORs=2)),
    "255planes": (128, 64, 11, 40, 32, 40, 255, 24, 24, 2.0, {}),
    "zoom2": (10, 64, 3, 9, 32, 48, 38, 48, 48, 1.0, {}),
    "no_symmetries": (20, 64, 3, 11, 32, 47, 39, 31, 31, 2.0,
                      dict(do_symmetry_90degrees_min_phi=False, do_symmetry_180degrees_min_phi=False,
                           do_symmetry_swap_segment=False, do_symmetry_swap_s=False)),
}


@pytest.fixture(scope="module", params=sorted(CASES))
def case(request):
    rings, crystals, span, mrd, views, tang, nz, ny, nx, vz, pm = CASES[request.param]
    sc = Scanner.cylindrical(rings, crystals, 100.0, 4.0, name=request.param)
    pdi = ProjDataInfoCylindrical.construct(sc, span=span, max_delta=mrd, num_views=views, num_tangential_poss=tang)
    img = VoxelsOnCartesianGrid(nz, ny, nx, vz, 2.5, 2.5)
    print(f"[tile] {request.param}: {pdi.num_bins} bins, image {img.shape}", flush=True)
    out = []
    for quad in (0, 1):
        P = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(RayTracingMatrixParameters(**pm)))
        P.context.set_tuning(_native.MI_TUNE_BP_QUAD, quad)
        P.set_up(pdi, img, num_subsets=4)
        P.context.set_tuning(_native.MI_TUNE_BP_QUAD, 0)
        out.append(P)
    yield pdi, img, out[0], out[1]
    for P in out:
        P.close()


def test_back_projection_bit_identical(case):
    pdi, img, T, C = case
    y = np.random.default_rng(51).uniform(0.0, 2.0, pdi.num_bins).astype(np.float32)
    for subset in (-1, 0, 3):
        a, b = T.back_project(y, subset=subset), C.back_project(y, subset=subset)
        assert b.max() > 0
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), subset


def test_infinite_value_stays_in_its_voxels(case):
    pdi, img, T, C = case
    y = np.random.default_rng(52).uniform(0.0, 2.0, pdi.num_bins).astype(np.float32)
    y[pdi.bin_index(0, 5, pdi.num_axial_poss_of(0) // 2, 1)] = np.inf
    a, b = T.back_project(y), C.back_project(y)
    assert np.isinf(b).any() and not np.isnan(a).any()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_osem_update_bit_identical(case):
    pdi, img, T, C = case
    y = np.random.default_rng(53).poisson(3.0, pdi.num_bins).astype(np.float32)
    x = np.random.default_rng(54).uniform(0.5, 1.5, img.shape).astype(np.float32)
    out = []
    for P in (T, C):
        obj = PoissonLogLikelihoodWithLinearModelForMeanAndProjData(P)
        obj.set_up(y, 0.1)
        obj.set_estimate(x)
        recon = OSMAPOSLReconstruction(obj, 2)
        recon.update_estimate(1, 1)
        recon.update_estimate(2, 2)
        out.append(obj.get_estimate())
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
