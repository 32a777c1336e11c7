"""Forward projection by row groups against tasks, with the kernel that runs on
either side named by the library (MI_TUNE_FP_ROW_GROUPS 2 and 0), GPU; and which
of them the default takes for projections of all subsets and of one.

Both sum every bin over its row in row order: the same bits, and the same
log-likelihood values within FP64 rounding of another order (1e-12).
"""
import numpy as np
import pytest

import test_gpu_rows
from stir_amd import _native
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid
from stir_amd.projectors import (PoissonLogLikelihoodWithLinearModelForMeanAndProjData, ProjectorByBinPairMI355X,
                                 ProjMatrixByBinUsingRayTracing)

pytestmark = pytest.mark.gpu

TASKS, ROWS = _native.MI_FORWARD_TASKS, _native.MI_FORWARD_ROW_GROUPS


def make(pdi, img, pm, rows, num_subsets):
    P = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(RayTracingMatrixParameters(**pm)))
    P.context.set_tuning(_native.MI_TUNE_FP_ROW_GROUPS, rows)
    P.set_up(pdi, img, num_subsets=num_subsets)
    return P


@pytest.mark.parametrize("name", sorted(test_gpu_rows.CASES) + ["40rings_long_families"])
def test_row_groups_against_tasks(name):
    rings, span, mrd, nz, n, pm = test_gpu_rows.CASES.get(name, (40, 3, 10, 79, 40, {}))
    sc = Scanner.cylindrical(rings, 64, 100.0, 4.0, name=name)
    pdi = ProjDataInfoCylindrical.construct(sc, span=span, max_delta=mrd, num_views=32, num_tangential_poss=43)
    img = VoxelsOnCartesianGrid(nz, n, n, 2.0, 2.5, 2.5)
    print(f"[rows paths] {name}: {pdi.num_bins} bins, image {img.shape}", flush=True)
    R, T = make(pdi, img, pm, 2, 4), make(pdi, img, pm, 0, 4)
    x = np.random.default_rng(64).uniform(0.0, 2.0, img.shape).astype(np.float32)
    for subset in (-1, 0, 3):
        assert R.context.projection_kernels(subset)[0] == ROWS and T.context.projection_kernels(subset)[0] == TASKS
        a, b = R.forward_project(x, subset=subset), T.forward_project(x, subset=subset)
        assert b.max() > 0 and np.array_equal(a.view(np.uint32), b.view(np.uint32)), subset
    y = np.random.default_rng(65).poisson(3.0, pdi.num_bins).astype(np.float32)
    values = []
    for P in (R, T):
        obj = PoissonLogLikelihoodWithLinearModelForMeanAndProjData(P)
        obj.set_up(y, 0.25, compute_sensitivities=False)
        values.append(obj.compute_objective_function_without_penalty(x))
    est = np.maximum(T.forward_project(x) + np.float32(0.25), y / np.float32(10000)).astype(np.float64)
    scale = np.abs(np.where(y > 0, y * np.log(est), 0.0) - est).sum()
    assert abs(values[0] - values[1]) <= 1e-12 * scale
    R.close()
    T.close()


# rings, crystals, span, maximum ring difference, image side, subsets, kernels of all subsets and of one: short
# families, groups that save a factor of two (whole projections only, where a subset is one round of waves), an image
# that does not fit the L2, and long families
DEFAULTS = [(8, 192, 1, 3, 60, 8, ROWS, ROWS), (16, 288, 3, 15, 200, 16, ROWS, TASKS),
            (20, 96, 3, 7, 300, 4, TASKS, TASKS), (32, 96, 5, 22, 60, 4, TASKS, TASKS)]


@pytest.mark.parametrize("rings,crystals,span,mrd,n,num_subsets,whole,subset", DEFAULTS)
def test_default_takes_row_groups_only_where_they_are_faster(rings, crystals, span, mrd, n, num_subsets, whole, subset):
    sc = Scanner.cylindrical(rings, crystals, 350.0, 4.0, name="default")
    pdi = ProjDataInfoCylindrical.construct(sc, span=span, max_delta=mrd, num_views=crystals // 2,
                                            num_tangential_poss=crystals // 2)
    img = VoxelsOnCartesianGrid(2 * rings - 1, n, n, 2.0, 350.0 / n, 350.0 / n)
    print(f"[rows paths] {rings} rings, span {span}, {n} x {n}", flush=True)
    D, T = make(pdi, img, {}, 1, num_subsets), make(pdi, img, {}, 0, num_subsets)
    x = np.random.default_rng(66).uniform(0.0, 2.0, img.shape).astype(np.float32)
    for s, kernel in ((-1, whole), (1, subset)):
        assert D.context.projection_kernels(s)[0] == kernel
        a, b = D.forward_project(x, subset=s), T.forward_project(x, subset=s)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    D.close()
    T.close()
