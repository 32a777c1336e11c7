"""Batches: every limit of the forward projection's row groups gives the same
images, GPU. Problems whose longest families lie under, between and over the
limits (15, 31, 47 and 63 axial positions); bins are summed in row order by
every kernel, so the images agree bit for bit.
"""
import numpy as np
import pytest

from stir_amd.batch import BatchedOSMAPOSL
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid

pytestmark = pytest.mark.gpu


def test_row_group_limits_give_the_same_images():
    problems = []
    for rings, span in ((8, 3), (16, 3), (24, 3), (32, 3), (12, 1)):
        sc = Scanner.cylindrical(rings, 64, 100.0, 4.0, name=f"{rings} rings")
        pdi = ProjDataInfoCylindrical.construct(sc, span=span, max_delta=rings - 1, num_views=32, num_tangential_poss=33)
        problems.append((pdi, VoxelsOnCartesianGrid(2 * rings - 1, 40, 40, 2.0, 2.5, 2.5), RayTracingMatrixParameters()))
    B = BatchedOSMAPOSL(problems, 4)
    for i, (pdi, img, pm) in enumerate(problems):
        B.set_data(i, np.random.default_rng(i).poisson(3.0, pdi.num_bins).astype(np.float32), 0.1)
    ref = None
    for limit in (32, 0, 8, 16, 27, 28, 31, 48, 64):
        B.set_launch(row_groups=limit)
        for i, (pdi, img, pm) in enumerate(problems):
            B.set_estimate(i, np.ones(img.shape, np.float32))
        B.run(4)
        got = [B.get_estimate(i) for i in range(len(B))]
        assert all(g.max() > 0 and np.isfinite(g).all() for g in got)
        if ref is None:
            ref = got
        for a, b in zip(ref, got):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), limit
    B.close()
