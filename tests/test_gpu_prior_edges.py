"""Neighbourhood priors and the two-stage sum of their values at image sizes
where the kernel's edges lie, against float64 on the host, GPU.

Tolerances: a term is two or three float32 operations on values of order 1, so
a gradient (26 terms) is within 26 x 4 x 2^-24 of the largest term's size, and
the value, summed in float64, within 4 x 2^-24 of itself: all terms are >= 0.
"""
import numpy as np
import pytest
import torch

from stir_amd.autograd import QuadraticPriorLoss, RelativeDifferencePriorLoss
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid
from stir_amd.projectors import ProjectorByBinPairMI355X, ProjMatrixByBinUsingRayTracing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 2, 65), (1, 5, 64), (2, 9, 63), (17, 132, 520)])
@pytest.mark.parametrize("kind", ["quadratic", "rdp"])
@pytest.mark.parametrize("with_kappa,only_2d", [(False, False), (True, True)])
def test_prior(shape, kind, with_kappa, only_2d):
    nz, ny, nx = shape
    sc = Scanner.cylindrical(1, 16, 2000.0, 4.0)
    pdi = ProjDataInfoCylindrical.construct(sc, span=1, max_delta=0, num_views=8, num_tangential_poss=4)
    img = VoxelsOnCartesianGrid(nz, ny, nx, 2.0, 2.5, 3.0)
    P = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(RayTracingMatrixParameters()))
    P.set_up(pdi, img, num_subsets=1)
    rng = np.random.default_rng(81)
    x = rng.uniform(0.5, 1.5, shape).astype(np.float32)
    kappa = rng.uniform(0.5, 1.5, shape).astype(np.float32) if with_kappa else None
    kt = None if kappa is None else torch.from_numpy(kappa).cuda()
    beta, gamma, eps = 0.7, 2.0, 0.1
    if kind == "quadratic":
        loss = QuadraticPriorLoss(P, beta, kt, only_2d)
    else:
        loss = RelativeDifferencePriorLoss(P, beta, gamma, eps, kt, only_2d)
    xt = torch.from_numpy(x).cuda().requires_grad_(True)
    value = loss(xt)
    value.backward()
    grad = xt.grad.cpu().numpy().astype(np.float64)
    ref_v, ref_g = 0.0, np.zeros(shape)
    x64 = x.astype(np.float64)
    k64 = np.ones(shape) if kappa is None else kappa.astype(np.float64)
    for dz in (0,) if only_2d else (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                if dz == dy == dx == 0:
                    continue
                w = 3.0 / np.sqrt((2.0 * dz) ** 2 + (2.5 * dy) ** 2 + (3.0 * dx) ** 2)
                a = tuple(slice(max(-d, 0), n - max(d, 0)) for d, n in zip((dz, dy, dx), shape))
                b = tuple(slice(max(d, 0), n - max(-d, 0)) for d, n in zip((dz, dy, dx), shape))
                if any(s.stop <= s.start for s in a):
                    continue
                xa, xb, kk = x64[a], x64[b], k64[a] * k64[b]
                d = xa - xb
                if kind == "quadratic":
                    ref_v += (w * d * d / 4 * kk).sum()
                    ref_g[a] += w * d * kk
                else:
                    den = xa + xb + gamma * np.abs(d) + eps
                    ref_v += (w * 0.5 * d * d / den * kk).sum()
                    ref_g[a] += w * d * (gamma * np.abs(d) + xa + 3 * xb + 2 * eps) / den ** 2 * kk
    P.close()
    ref_v *= beta
    ref_g *= beta
    assert abs(value.item() - ref_v) <= 4 * 2.0 ** -24 * abs(ref_v)
    # the largest term: w <= 1.2, |d| < 1, kappa^2 < 2.25, the fraction of the relative difference <= 4
    assert np.abs(grad - ref_g).max() <= 26 * 4 * 2.0 ** -24 * beta * 1.2 * 2.25 * (1.0 if kind == "quadratic" else 4.0)
