"""The region form of the coil-estimation loops (several iterations per launch)
against the FP64 oracle: images that the regions do not divide, thinner than a
region's halo, iteration counts that the launches do not divide, and grids on
both sides of the sizes that pick small and large regions.  Tolerance 1e-4 as
for the other coil steps (float32 loops)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _problem(W, H, C, seed):
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:H, 0:W]
    u = 100 * (1 + np.exp(-((x - W / 2) ** 2 / W**2 + (y - H / 2) ** 2 / H**2) * 4)) * np.exp(0.3j * x / W)
    b = np.stack([np.exp(1j * rng.uniform(0, 6) + (0.5 + 0.2j) * np.cos(x / W * 3 + c) + 0.2j * y / H) for c in range(C)])
    crec = b * u + 0.5 * (rng.standard_normal((C, H, W)) + 1j * rng.standard_normal((C, H, W)))
    c = lambda a: np.asarray(a, np.complex64).astype(np.complex128)
    return c(u), c(crec), c(b)


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("W,H,C,its", [(33, 17, 1, 9), (5, 70, 2, 8), (64, 1, 1, 12), (1, 40, 2, 7),
                                       (120, 100, 24, 21), (200, 90, 3, 16)])
def test_b1_recon_regions(gpu, W, H, C, its):
    print(f"[gpu coil regions] b1 W={W} H={H} C={C} its={its}", flush=True)
    u, crec, _ = _problem(W, H, C, W + its)
    got = gpu.coil_b1_recon(u, crec, its, 2.0)
    assert _rel(got, O.coil_b1_recon(u, crec, its, 2.0)) < 1e-4


@pytest.mark.parametrize("W,H", [(33, 17), (12, 50), (1, 30), (30, 1), (528, 520)])
def test_utgv2_regions(gpu, W, H):
    print(f"[gpu coil regions] utgv2 W={W} H={H}", flush=True)
    u, crec, b1 = _problem(W, H, 2, W)
    x0 = np.zeros((H, W), np.complex128)
    assert _rel(gpu.coil_utgv2(b1, crec, [1, 0], x0), O.coil_utgv2(b1, crec, [1, 0], x0)) < 1e-4
