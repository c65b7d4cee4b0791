"""Transforms of the standalone 2D FFT and the gridding passes on runtime
plans, against the FP64 oracle: lengths whose stages cover every plan radix
(two-stage, narrow and wide kinds, one-stage lengths with their radix-1
partner), and image and grid sizes that leave partial tiles.  FFT tolerance:
2e-6 as for the other FFT cases; gridding: 2e-5 as for the other geometries
(the float32 kernel weights)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _c(rng, *s):
    return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64).astype(np.complex128)


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("W,H", [(1, 1), (7, 1), (1, 270), (13, 16), (225, 100), (300, 432),
                                 (486, 250), (245, 320), (605, 336), (845, 30), (480, 512)])
@pytest.mark.parametrize("centered", [False, True])
def test_fft2_plan_radices(gpu, W, H, centered):
    print(f"[gpu fft2] W={W} H={H} centered={centered}", flush=True)
    a = _c(np.random.default_rng(W + H), 2, H, W)
    got = gpu.fft2(a, -1, centered)
    ref = np.stack([O.fft2(a[i], -1, centered) for i in range(2)])
    assert _rel(got, ref) < 2e-6


# (W, H, C, T, nFE, spokes, osf): grids 240 x 210, 288 x 252, 448 x 336, 300 x 12, 143 x 130,
# 528 x 90 (wide), 225 x 14
@pytest.mark.parametrize("W,H,C,T,nfe,spf,osf", [
    (160, 140, 3, 2, 96, 7, 1.5), (192, 168, 2, 1, 96, 5, 1.5), (224, 168, 3, 1, 128, 5, 2.0),
    (200, 8, 2, 2, 64, 4, 1.5), (110, 100, 2, 2, 64, 5, 1.3), (264, 45, 2, 1, 96, 5, 2.0),
    (150, 9, 4, 1, 64, 3, 1.5)])
def test_gridding_runtime_plans(gpu, W, H, C, T, nfe, spf, osf):
    print(f"[gpu gridding] W={W} H={H} C={C} T={T} osf={osf}", flush=True)
    rng = np.random.default_rng(W)
    tr = O.radial_trajectory(nfe, spf, T).astype(np.float32).astype(np.float64)
    dcf = (np.sqrt(tr[:, 0] ** 2 + tr[:, 1] ** 2) + 0.01).astype(np.float32).astype(np.float64)
    op = gpu.A.NoncartesianOperator(W, H, C, T, nfe, spf, gpu._r(tr), gpu._r(dcf), kernel_width=3,
                                    osf=osf)
    x, b1, z = _c(rng, T, H, W), _c(rng, C, H, W), _c(rng, T, C, nfe * spf)
    got = gpu._n(op.BackwardOperation(gpu._t(x), gpu._t(b1)))
    assert _rel(got, O.nufft_K(x, b1, tr, dcf, 3, osf)) < 2e-5
    got = gpu._n(op.ForwardOperation(gpu._t(z), gpu._t(b1)))
    assert _rel(got, O.nufft_KH(z, b1, tr, dcf, 3, osf)) < 2e-5
