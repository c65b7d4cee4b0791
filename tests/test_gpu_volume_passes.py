"""The volumetric operator's separable passes against numpy's FFT in float64:
axes on two-stage, narrow and wide plans, partial row and column tiles, coil
counts that the adjoint's waves do not divide, with and without a mask.
(The dual update runs in the reconstruction cases of test_gpu_3d.py.)
Tolerance 2e-6 as for the other volume cases (float32 transforms)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,D,C", [(128, 20, 12, 1), (30, 32, 7, 2), (300, 5, 3, 3), (9, 6, 270, 5),
                                     (22, 143, 4, 6), (605, 3, 2, 4), (16, 16, 16, 9)])
@pytest.mark.parametrize("masked", [False, True])
def test_volume_pair(gpu, W, H, D, C, masked):
    print(f"[gpu volume] W={W} H={H} D={D} C={C} masked={masked}", flush=True)
    rng = np.random.default_rng(W + D)
    c = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    u, b1, z = c(D, H, W), c(C, D, H, W), c(C, D, H, W)
    m = (rng.random((D, H, W)) < 0.5).astype(np.float32) if masked else np.ones((D, H, W), np.float32)
    op = gpu.A.CartesianOperator3D(W, H, D, C, mask=gpu._r(m) if masked else None)
    ax = (1, 2, 3)
    u64, b64, z64 = u.astype(np.complex128), b1.astype(np.complex128), z.astype(np.complex128)
    got = gpu._n(op.BackwardOperation(gpu._t(u), gpu._t(b1)))
    ref = np.fft.ifftn(b64 * u64, axes=ax, norm="ortho") * m
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2e-6
    got = gpu._n(op.ForwardOperation(gpu._t(z), gpu._t(b1)))
    ref = (b64.conj() * np.fft.fftn(z64 * m, axes=ax, norm="ortho")).sum(0)
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2e-6
