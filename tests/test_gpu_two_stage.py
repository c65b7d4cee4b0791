"""The two-stage Cartesian passes (cart_two.hpp) against the FP64 oracle at
lengths that use every radix from 1 to 16 in either stage, with column tiles
and row blocks that do not divide the image.  A float32 transform of at most
2^16 points is within a few 1e-7 of the exact one (rounding of 4 radix stages,
6e-8 each, and of the twiddles): 2e-6 holds it with room."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(256, 128), (225, 240), (210, 196), (182, 168), (169, 143), (121, 110), (132, 144),
         (81, 90), (63, 72), (56, 49), (36, 42), (25, 30), (20, 16), (9, 12), (4, 6), (3, 2),
         (1, 5), (11, 13), (154, 14), (7, 1), (15, 8)]


@pytest.mark.parametrize("W,H", SIZES)
@pytest.mark.parametrize("centered", [False, True])
def test_operator_pair_every_radix(gpu, W, H, centered):
    print(f"[gpu two-stage] W={W} H={H} centered={centered}", flush=True)
    rng = np.random.default_rng(W * 1000 + H)
    c = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64).astype(np.complex128)
    T, C = 3, 5
    x, b1, z = c(T, H, W), c(C, H, W), c(T, C, H, W)
    mask = np.repeat((rng.random((T, H, 1)) < 0.4).astype(np.float64), W, axis=2)
    mask[0] = 0.0  # a frame with no sampled row
    for m in (None, mask):
        for got, ref in ((gpu.cart_K(x, b1, m, centered), O.cart_K(x, b1, m, centered)),
                         (gpu.cart_KH(z, b1, m, centered), O.cart_KH(z, b1, m, centered))):
            if not np.any(ref):
                assert not np.any(got)
            else:
                assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2e-6


@pytest.mark.parametrize("W,H,T,C", [(40, 36, 2, 1), (40, 36, 2, 2), (40, 36, 2, 3), (40, 36, 2, 4),
                                     (48, 256, 2, 7), (50, 225, 3, 9), (16, 64, 90, 4), (72, 64, 170, 3)])
def test_operator_pair_coil_groups(gpu, W, H, T, C):
    """Coil counts that the blocks' coil groups do not divide, a group without
    a coil, and grids on both sides of the sizes where the groups start."""
    print(f"[gpu coil groups] W={W} H={H} T={T} C={C}", flush=True)
    rng = np.random.default_rng(C)
    c = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64).astype(np.complex128)
    x, b1, z = c(T, H, W), c(C, H, W), c(T, C, H, W)
    mask = np.repeat((rng.random((T, H, 1)) < 0.5).astype(np.float64), W, axis=2)
    for got, ref in ((gpu.cart_K(x, b1, mask, False), O.cart_K(x, b1, mask, False)),
                     (gpu.cart_KH(z, b1, mask, False), O.cart_KH(z, b1, mask, False))):
        assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2e-6
