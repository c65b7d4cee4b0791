"""K^H of the gridding operator with one and two coils per column block (runtime
plans, narrow and wide) on either side of the block count where two are taken,
odd coil counts among them, against the FP64 oracle (2e-5, as for the operator's
other cases: the float32 kernel weights)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


# grid length (plan), one-coil blocks: 288 (narrow) 108 / 3240, 312 (wide) 117 / 2925,
# 840 (wide, large tiles) 210 / 2940
@pytest.mark.parametrize("n,osf,T,C", [(96, 3.0, 1, 3), (96, 3.0, 10, 9), (104, 3.0, 1, 3),
                                       (104, 3.0, 15, 5), (210, 4.0, 1, 1), (210, 4.0, 2, 7)])
def test_adjoint_coils(gpu, n, osf, T, C):
    print(f"[gpu adjoint coils] n={n} osf={osf} T={T} C={C}", flush=True)
    rng = np.random.default_rng(n + C)
    c = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64).astype(np.complex128)
    nfe, spf = 48, 3
    tr = O.radial_trajectory(nfe, spf, T).astype(np.float32).astype(np.float64)
    dcf = (np.sqrt(tr[:, 0] ** 2 + tr[:, 1] ** 2) + 0.01).astype(np.float32).astype(np.float64)
    op = gpu.A.NoncartesianOperator(n, n, C, T, nfe, spf, gpu._r(tr), gpu._r(dcf), kernel_width=3, osf=osf)
    b1, z = c(C, n, n), c(T, C, nfe * spf)
    got = gpu._n(op.ForwardOperation(gpu._t(z), gpu._t(b1)))
    ref = O.nufft_KH(z, b1, tr, dcf, 3, osf)
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 2e-5
