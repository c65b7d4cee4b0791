"""The Cartesian passes as the solvers run them, at lengths that use every radix
from 1 to 16 in either stage: K and K^H on wide column tiles, where a lane runs
several butterflies of the second stage; the dual update with both transforms in
one pass, the step rule's norms (K of a difference) and the data residual against
the FP64 oracle; and launch sets whose column tiles differ, bit for bit.
Volumes: the dual update on narrow and wide depth plans.

Tolerances: 2e-6 for one transform pair as in test_gpu_two_stage.py; 1e-5 for three
step-rule iterations as for the engine's full-size reconstructions (three pairs and
the stencils between); 1e-5 for the residual, a float32 K minus data of its size."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(256, 128), (225, 240), (210, 196), (182, 168), (169, 143), (121, 110), (132, 144),
         (81, 90), (63, 72), (56, 49), (36, 42), (25, 30), (20, 16), (9, 12), (4, 6), (11, 13),
         (154, 14), (15, 8), (128, 32), (39, 45)]


def _c(rng, *s):
    return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64).astype(np.complex128)


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# heights whose two radices need different powers of two of lanes, at least 512 wide
# tiles: 8 x 4, 13 x 3, 9 x 5, 13 x 4, 12 x 8, 14 x 8
@pytest.mark.parametrize("H,T", [(32, 256), (39, 256), (45, 171), (52, 256), (96, 171), (112, 171)])
@pytest.mark.parametrize("centered", [False, True])
def test_operator_pair_wide_tiles(gpu, H, T, centered):
    print(f"[gpu wide tiles] H={H} T={T} centered={centered}", flush=True)
    W, C = 70, 2
    rng = np.random.default_rng(H)
    x, b1, z = _c(rng, T, H, W), _c(rng, C, H, W), _c(rng, T, C, H, W)
    mask = np.repeat((rng.random((T, H, 1)) < 0.4).astype(np.float64), W, axis=2)
    mask[3] = 0.0
    assert _rel(gpu.cart_K(x, b1, mask, centered), O.cart_K(x, b1, mask, centered)) < 2e-6
    assert _rel(gpu.cart_KH(z, b1, mask, centered), O.cart_KH(z, b1, mask, centered)) < 2e-6


def _problem(W, H, seed):
    rng = np.random.default_rng(seed)
    T, C = 3, 3
    mask = np.repeat((rng.random((T, H, 1)) < 0.5).astype(np.float64), W, axis=2)
    mask[:, 0] = 1.0
    b1, x0 = _c(rng, C, H, W), _c(rng, T, H, W)
    data = (_c(rng, T, C, H, W) * mask[:, None]).astype(np.complex64).astype(np.complex128)
    return data, b1, mask, x0


@pytest.mark.parametrize("W,H", SIZES)
@pytest.mark.parametrize("centered", [False, True])
def test_iterations_every_radix(gpu, W, H, centered):
    import torch
    print(f"[gpu iterations] W={W} H={H} centered={centered}", flush=True)
    data, b1, mask, x0 = _problem(W, H, W * 1000 + H)
    p = O.default_params("tv")
    p.update(maxIt=3, lambda_=2.0, centered=int(centered))
    ref = O.recon(p, data, b1, mask, x0, logs=True)
    got = gpu.recon_logs(p, data, b1, mask, x0)
    assert _rel(got["x"], ref["x"]) < 1e-5
    np.testing.assert_allclose(got["sigma"], ref["sigma"], rtol=1e-5)
    # the residual of the image that one iteration leaves, through the engine
    e = gpu.A.Engine(use_graphs=False)
    c64 = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.complex64)).to("cuda")
    rid = e.submit(gpu.A.Request(0, c64(data), c64(b1), mask=gpu._r(mask), x0=c64(x0), centered=centered,
                                 params={"maxIt": 1, "lambda": 2.0, "adaptLambda": 0}, debug=True))
    e.step()
    fid = e.gap_log(rid)[2][0]
    x = torch.empty(x0.shape, dtype=torch.complex64, device="cuda")
    assert e.poll(rid, x)
    u = x.cpu().numpy().astype(np.complex128)
    want = 2.0 / 2.0 * np.linalg.norm(O.cart_K(u, b1, mask, centered) - data)
    assert abs(fid - want) <= 1e-5 * want


# one request alone (narrow column tiles) and thirty of it (wide ones)
@pytest.mark.parametrize("W,H", [(70, 32), (64, 39), (48, 45), (72, 96), (50, 112)])
def test_results_do_not_depend_on_the_tiles(gpu, W, H):
    import torch
    print(f"[gpu tiles] W={W} H={H}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(H)
    T, C, n = 20, 2, 30
    r = lambda *s: torch.randn(*s, dtype=torch.complex64, device="cuda", generator=g)
    m = (torch.rand(T, H, 1, device="cuda", generator=g) < 0.5).float()
    m[:, 0] = 1.0
    m = m.expand(T, H, W).contiguous()
    d, b1, x0 = r(T, C, H, W) * m[:, None], r(C, H, W), r(T, H, W)

    def run(count):
        e = gpu.A.Engine(use_graphs=False)
        ids = [e.submit(gpu.A.Request(0, d, b1, mask=m, x0=x0,
                                      params={"maxIt": 12, "lambda": 2.0, "adaptLambda": 0}))
               for _ in range(count)]
        outs = [torch.empty_like(x0) for _ in ids]
        left = set(range(count))
        while left:
            e.step()
            left = {i for i in left if not e.poll(ids[i], outs[i])}
        return [o.cpu().numpy() for o in outs]

    alone = run(1)[0]
    assert np.isfinite(alone).all()
    for x in run(n):
        assert np.array_equal(x, alone)


# depths on two-stage, narrow and wide plans (two LDS tiles in the dual update)
@pytest.mark.parametrize("D,H,W,C", [(48, 5, 9, 2), (270, 3, 5, 2), (605, 2, 3, 3), (143, 4, 6, 1), (1024, 2, 2, 2)])
def test_volume_iterations(gpu, D, H, W, C):
    print(f"[gpu volume iterations] D={D} H={H} W={W} C={C}", flush=True)
    rng = np.random.default_rng(D)
    b1, x0 = _c(rng, C, D, H, W), _c(rng, D, H, W)
    mask = (rng.random((D, H, W)) < 0.5).astype(float)
    data = _c(rng, C, D, H, W) * mask[None]
    p = O.default_params("tgv2_3d")
    p.update(maxIt=3, lambda_=2.0, dx=1.0, dy=1.0, dz=2.0)
    ref = O.recon3(p, data, b1, mask, x0)
    rec = gpu.A.TGV2_3D(W, H, C, D, gpu.A.CartesianOperator3D(W, H, D, C, gpu._r(mask)), None)
    q = rec.GetParams()
    q.update(maxIt=3, adaptLambda=0, dx=1.0, dy=1.0, dz=2.0)
    q["lambda"] = 2.0
    rec.SetParams(q)
    x = gpu._t(x0)
    rec.IterativeReconstruction(gpu._t(data), x, gpu._t(b1))
    assert _rel(gpu._n(x), ref["x"]) < 1e-5
    np.testing.assert_allclose(rec.sigma_log(), ref["sigma"], rtol=1e-5)
