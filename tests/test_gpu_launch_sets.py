"""Requests whose launch set decides which kernels and tiles run them: every
result is bit for bit that of the same request alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _data(torch, W, H, T, C, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = lambda *s: torch.randn(*s, dtype=torch.complex64, device="cuda", generator=g)
    m = (torch.rand(T, H, 1, device="cuda", generator=g) < 0.4).float()
    m[:, 0] = 1.0
    m = m.expand(T, H, W).contiguous()
    return r(T, C, H, W) * m[:, None], r(C, H, W), m, r(T, H, W)


def _run(A, torch, sizes, centered, its=13):
    e = A.Engine(use_graphs=False)
    ids, outs = [], []
    for s in sizes:
        d, b1, m, x0 = _data(torch, *s, seed=sum(s))
        ids.append(e.submit(A.Request(1, d, b1, mask=m, x0=x0, centered=centered,
                                      params={"maxIt": its, "lambda": 2.0, "adaptLambda": 0})))
        outs.append(torch.empty_like(x0))
    left = set(range(len(ids)))
    while left:
        e.step()
        left = {i for i in left if not e.poll(ids[i], outs[i])}
    return [o.cpu().numpy() for o in outs]


# (W, H, frames, coils): rows of 256 beside other two-stage rows, either the larger part
@pytest.mark.parametrize("sizes", [
    [(256, 40, 4, 3), (128, 36, 3, 2), (70, 63, 2, 2)],
    [(256, 30, 2, 2), (192, 96, 5, 4), (240, 48, 3, 2), (200, 33, 2, 2)]])
@pytest.mark.parametrize("centered", [False, True])
def test_row_kernels(gpu, sizes, centered):
    import torch
    print(f"[gpu launch sets] rows {sizes} centered={centered}", flush=True)
    for s, x in zip(sizes, _run(gpu.A, torch, sizes, centered)):
        assert np.isfinite(x).all()
        assert np.array_equal(x, _run(gpu.A, torch, [s], centered)[0]), s


# columns of 256 beside other two-stage columns: few, in the kernel of those; and
# 1600 blocks of them, in their own
@pytest.mark.parametrize("sizes", [
    [(39, 256, 3, 3), (96, 192, 3, 2), (33, 225, 2, 2)],
    [(256, 256, 100, 1), (64, 256, 4, 3), (80, 128, 3, 2)]])
@pytest.mark.parametrize("centered", [False, True])
def test_column_kernels(gpu, sizes, centered):
    import torch
    print(f"[gpu launch sets] columns {sizes} centered={centered}", flush=True)
    for s, x in zip(sizes, _run(gpu.A, torch, sizes, centered)):
        assert np.isfinite(x).all()
        assert np.array_equal(x, _run(gpu.A, torch, [s], centered)[0]), s
