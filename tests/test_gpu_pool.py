"""Reconstructions whose state lands in memory that an earlier one used: the
results stay bit for bit those of the first run, through the solver classes
(other sizes and methods in between, the solver destroyed and made again, two
host threads with streams of their own) and through the engine (after a cancel
of a running request); sampling masks whose rows are read on the GPU against
the oracle's K."""
import threading

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _data(torch, W, H, T, C, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = lambda *s: torch.randn(*s, dtype=torch.complex64, device="cuda", generator=g)
    mask = (torch.rand(T, H, 1, device="cuda", generator=g) < 0.5).float().expand(T, H, W).contiguous()
    return r(T, C, H, W) * mask[:, None], r(C, H, W), mask, r(T, H, W)


def _run(A, torch, cls, W, H, T, C, seed, its=12):
    d, b1, mask, x0 = _data(torch, W, H, T, C, seed)
    op = A.CartesianOperator(W, H, C, T, mask=mask, centered=False)
    rec = cls(W, H, C, T, op)
    rec.SetParams({"maxIt": its, "lambda": 2.0, "adaptLambda": 0})
    return rec.IterativeReconstruction(d, x0.clone(), b1).cpu().numpy()


def test_solver_state_in_reused_memory(gpu):
    import torch
    A = gpu.A
    print("[gpu pool] solvers", flush=True)
    first = _run(A, torch, A.TGV2, 48, 40, 5, 3, 1)
    keep = A.TV(8, 8, 1, 1, A.CartesianOperator(8, 8, 1, 1))  # a solver alive: blocks are kept
    for k in range(3):
        _run(A, torch, A.ICTGV2, 40, 36, 4, 2, 10 + k)
        _run(A, torch, A.TV, 64, 50, 6, 2, 20 + k)
        assert np.array_equal(_run(A, torch, A.TGV2, 48, 40, 5, 3, 1), first)
    del keep
    assert np.array_equal(_run(A, torch, A.TGV2, 48, 40, 5, 3, 1), first)


def test_solver_threads(gpu):
    import torch
    A = gpu.A
    print("[gpu pool] threads", flush=True)
    ref = {s: _run(A, torch, A.TGV2, 40, 40, 4, 2, s) for s in (1, 2)}
    bad = []

    def work(seed):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(6):
                if not np.array_equal(_run(A, torch, A.TGV2, 40, 40, 4, 2, seed), ref[seed]):
                    bad.append(seed)
    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_engine_state_in_reused_memory(gpu):
    import torch
    A = gpu.A
    print("[gpu pool] engine", flush=True)
    d, b1, mask, x0 = _data(torch, 48, 40, 5, 3, 7)
    other = _data(torch, 48, 40, 5, 3, 8)
    req = lambda v, its: A.Request(1, v[0], v[1], mask=v[2], x0=v[3],
                                   params={"maxIt": its, "lambda": 2.0, "adaptLambda": 0})
    e = A.Engine()

    def one():
        rid, out = e.submit(req((d, b1, mask, x0), 12)), torch.empty_like(x0)
        while not e.poll(rid, out):
            e.step()
        return out.cpu().numpy()
    first = one()
    for _ in range(3):
        rid = e.submit(req(other, 50))
        e.step()
        e.cancel(rid)
        assert np.array_equal(one(), first)


@pytest.mark.parametrize("kind", ["none", "one", "negative", "partial"])
def test_mask_rows(gpu, kind):
    print(f"[gpu pool] mask {kind}", flush=True)
    rng = np.random.default_rng(3)
    T, C, H, W = 3, 2, 20, 300
    m = np.zeros((T, H, W), np.float32)
    if kind == "one":
        m[1, 7, 299] = 1.0  # one value of one row
    elif kind == "negative":
        m[:, ::3] = -0.5
    elif kind == "partial":
        m[rng.random((T, H, W)) < 0.02] = 1.0
    c = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64).astype(np.complex128)
    x, b1 = c(T, H, W), c(C, H, W)
    got, ref = gpu.cart_K(x, b1, m, False), O.cart_K(x, b1, m.astype(np.float64), False)
    assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(ref)
