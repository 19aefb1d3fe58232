"""Several right-hand sides of plans that store FP64 values beside compressed
ones, in both directions, against the oracle on the stored factors; and
infinities and NaN in the vectors, for every kind of plan.

Tolerances: as for the plans without FP64 values, the bar of FP32-accumulated
products (2e-6); FP32 vectors add one rounding of the result."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from hlr_amd import _native as N
from hlr_amd.hmatrix import INVR_SPHERE, HMatrix, random_vector
from hlr_amd.plan import Plan
from tests.golden_data import load
from tests.helpers import dequantized_arena, rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ragged():
    return HMatrix(INVR_SPHERE.with_(n=2999))


@pytest.mark.parametrize("vec", ["f64", "f32"])
@pytest.mark.parametrize("prec", ["valr", "bfp", "afl"])
@pytest.mark.parametrize("op", [N.OP_NORMAL, N.OP_TRANSPOSED])
def test_fp64_beside_compressed(cuda, ragged, prec, op, vec):
    import torch
    hm = ragged
    p = Plan.from_hmatrix(hm, precision=prec, eps=1e-6, dense_prec="fp64")
    assert p.arena_elems(0) > 0 and sum(p.arena_elems(f) for f in range(1, N.NFMT)) > 0
    deq = dequantized_arena(p, hm)
    dt = torch.float64 if vec == "f64" else torch.float32
    tol = 2e-6 + (0 if vec == "f64" else 2.0 ** -23)
    for nrhs in (2, 13, 40, 64):
        print(f"[gpu] mrhs kinds {prec}+fp64 {vec} op={op} nrhs={nrhs}", flush=True)
        X = np.stack([random_vector(hm.n, 60 + j) for j in range(nrhs)]).astype(np.float32).astype(np.float64)
        Y0 = np.stack([random_vector(hm.n, 160 + j) for j in range(nrhs)]).astype(np.float32).astype(np.float64)
        Y = torch.as_tensor(Y0, dtype=dt, device=cuda)
        p.apply(0.75, op, torch.as_tensor(X, dtype=dt, device=cuda), Y)
        out = Y.double().cpu().numpy()
        for j in range(nrhs):
            yr = Y0[j].copy()
            oracle.mul_vec(hm.blocks, deq, 0.75, op, X[j], yr)
            assert rel(out[j], yr) <= tol, (nrhs, j)
    p.close()


@pytest.mark.parametrize("prec,dense", [("fp64", "auto"), ("fp32", "auto"), ("valr", "auto"), ("valr", "fp64"),
                                        ("bfp", "auto"), ("bfp", "fp64"), ("afl", "auto"), ("afl", "fp64")])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_values_that_are_not_finite(cuda, prec, dense, bad):
    """A column with such a value: the other columns keep their bits, and it is
    finite in the rows where the product of one right-hand side is.  The
    first, the last and the middle index: ends of panels, remainders."""
    import torch
    g = load("h_ragged")
    p = Plan(g["blocks"], g["arena"], g["nrows"], g["ncols"], precision=prec, eps=1e-6, dense_prec=dense)
    for op, x, y0 in ((N.OP_NORMAL, "x", "y0"), (N.OP_TRANSPOSED, "xt", "yt0")):
        n = len(g[x])
        for nrhs in (2, 5, 19, 37, 64):
            print(f"[gpu] mrhs nonfinite {prec} {dense} {bad} op={op} nrhs={nrhs}", flush=True)
            c = (np.arange(nrhs) % 7 - 3.0)[:, None]
            X = torch.as_tensor(c * g[x], device=cuda)
            Y0 = torch.as_tensor(np.repeat(g[y0][None].astype(np.float64), nrhs, 0), device=cuda)
            clean = Y0.clone()
            p.apply(g["alpha"], op, X, clean)
            for at, col in ((0, nrhs - 1), (n - 1, 0), (n // 2, nrhs // 2)):
                Xb = X.clone()
                Xb[col, at] = bad
                Y = Y0.clone()
                p.apply(g["alpha"], op, Xb, Y)
                one = Y0[col].clone()
                p.apply(g["alpha"], op, Xb[col], one)
                rest = [j for j in range(nrhs) if j != col]
                assert torch.equal(Y[rest], clean[rest]), (op, nrhs, at)
                assert torch.equal(torch.isfinite(Y[col]), torch.isfinite(one)), (op, nrhs, at)
                assert not bool(torch.isfinite(one).all())
    p.close()
