"""Several right-hand sides of plans whose workspace rows are FP32: the range
of the vectors is that of the product of one right-hand side.

The integer fixtures with factors and vectors scaled by powers of two: no
rounding anywhere, so the products are the scaled integer results bit for bit
where every FP32 sum stays in FP32's range, as it does here.  What leaves it
are the partial sums and t alone, when one factor is large and the other
small."""
from __future__ import annotations

import numpy as np
import pytest

from hlr_amd import _native as N
from hlr_amd.batch import Batch
from hlr_amd.plan import FORMAT_NAMES, Plan
from tests.golden_data import CASES, load

pytestmark = pytest.mark.gpu

FORMATS = [("valr", "fp8_e4m3"), ("bfp", "bfp8"), ("bfp", "bfp16"), ("bfp", "bfp25")]


def _scaled(g, ea, eb):
    """the fixture's arena with U scaled by 2^ea, V by 2^eb"""
    ar = np.array(g["arena"], dtype=np.float64)
    for blk in g["blocks"]:
        k = int(blk["rank"])
        if int(blk["kind"]) == N.BLOCK_DENSE:
            continue
        ar[int(blk["off_a"]):][:int(blk["nrows"]) * k] *= 2.0 ** ea
        ar[int(blk["off_b"]):][:int(blk["ncols"]) * k] *= 2.0 ** eb
    return ar


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("prec,force", FORMATS)
@pytest.mark.parametrize("ea,ex", [(-40, 90), (40, 90), (-55, -85), (55, -85)])
def test_unbalanced_factors(cuda, case, prec, force, ea, ex):
    """U 2^ea and V 2^-ea, vectors 2^ex: t lies beyond FP32's range"""
    import torch
    g = load(case)
    p = Plan(g["blocks"], _scaled(g, ea, -ea), g["nrows"], g["ncols"], precision=prec, eps=1e-6, force_format=force,
             dense_prec="fp32")
    for op, x, y0, y in ((N.OP_NORMAL, "x", "y0", "y"), (N.OP_TRANSPOSED, "xt", "yt0", "yt")):
        want = 2.0 ** ex * g[y].astype(np.float64)
        for nrhs in (1, 3, 20):
            print(f"[gpu] mrhs range {case} {force} 2^{ea} 2^{ex} op={op} nrhs={nrhs}", flush=True)
            X = torch.as_tensor(np.repeat(2.0 ** ex * g[x][None].astype(np.float64), nrhs, 0), device=cuda)
            Y = torch.as_tensor(np.repeat(2.0 ** ex * g[y0][None].astype(np.float64), nrhs, 0), device=cuda)
            if nrhs == 1:
                X, Y = X[0], Y[0]
            p.apply(g["alpha"], op, X, Y)
            assert np.array_equal(Y.cpu().numpy(), np.broadcast_to(want, Y.shape)), (op, nrhs)
    # the batched passes
    X = torch.as_tensor(np.repeat(2.0 ** ex * g["x"][None].astype(np.float64), 5, 0), device=cuda)
    Y = torch.as_tensor(np.repeat(2.0 ** ex * g["y0"][None].astype(np.float64), 5, 0), device=cuda)
    b = Batch([p], [5])
    b.apply([X], [Y], [g["alpha"]])
    b.check()
    assert np.array_equal(Y.cpu().numpy(), np.broadcast_to(2.0 ** ex * g["y"].astype(np.float64), Y.shape))
    b.close()
    p.close()


@pytest.mark.parametrize("force", ["bfp8", "bfp16", "bfp25"])
@pytest.mark.parametrize("op,ed,ex", [(N.OP_NORMAL, -60, 140), (N.OP_TRANSPOSED, 50, 90), (N.OP_TRANSPOSED, -60, -80)])
def test_dense_leaves_in_scaled_formats(cuda, force, op, ed, ex):
    """One dense leaf of integers times 2^ed, vectors 2^ex: x is scaled
    before it is rounded (forward), the partials of x are scaled after their
    sums (transposed)."""
    import torch
    rng = np.random.default_rng(3)
    m, n = 150, 90
    A = rng.integers(-9, 10, (m, n)).astype(np.float64)
    b = np.zeros(1, dtype=N.block_dtype())
    b["nrows"], b["ncols"], b["kind"], b["off_b"], b["off_s"] = m, n, N.BLOCK_DENSE, -1, -1
    # an odd value in every column that needs the format's width
    A[rng.integers(0, m, n), np.arange(n)] = {"bfp8": 9, "bfp16": 301, "bfp25": 40001}[force]
    p = Plan(b, (2.0 ** ed * A).T.reshape(-1), m, n, precision="bfp", eps=1e-6)
    assert [FORMAT_NAMES[f] for f in range(N.NFMT) if p.arena_elems(f)] == [force]
    trans = op == N.OP_TRANSPOSED
    nin, nout = (m, n) if trans else (n, m)
    x = rng.integers(-5, 6, nin).astype(np.float64)
    want = 2.0 ** (ed + ex) * ((A.T if trans else A) @ x)
    for nrhs in (1, 2, 7):
        print(f"[gpu] mrhs range dense {force} op={op} nrhs={nrhs}", flush=True)
        X = torch.as_tensor(np.repeat(2.0 ** ex * x[None], nrhs, 0), device=cuda)
        Y = torch.zeros(nrhs, nout, dtype=torch.float64, device=cuda)
        if nrhs == 1:
            X, Y = X[0], Y[0]
        p.apply(1.0, op, X, Y)
        assert np.array_equal(Y.cpu().numpy(), np.broadcast_to(want, Y.shape)), nrhs
    p.close()


def test_zero_columns_beside_tiny_ones(cuda):
    """A column that is zero in one row panel (scale 1) and near the smallest
    FP8 scales in the other: the quotient of the scales is finite."""
    import torch
    m, n, e = 128, 70, -130
    rng = np.random.default_rng(4)
    U, V = rng.integers(-4, 5, (m, 2)).astype(np.float64), rng.integers(-4, 5, (n, 2)).astype(np.float64)
    U[:64, 0] = 0
    U[64:, 1] = 0
    b = np.zeros(1, dtype=N.block_dtype())
    b["nrows"], b["ncols"], b["rank"], b["kind"] = m, n, 2, N.BLOCK_LOWRANK
    b["off_b"], b["off_s"] = 2 * m, -1
    arena = np.concatenate([2.0 ** e * U.T.reshape(-1), V.T.reshape(-1)])
    p = Plan(b, arena, m, n, precision="valr", eps=1e-6, force_format="fp8_e4m3")
    x = rng.integers(-5, 6, n).astype(np.float64)
    want = 2.0 ** (e + 60) * (U @ (V.T @ x))
    for nrhs in (1, 3, 17):
        print(f"[gpu] mrhs range zero columns nrhs={nrhs}", flush=True)
        X = torch.as_tensor(np.repeat(2.0 ** 60 * x[None], nrhs, 0), device=cuda)
        Y = torch.zeros(nrhs, m, dtype=torch.float64, device=cuda)
        if nrhs == 1:
            X, Y = X[0], Y[0]
        p.apply(1.0, N.OP_NORMAL, X, Y)
        assert np.array_equal(Y.cpu().numpy(), np.broadcast_to(want, Y.shape)), nrhs
    p.close()
