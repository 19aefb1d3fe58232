"""Batches whose members are stored in different kinds of formats (GPU): every
member gets bit for bit the product that its plan computes alone, eagerly and
from a captured graph, whatever the other members are."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from hlr_amd import _native as N
from hlr_amd.batch import Batch
from hlr_amd.hmatrix import INVR_SPHERE, HMatrix, random_vector
from hlr_amd.plan import Plan
from tests.helpers import rel

pytestmark = pytest.mark.gpu

#: n, precision, dense_prec, nrhs: one and several kinds of arithmetic and
#: tile counts, plans with few and with many row panels
MEMBERS = [(1500, "fp64", "auto", 20), (1500, "valr", "auto", 20), (9000, "fp64", "auto", 5), (2999, "valr", "fp64", 40),
           (9000, "bfp", "auto", 17), (1500, "bfp", "fp64", 3), (2999, "afl", "auto", 64), (2999, "valr", "auto", 1),
           (1500, "fp64", "auto", 1), (2999, "fp32", "auto", 2), (2999, "valr", "auto", 49)]


@pytest.fixture(scope="module")
def matrices():
    return {n: HMatrix(INVR_SPHERE.with_(n=n)) for n in {m[0] for m in MEMBERS}}


@pytest.mark.parametrize("vec", ["f64", "f32"])
@pytest.mark.parametrize("pick", [list(range(len(MEMBERS))), [0, 1], [4, 2], [6, 3], [1, 5, 7]])
def test_members_keep_their_bits(cuda, matrices, pick, vec):
    import torch
    members = [MEMBERS[i] for i in pick]
    dt = torch.float64 if vec == "f64" else torch.float32
    plans = [Plan.from_hmatrix(matrices[n], precision=p, eps=1e-6, dense_prec=d) for n, p, d, _ in members]
    alphas = [0.5 + 0.25 * i for i in range(len(members))]
    xs, refs = [], []
    for i, ((n, _, _, r), p, a) in enumerate(zip(members, plans, alphas)):
        X = np.stack([random_vector(n, 70 + 100 * i + j) for j in range(r)])
        xs.append(torch.as_tensor(X if r > 1 else X[0], dtype=dt, device=cuda))
        y = torch.zeros_like(xs[-1])
        p.apply(a, N.OP_NORMAL, xs[-1], y)
        refs.append(y)
    ys = [torch.zeros_like(x) for x in xs]
    b = Batch(plans, [m[3] for m in members], N.F64 if vec == "f64" else N.F32)
    print(f"[gpu] mixed batch {members} {vec}", flush=True)
    b.apply(xs, ys, alphas)
    b.check()
    for m, y, ref in zip(members, ys, refs):
        assert torch.equal(y, ref), m
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        b.capture(xs, ys, alphas, stream=stream)
    stream.synchronize()
    for rep in range(3):
        for y in ys:
            y.zero_()
        torch.cuda.synchronize()
        _ = torch.ones(1024, device=cuda).sum().item()       # eager work between replays
        b.replay(stream=stream)
        b.check(stream=stream)
        for m, y, ref in zip(members, ys, refs):
            assert torch.equal(y, ref), (rep, m)
    b.close()
    if vec == "f64":
        for (n, prec, _, r), x, y, a, p in zip(members, xs, ys, alphas, plans):
            hm, X = matrices[n], x.cpu().numpy()
            ref = np.zeros_like(X)
            oracle.mul_vec(hm.blocks, hm.arena, a, N.OP_NORMAL, X, ref)
            assert rel(y.cpu().numpy(), ref) <= (1e-13 if prec == "fp64" else 2e-6), (n, prec, r)
    for p in plans:
        p.close()
