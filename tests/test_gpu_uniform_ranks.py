"""H^2 products with clusters of rank 0 (GPU) against the oracle: leaf and
inner clusters without a basis beside others that have one, in plans that hold
bases and transfers in both orientations (FP64) and in the others."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

import oracle
from hlr_amd import _native as N
from hlr_amd.hmatrix import HMatrix, INVR_SPHERE, random_vector
from hlr_amd.uniform import UPlan, build_uniform
from tests.helpers import rel

pytestmark = pytest.mark.gpu


def _drop(cb, rng, share):
    """cb with rank 0 at a share of its clusters, and where nothing is left
    that feeds a cluster"""
    cb = cb.copy()
    cb["rank"][rng.random(len(cb)) < share] = 0
    while True:
        fed = np.zeros(len(cb), bool)
        sons = (cb["rank"] > 0) & (cb["off_transfer"] >= 0)
        fed[cb["parent"][sons]] = True
        unfed = (cb["rank"] > 0) & (cb["off_basis"] < 0) & ~fed
        if not unfed.any():
            return cb
        cb["rank"][unfed] = 0


@pytest.mark.parametrize("share", [0.1, 0.6, 1.0])
@pytest.mark.parametrize("prec,bar", [("fp64", 1e-13), ("fp32", 2e-6)])
def test_rank_zero_clusters(cuda, share, prec, bar):
    import torch
    hm = HMatrix(INVR_SPHERE.with_(n=3000))
    um = build_uniform(hm, 1e-6, nested=True)
    hm.close()
    rng = np.random.default_rng(2)
    um = dataclasses.replace(um, rowcb=_drop(um.rowcb, rng, share), colcb=_drop(um.colcb, rng, share))
    zero = [int((cb["rank"] == 0).sum()) for cb in (um.rowcb, um.colcb)]
    assert min(zero) > 0
    plan = UPlan(um, precision=prec)
    x, y0 = random_vector(um.ncols, 3), random_vector(um.nrows, 4)
    for op in (N.OP_NORMAL, N.OP_TRANSPOSED):
        print(f"[gpu] uplan ranks {prec} share={share} zero={zero} of {len(um.rowcb)} op={op}", flush=True)
        yt = torch.as_tensor(y0, device=cuda).clone()
        plan.apply(1.5, op, torch.as_tensor(x, device=cuda), yt)
        yr = y0.copy()
        oracle.uniform_mul_vec(um.rowcb, um.colcb, um.blocks, um.arena, 1.5, op, x, yr)
        assert rel(yt.cpu().numpy(), yr) <= bar
    plan.close()
