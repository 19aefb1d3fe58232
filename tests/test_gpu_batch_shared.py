"""Batch members that act on the same y (GPU): members of different counts of
right-hand-side tiles act in the order of these counts, as products one after
the other do, eagerly and from a captured graph."""
from __future__ import annotations

import numpy as np
import pytest

from hlr_amd import _native as N
from hlr_amd.batch import Batch
from hlr_amd.hmatrix import INVR_SPHERE, HMatrix, random_vector
from hlr_amd.plan import Plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precs", [("fp64",) * 4, ("valr", "fp64", "bfp", "valr")])
def test_members_on_one_y(cuda, precs):
    import torch
    hm = HMatrix(INVR_SPHERE.with_(n=1500))
    plans = [Plan.from_hmatrix(hm, precision=p, eps=1e-6) for p in precs]
    nrhs = [33, 1, 5, 17]                       # in the batch's order; they act as 1, 5, 17, 33
    big = torch.as_tensor(np.stack([random_vector(hm.n, 9 + j) for j in range(40)]), device=cuda)
    xs = [torch.as_tensor(np.stack([random_vector(hm.n, 50 * (i + 2) + j) for j in range(r)]), device=cuda)
          for i, r in enumerate(nrhs)]
    xs[1] = xs[1][0]
    # rows of one block; the single member's x is a column that others write
    def ys(Y):
        return [Y[:33], Y[3], Y[2:7], Y[1:18]]
    ref = big.clone()
    xs[1] = ref[5].clone()
    yr = ys(ref)
    for i in np.argsort(nrhs):
        plans[i].apply(0.5 + i, N.OP_NORMAL, xs[i], yr[i])
    alphas = [0.5 + i for i in range(4)]
    b = Batch(plans, nrhs)
    Y = big.clone()
    args = [xs[0], Y[5], xs[2], xs[3]]
    print(f"[gpu] batch on one y {precs}", flush=True)
    b.apply(args, ys(Y), alphas)
    b.check()
    assert torch.equal(Y, ref)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        b.capture(args, ys(Y), alphas, stream=stream)
    stream.synchronize()
    for rep in range(3):
        Y.copy_(big)
        torch.cuda.synchronize()
        b.replay(stream=stream)
        b.check(stream=stream)
        assert torch.equal(Y, ref), rep
        _ = torch.ones(1024, device=cuda).sum().item()       # eager work between replays
    b.close()
    for p in plans:
        p.close()
    hm.close()
