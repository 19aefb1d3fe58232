"""Several right-hand sides of a matrix whose workspace rows pass the kernels'
32-bit byte offsets (GPU): 8.5 M low-rank columns, 64 right-hand sides of FP64.
The call takes fewer per pass and the batch cuts the member into parts; both
are held to the dense product and to each other bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from hlr_amd import _native as N
from hlr_amd.batch import Batch
from hlr_amd.plan import Plan

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(300)]

B, NT = 4, 1456                    # tiles of 4 x 4 and rank 4


@pytest.fixture(scope="module")
def tiles():
    rng = np.random.default_rng(11)
    arena = rng.uniform(-1, 1, 1 << 16)
    i, j = (a.reshape(-1) for a in np.meshgrid(np.arange(NT), np.arange(NT), indexing="ij"))
    b = np.zeros(NT * NT, dtype=N.block_dtype())
    b["row_ofs"], b["col_ofs"], b["nrows"], b["ncols"], b["rank"] = i * B, j * B, B, B, B
    b["kind"] = N.BLOCK_LOWRANK
    b["off_a"], b["off_b"] = rng.integers(0, arena.size - B * B, b.size), rng.integers(0, arena.size - B * B, b.size)
    b["off_s"] = -1
    # (tile, column l, row): the tile is U V^T
    at = np.arange(B * B)
    U = arena[b["off_a"][:, None] + at].reshape(-1, B, B)
    V = arena[b["off_b"][:, None] + at].reshape(-1, B, B)
    T = np.einsum("tli,tlj->tij", U, V).reshape(NT, NT, B, B)
    return b, arena, T.transpose(0, 2, 1, 3).reshape(NT * B, NT * B)


def test_beyond_32_bit_offsets(cuda, tiles):
    import torch
    blocks, arena, A = tiles
    n, nrhs = NT * B, 64
    assert (B * NT * NT + n + 1) * nrhs * 8 > 1 << 32
    p = Plan(blocks, arena, n, n, precision="fp64")
    gen = torch.Generator(device="cuda").manual_seed(5)
    X = torch.rand((nrhs, n), generator=gen, dtype=torch.float64, device=cuda) * 2 - 1
    At = torch.as_tensor(A, device=cuda)
    for op in (N.OP_NORMAL, N.OP_TRANSPOSED):
        print(f"[gpu] mrhs offsets op={op} workspace {p.workspace_bytes(op, nrhs)}", flush=True)
        Y = torch.zeros_like(X)
        p.apply(2.0, op, X, Y)
        ref = 2.0 * (X @ (At.T.contiguous() if op == N.OP_NORMAL else At))
        assert float((Y - ref).norm() / ref.norm()) <= 1e-13
        if op == N.OP_NORMAL:
            print("[gpu] mrhs offsets batch", flush=True)
            Z = torch.zeros_like(X)
            b = Batch([p], [nrhs])
            b.apply([X], [Z], [2.0])
            b.check()
            assert torch.equal(Z, Y)
            b.close()
    p.close()
