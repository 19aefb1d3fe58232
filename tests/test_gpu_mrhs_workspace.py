"""Several right-hand sides with less workspace than a whole pass takes: the
factors are read more often, every column keeps its bits.

hmvm_apply_noalloc is held to hmvm_apply bit for bit at sizes where its fixed
array holds only a part of the columns; hmvm_apply_ws to the same with every
workspace that holds one column on the matrix cores."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from hlr_amd import _native as N
from hlr_amd.hmatrix import HMatrix, INVR_SPHERE, random_vector
from hlr_amd.plan import Plan, _stream_handle

pytestmark = pytest.mark.gpu


def _vectors(n, nrhs, cuda, dtype):
    import torch
    X = torch.as_tensor(np.stack([random_vector(n, 60 + j) for j in range(nrhs)]), dtype=dtype, device=cuda)
    Y = torch.as_tensor(np.stack([random_vector(n, 460 + j) for j in range(nrhs)]), dtype=dtype, device=cuda)
    return X, Y


@pytest.fixture(scope="module")
def sphere16k():
    return HMatrix(INVR_SPHERE.with_(n=16384))


@pytest.mark.parametrize("prec,op,nrhs", [("fp64", N.OP_NORMAL, 39), ("fp64", N.OP_TRANSPOSED, 39),
                                          ("fp64", N.OP_TRANSPOSED, 65), ("valr", N.OP_TRANSPOSED, 64),
                                          ("valr", N.OP_TRANSPOSED, 130)])
def test_noalloc_in_parts(cuda, sphere16k, prec, op, nrhs):
    import torch
    hm = sphere16k
    p = Plan.from_hmatrix(hm, precision=prec, eps=1e-6)
    print(f"[gpu] noalloc parts {prec} op={op} nrhs={nrhs} full {p.workspace_bytes(op, nrhs)}", flush=True)
    assert p.workspace_bytes(op, nrhs) > N.NOALLOC_MAX_BYTES
    X, Y = _vectors(hm.n, nrhs, cuda, torch.float64)
    ref = Y.clone()
    p.apply(1.5, op, X, ref)
    rc = N.hmvm().hmvm_apply_noalloc(p.handle, 1.5, op, C.c_void_p(X.data_ptr()), hm.n, C.c_void_p(Y.data_ptr()), hm.n,
                                     nrhs, N.F64, _stream_handle(None))
    torch.cuda.synchronize()
    assert rc == 0
    assert torch.equal(Y, ref)
    p.close()


@pytest.mark.parametrize("vec", ["f64", "f32"])
@pytest.mark.parametrize("prec", ["fp64", "valr", "afl"])
@pytest.mark.parametrize("op", [N.OP_NORMAL, N.OP_TRANSPOSED])
def test_workspaces_between_smallest_and_full(cuda, prec, op, vec):
    import torch
    hm = HMatrix(INVR_SPHERE.with_(n=2999))
    p = Plan.from_hmatrix(hm, precision=prec, eps=1e-6)
    dt, code = (torch.float64, N.F64) if vec == "f64" else (torch.float32, N.F32)
    for nrhs in (3, 19, 65):
        X, Y0 = _vectors(hm.n, nrhs, cuda, dt)
        ref = Y0.clone()
        p.apply(0.5, op, X, ref)
        full, one = p.workspace_bytes(op, nrhs), p.workspace_bytes(op, 1)
        ws = torch.empty(full // 8 + 1, dtype=torch.float64, device=cuda)
        taken = 0
        for nb in sorted({full, full - 16, full * 99 // 100 // 8 * 8, full * 9 // 10 // 8 * 8, full // 2 // 8 * 8,
                          full // 3 // 8 * 8, full // 7 // 8 * 8, one}, reverse=True):
            if nb < one:
                continue
            Y = Y0.clone()
            rc = N.hmvm().hmvm_apply_ws(p.handle, 0.5, op, C.c_void_p(X.data_ptr()), hm.n, C.c_void_p(Y.data_ptr()),
                                        hm.n, nrhs, code, C.c_void_p(ws.data_ptr()), nb, _stream_handle(None))
            torch.cuda.synchronize()
            print(f"[gpu] mrhs workspace {prec} {vec} op={op} nrhs={nrhs} {nb} of {full}: {rc}", flush=True)
            # forward calls need the columns of a pass in rows without padding
            assert rc == 0 or (op == N.OP_NORMAL and nb < full and N.ERRORS[rc] == "HMVM_ERR_INVALID_ARG")
            if rc == 0:
                taken += 1
                assert torch.equal(Y, ref), (nrhs, nb)
            else:
                assert torch.equal(Y, Y0)
        assert taken >= (2 if op == N.OP_TRANSPOSED else 1)
    p.close()
    hm.close()
