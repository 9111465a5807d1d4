"""fdfd_solve_static (the solve without a workspace argument) through the C
ABI: the same fields, bit for bit, as fdfd_solve with a caller workspace, on
two calls in a row, the second on a smaller grid; oversized solves are
refused with FDFD_ERR_ARG."""

import ctypes

import numpy as np
import pytest
import torch

from fdfdpy_amd import _lib as L
from fdfdpy_amd import configs as C
from fdfdpy_amd.device import DeviceOperator, _stream, _vp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _solve_both(n, precision, nrhs, blocks, transpose=0):
    p = C.c3_request(300 + n, n=n)
    op = DeviceOperator(p.shape, p.omega, p.dl, p.npml, p.pol, p.L0, DEV)
    op.set_eps(p.eps)
    fac = op.factor(precision, stepwise=blocks)
    assert (fac.numel() != op.nd_bytes[precision]) == blocks
    lib = L.lib()
    g = ctypes.byref(op.grid)
    pr = L.PREC[precision]
    rng = np.random.default_rng(n)
    b = torch.tensor(rng.standard_normal((nrhs,) + p.shape) + 1j * rng.standard_normal((nrhs,) + p.shape),
                     device=DEV)
    bs = op.to_solver(b)
    x_ref = torch.empty_like(bs)
    x_st = torch.full_like(bs, float("nan"))
    work = torch.empty(lib.fdfd_solve_workspace_bytes(g, pr, nrhs), dtype=torch.uint8, device=DEV)
    st_ref, st_st = L.FdfdSolveStats(), L.FdfdSolveStats()
    rel_ref, rel_st = (ctypes.c_double * nrhs)(), (ctypes.c_double * nrhs)()
    L.check(lib.fdfd_solve(g, _vp(op.op), _vp(fac), pr, _vp(bs), _vp(x_ref), nrhs, transpose, 1e-10, 60,
                           _vp(work), ctypes.byref(st_ref), rel_ref, _stream(DEV)))
    L.check(lib.fdfd_solve_static(g, _vp(op.op), _vp(fac), pr, _vp(bs), _vp(x_st), nrhs, transpose, 1e-10, 60,
                                  ctypes.byref(st_st), rel_st, _stream(DEV)))
    torch.cuda.synchronize()
    assert st_st.converged and st_st.iterations == st_ref.iterations
    assert list(rel_st) == list(rel_ref)
    return x_ref.cpu().numpy(), x_st.cpu().numpy()


@pytest.mark.parametrize("precision", ["c64", "fp64"])
@pytest.mark.parametrize("blocks", [False, True])
def test_static_solve_equals_workspace_solve(precision, blocks):
    # two calls in a row on the shared static workspace, the second smaller
    for n, nrhs in ((256, 3), (128, 1)):
        a, b = _solve_both(n, precision, nrhs, blocks)
        assert np.array_equal(a, b), f"{precision} n={n}: max difference {np.abs(a - b).max()}"
    a, b = _solve_both(192, precision, 2, blocks, transpose=1)
    assert np.array_equal(a, b)


def test_static_solve_refuses_oversized_work():
    lib = L.lib()
    p = C.c3_request(3, n=768)
    g = L.FdfdGrid(768, 768, 25, 25, 0, 0, p.omega, p.dl, p.L0)
    assert lib.fdfd_solve_workspace_bytes(ctypes.byref(g), 0, 4) > 64 << 20
    dummy = torch.zeros(16, dtype=torch.float64, device=DEV)
    st = L.FdfdSolveStats()
    rc = lib.fdfd_solve_static(ctypes.byref(g), _vp(dummy), _vp(dummy), 0, _vp(dummy), _vp(dummy), 4, 0,
                               1e-10, 10, ctypes.byref(st), None, _stream(DEV))
    assert rc == L.FDFD_ERR_ARG
    assert b"64" in lib.fdfd_last_error() or b"static" in lib.fdfd_last_error()
    rc = lib.fdfd_solve_static(ctypes.byref(g), _vp(dummy), _vp(dummy), 0, _vp(dummy), _vp(dummy), 17, 0,
                               1e-10, 10, ctypes.byref(st), None, _stream(DEV))
    assert rc == L.FDFD_ERR_ARG
