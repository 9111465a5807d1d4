"""The nested-dissection factor: its tree and index maps on the CPU, the factor
and solve on the GPU against the oracle.

The CPU half eliminates the oracle's operator front by front with numpy, in
the library's own tree and maps (fdfd_nd_front), and compares the solution
with SuperLU: every cell is eliminated once, every index lies inside its
array, and the fronts add up to the whole periodic operator.
"""

import ctypes

import numpy as np
import pytest
import torch

from fdfdpy_amd import _lib as L
from fdfdpy_amd import configs as C
from oracle import construct_A, solver_direct

OMEGA = C.omega_of(1.55e-6)
DEV = "cuda:0"


def relerr(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


def _eps(rng, N):
    return 1 + 11.25 * (rng.random(N) < 0.5)


def _front(g, level, box):
    lib = L.lib()
    info = (ctypes.c_int32 * 8)()
    L.check(lib.fdfd_nd_front(ctypes.byref(g), level, box, info, None, None))
    n = info[3] + info[4]
    cells, maps = np.zeros(n, np.int64), np.zeros((n, 2), np.int32)
    L.check(lib.fdfd_nd_front(ctypes.byref(g), level, box, info, cells.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)),
                              maps.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))))
    return list(info), cells, maps


def _multifrontal(nx, ny, A, b):
    g = L.FdfdGrid(nx, ny, 10, 10, 0, 0, OMEGA, 0.02, 1e-6)
    levels = _front(g, -1, 0)[0][0]
    A = A.tocsr()
    updates, done = [], []
    eliminated = np.zeros(nx * ny, int)
    for level in range(-1, levels + 1):
        new, fronts = [], []
        for k in range(_front(g, level, 0)[0][1]):
            info, cells, maps = _front(g, level, k)
            s, n = info[3], len(cells)
            assert cells.min() >= 0 and cells.max() < nx * ny
            eliminated[cells[:s]] += 1
            # the front's own entries: rows and columns of its separator
            F = np.zeros((n, n), complex)
            F[:s, :] = A[cells[:s]][:, cells].toarray()
            F[s:, :s] = A[cells[s:]][:, cells[:s]].toarray()
            if len(set(cells)) != n:          # no cell twice in a front
                raise AssertionError(f"level {level} box {k}: a cell appears twice")
            f = np.concatenate([b[cells[:s]], np.zeros(n - s)]).astype(complex)
            if level >= 0:
                for t in range(2):
                    v = np.nonzero(maps[:, t] >= 0)[0]
                    if len(v):
                        Cc, uc, border = updates[info[5 + t]]
                        at = maps[v, t]
                        assert np.array_equal(border[at], cells[v])   # the same cells on both sides
                        F[np.ix_(v, v)] += Cc[np.ix_(at, at)]
                        f[v] += uc[at]
            X = np.linalg.inv(F[:s, :s])
            W = X @ F[:s, s:]
            z = X @ f[:s]
            new.append((F[s:, s:] - F[s:, :s] @ W, f[s:] - F[s:, :s] @ z, cells[s:]))
            fronts.append((cells, s, z, W))
        updates = new
        done.append(fronts)
    assert (eliminated == 1).all()
    x = np.zeros(nx * ny, complex)
    for fronts in reversed(done):
        for cells, s, z, W in fronts:
            x[cells[:s]] = z - W @ x[cells[s:]]
    return x


@pytest.mark.parametrize("N,npml,pol", [((64, 64), [8, 8], "Ez"), ((65, 97), [9, 0], "Hz"), ((200, 64), [10, 10], "Ez"),
                                        ((71, 130), [0, 0], "Ez"), ((64, 230), [8, 12], "Hz"), ((16, 16), [4, 4], "Ez"),
                                        ((17, 90), [0, 9], "Hz"), ((31, 23), [5, 5], "Ez")])
def test_tree_and_maps_solve_the_periodic_operator(N, npml, pol):
    rng = np.random.default_rng(N[0] + N[1])
    A, _ = construct_A(OMEGA, [0, N[0] * 0.02], [0, N[1] * 0.02], _eps(rng, N), npml, pol, 1e-6)
    b = rng.standard_normal(N[0] * N[1]) + 1j * rng.standard_normal(N[0] * N[1])
    assert relerr(_multifrontal(N[0], N[1], A, b), solver_direct(A, b)) < 1e-9


def test_range_and_sizes():
    """Every grid whose shorter side has 16 cells or more (64 in complex64) is
    in the range, smaller ones are not; flags that exclude each other are
    refused; the two kinds of factor never have one size."""
    lib = L.lib()

    def grid(nx, ny):
        return ctypes.byref(L.FdfdGrid(nx, ny, 10, 10, 0, 0, OMEGA, 0.02, 1e-6))
    for n in list(range(16, 460)) + [511, 512, 513, 768, 1023, 1500, 2047, 2048]:
        for m in (16, 64, n, n + 1, 2 * n + 1):
            ny, nx = min(n, m), max(n, m)
            for prec in (0, 1):
                assert lib.fdfd_nd_supported(grid(nx, ny), prec) == (prec == 0 or ny >= 64), (nx, ny)
                if prec == 1 and ny < 64:
                    continue
                nd = lib.fdfd_factor_bytes(grid(nx, ny), prec | L.FACTOR_ND)
                assert nd > 0 and nd != lib.fdfd_factor_bytes(grid(nx, ny), prec)
    for shape, prec in (((63, 64), 1), ((64, 63), 1), ((500, 15), 0), ((15, 16), 0), ((2, 2), 0)):
        assert lib.fdfd_nd_supported(grid(*shape), prec) == 0
        assert lib.fdfd_factor_bytes(grid(*shape), prec | L.FACTOR_ND) == 0
    for bad in (L.FACTOR_ND | L.FACTOR_PIVOT, L.FACTOR_ND | L.FACTOR_STEPWISE):
        assert lib.fdfd_factor_bytes(grid(128, 128), bad) == 0
    prev = lib.fdfd_set_twist(0)
    try:   # the one-chain order is a block factorization
        assert lib.fdfd_nd_supported(grid(128, 128), 0) == 0
    finally:
        lib.fdfd_set_twist(prev)


@pytest.mark.parametrize("longest,short", [(8192, 16), (8192, 32), (11585, 33), (11585, 64), (16384, 128), (32768, 512)])
def test_long_grids_are_block_factors(longest, short):
    """The root front grows with the square of the long side, a block factor
    with the side: beyond the line the block factor is the one of choice, and
    the tree stays there for who asks for it."""
    lib = L.lib()
    for nx, want in ((longest, 1), (longest + 1, 0), (10 * longest, 0)):
        g = ctypes.byref(L.FdfdGrid(nx, short, 8, 8, 0, 0, OMEGA, 0.02, 1e-6))
        assert lib.fdfd_nd_supported(g, 0) == want
        assert lib.fdfd_nd_supported(g, 1) == (want if short >= 64 else 0)
    g = ctypes.byref(L.FdfdGrid(longest + 1, short, 8, 8, 0, 0, OMEGA, 0.02, 1e-6))
    assert lib.fdfd_factor_bytes(g, L.FACTOR_ND) > 0


@pytest.mark.parametrize("nx,ny", [(16, 16), (64, 64), (200, 96), (512, 512), (1000, 64)])
@pytest.mark.parametrize("es", [8, 4])
def test_workspace_holds_what_the_launches_use(nx, ny, es):
    """The bands and the updates of two levels; pivot inverses, fronts and
    panels only of the levels that are eliminated step by step (a separator
    over one tile, or a border over 2 tiles, 3 in complex64, and the root)."""
    if es == 4 and ny < 64:
        pytest.skip("complex64 factors of grids below 64 cells are block factors")
    lib, pad = L.lib(), lambda n: -(-n // 32) * 32
    g = L.FdfdGrid(nx, ny, 8, 8, 0, 0, OMEGA, 0.02, 1e-6)
    levels = _front(g, -1, 0)[0][0]
    info = (ctypes.c_int32 * 8)()
    boxes = ss = sb = panels = updates = 0
    for level in range(-1, levels + 1):
        s = b = k = 0
        while k == 0 or k < info[1]:
            L.check(lib.fdfd_nd_front(ctypes.byref(g), level, k, info, None, None))
            s, b, k = max(s, info[3]), max(b, info[4]), k + 1
        sp, bp = (32, 32) if level == -1 else (pad(s), pad(b))
        updates = max(updates, k * bp * bp)
        if level == -1 or (level < levels and sp == 32 and bp <= (64 if es == 8 else 96)):
            continue
        boxes, panels = max(boxes, k), max(panels, k * sp * bp)
        if sp > 32:
            ss, sb = max(ss, k * sp * sp), max(sb, k * sp * bp)
    need = 2 * es * (3 * nx * ny + 2 * boxes * 32 * 32 + 2 * ss + 2 * sb + panels + sb + 2 * updates)
    got = lib.fdfd_factor_workspace_bytes(ctypes.byref(g), (0 if es == 8 else 1) | L.FACTOR_ND)
    assert 0 <= got - need <= 1024 + 11 * 256      # the status header, and the parts' alignment


def _device(N, npml, pol, eps, precision):
    from fdfdpy_amd.device import DeviceOperator
    op = DeviceOperator(N, OMEGA, 0.02, npml, pol, 1e-6, DEV)
    op.set_eps(eps)
    assert op.nested(precision)
    return op


@pytest.mark.gpu
@pytest.mark.parametrize("N,npml,pol,nrhs", [
    ((64, 64), [8, 8], "Ez", 1), ((65, 97), [9, 12], "Hz", 2), ((128, 66), [10, 0], "Ez", 3),
    ((129, 70), [0, 0], "Hz", 5), ((64, 300), [8, 15], "Ez", 8), ((257, 96), [20, 10], "Hz", 9),
    ((16, 16), [4, 4], "Ez", 1), ((17, 120), [0, 10], "Hz", 4), ((33, 32), [6, 6], "Ez", 5), ((47, 63), [9, 9], "Hz", 2),
    ((301, 290), [12, 12], "Ez", 4)])
@pytest.mark.parametrize("precision", ["fp64", "c64"])
def test_solves_match_the_oracle(N, npml, pol, nrhs, precision):
    """Edges of the tree (power-of-two sides and their neighbours, long
    grids), both polarizations, periodic axes, a lossy cell, every count of
    right-hand sides per pass, separators and borders over 512 cells (more than
    one batch of a sweep's rows); forward and transposed."""
    if precision == "c64" and min(N) < 64:
        pytest.skip("complex64 factors of grids below 64 cells are block factors")
    rng = np.random.default_rng(sum(N) + nrhs)
    eps = _eps(rng, N).astype(complex)
    eps[N[0] // 2:, N[1] // 2:] += 0.3j
    op = _device(N, npml, pol, eps, precision)
    A, _ = construct_A(OMEGA, [0, N[0] * 0.02], [0, N[1] * 0.02], eps, npml, pol, 1e-6)
    b = rng.standard_normal((nrhs,) + N) + 1j * rng.standard_normal((nrhs,) + N)
    for transpose, M in ((False, A), (True, A.T.tocsr())):
        x, rep = op.solve(torch.tensor(b, device=DEV), precision=precision, tol=1e-12, transpose=transpose)
        assert rep.converged and not rep.fell_back
        assert op.factors[precision][0].numel() == op.nd_bytes[precision]
        for q in {0, nrhs - 1}:
            assert relerr(x[q].cpu().numpy(), solver_direct(M, b[q].reshape(-1)).reshape(N)) < 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("N,cells", [((29, 21), {8, 10, 12, 15}), ((19, 19), {9, 12, 16}), ((16, 16), {21}),
                                     ((21, 21), {16, 20, 25}), ((17, 17), {21, 24, 28, 32})])
def test_leaves_of_every_size(N, cells):
    """The leaf inverse from 8 cells to a full tile, odd counts (a pivot pair
    half padding) among them. An exact factor leaves the first residual at
    eps ||A|| ||x|| ~ 1e-16 * 1e3: one sweep meets 1e-12."""
    g = L.FdfdGrid(*N, 4, 4, 0, 0, OMEGA, 0.02, 1e-6)
    assert {_front(g, -1, k)[0][3] for k in range(_front(g, -1, 0)[0][1])} == cells
    rng = np.random.default_rng(N[0])
    eps = _eps(rng, N)
    op = _device(N, [4, 4], "Ez", eps, "fp64")
    b = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    x, rep = op.solve(torch.tensor(b, device=DEV), precision="fp64", tol=1e-12, max_iter=1)
    assert rep.converged and rep.sweeps == 1
    A, _ = construct_A(OMEGA, [0, N[0] * 0.02], [0, N[1] * 0.02], eps, [4, 4], "Ez", 1e-6)
    assert relerr(x.cpu().numpy(), solver_direct(A, b.reshape(-1)).reshape(N)) < 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "c64"])
def test_kinds_are_told_apart_and_repeat_to_the_bit(precision):
    """fdfd_solve without a kind in its precision reads the tag; fdfd_sweep on
    this kind adds A^-1 r; two factorizations and solves have equal bits; a
    zero right-hand side gives zeros without a sweep."""
    N = (90, 101)
    rng = np.random.default_rng(7)
    op = _device(N, [10, 10], "Ez", _eps(rng, N), precision)
    lib, g, pr = L.lib(), ctypes.byref(op.grid), L.PREC[precision]
    fac = op.factor(precision)
    b = op.to_solver(torch.tensor(rng.standard_normal((2,) + N) + 1j * rng.standard_normal((2,) + N), device=DEV))
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    work = torch.empty(lib.fdfd_solve_workspace_bytes(g, pr, 2), dtype=torch.uint8, device=DEV)
    xs = []
    for flag in (0, L.FACTOR_ND):
        x, st = torch.full_like(b, float("nan")), L.FdfdSolveStats()
        L.check(lib.fdfd_solve(g, ptr(op.op), ptr(fac), pr | flag, ptr(b), ptr(x), 2, 0, 1e-10, 20, ptr(work),
                               ctypes.byref(st), None, None))
        torch.cuda.synchronize()
        xs.append(x)
    assert torch.equal(xs[0], xs[1])
    y = torch.zeros_like(b)
    torch.cuda.synchronize()
    L.check(lib.fdfd_sweep(g, ptr(op.op), ptr(fac), pr, ptr(b), ptr(y), 2, ptr(work), None))
    assert relerr(y.cpu().numpy(), xs[0].cpu().numpy()) < (1e-10 if precision == "fp64" else 1e-2)
    op.drop_factor()
    del fac
    x, rep = op.solve(op.to_user(b), precision=precision, tol=1e-10)     # a new factor, the same bits
    assert torch.equal(op.to_solver(x), xs[0])
    x, rep = op.solve(torch.zeros(N, dtype=torch.complex128, device=DEV), precision=precision)
    assert not x.any() and rep.sweeps == 0 and rep.converged
    # a block factor of the same grid goes the block path
    op.drop_factor()
    op.factor(precision, stepwise=True)
    xb, rep = op.solve(torch.tensor(np.ones(N) + 0j, device=DEV), precision=precision, tol=1e-10)
    assert rep.converged and op.factors[precision][0].numel() != op.nd_bytes[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("N,npml", [((64, 80), [8, 8]), ((129, 96), [10, 10])])
def test_a_solve_that_met_its_tolerance_stays_converged(N, npml):
    """The tolerance is the smallest residual that the complex64 refinement
    passes through, at its floor: the sweep that follows such an iterate lies
    above it, and the solve ends with the iterate that met it."""
    lib, found = L.lib(), 0
    for seed in range(8):
        rng = np.random.default_rng(seed)
        op = _device(N, npml, "Ez", _eps(rng, N), "c64")
        g, fac = ctypes.byref(op.grid), op.factor("c64")
        b = op.to_solver(torch.tensor(rng.standard_normal(N) + 1j * rng.standard_normal(N), device=DEV))
        work = torch.empty(lib.fdfd_solve_workspace_bytes(g, 1, 1), dtype=torch.uint8, device=DEV)

        def solve(tol, steps):
            x, st, ptr = torch.empty_like(b), L.FdfdSolveStats(), lambda t: ctypes.c_void_p(t.data_ptr())
            torch.cuda.synchronize()
            rc = lib.fdfd_solve(g, ptr(op.op), ptr(fac), 1 | L.FACTOR_ND, ptr(b), ptr(x), 1, 0, tol, steps, ptr(work),
                                ctypes.byref(st), None, None)
            return rc, x, st
        seq = [solve(1e-30, k) for k in range(1, 13)]
        res = [st.max_rel_residual for _, _, st in seq]
        k = int(np.argmin(res))
        if seq[k][2].iterations != k + 1 or k + 1 >= seq[-1][2].iterations:
            continue                   # the smallest one is the last before the stall
        found += 1
        rc, x, st = solve(res[k], 20)
        assert rc == L.FDFD_OK and st.converged and st.max_rel_residual <= res[k]
        assert torch.equal(x, seq[k][1])
    assert found


@pytest.mark.gpu
@pytest.mark.parametrize("n,seed,precision,tol", [(128, 24, "fp64", 1e-12), (96, 10, "c64", 1e-12),
                                                  (192, 38, "c64", 1e-12), (128, 15, "c64", 1e-10)])
def test_solves_are_as_exact_as_the_block_factors(n, seed, precision, tol):
    """Operators whose first iterate within the tolerance is 9 to 28 times
    as far from the solution as the block factor's result at that tolerance.
    The solution is FP64 refinement run to its floor, good to the rounding of
    the residual, 1e-16 ||A|| ||x|| / ||b|| ~ 1e-14, times the amplification
    seen above (10): the block factor's error is above 1e-13 in every case."""
    lib = L.lib()
    p = C.c3_request(seed, n=n)
    op = _device(p.shape, p.npml, p.pol, p.eps, "fp64")
    assert (p.dl, p.L0) == (0.02, 1e-6)
    op.grid.omega = op.grid_user.omega = p.omega
    op.set_eps(p.eps)
    b = torch.tensor(p.rhs(), device=DEV)

    def error(x):
        return max(relerr(x[q].cpu().numpy(), ref[q].cpu().numpy()) for q in range(b.shape[0]))
    bs, fac, g = op.to_solver(b), op.factor("fp64"), ctypes.byref(op.grid)
    work = torch.empty(lib.fdfd_solve_workspace_bytes(g, L.FACTOR_ND, b.shape[0]), dtype=torch.uint8, device=DEV)
    ref, ptr = torch.empty_like(bs), lambda t: ctypes.c_void_p(t.data_ptr())
    torch.cuda.synchronize()
    lib.fdfd_solve(g, ptr(op.op), ptr(fac), L.FACTOR_ND, ptr(bs), ptr(ref), b.shape[0], 0, 1e-30, 5, ptr(work), None, None,
                   None)
    ref = op.to_user(ref)
    op.drop_factor()
    x, rep = op.solve(b, precision=precision, tol=tol, fallback=False)
    assert op.factors[precision][0].numel() == op.nd_bytes[precision]
    op.drop_factor()
    op.factor(precision, stepwise=True)
    y, _ = op.solve(b, precision=precision, tol=tol, fallback=False)
    assert op.factors[precision][0].numel() != op.nd_bytes[precision]
    print(f"{n} {seed} {precision} {tol:g}: error {error(x):.1e} in {rep.sweeps} sweeps, block {error(y):.1e}")
    assert error(y) > 1e-13 and error(x) <= error(y)


@pytest.mark.gpu
def test_memory_for_a_block_factor_alone_gets_one(monkeypatch):
    """Where the device has no room for the nested-dissection factor and its
    workspace (an allocation over the block factor's size fails here), the
    block factor solves."""
    N = (64, 64)
    rng = np.random.default_rng(5)
    eps = _eps(rng, N)
    op = _device(N, [8, 8], "Ez", eps, "fp64")
    most, real = op.lib.fdfd_factor_bytes(ctypes.byref(op.grid), 0), torch.empty

    def limited(*a, **k):
        if k.get("dtype") is torch.uint8 and a[0] > most:
            raise torch.cuda.OutOfMemoryError("no room")
        return real(*a, **k)
    monkeypatch.setattr(torch, "empty", limited)
    b = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    x, rep = op.solve(torch.tensor(b, device=DEV), precision="fp64", tol=1e-12)
    assert rep.converged and not rep.fell_back and op.factors["fp64"][0].numel() == most < op.nd_bytes["fp64"]
    A, _ = construct_A(OMEGA, [0, N[0] * 0.02], [0, N[1] * 0.02], eps, [8, 8], "Ez", 1e-6)
    assert relerr(x.cpu().numpy(), solver_direct(A, b.reshape(-1)).reshape(N)) < 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("stepwise,tries", [(False, 2), (True, 1)])
def test_no_factor_is_tried_twice(monkeypatch, stepwise, tries):
    """fallback=False and a tolerance out of reach: the nested-dissection and
    the block factor once each, a resident block factor once."""
    from fdfdpy_amd.device import DeviceOperator
    N = (80, 72)
    rng = np.random.default_rng(3)
    op = _device(N, [9, 9], "Ez", _eps(rng, N), "c64")
    op.factor("c64", stepwise=stepwise)
    real, calls = DeviceOperator._solve_one, []
    monkeypatch.setattr(DeviceOperator, "_solve_one", lambda self, *a: calls.append(1) or real(self, *a))
    b = torch.tensor(rng.standard_normal(N) + 0j, device=DEV)
    with pytest.raises(L.NotConverged):
        op.solve(b, precision="c64", tol=1e-15, max_iter=1, fallback=False)
    assert len(calls) == tries


@pytest.mark.gpu
def test_stall_without_fallback_takes_the_block_factor(monkeypatch):
    """fallback=False keeps the precision: when the nested-dissection factor
    does not refine (its report forced here), the block factor does."""
    from fdfdpy_amd.device import DeviceOperator
    N = (80, 72)
    rng = np.random.default_rng(3)
    eps = _eps(rng, N)
    op = _device(N, [9, 9], "Ez", eps, "c64")
    real = DeviceOperator._solve_one

    def stalled(self, *a, **k):
        rep = real(self, *a, **k)
        if self.factors["c64"][0].numel() == self.nd_bytes["c64"]:
            rep.converged = False
        return rep
    monkeypatch.setattr(DeviceOperator, "_solve_one", stalled)
    b = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    x, rep = op.solve(torch.tensor(b, device=DEV), precision="c64", tol=1e-10, fallback=False)
    assert rep.converged and rep.precision == "c64"
    assert op.factors["c64"][0].numel() != op.nd_bytes["c64"]
    A, _ = construct_A(OMEGA, [0, N[0] * 0.02], [0, N[1] * 0.02], eps, [9, 9], "Ez", 1e-6)
    assert relerr(x.cpu().numpy(), solver_direct(A, b.reshape(-1)).reshape(N)) < 1e-8
