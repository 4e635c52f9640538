"""Marching PCG rounds (csrc/pf_march.hpp): cavities with several regions per
workgroup evaluate the two-iteration round by waves that march up column
strips. Their vectors are those of the regions; only the order of the FP64
sums differs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ITS = 12


def _solve(nx, ny, dx, dy, op, jacobi, cap, iterate64, b):
    from pyflow import _hip as H
    from pyflow._device import DeviceBatch, cavity_params
    p = cavity_params(nx, ny, dx=dx, dy=dy, disable_advection=True, lin_tol=1e-14, lin_maxiter=ITS, jacobi=jacobi,
                      op=H.OP_NEG_LAP_PINNED if op == "pinned" else H.OP_POS_LAP_DIRICHLET, mode=H.MODE_SOLVE)
    p.max_workgroups, p.pcg_per_round, p.iterate64 = cap, 2, iterate64
    batch = DeviceBatch([p], "mixed")
    try:
        batch.set_rhs(0, b)
        d = batch.run(1)[0]
        return batch.solution(0), d.rp_iterations, d.outer_passes
    finally:
        batch.close()


def _cg64(nx, ny, dx, dy, op, jacobi, b, inv_diag):
    """ITS iterations of PCG in float64."""
    def apply(x):
        g = np.pad(x, 1, mode="edge")
        q = (g[1:-1, 2:] - 2 * x + g[1:-1, :-2]) / dx ** 2 + (g[2:, 1:-1] - 2 * x + g[:-2, 1:-1]) / dy ** 2
        if op == "pinned":
            q = -q
            q[0, 0] = x[0, 0]
        else:
            q[0], q[-1], q[:, 0], q[:, -1] = x[0], x[-1], x[:, 0], x[:, -1]
        return q

    m = np.ones((ny, nx))
    if jacobi:
        m[1:-1, 1:-1] = inv_diag
    x, r = np.zeros_like(b), b.copy()
    p = m * r
    rho = np.sum(r * p)
    for _ in range(ITS):
        q = apply(p)
        a = rho / np.sum(p * q)
        x += a * p
        r -= a * q
        z = m * r
        rho, old = np.sum(r * z), rho
        p = z + (rho / old) * p
    return x


# Strips of 120 columns at most: narrower than a pair's halo, one, one and a
# little, cut pairs (odd nx); segments of one row and more; strips and segments
# inside the domain; an FP64 iterate marches above 2048^2 cells.
@pytest.mark.parametrize("nx,ny,cap,iterate64", [
    (2, 300, 2, 1), (3, 131, 1, 1), (70, 9, 1, 1), (120, 70, 1, 1), (121, 66, 1, 1), (128, 9, 1, 1), (245, 61, 1, 1),
    (400, 90, 2, 1), (497, 203, 3, 1), (361, 30, 2, 1), (1201, 64, 2, 1), (1100, 1031, 256, 1),
    (4161, 1031, 256, 2), (2050, 2047, 256, 2)])
@pytest.mark.parametrize("op,jacobi,dx,dy", [("pinned", True, 1.0, 1.0), ("pinned", False, 0.5, 1.25),
                                             ("dirichlet", True, 1.0, 0.75)])
def test_marching_rounds(nx, ny, cap, iterate64, op, jacobi, dx, dy):
    """ITS iterations equal those on one region per workgroup, and float64 PCG.

    Bounds: where two orders of a sum differ, a step length may round to the
    next float (2^-23); 2 ITS of them move the iterate by at most 2 ITS 2^-23
    times a growth of a few, below 2e-5. Against float64 the FP32 vectors add
    a rounding of the same size per iteration and neighbour: 1e-4."""
    rng = np.random.default_rng(nx * 7 + ny)
    b = rng.standard_normal((ny, nx))
    if op == "pinned":
        b -= b.mean()
        b[0, 0] = 0.0
    else:
        b[0] = b[-1] = 0.0
        b[:, 0] = b[:, -1] = 0.0
    x, its, passes = _solve(nx, ny, dx, dy, op, jacobi, cap, iterate64, b)
    y, its_y, _ = _solve(nx, ny, dx, dy, op, jacobi, 1 << 20, iterate64, b)
    assert its == its_y
    assert np.linalg.norm(x - y) <= 2e-5 * np.linalg.norm(y)
    if its == ITS and passes == 1:  # one PCG from the start
        from pyflow._device import cavity_params
        z = _cg64(nx, ny, dx, dy, op, jacobi, b, cavity_params(nx, ny, dx=dx, dy=dy).inv_diag)
        assert np.linalg.norm(x - z) <= 1e-4 * np.linalg.norm(z)
