"""Resident solves (csrc/pf_resident.hpp): the CG iterations of a single cavity
run inside one launch by workgroups that exchange their sums and region edges
through memory, and FP64 divisions by the spacings are exact multiply-adds
(div_fast). Both must give the bits of one phase per launch with true
divisions (PYFLOW_RESIDENT=0; PYFLOW_FASTDIV=0), whatever the grid, operator,
iteration cap and values."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(params, precision, resident, fastdiv=True):
    from pyflow._device import DeviceBatch
    want = {"PYFLOW_RESIDENT": "1" if resident else "0", "PYFLOW_FASTDIV": "1" if fastdiv else "0"}
    old = {k: os.environ.get(k) for k in want}
    os.environ.update(want)  # read when cavities are added and tables built
    try:
        b = DeviceBatch([params], precision)
        if params.mode == 2:
            b.set_rhs(0, np.zeros((params.ny, params.nx)))
        b.run(1)  # builds the tables; from rest this step (or a zero solve) leaves no trace
        return b
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


def _solve(nx, ny, dx, dy, op, b, maxiter, precision, resident, fastdiv=True, tol=1e-12, rows=0, jacobi=True):
    from pyflow import _hip as H
    from pyflow._device import cavity_params
    p = cavity_params(nx, ny, dx=dx, dy=dy, disable_advection=True, lin_tol=tol, lin_maxiter=maxiter, jacobi=jacobi,
                      op=H.OP_NEG_LAP_PINNED if op == "pinned" else H.OP_POS_LAP_DIRICHLET, mode=H.MODE_SOLVE)
    p.tile_rows = rows
    batch = _batch(p, precision, resident, fastdiv)
    try:
        batch.set_rhs(0, b)
        d = batch.run(1)[0]
        return batch.solution(0), (d.rp_iterations, d.rp_info, d.bnorm, d.rp_residual, d.outer_passes), batch.rounds()
    finally:
        batch.close()


def _rhs(kind, ny, nx):
    rng = np.random.default_rng(3)
    b = rng.standard_normal((ny, nx))
    if kind == "source":  # Krylov vectors fade out towards the far corner, zeros beyond the front
        b[:] = 0.0
        b[ny // 2, 1] = -1.0
    elif kind == "tiny":
        b *= 1e-290
    elif kind == "subnormal":
        b *= 1e-312
    elif kind == "wide":
        b *= 10.0 ** rng.integers(-200, 140, size=b.shape)
        b[rng.random(b.shape) < 0.3] = -0.0
    elif kind == "huge":
        b *= 1e150
    elif kind == "inf":
        b[ny // 3, nx // 2] = np.inf
    return b


def _same(a, b):
    for x, y in zip(a[:2], b[:2]):
        assert np.array_equal(x, y, equal_nan=True)
    x, y = np.asarray(a[0]), np.asarray(b[0])
    fin = np.isfinite(x)
    assert np.array_equal(np.signbit(x[fin]), np.signbit(y[fin]))


@pytest.mark.parametrize("kind", ["normal", "source", "tiny", "subnormal", "wide", "huge", "inf"])
@pytest.mark.parametrize("nx,ny,dx,dy,op", [
    (64, 40, 1.0 / 63, 0.1, "pinned"),        # one region
    (130, 97, 1.0, 1.25, "pinned"),           # several regions, ragged
    (129, 33, 1e-3, 7.3, "dirichlet"),
    (70, 20, 1e30, 0.3, "pinned"),            # a spacing out of range: true divisions
])
def test_fp64_values_bitwise(nx, ny, dx, dy, op, kind):
    b = _rhs(kind, ny, nx)
    print(f"[resident] {nx}x{ny} dx={dx} dy={dy} {op} {kind}", flush=True)
    ref = _solve(nx, ny, dx, dy, op, b, 150, "fp64", False)
    _same(_solve(nx, ny, dx, dy, op, b, 150, "fp64", True), ref)
    _same(_solve(nx, ny, dx, dy, op, b, 150, "fp64", True, fastdiv=False), ref)


@pytest.mark.parametrize("nx,ny,rows,maxiter,jacobi", [
    (65, 17, 0, 400, True),      # a one-column region, a one-row tile
    (2, 300, 0, 900, True),      # narrow: neighbours above and below only
    (300, 2, 0, 900, True),      # flat: neighbours left and right only
    (128, 128, 1, 2000, True),   # full regions of one tile
    (127, 129, 2, 2000, False),  # regions of two tiles, one cell short and one over
    (192, 96, 4, 37, True),      # stopped at the cap
    (192, 96, 4, 1, True),       # a single iteration
    (512, 448, 4, 9000, True),   # several thousand iterations, 56 workgroups
    (1024, 1024, 4, 60, True),   # one workgroup per CU
])
def test_fp64_shapes_bitwise(nx, ny, rows, maxiter, jacobi):
    b = _rhs("normal", ny, nx)
    print(f"[resident] {nx}x{ny} rows={rows} cap={maxiter} jacobi={jacobi}", flush=True)
    ref = _solve(nx, ny, 1.0, 1.0, "pinned", b, maxiter, "fp64", False, rows=rows, jacobi=jacobi)
    new = _solve(nx, ny, 1.0, 1.0, "pinned", b, maxiter, "fp64", True, rows=rows, jacobi=jacobi)
    _same(new, ref)
    if maxiter > 1:
        assert new[2] < ref[2]


@pytest.mark.parametrize("nx,ny,rows,maxiter,op,jacobi", [
    (2, 2, 0, 50, "pinned", True),
    (5, 3, 0, 50, "dirichlet", True),
    (64, 16, 1, 500, "pinned", True),      # one full region of one tile
    (65, 17, 0, 800, "pinned", True),      # frames with one-cell neighbours
    (67, 66, 4, 1500, "dirichlet", True),  # neighbours narrower than the frame
    (2, 300, 0, 1500, "pinned", True),
    (300, 3, 0, 1500, "pinned", False),
    (130, 33, 1, 2000, "pinned", True),
    (131, 97, 2, 2000, "pinned", True),
    (192, 128, 4, 3000, "pinned", False),
    (256, 192, 4, 3000, "dirichlet", True),
    (255, 193, 4, 7, "pinned", True),      # odd cap: a last round of one iteration
    (255, 193, 4, 2, "pinned", True),
    (449, 389, 4, 6000, "pinned", True),
    (1024, 1024, 4, 200, "pinned", True),  # one workgroup per CU
])
def test_mixed_shapes_bitwise(nx, ny, rows, maxiter, op, jacobi):
    b = _rhs("normal", ny, nx)
    print(f"[resident] mixed {nx}x{ny} rows={rows} cap={maxiter} {op} jacobi={jacobi}", flush=True)
    ref = _solve(nx, ny, 1.0, 1.25, op, b, maxiter, "mixed", False, rows=rows, jacobi=jacobi, tol=1e-9)
    new = _solve(nx, ny, 1.0, 1.25, op, b, maxiter, "mixed", True, rows=rows, jacobi=jacobi, tol=1e-9)
    _same(new, ref)


@pytest.mark.parametrize("kind", ["source", "tiny", "wide", "inf"])
def test_mixed_values_bitwise(kind):
    b = _rhs(kind, 97, 130)
    if kind == "wide":
        b = np.clip(b, -1e30, 1e30)
    print(f"[resident] mixed values {kind}", flush=True)
    ref = _solve(130, 97, 1.0, 1.0, "pinned", b, 200, "mixed", False)
    new = _solve(130, 97, 1.0, 1.0, "pinned", b, 200, "mixed", True)
    _same(new, ref)


@pytest.mark.parametrize("nx,ny,precision", [(100, 70, "fp64"), (64, 64, "fp64"), (100, 70, "mixed"), (300, 200, "mixed")])
def test_steps_bitwise(nx, ny, precision):
    """Steps of a lid-driven cavity, several per run and one per run."""
    from pyflow._device import cavity_params
    out = []
    for resident in (False, True):
        p = cavity_params(nx, ny, dx=1.0, dy=1.0, scheme="quick", lid_velocity=1.0, Re=400.0, lin_tol=1e-8,
                          lin_maxiter=2000)
        print(f"[resident] steps {nx}x{ny} resident={resident}", flush=True)
        b = _batch(p, precision, resident)
        try:
            ds = [b.run(n)[0] for n in (3, 1, 2)]
            f = [np.zeros((ny + 2, nx + 2)) for _ in range(3)]
            b.download(0, *f)
        finally:
            b.close()
        out.append((f, [(d.dt, d.rp_iterations, d.rp_iterations_run, d.rp_residual, d.continuity, d.ru) for d in ds]))
    assert np.array_equal(np.array(out[0][0]), np.array(out[1][0]))
    assert out[0][1] == out[1][1]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_meeting_fails_bitwise(monkeypatch, precision):
    """Workgroups that do not wait for each other (PYFLOW_MEET_US=0) run
    ordinary rounds wherever they did not all arrive at once: the same bits."""
    b = _rhs("normal", 260, 330)
    ref = _solve(330, 260, 1.0, 1.0, "pinned", b, 300, precision, False)
    monkeypatch.setenv("PYFLOW_MEET_US", "0")
    new = _solve(330, 260, 1.0, 1.0, "pinned", b, 300, precision, True)
    print(f"[resident] no waiting {precision}: {new[2]} launches, one phase per launch {ref[2]}", flush=True)
    _same(new, ref)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_concurrent_streams_bitwise(precision):
    """Two threads solve on two streams at once, each with more than half of
    the GPU's CUs as workgroups: whoever cannot gather its workgroups runs
    ordinary rounds, and both get the bits they get alone."""
    import threading

    import torch
    from pyflow import _hip as H
    from pyflow._device import DeviceBatch, cavity_params
    nx, ny = 832, 768  # 13 x 12 regions
    b = _rhs("normal", ny, nx)
    p = cavity_params(nx, ny, dx=1.0, dy=1.0, disable_advection=True, lin_tol=1e-9, lin_maxiter=400, mode=H.MODE_SOLVE)

    def go(out, k):
        with torch.cuda.stream(torch.cuda.Stream()):
            batch = DeviceBatch([p], precision)
            try:
                for _ in range(3):
                    batch.set_rhs(0, b)
                    batch.run(1)
                    out[k].append(batch.solution(0))
            finally:
                batch.close()

    alone, both = [[]], [[], []]
    go(alone, 0)
    ts = [threading.Thread(target=go, args=(both, k)) for k in range(2)]
    print(f"[resident] two streams {precision}", flush=True)
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(len(r) == 3 for r in both)
    for r in both:
        for x in r:
            assert np.array_equal(x, alone[0][0])


@pytest.mark.parametrize("sizes", [
    [(512, 512), (449, 300), (64, 64), (33, 40), (512, 384), (200, 640), (96, 96), (512, 448)],  # more workgroups than CUs
    [(130, 97), (16, 16), (65, 17)],
])
def test_batch_bitwise(sizes):
    """A batch whose cavities run their PCG in turns, against one phase per
    launch for all: three steps, then one more."""
    from pyflow._device import DeviceBatch, cavity_params
    out = []
    for resident in ("0", "1"):
        ps = [cavity_params(nx, ny, dx=1.0, dy=1.0, scheme="quick", lid_velocity=1.0, Re=300.0 * (k + 1), lin_tol=1e-6,
                            lin_maxiter=3000) for k, (nx, ny) in enumerate(sizes)]
        print(f"[resident] batch of {len(sizes)} resident={resident}", flush=True)
        old = os.environ.get("PYFLOW_RESIDENT")
        os.environ["PYFLOW_RESIDENT"] = resident
        try:
            b = DeviceBatch(ps, "mixed")
            d = [b.run(n) for n in (3, 1)]
        finally:
            if old is None:
                del os.environ["PYFLOW_RESIDENT"]
            else:
                os.environ["PYFLOW_RESIDENT"] = old
        f = []
        for k, (nx, ny) in enumerate(sizes):
            a = [np.zeros((ny + 2, nx + 2)) for _ in range(3)]
            b.download(k, *a)
            f += a
        b.close()
        out.append((f, [(x[k].rp_iterations_run, x[k].rp_residual, x[k].continuity) for x in d for k in range(len(sizes))]))
    for x, y in zip(out[0][0], out[1][0]):
        assert np.array_equal(x, y)
    assert out[0][1] == out[1][1]
