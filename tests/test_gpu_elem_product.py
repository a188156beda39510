"""FP64 solves of an assembled system take their products in element form; the
rows (CISMGPU_SPMV_FULL=1) are the reference.  Sides around the 63 x 7 vertex
tile, two to seventeen levels, an ice-free rim, floating ice.  Systems that
the element form does not stand for keep the rows: prescribed velocities,
periodic grids (the images of an element have other coordinates, and so other
last bits), a bent grid, inactive vertices inside the ice, a restored matrix.

Bar: the iterates after 7 Chronopoulos-Gear (6 standard) iterations.  Each
product of either form sums a few hundred terms, so it is off by some 1e-14 of
sum |A| |x| at most, and the iterates add a handful of such errors: 1e-12."""
import os

import numpy as np
import pytest

from cism_amd import pcg, synthetic
from cism_amd.velo import BPSolver

pytestmark = pytest.mark.gpu

PROBLEMS = {
    "stream62": lambda: synthetic.ice_stream(62, nz=3, seed=1),
    "stream63": lambda: synthetic.ice_stream(63, nz=11, seed=2),
    "stream64": lambda: synthetic.ice_stream(64, nz=2, seed=3),
    "stream128": lambda: synthetic.ice_stream(128, nz=5, seed=4),
    "stream20": lambda: synthetic.ice_stream(20, nz=17, seed=5),
    "ismip_c": lambda: synthetic.ismip_hom("c", n=40, nz=6),
    "yield_stream": lambda: synthetic.yield_stress_stream("raymond"),
    "marine": lambda: synthetic.marine_sheet(70, nz=7, seed=6),
}
# what a problem's FP64 products are read from when nothing forces the full rows
ROWS = {"yield_stream": "half rows", "ismip_c": "half rows"}


def _iterate(prob, full, algo, bend=False):
    os.environ["CISMGPU_SPMV_FULL"] = "1" if full else "0"
    try:
        s = BPSolver(prob)
        if bend:                       # one vertex off the rectilinear grid: the rows are the only form
            s.xV[s.grid.nvx // 2, s.grid.nvy // 2] += 1.0
        s.assemble(prob.uvel, prob.vvel)
        s.sys.zero_x()
        r = s.sys.solve(algo=algo, precond=2, tolerance=0.0, maxiters=7 if algo == pcg.ALGO_CHRONGEAR else 6,
                        raise_on_error=False)
        x = np.stack(s.sys.get_x())
        r["form"] = s.sys.fp64_product
        r["L2"] = s.residual()[0]
        s.sys.close()
        return r, x
    finally:
        os.environ.pop("CISMGPU_SPMV_FULL", None)


@pytest.mark.parametrize("algo", [pcg.ALGO_CHRONGEAR, pcg.ALGO_STANDARD])
@pytest.mark.parametrize("name", list(PROBLEMS))
def test_element_form_matches_rows(require_gpu, name, algo):
    prob = PROBLEMS[name]()
    r1, x1 = _iterate(prob, True, algo)
    r0, x0 = _iterate(prob, False, algo)
    assert r1["spmv_kind"] == 0 and r1["form"] == "full rows"
    assert r0["form"] == ROWS.get(name, "element form")
    rel = np.linalg.norm(x0 - x1) / np.linalg.norm(x1)
    print(name, algo, f"rel {rel:.2e}, err {r0['err']:.6e} / {r1['err']:.6e}, same bits {np.array_equal(x0, x1)}")
    assert np.linalg.norm(x1) > 0 and rel < 1e-12
    assert r0["err"] == pytest.approx(r1["err"], rel=1e-10)
    # one product each on iterates that differ by rel: |A dx| <= |A| |dx|, and |A||x| is within 1e4 of the residual here
    assert r0["L2"] == pytest.approx(r1["L2"], rel=1e-8)


def test_bent_grid_keeps_the_rows(require_gpu):
    prob = PROBLEMS["stream63"]()
    (_, x1), (_, x0) = _iterate(prob, True, pcg.ALGO_CHRONGEAR, True), _iterate(prob, False, pcg.ALGO_CHRONGEAR, True)
    assert np.array_equal(x0, x1)
    assert not np.array_equal(_iterate(prob, False, pcg.ALGO_CHRONGEAR)[1],
                              _iterate(prob, True, pcg.ALGO_CHRONGEAR)[1])


def test_restored_assembly_keeps_the_rows(require_gpu):
    """The element form belongs to the last assembly: after a restore the
    products are the rows of the restored matrix, with the bits of a run that
    had no other form, until the next assembly."""
    prob = PROBLEMS["stream20"]()
    out = []
    for full in (True, False):
        os.environ["CISMGPU_SPMV_FULL"] = "1" if full else "0"
        try:
            s = BPSolver(prob)
            s.assemble(prob.uvel, prob.vvel)
            s.save_assembly()
            s.assemble(2.0 * prob.uvel, 2.0 * prob.vvel)
            s.restore_assembly()
            s.sys.zero_x()
            s.sys.solve(precond=2, tolerance=0.0, maxiters=7, raise_on_error=False)
            assert s.sys.fp64_product == ("full rows" if full else "half rows")
            out.append((np.stack(s.sys.get_x()), *s.residual()))
            s.assemble(prob.uvel, prob.vvel)
            s.sys.solve(precond=2, tolerance=0.0, maxiters=7, raise_on_error=False)
            assert s.sys.fp64_product == ("full rows" if full else "element form")
            s.sys.close()
        finally:
            os.environ.pop("CISMGPU_SPMV_FULL", None)
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1:] == out[1][1:]


def test_accelerated_picard_matches_the_rows(require_gpu):
    """Accelerated iterations that reject an extension solve a restored
    matrix: the same decisions and iteration counts as on full rows, and the
    same velocity to what the linear tolerance leaves (1e-8 relative residual,
    condition number below 1e2 after the column preconditioner)."""
    prob = PROBLEMS["stream63"]()
    out = []
    for full in (True, False):
        os.environ["CISMGPU_SPMV_FULL"] = "1" if full else "0"
        try:
            s = BPSolver(prob)
            out.append(s.picard(maxiter=8, resid_target=1e-12, linear_maxiters=2000, accelerate=True))
            s.sys.close()
        finally:
            os.environ.pop("CISMGPU_SPMV_FULL", None)
    a, b = out
    assert a.alpha == b.alpha and a.linear_iters == b.linear_iters
    rejected = sum(1 for q in range(1, len(a.alpha)) if a.alpha[q] == 1.0 and a.alpha[q - 1] > 1.0 and
                   a.L2_norm[q + 1] >= a.L2_norm[q])
    assert rejected > 0
    u, v = np.stack([a.uvel, a.vvel]), np.stack([b.uvel, b.vvel])
    assert np.linalg.norm(u - v) < 1e-6 * np.linalg.norm(u)


def _masked(env, drop):
    """Assembled stream with inactive vertices inside the ice: nnz, pairs, two solves, residual."""
    os.environ.update(env)
    try:
        prob = synthetic.ice_stream(40, nz=5, seed=9)
        s = BPSolver(prob)
        for i, j in drop:
            assert s.active_vertex[i, j] == 1
            s.active_vertex[i, j] = 0
        info = s.assemble(prob.uvel, prob.vvel)
        out = [info["nnz"], info["asym_pairs"], *s.residual()]
        for kw in (dict(), dict(precision=pcg.MIXED_FP32, inner_tol=1e-4, max_outer=20)):
            s.sys.zero_x()
            r = s.sys.solve(precond=2, tolerance=1e-9, maxiters=1000, raise_on_error=False, **kw)
            assert r["status"] == 0 and r["err"] < 1e-9, r
            out.append(np.stack(s.sys.get_x()))
        s.sys.close()
        return out
    finally:
        for k in env:
            os.environ.pop(k, None)


def test_inactive_vertices_inside_the_ice(require_gpu):
    """Their rows are zero and their neighbours' rows are not, so neither the
    element form nor half storage stands for that matrix: the full rows do,
    and every row is counted.  One vertex in a wavefront's middle, one at a
    tile's edge, two neighbours."""
    drop = [(12, 17), (20, 9), (21, 9), (33, 30)]
    out = _masked({}, drop)
    ref = _masked({"CISMGPU_SPMV_FULL": "1", "CISMGPU_SYMCHECK": "full"}, drop)
    assert out[:2] == ref[:2] and out[1] > 0
    assert out[2] == pytest.approx(ref[2], rel=1e-12) and out[3] == pytest.approx(ref[3], rel=1e-12)
    assert all(np.array_equal(a, b) for a, b in zip(out[4:], ref[4:]))
