"""The FP32 product that reads every half-stored slot once (marching along j)
against the one that re-reads the partner rows and the full rows: the same
bits.  Column counts around the 64-lane tile (a last tile of one column among
them), level counts around the 12 wavefronts of a workgroup, periodic images,
fewer rows than a share."""
import os

import numpy as np
import pytest

from cism_amd import pcg
from cism_amd.grid import BC_NO_ICE, BC_OUTFLOW, BC_PERIODIC
from systems import random_spd_system

pytestmark = pytest.mark.gpu

CASES = [(63, 6, 12, BC_NO_ICE), (64, 9, 13, BC_PERIODIC), (65, 5, 2, BC_PERIODIC), (66, 7, 5, BC_OUTFLOW),
         (6, 40, 23, BC_PERIODIC), (129, 4, 3, BC_PERIODIC)]


def _solve(g, act, A, bu, bv, **env):
    os.environ.update(env)
    try:
        with pcg.System(g) as s:
            s.set_matrix(act, *A, bu, bv)
            s.set_x(g.zeros_vec(), g.zeros_vec())
            r = s.solve(precond=2, tolerance=1e-10, maxiters=3000, precision=pcg.MIXED_FP32, inner_tol=1e-3,
                        max_outer=30)
            return r, np.stack(s.get_x())
    finally:
        for k in env:
            os.environ.pop(k, None)


@pytest.mark.parametrize("nx,ny,nz,bc", CASES)
def test_marching_product_same_bits(require_gpu, nx, ny, nz, bc):
    sys = random_spd_system(n=nx, ny=ny, nz=nz, bc=bc, seed=nx + nz)
    r1, x1 = _solve(*sys, CISMGPU_SPMV_SYMX="1")
    r0, x0 = _solve(*sys, CISMGPU_SPMV_SYMX="0")
    rf, xf = _solve(*sys, CISMGPU_SPMV_FULL="1")
    assert (r1["spmv_kind"], r0["spmv_kind"], rf["spmv_kind"]) == (3, 3, 1)
    assert r1["niters"] == r0["niters"] == rf["niters"] and r1["err"] < 1e-10
    assert np.array_equal(x1, x0) and np.array_equal(x1, xf)
