"""cismgpu_residual_vector_3d_noalloc over its 64-node tiles: fewer nodes than
a tile, a partial last tile, and more tiles than workgroups, against the same
sums by numpy.  A coefficient that couples outside the levels or belongs to a
row without an active vertex holds NaN: it must not be used."""
import ctypes

import numpy as np
import pytest
import torch

from cism_amd import _lib
from cism_amd.grid import Grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx_own,ny_own,nz", [(2, 3, 1), (5, 9, 2), (9, 6, 3), (131, 100, 11)])
def test_residual_tiles(require_gpu, nx_own, ny_own, nz):
    g = Grid.from_owned(nx_own, ny_own, nz)
    rng = np.random.default_rng(nz)
    act = np.asfortranarray(rng.random((g.nvx, g.nvy)) < 0.8).astype(np.int32, order="F")
    own = np.zeros_like(act)
    own[g.ilo - 1:g.ihi, g.jlo - 1:g.jhi] = 1
    on = (act * own) == 1
    A = [np.asfortranarray(rng.standard_normal(g.mat_shape)) for _ in range(4)]
    for a in A:
        a[:, :, ~on] = np.nan
        a[0:9, 0] = np.nan
        a[18:27, nz - 1] = np.nan
    b, x = ([np.asfortranarray(rng.standard_normal(g.vec_shape)) for _ in range(2)] for _ in range(2))
    want = [np.zeros(g.vec_shape) for _ in range(2)]
    size = np.zeros(g.vec_shape)                          # sum of |a x|: the scale of the rounding
    pad = [np.pad(v, 1) for v in x]
    for m in range(27):
        o = (m // 9, m % 3, (m // 3) % 3)                 # level, i, j offsets + 1
        n = [p[o[0]:o[0] + nz, o[1]:o[1] + g.nvx, o[2]:o[2] + g.nvy] for p in pad]
        with np.errstate(invalid="ignore"):
            for blk in range(4):
                t = np.nan_to_num(A[blk][m]) * n[blk % 2]
                want[blk // 2] += t
                size += np.abs(t)
    want = [(w - r) * on for w, r in zip(want, b)]
    dev = lambda a: torch.from_numpy(a.ravel(order="F").copy()).cuda()
    d = [dev(a) for a in [act] + A + b + x]
    out = [torch.full((int(np.prod(g.vec_shape)),), 7.0, dtype=torch.float64, device="cuda") for _ in range(2)]
    norms = torch.zeros(2, dtype=torch.float64, device="cuda")
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    st = _lib.load().cismgpu_residual_vector_3d_noalloc(ctypes.byref(g.cstruct()), *[P(t) for t in d],
                                                        *[P(t) for t in out], P(norms), None)
    assert st == 0, _lib.last_error()
    torch.cuda.synchronize()
    # 54 products and adds and the rhs: at most 55 roundings of the sum of the magnitudes
    bound = 56 * 2.0 ** -53 * (size + np.abs(b[0]) + np.abs(b[1])) * on
    for o, w in zip(out, want):
        r = o.cpu().numpy().reshape(g.vec_shape, order="F")
        assert np.all(np.abs(r - w) <= bound)
    L2 = np.sqrt(sum(np.sum(w ** 2) for w in want))
    L2b = np.sqrt(sum(np.sum((v * on) ** 2) for v in b))
    assert norms[0].item() == pytest.approx(L2, rel=1e-12)
    assert norms[1].item() == pytest.approx(L2 / L2b, rel=1e-12)
