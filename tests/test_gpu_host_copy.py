"""Vectors out of the device: the runtime's copy below 6 MiB, and above it the
chunked copy of several host threads (2 MiB chunks, a partial last one, and
fewer chunks than two rounds of the threads)."""
import numpy as np
import pytest

from cism_amd import pcg
from cism_amd.grid import Grid

pytestmark = pytest.mark.gpu


# bytes of both components: 0.2, 6.0 (just under 6 MiB), 6.6, 8.4 and 36 MB
@pytest.mark.parametrize("nx,ny,nz", [(30, 30, 11), (180, 183, 11), (190, 193, 11), (201, 250, 10), (333, 401, 17)])
def test_velocity_round_trip(require_gpu, nx, ny, nz):
    g = Grid.from_owned(nx, ny, nz)
    rng = np.random.default_rng(nx)
    u, v = (np.asfortranarray(rng.standard_normal(g.vec_shape)) for _ in range(2))
    with pcg.System(g) as s:
        for _ in range(2):
            s.set_x(u, v)
            a, b = s.get_x()
            assert np.array_equal(a, u) and np.array_equal(b, v)
            u, v = v, u
