"""The periodic fill (in place: ghosts, then sets of shared vertices) against
the oracle's, bit for bit, on blocks of their own sizes in one batch; a batch
with a block under four cells along an axis goes through a snapshot."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import oracle as orc  # noqa: E402
from z4c_amd import Params  # noqa: E402
from z4c_amd.z4c import MeshBlockGeom, Z4c  # noqa: E402


@pytest.mark.parametrize("sizes", [[(4, 4, 4), (5, 4, 17), (16, 16, 16), (33, 6, 7)],
                                   [(21, 17, 13)], [(4, 30, 5), (2, 9, 5)], [(3, 3, 3)]])
@pytest.mark.parametrize("nvar", [1, 3, 22])
def test_fill_equals_oracle(sizes, nvar):
    gs = [MeshBlockGeom(n, (0.1, 0.1, 0.1), (0.0, 0.0, 0.0)) for n in sizes]
    z = Z4c(gs, Params())
    rng = np.random.default_rng(nvar)
    host = [rng.standard_normal((nvar,) + g.shape) for g in gs]
    u = z.upload(host)
    for _ in range(2):
        z.periodic_fill(u, nvar)
        host = [orc.periodic_fill(orc.Geom.block(g.nx, g.dx, g.xmin), h) for g, h in zip(gs, host)]
    for got, exp in zip(z.download(u, nvar), host):
        assert np.array_equal(got, exp)
    z.close()
