"""The device sum of the history partials over several chunks of 256 tiles
(whole, one tile over, one under) equals the host loop's bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from z4c_amd import Params  # noqa: E402
from z4c_amd.z4c import MeshBlockGeom, Z4c  # noqa: E402


# interior tiles of 256 vertices: 128 of 32*32*32, 1 of 6*6*7, 20 of 17^3
@pytest.mark.parametrize("cells", [[(31, 31, 31)] * 2, [(31, 31, 31)] * 2 + [(5, 5, 6)],
                                   [(31, 31, 31)] * 4 + [(16, 16, 16)] * 13, [(5, 5, 6)],
                                   [(5, 5, 6)] * 255, [(5, 5, 6)] * 513])
def test_sum_in_chunks_equals_host_loop(cells):
    z = Z4c([MeshBlockGeom(n, (0.1, 0.1, 0.1), (0.1 * b, 0.0, 0.0)) for b, n in enumerate(cells)],
            Params())
    gen = torch.Generator(device="cuda").manual_seed(len(cells))
    u = torch.randn(22 * z.total_points, dtype=torch.float64, device="cuda", generator=gen)
    con = torch.randn(7 * z.total_points, dtype=torch.float64, device="cuda", generator=gen)
    out = torch.full((8,), float("nan"), dtype=torch.float64, device="cuda")
    z.history_noalloc(u, con, out)
    assert np.array_equal(np.array(z.history(u, con)), out.cpu().numpy())
    z.close()
