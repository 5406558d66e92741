"""crowding_distance where its two forms change hands (one workgroup up to 1024
points, radix sorts beyond) and at the powers of two below.  Bit for bit with the
oracle."""
import numpy as np
import pytest

import oracle as O
import pagmo2_amd as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [64, 65, 1023, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("m", [2, 3, 7])
def test_crowding(n, m):
    pts = np.random.default_rng(n + m).integers(0, n, (n, m)).astype(float)
    ws = P.Fnds()
    out = torch.empty(n, dtype=torch.float64, device="cuda:0")
    ws.crowding_distance(torch.from_numpy(pts).to("cuda:0"), out)
    ws.close()
    ref = O.crowding_distance(pts, stable=True)
    assert np.array_equal(out.cpu().numpy(), ref, equal_nan=True)
    assert np.array_equal(P.crowding_distance_host(pts), ref, equal_nan=True)
