"""What the benchmark times as one fast_non_dominated_sorting ends with every output, the
domination lists among them, in the buffers it gives."""
import numpy as np
import pytest

import bench
import oracle as O
import pagmo2_amd as P

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,m", [(300, 2), (700, 5)])
def test_every_output_is_written(n, m):
    objs = np.random.default_rng(n).uniform(0, 1, (n, m))
    out = bench.fnds_buffers(torch, n)
    for t in out.values():
        t.fill_(-1)
    ws = P.Fnds()
    bench.fnds_call(P, ws, torch.from_numpy(objs).to("cuda:0"), out)
    torch.cuda.synchronize()
    ws.close()
    for k, ref in O.fnds(objs).items():
        got = out[k].cpu().numpy()
        assert np.array_equal(got[: len(ref)].astype(np.uint64), ref), k
        assert (got[len(ref):] == -1).all(), k
