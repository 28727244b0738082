"""rmi_topk at the edges of its work split: one 64-key register, one 256-logit slice, one workgroup's 2048 logits, the
eight lists of a merge wave, a part-full last list, lists of more slices per wave, and the k where popped lists give
way to sorted ones.  The result is exact."""
import numpy as np
import pytest

from tests.gpu_util import dev, empty, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 64, 65, 255, 257, 2047, 2049, 8 * 2048, 8 * 2048 + 1, 65 * 2048 - 3, 300001])
def test_topk_edges(orc, n):
    import rapier_amd as rmi
    rng = np.random.default_rng(n)
    l = (rng.integers(-2000, 2000, n) / 8.0).astype(np.float32)   # ties, some of them across lists
    l[-1] = 1e4
    for k in sorted({1, min(n, 16), min(n, 17), min(n, 63), min(n, 64)}):
        ws = empty(rmi.topk_workspace_bytes(n) // 4)
        ids, vals = empty(k, "int32"), empty(k)
        rmi.topk(dev(l), n, k, ids, vals, ws)
        assert list(zip(host(ids).tolist(), host(vals).tolist())) == orc.topk(l, k), (n, k)
