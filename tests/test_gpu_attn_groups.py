"""Several slot groups of a (chunk, KV head) pair as consecutive workgroups of one XCD: the pairs are padded to a
multiple of 8, so pair counts around that multiple, odd group counts and a last group that is part full are the edges.
Each token's gated output and Q8_1 blocks are bitwise the one-token launch at its position (one group, no padding)."""
import numpy as np
import pytest

from tests.gpu_util import dev, empty, host

pytestmark = pytest.mark.gpu

HD = 256


def flash(rmi, q, kc, vc, p0, gate, nh, nkv, ntok, ctx, nsub):
    ws = empty(rmi.gqa_workspace_bytes(ctx, nkv, nsub), "uint8")
    y, q8 = empty(ntok * nh * HD), empty(ntok * nh * HD // 32 * 36, "uint8")
    rmi.gqa_flash_decode(q, kc, vc, dev(np.array([p0], np.int32)), gate, 2 * nh * HD, y, nh * HD, q8, nh * HD // 32 * 36,
                         ws, nh, nkv, HD, ntok, ctx, nsub, 1.0 / 16.0)
    return host(y).view(np.uint32), host(q8)


@pytest.mark.parametrize("nh,nkv,ctx,nsub,ntok", [
    (4, 1, 64, 1, 3),       # one pair, two groups (the second half full)
    (4, 1, 448, 1, 16),     # 7 pairs
    (8, 2, 256, 1, 5),      # 8 pairs, three groups
    (9, 3, 192, 1, 3),      # 9 pairs, G = 3: a token spans two groups
    (16, 4, 576, 2, 11),    # 20 pairs, the last chunk part full
])
def test_chunk_groups_equal_single_queries(rmi_mod, nh, nkv, ctx, nsub, ntok):
    rng = np.random.default_rng(ctx + ntok)
    kc, vc = (dev(rng.standard_normal(ctx * nkv * HD).astype(np.float16).view(np.uint16)) for _ in range(2))
    q, g = (dev(rng.standard_normal(ntok * nh * HD * m).astype(np.float32)) for m in (1, 2))
    p0 = ctx - ntok
    y, q8 = flash(rmi_mod, q, kc, vc, p0, g, nh, nkv, ntok, ctx, nsub)
    blk = nh * HD // 32 * 36
    for t in range(ntok):
        y1, q81 = flash(rmi_mod, q[t * nh * HD:], kc, vc, p0 + t, g[t * 2 * nh * HD:], nh, nkv, 1, ctx, nsub)
        assert np.array_equal(y1, y[t * nh * HD:(t + 1) * nh * HD]), f"token {t}"
        assert np.array_equal(q81, q8[t * blk:(t + 1) * blk]), f"q8 token {t}"


@pytest.fixture(scope="module")
def rmi_mod():
    import rapier_amd
    rapier_amd.lib()
    return rapier_amd
