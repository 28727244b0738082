"""Prompts of 64 tokens and more run in wide chunks (up to 1024 tokens per weight pass): the state, caches and hidden
are those of the narrow chunks bit for bit, and the packed GEMM behind them gives the single-column GEMV's bits."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_ingest import assert_same, snapshot

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def E():
    import rapier_amd.engine as eng
    from tests.gpu_util import torch
    torch()
    return eng


# 64: the shortest wide chunk; 79: a narrow graph chunk's remainder behind it would be shorter than a chunk; 129: one
# column past a GEMM tile; 1024 / 1025: a whole chunk, and one token behind it; 1100: a second wide chunk
@pytest.mark.parametrize("n", [64, 79, 129, 1024, 1025, 1100])
def test_wide_prefill_equals_narrow_chunks(E, n):
    eng = E.Engine(E.small_config(ssm_h_k=8, ssm_h_v=16), seed=5, max_ctx=1280)
    rng = np.random.default_rng(n)
    prompt = [int(t) for t in rng.integers(0, 5000, size=n)]
    first = eng.prefill(prompt, batch=8)
    ref = snapshot(E, eng, n)
    greedy, _ = eng.generate(6, mode=E.GREEDY)
    assert eng.prefill(prompt, batch=16) == first
    assert_same(snapshot(E, eng, n), ref, "wide")
    toks, _ = eng.generate(6, mode=E.GREEDY)
    assert toks == greedy
    eng.close()


def test_wide_ingest_continues_a_context(E):
    """behind a generation: the positions, the live GDN buffers and the draft's hidden are the narrow chunks'"""
    eng = E.Engine(E.small_config(ssm_h_k=8, ssm_h_v=16), seed=7, max_ctx=512)
    rng = np.random.default_rng(3)
    a = [int(t) for t in rng.integers(0, 5000, size=90)]
    b = [int(t) for t in rng.integers(0, 5000, size=131)]
    snaps = []
    for batch in (4, 16):
        eng.prefill(a, batch=batch)
        eng.generate(9, mode=E.MTP)
        eng.ingest(b, batch=batch)
        snaps.append(snapshot(E, eng, eng.state()[0]))
    assert_same(snaps[1], snaps[0], "wide ingest")
    eng.close()


# behind a long context: the attention chunks (64 nsub positions: 256, 512 and 1024 here) that a wide chunk's tokens span,
# the host's cut of the grid, and the merge of many chunks, at two, eight and four heads per KV head
@pytest.mark.parametrize("n_head,n_kv,max_ctx,nsub", [(8, 4, 16384, 4), (16, 2, 65536, 8), (8, 4, 65536, 16)])
def test_wide_ingest_behind_a_long_context(E, n_head, n_kv, max_ctx, nsub):
    eng = E.Engine(E.small_config(n_head=n_head, n_kv=n_kv), seed=11, max_ctx=max_ctx)
    assert eng.info()["attn_chunk"] == 64 * nsub
    ctx = max_ctx // 2 + 400
    cur = eng.synth_context(ctx, seed=3, last_token=77)
    eng.save_state()
    toks = [int(t) for t in np.random.default_rng(n_kv).integers(0, 5000, size=1101)]
    row = 2 * n_kv * 256
    c = eng.cfg

    def ingest(batch):
        eng.restore_state(ctx, cur)
        first = eng.ingest(toks, batch=batch)
        out = {"first": first, "state": eng.state()}
        for which, il in [(w, l) for l in (3, 4) for w in (E.BUF_K_CACHE, E.BUF_V_CACHE)]:
            out[which, il] = eng.read(which, il, len(toks) * row, offset=ctx * row).tobytes()
        for il in range(3):
            out["state", il] = eng.read(E.BUF_GDN_STATE, il, 4 * 128 * c.ssm_h_v * 128).tobytes()
            out["hist", il] = eng.read(E.BUF_GDN_HIST, il, 4 * c.ssm_h_v * 9 * 128).tobytes()
        out["hidden"] = eng.read(E.BUF_HIDDEN, 0, 4 * c.n_embd).tobytes()
        return out

    narrow, wide = ingest(8), ingest(16)
    assert [k for k in narrow if narrow[k] != wide[k]] == []
    eng.close()


def test_wide_prefill_9b(E):
    eng = E.Engine(E.qwen35_9b_config(), seed=2024, max_ctx=512)
    prompt = [int(t) for t in np.random.default_rng(1).integers(0, 248320, size=141)]
    first = eng.prefill(prompt, batch=8)
    ref = snapshot(E, eng, len(prompt))
    assert eng.prefill(prompt, batch=16) == first
    assert_same(snapshot(E, eng, len(prompt)), ref, "wide")
    eng.close()


# res "y": the residual in place, as the engine's output and down projections take it
@pytest.mark.parametrize("n_in,n_out,ncols,res", [(2048, 33, 1, True), (2048, 64, 17, False), (4096, 65, 128, True),
                                                  (4096, 100, 129, False), (6144, 130, 31, True), (12288, 70, 130, True),
                                                  (2048, 66, 130, "y"), (4096, 132, 65, "y")])
def test_packed_gemm_is_the_gemv(n_in, n_out, ncols, res):
    import oracle
    import rapier_amd as rmi
    from tests.gpu_util import torch
    T = torch()
    L = rmi.lib()
    st = T.cuda.Stream()
    h = ctypes.c_void_p(st.cuda_stream)
    dev = lambda a: T.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    w = dev(oracle.gen_q6k(n_out, n_in, seed=n_out))
    wp = T.empty(rmi.q6_k_packed_bytes(n_in, n_out), dtype=T.uint8, device="cuda")
    xq = dev(oracle.quantize_q8_1(oracle.normal(n_in * ncols, seed=3), n_in, ncols))
    r = dev(oracle.normal(n_out * ncols, seed=4)) if res else None
    np_ = (n_out + 3) // 4
    y, y1 = r.clone() if res == "y" else T.full((ncols * n_out,), 7.0, device="cuda"), T.zeros(ncols * n_out, device="cuda")
    part, part1 = T.full((ncols * np_,), 7.0, device="cuda"), T.zeros(ncols * np_, device="cuda")
    ws = T.empty(rmi.q6_k_gemm_workspace_bytes(n_in, ncols), dtype=T.uint8, device="cuda")
    T.cuda.synchronize()
    p = lambda t, o=0: ctypes.c_void_p(t.data_ptr() + o if t is not None else None)  # noqa: E731
    rmi.q6_k_pack(w, wp, n_in, n_out, stream=st)
    rmi.q6_k_gemm_packed(wp, xq, y, y if res == "y" else r, part if res else None, n_in, n_out, ncols, ws, stream=st)
    for j in range(ncols):
        xj = p(xq, j * (n_in // 32) * 36)
        if res:
            rmi._check(L.rmi_native_q6_k_mmvq_packed_res_n(p(wp), xj, p(y1, 4 * j * n_out), p(r, 4 * j * n_out),
                                                           p(part1, 4 * j * np_), n_in, n_out, 1, h))
        else:
            rmi._check(L.rmi_native_q6_k_mmvq_packed(p(wp), xj, p(y1, 4 * j * n_out), n_in, n_out, 1, h))
    T.cuda.synchronize()
    assert T.equal(y, y1)
    if res:
        assert T.equal(part, part1)
