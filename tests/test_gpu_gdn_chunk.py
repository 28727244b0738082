"""Chunks of 3..5 tokens on one workgroup per value head and of 6..16 on four: the bits of the single-token steps for head
counts that are no multiple of eight, the second buffer live, rows wider than their data, and no Q8_1 output."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
S, EPS = 128, 1e-6


@pytest.mark.parametrize("h_k,h_v,ntok,sel,q8", [(1, 2, 3, 0, True), (3, 6, 4, 1, True), (6, 6, 15, 1, False), (2, 8, 16, 0, True),
                                                 (16, 32, 5, 1, True), (2, 4, 6, 1, True), (5, 10, 7, 0, True)])
def test_chunk_is_its_single_steps(h_k, h_v, ntok, sel, q8):
    import rapier_amd as rmi
    from tests.gpu_util import torch
    T = torch()
    g = T.Generator(device="cuda")
    g.manual_seed(h_v + ntok)
    rnd = lambda *s, std=1.0: T.randn(*s, generator=g, device="cuda") * std  # noqa: E731
    ch = 2 * h_k * S + h_v * S
    row, ab_row, y_row, q_row = ch + h_v * S + 5, 2 * h_v + 3, h_v * S + 7, h_v * S // 32 * 36 + 4
    x, ab = rnd(ntok, row), rnd(ntok, ab_row)
    conv_w, dt = rnd(ch, 4, std=0.5), rnd(h_v, std=0.1)
    ssm_a, gamma = -T.exp(rnd(h_v, std=0.5)), 1 + rnd(S, std=0.1)
    state0 = rnd(S, h_v, S, std=0.05)
    base = rnd(2 * h_k + h_v, S, 3, std=0.5)
    q = T.arange(h_v, device="cuda") % h_k
    hist0 = T.stack([base[q], base[h_k + q], base[2 * h_k:]], 1).contiguous()
    st = T.cuda.Stream()
    sel_t = T.full((1,), sel, dtype=T.int32, device="cuda")

    def run(n_per_call):
        live, other = state0.clone(), T.zeros_like(state0)
        hl, ho = hist0.clone(), T.zeros_like(hist0)
        a, b, c, d = (other, live, ho, hl) if sel else (live, other, hl, ho)
        y = T.full((ntok, y_row), 3.0, device="cuda")
        o = T.zeros(ntok, q_row, dtype=T.uint8, device="cuda")
        xch = T.zeros(rmi.gdn_exchange_bytes(h_v), dtype=T.uint8, device="cuda")
        T.cuda.synchronize()
        for t in range(0, ntok, n_per_call):
            rmi.gdn_layer_tokens_x(a, b, c, d, sel_t, x[t], row, ab[t], ab_row, conv_w, dt, ssm_a, gamma, EPS, y[t], y_row,
                                   o[t] if q8 else None, q_row, h_k, h_v, n_per_call, xch, stream=st)
        T.cuda.synchronize()
        assert not other.any() and not ho.any()
        return y, o, live, hl

    for u, v in zip(run(ntok), run(1)):
        assert T.equal(u, v)


@pytest.mark.parametrize("over,h_k,h_v,ntok", [("z", 16, 32, 16), ("z", 3, 6, 7), ("v", 16, 32, 9), ("v", 2, 4, 16),
                                               ("one row", 4, 8, 8)])
def test_chunk_output_over_its_inputs(over, h_k, h_v, ntok):
    """y laid over the z or v rows, or one y row for every token (only its Q8_1 wanted): the same results"""
    import rapier_amd as rmi
    from tests.gpu_util import torch
    T = torch()
    g = T.Generator(device="cuda")
    g.manual_seed(h_v)
    rnd = lambda *s, std=1.0: T.randn(*s, generator=g, device="cuda") * std  # noqa: E731
    ch = 2 * h_k * S + h_v * S
    row = ch + h_v * S
    x0, ab = rnd(ntok, row), rnd(ntok, 2 * h_v)
    conv_w, dt = rnd(ch, 4, std=0.5), rnd(h_v, std=0.1)
    ssm_a, gamma = -T.exp(rnd(h_v, std=0.5)), 1 + rnd(S, std=0.1)
    state0, hist0 = rnd(S, h_v, S, std=0.05), rnd(h_v, 3, S, 3, std=0.5)
    st = T.cuda.Stream()
    sel = T.zeros(1, dtype=T.int32, device="cuda")

    def run(y_of):
        x, live, hist = x0.clone(), state0.clone(), hist0.clone()
        y, stride = y_of(x)
        o = T.zeros(ntok, h_v * S // 32 * 36, dtype=T.uint8, device="cuda")
        T.cuda.synchronize()
        rmi.gdn_layer_tokens(live, T.zeros_like(live), hist, T.zeros_like(hist), sel, x, row, ab, 2 * h_v, conv_w, dt, ssm_a,
                             gamma, EPS, y, stride, o, o.shape[1], h_k, h_v, ntok, stream=st)
        T.cuda.synchronize()
        return y, o, live, hist

    ref = run(lambda x: (T.zeros(ntok, h_v * S, device="cuda"), h_v * S))
    if over == "one row":
        got = run(lambda x: (T.zeros(h_v * S, device="cuda"), 0))
    else:
        at = ch if over == "z" else 2 * h_k * S
        got = run(lambda x: (x[:, at:at + h_v * S], row))
        assert T.equal(got[0], ref[0])
    for u, v in zip(got[1:], ref[1:]):
        assert T.equal(u, v)
