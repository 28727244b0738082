"""The packed Q6_K GEMV with column counts that fill no pass: the ingest kernel's part-full 8- and 16-column passes, in
every form of it (a wave per quad, column-split pairs, two K halves, passes of 8 plus a rest), give the single-column
bits and write nothing past the last column."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,n_out,cols", [(2048, 33, (5, 8, 15)), (4096, 1026, (3, 5, 7, 9, 12, 16)), (4096, 12350, (6, 13)),
                                             (8192, 514, (5, 9, 14)), (12288, 258, (4, 7, 9, 11)), (10240, 130, (5, 9, 13))])
@pytest.mark.parametrize("res", [False, True])
def test_part_full_passes_are_the_single_column_bits(n_in, n_out, cols, res):
    import oracle
    import rapier_amd as rmi
    from tests.gpu_util import torch
    T = torch()
    L = rmi.lib()
    st = T.cuda.Stream()
    h = ctypes.c_void_p(st.cuda_stream)
    dev = lambda a: T.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    w = dev(np.asarray(oracle.gen_q6k(n_out, n_in, seed=n_out)).reshape(-1).view(np.uint8))
    wp = T.zeros(rmi.lib().rmi_q6_k_packed_bytes(n_in, n_out), dtype=T.uint8, device="cuda")
    q, np_ = n_in // 32 * 36, (n_out + 3) // 4
    xq = dev(oracle.quantize_q8_1(oracle.normal(n_in * 16, seed=n_in), n_in, 16))
    r = dev(oracle.normal(n_out * 16, seed=4))
    y1, part1 = T.zeros(16 * n_out, device="cuda"), T.zeros(16 * np_, device="cuda")
    T.cuda.synchronize()
    p = lambda t, o=0: ctypes.c_void_p(t.data_ptr() + o)  # noqa: E731
    rmi._check(L.rmi_q6_k_pack(p(w), p(wp), n_in, n_out, h))

    def go(n, j, yy, pp):
        a = (p(wp), p(xq, j * q), p(yy, 4 * j * n_out))
        if res:
            rmi._check(L.rmi_native_q6_k_mmvq_packed_res_n(*a, p(r, 4 * j * n_out), p(pp, 4 * j * np_), n_in, n_out, n, h))
        else:
            rmi._check(L.rmi_native_q6_k_mmvq_packed(*a, n_in, n_out, n, h))

    for j in range(16):
        go(1, j, y1, part1)
    for n in cols:
        y, part = T.full((16 * n_out,), 7.0, device="cuda"), T.full((16 * np_,), 7.0, device="cuda")
        T.cuda.synchronize()
        go(n, 0, y, part)
        T.cuda.synchronize()
        assert T.equal(y[:n * n_out], y1[:n * n_out]) and bool((y[n * n_out:] == 7.0).all()), n
        if res:
            assert T.equal(part[:n * np_], part1[:n * np_]) and bool((part[n * np_:] == 7.0).all()), n
