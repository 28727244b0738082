"""The one-pass GEMV over several columns (mmvq_cols.hip) gives the single-column kernel's bits: rows that end inside a
slab, tiles with rows and columns missing, one to six slabs, several tiles per workgroup, both lane splits of Q6_K at each
of them, and the fewest columns and rows each type takes it from (with the calls just below, which keep the passes)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TYPES = {"q4_k": 12, "q5_k": 13, "q6_k": 14, "q8_0": 8}


def blocks(oracle, name, n_out, n_in, seed):
    if name == "q6_k":
        return oracle.gen_q6k(n_out, n_in, seed=seed)
    if name == "q8_0":
        return oracle.gen_q8_0(n_out, n_in, seed=seed)
    rng = np.random.default_rng(seed)
    b = rng.integers(0, 256, (n_out * (n_in // 256), 144 if name == "q4_k" else 176), dtype=np.uint8)
    b[:, :4] = rng.normal(0, 1e-2, (b.shape[0], 2)).astype(np.float16).view(np.uint8)   # d, dmin
    return b.reshape(-1)


# off 4: a matrix 4 bytes off 16 (Q6_K: off its streaming kernels)
@pytest.mark.parametrize("name,off", [(n, 0) for n in TYPES] + [("q6_k", 4), ("q8_0", 4)])
@pytest.mark.parametrize("n_in,n_out,ncols,res", [
    (256, 17, 9, True), (1280, 33, 16, False), (2048, 40, 12, True), (4096, 2051, 5, False), (4096, 4300, 16, True),
    (6144, 70, 13, True), (8192, 1100, 8, False), (11008, 50, 11, False), (12288, 16, 16, True), (12288, 100, 9, False),
    (768, 2560, 5, True), (768, 2559, 5, False), (1024, 2561, 3, True), (5120, 1700, 3, False), (5120, 70, 13, True),
    (5120, 5000, 4, False), (4096, 8200, 3, True), (4096, 10241, 5, False), (3072, 10240, 3, False), (4096, 5700, 4, True),
    (12288, 4608, 5, False), (12288, 5633, 3, True)])
def test_columns_are_the_single_column_bits(name, n_in, n_out, ncols, res, off):
    import oracle
    import rapier_amd as rmi
    from tests.gpu_util import torch
    T = torch()
    L = rmi.lib()
    st = T.cuda.Stream()
    h = ctypes.c_void_p(st.cuda_stream)
    dev = lambda a: T.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    w = dev(np.concatenate([np.zeros(off, np.uint8), blocks(oracle, name, n_out, n_in, n_out)]))[off:]
    q = n_in // 32 * 36
    xq = dev(oracle.quantize_q8_1(oracle.normal(n_in * ncols, seed=n_in), n_in, ncols))
    np_ = (n_out + 3) // 4
    r = dev(oracle.normal(n_out * ncols, seed=4))
    y, y1 = T.full((ncols * n_out,), 7.0, device="cuda"), T.zeros(ncols * n_out, device="cuda")
    part, part1 = T.full((ncols * np_,), 7.0, device="cuda"), T.zeros(ncols * np_, device="cuda")
    T.cuda.synchronize()
    p = lambda t, o=0: ctypes.c_void_p(t.data_ptr() + o)  # noqa: E731

    def go(n, j, yy, pp):
        if res:
            rmi._check(getattr(L, f"rmi_native_{name}_mmvq_res_n")(p(w), p(xq, j * q), p(yy, 4 * j * n_out), p(r, 4 * j * n_out),
                                                                   p(pp, 4 * j * np_), n_in, n_out, n, h))
        else:
            rmi._check(L.rmi_native_mmvq(TYPES[name], p(w), p(xq, j * q), p(yy, 4 * j * n_out), n_in, n_out, n, h))

    go(ncols, 0, y, part)
    for j in range(ncols):
        go(1, j, y1, part1)
    T.cuda.synchronize()
    assert T.equal(y, y1)
    if res:
        assert T.equal(part, part1)
