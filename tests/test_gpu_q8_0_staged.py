"""The Q8_0 GEMV that stages its columns and row pieces in LDS (one or two columns, whole 16-byte pieces, aligned
operands) gives the general kernel's bits; a matrix 4 bytes off its alignment takes the general kernel.  Rows of
half a step, of whole steps and with a part-full last step; row counts off each workgroup size; both sides of the lines on
size and on the columns' LDS."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncols,res", [(1, False), (1, True), (2, False), (2, True)])
@pytest.mark.parametrize("n_in,n_out", [(2048, 5121), (4096, 2561), (4096, 4096), (4352, 4099), (12288, 1001),
                                        (28928, 402), (29184, 401), (2048, 4882), (2048, 4883), (2048, 5371), (2048, 5441),
                                        (2304, 4341)])
def test_staged_is_the_general_kernel(ncols, res, n_in, n_out):
    import oracle
    import rapier_amd as rmi
    from tests.gpu_util import torch
    T = torch()
    L = rmi.lib()
    st = T.cuda.Stream()
    h = ctypes.c_void_p(st.cuda_stream)
    wb = np.asarray(oracle.gen_q8_0(n_out, n_in, seed=n_out)).reshape(-1).view(np.uint8)
    w = T.from_numpy(wb.copy()).cuda()
    off = T.zeros(wb.size + 4, dtype=T.uint8, device="cuda")
    off[4:] = w
    x = T.from_numpy(np.ascontiguousarray(oracle.quantize_q8_1(oracle.normal(n_in * ncols, seed=n_in), n_in, ncols))).cuda()
    r = T.from_numpy(np.ascontiguousarray(oracle.normal(n_out * ncols, seed=4))).cuda()
    y = T.full((2, ncols * n_out), 7.0, device="cuda")
    part = T.full((2, ncols * ((n_out + 3) // 4)), 7.0, device="cuda")
    T.cuda.synchronize()
    p = lambda t, o=0: ctypes.c_void_p(t.data_ptr() + o)  # noqa: E731
    for i, wp in enumerate((p(w), p(off, 4))):
        if res:
            rmi._check(L.rmi_native_q8_0_mmvq_res_n(wp, p(x), p(y[i]), p(r), p(part[i]), n_in, n_out, ncols, h))
        else:
            rmi._check(L.rmi_native_q8_0_mmvq(wp, p(x), p(y[i]), n_in, n_out, ncols, h))
    T.cuda.synchronize()
    assert T.isfinite(y).all() and not (y == 7.0).any()
    assert T.equal(y[0], y[1])
    if res:
        assert T.equal(part[0], part[1])


@pytest.mark.parametrize("ncols", [5, 6])
@pytest.mark.parametrize("n_in,n_out", [(16384, 1279), (16384, 1281)])   # both sides of the line for a last pass
def test_last_pass_of_more_columns(ncols, n_in, n_out):
    test_staged_is_the_general_kernel(ncols, True, n_in, n_out)
