"""GPU: sbi_newton_eval_f64_gemm, the FP64 Newton form of several outputs in one call.

The same kernels as sbi_newton_basis_rows and sbi_contract_f64_ws, so the same bits: with all of its
workspace, with the basis matrix alone, in memory_limit chunks, and one point alone."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import indices as OI

pytestmark = pytest.mark.gpu


def build(d, d_out, m, **kw):
    from smolyax_amd import nodes as SN
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator

    k = np.log((2 + np.arange(d)) / np.log(2))
    t = OI.find_approximate_threshold(k, m, True)
    a = np.random.default_rng(d + m).standard_normal((d_out, d)) / (np.arange(d) + 1.0)
    return SmolyakBarycentricInterpolator(d_out=d_out, node_gen=SN.Leja(dim=d), k=k, t=t,
                                          f=lambda x: np.cos(a @ np.asarray(x) + 0.3), **kw)


@pytest.mark.parametrize("d,d_out,m,P", [(2, 2, 12, 1), (3, 9, 200, 63), (6, 33, 250, 64),
                                         (10, 15, 900, 130), (40, 16, 1500, 65), (12, 3, 4000, 7),
                                         (400, 2, 1500, 131), (330, 3, 1030, 1), (1000, 17, 2000, 64)])
def test_one_call_has_the_bits_of_its_parts(gpu, d, d_out, m, P):
    from smolyax_amd import _native as N

    ip = build(d, d_out, m)
    S, n = ip._surpluses("f64", gemm=True), ip._nlayout.basis_n
    wide = torch.rand((P, d + 3), dtype=torch.float64, device="cuda") * 2 - 1
    x, ldx = wide[:, :d], d + 3
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    H = torch.empty((n, P + P % 2), dtype=torch.float64, device="cuda")
    N.check(N.fn["sbi_newton_basis_rows"](ip._nplan, x.data_ptr(), P, ldx, 0, n, H.data_ptr(),
                                          H.stride(0), 0, st), "basis")
    want = torch.empty((P, d_out), dtype=torch.float64, device="cuda")
    ld = d_out + d_out % 2
    N.check(N.fn["sbi_contract_f64_ws"](H.data_ptr(), H.stride(0), S.data_ptr(), ld, None,
                                        want.data_ptr(), d_out, P, d_out, n, None, 0, st), "contract")
    nb = N.c_i64()
    ws = N.fn["sbi_newton_eval_f64_gemm_workspace"](ip._nplan, P, ctypes.byref(nb))
    print(f"d={d} d_out={d_out} rows={n} P={P}: workspace {ws}, basis {nb.value}", flush=True)
    assert ws >= nb.value >= 8 * n * P
    for have in (ws, nb.value):
        W = torch.empty(have, dtype=torch.uint8, device="cuda")
        y = torch.full((P, d_out + 1), float("nan"), dtype=torch.float64, device="cuda")
        N.check(N.fn["sbi_newton_eval_f64_gemm"](ip._nplan, x.data_ptr(), P, ldx, S.data_ptr(), ld,
                                                 y.data_ptr(), d_out + 1, W.data_ptr(), have, st),
                "eval")
        assert torch.equal(y[:, :d_out], want) and torch.isnan(y[:, d_out]).all()
    assert torch.equal(ip.evaluate(x, "newton-fp64"), want)
    assert torch.equal(ip.evaluate(x[P // 2], "newton-fp64")[0], want[P // 2])
    assert (ip._table_rows() > 0) == (d > 300)  # (wide plans: basis from a table in global memory, or,
    # with the basis matrix alone and in the chunks below, factor by factor)
    ip._memory_limit = 64 * 8 * n / 1024**3  # chunks of 64 points
    assert torch.equal(ip.evaluate(x, "newton-fp64"), want)
    assert N.fn["sbi_newton_eval_f64_gemm"](ip._nplan, x.data_ptr(), P, ldx, S.data_ptr(), ld,
                                            y.data_ptr(), d_out + 1, W.data_ptr(), nb.value - 1,
                                            st) == -1
