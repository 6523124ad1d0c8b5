"""GPU: sbi_newton_jacobian_f64 on the forms of S and workspace that a C caller may pass.

More than 8 outputs: the rows of S are copied 16 bytes at a time where they start on 16 bytes (and,
for an odd number of outputs, where the caller promises the spare element), else in 4-byte pieces;
the sums are the same, so the results have to be the same bits."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import indices as OI

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [9, 16, 33, 64])
@pytest.mark.parametrize("P", [1, 67])
def test_same_bits_for_every_form_of_the_surpluses(gpu, n, P):
    from smolyax_amd import _native as N
    from smolyax_amd import nodes as SN
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator

    d, m = 7, 700  # (dims of several parts and dims of a few rows)
    k = np.log((2 + np.arange(d)) / np.log(2))
    t = OI.find_approximate_threshold(k, m, True)
    a = np.random.default_rng(n).standard_normal((n, d)) / (np.arange(d) + 1.0)
    ip = SmolyakBarycentricInterpolator(d_out=n, node_gen=SN.Leja(dim=d), k=k, t=t,
                                        f=lambda x: np.cos(a @ np.asarray(x) + 0.3))
    x = torch.rand((P, d), dtype=torch.float64, device="cuda") * 2 - 1
    want = ip.gradient(x)
    rows = ip._S["f64"].shape[0]
    nb = int(N.fn["sbi_newton_jacobian_workspace"](ip._nplan, P, n))
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    # (row stride, first element of S, first word of the workspace): as many elements as the rows need
    for lds, first, w0 in ((n, 0, 0), (n, 1, 0), (n + 1, 0, 1), (n + 2, 1, 1), (n + 3, 0, 0)):
        flat = torch.full((first + (rows - 1) * lds + n,), float("nan"), dtype=torch.float64,
                          device="cuda")
        S = flat[first:].as_strided((rows, n), (lds, 1))
        S.copy_(ip._S["f64"])
        W = torch.empty(w0 + (nb + 7) // 8, dtype=torch.float64, device="cuda")[w0:]
        J = torch.full((P, n, d), float("nan"), dtype=torch.float64, device="cuda")
        print(f"n={n} P={P} lds={lds} first={first} workspace + {8 * w0}", flush=True)
        N.check(N.fn["sbi_newton_jacobian_f64"](ip._nplan, x.data_ptr(), P, d, S.data_ptr(), lds, n,
                                                J.data_ptr(), W.data_ptr(), nb, st), "jacobian")
        torch.cuda.synchronize()
        assert torch.equal(J, want)
