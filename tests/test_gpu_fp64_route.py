"""GPU: precision "fp64" on nested nodes is served by the Newton form.

The same polynomial as the barycentric combination technique (the general path, still there for
non-nested nodes): both against each other over the inputs that evaluate() takes, with the
technique's own rounding as the bound, sum |zeta F| terms each rounded once: (number of entries)
* 2^-53 is far above it, so 1e-10 of max |y| is used for index sets of up to 1e5 entries; and the
Newton form is no further from the exact interpolant than the technique, or below 1e-14."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import indices as OI
from oracle import nodes as ON
from oracle import smolyak as OS

pytestmark = pytest.mark.gpu


def build(d, d_out, m, dom=False, f=None, kind="leja"):
    from smolyax_amd import nodes as SN
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator

    rng = np.random.default_rng(d + m)
    k = np.log((2 + np.arange(d)) / np.log(2))
    if kind == "gh":
        ong, sng = ON.gauss_hermite(dim=d), SN.GaussHermite(dim=d)
    elif dom:
        dm = np.sort(rng.random((d, 2)), axis=1) + [0, 0.3]
        ong, sng = ON.leja(domains=dm), SN.Leja(domains=dm)
    else:
        ong, sng = ON.leja(dim=d), SN.Leja(dim=d)
    t = OI.find_approximate_threshold(k, m, ong.is_nested)
    a = rng.standard_normal((d_out, d)) / (np.arange(d) + 1.0)
    f = f or (lambda x: np.cos(a @ np.asarray(x) + 0.3))
    ref = OS.Interpolant(d_out=d_out, node_gen=ong, k=k, t=t, f=f)
    return ref, SmolyakBarycentricInterpolator(d_out=d_out, node_gen=sng, k=k, t=t, f=f), ong, rng


def technique(ip, x):
    """The combination technique's own kernels on the same plan."""
    from smolyax_amd import _native as N

    xt = ip._validate_input(x)
    if ip.d_out >= 16:
        return ip._eval_bary_gemm(xt)
    y = torch.empty((xt.shape[0], ip.d_out), dtype=torch.float64, device="cuda")
    if ip._desc.n_share:  # 2 to 16 outputs on a plan without a Newton form in FP64
        nb = N.fn["sbi_bary_eval_few_workspace"](ip._plan, xt.shape[0])
        W = torch.empty(max(nb, 8), dtype=torch.uint8, device="cuda")
        N.check(N.fn["sbi_bary_eval_few_f64"](ip._plan, xt.data_ptr(), xt.shape[0], xt.stride(0),
                                              y.data_ptr(), W.data_ptr(), nb,
                                              ctypes.c_void_p(None)), "eval")
        torch.cuda.synchronize()
        return y
    N.check(N.fn["sbi_bary_eval_f64"](ip._plan, xt.data_ptr(), xt.shape[0], xt.stride(0),
                                      y.data_ptr(), ctypes.c_void_p(None)), "eval")
    torch.cuda.synchronize()
    return y


def rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("d,d_out,m,dom", [(1, 1, 61, False), (1, 3, 20, True), (2, 1, 90, True),
                                           (6, 5, 300, True), (10, 15, 700, False),
                                           (9, 16, 500, True), (40, 33, 900, False),
                                           (300, 1, 400, False)])
def test_same_values_as_the_combination_technique(gpu, d, d_out, m, dom):
    ref, ip, ong, rng = build(d, d_out, m, dom)
    assert ip._fp64_newton
    x = np.stack([g.scale(c) for g, c in zip(ong, rng.uniform(-1, 1, (131, d)).T)], axis=1)
    x[:2, 0] = ong[0](1)[:2]  # on nodes
    y, yt = ip.evaluate(x, "fp64").cpu().numpy(), technique(ip, x).cpu().numpy()
    assert y.shape == (131, d_out) and rel(y, yt) <= 1e-10
    ye = np.asarray(ref(x[:16], dtype=np.longdouble), dtype=np.float64)
    e, et = rel(y[:16], ye), rel(yt[:16], ye)
    print(f"d={d} d_out={d_out} m={m}: Newton {e:.1e}, combination technique {et:.1e} from exact")
    assert e <= max(et, 1e-14)
    # every form of input: strided rows, a transposed layout, float32, one point
    xt = torch.as_tensor(x, device="cuda")
    wide = torch.zeros((131, d + 3), dtype=torch.float64, device="cuda")
    wide[:, :d] = xt
    for other in (wide[:, :d], xt.t().contiguous().t(), wide[::2, :d]):
        want = ip.evaluate(other.contiguous(), "fp64")
        assert torch.equal(ip.evaluate(other, "fp64"), want)
    x32 = x.astype(np.float32)
    assert rel(ip.evaluate(x32, "fp64").cpu().numpy(),
               technique(ip, x32.astype(np.float64)).cpu().numpy()) <= 1e-10
    assert np.array_equal(ip.evaluate(x[5], "fp64").cpu().numpy()[0],
                          ip.evaluate(x[5:6], "fp64").cpu().numpy()[0])
    bad = x.copy()
    bad[7, 0] = np.nan
    yb = ip.evaluate(bad, "fp64").cpu().numpy()
    assert np.isnan(yb[7]).all() and np.array_equal(np.delete(yb, 7, 0), np.delete(y, 7, 0))


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_values_that_are_not_finite_keep_the_combination_technique(gpu, value):
    d = 4
    f = lambda x: value if np.asarray(x)[1] == 1.0 else float(np.sum(x))
    _, ip, _, rng = build(d, 1, 60, f=f)
    assert not ip._fp64_newton
    x = rng.uniform(-1, 1, (70, d))
    y = ip.evaluate(x, "fp64").cpu().numpy()
    assert np.array_equal(y, technique(ip, x).cpu().numpy(), equal_nan=True)


def test_non_nested_nodes_keep_the_combination_technique(gpu):
    _, ip, _, rng = build(5, 3, 200, kind="gh")
    assert not ip._fp64_newton
    x = rng.standard_normal((70, 5))
    assert torch.equal(ip.evaluate(x, "fp64"), technique(ip, x))
