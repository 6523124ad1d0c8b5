"""GPU: the smallest nested plans keep the walk over blocks in "fp64" (one launch instead of two).

On both sides of the line the values are those of the other route, up to the rounding of either: at
most 4 roundings per factor and entry, at most 500 entries whose |zeta F| are at most 3 for these f,
so 1e-12 of max |y| holds for both; and the route depends on the plan alone."""

import numpy as np
import pytest
import torch

from oracle import indices as OI

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,m,d_out,small", [(1, 1, 2, True), (1, 15, 3, True), (1, 40, 1, False),
                                             (2, 10, 15, True), (2, 40, 2, True), (3, 45, 2, True),
                                             (5, 20, 8, True), (40, 80, 1, True), (40, 80, 5, False),
                                             (2, 10, 16, False), (10, 160, 1, True),
                                             (10, 160, 2, False), (5, 160, 1, False)])
def test_route_of_small_plans(gpu, d, m, d_out, small):
    from smolyax_amd import nodes as SN
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator

    k = np.log((2 + np.arange(d)) / np.log(2))
    t = OI.find_approximate_threshold(k, m, True) if m > 1 else 0.1
    a = np.random.default_rng(d + m).standard_normal((d_out, d)) / (np.arange(d) + 1.0)
    f = lambda x: np.cos(a @ np.asarray(x) + 0.3)
    ip = SmolyakBarycentricInterpolator(d_out=d_out, node_gen=SN.Leja(dim=d), k=k, t=t, f=f)
    print(f"d={d} m={m} d_out={d_out}: {ip.layout.k_raw} entries, small {ip._small_plan}", flush=True)
    assert ip._small_plan == small
    wide = torch.rand((133, d + 3), dtype=torch.float64, device="cuda") * 2 - 1
    wide[0, :d] = 0.0  # a node
    x = wide[:, :d]
    y = ip.evaluate(x, "fp64")
    yn = ip.evaluate(x, "newton-fp64")
    assert float((y - yn).abs().max()) <= 1e-12 * float(yn.abs().max())
    if not small:
        assert torch.equal(y, yn)
    assert torch.equal(ip(x.contiguous()), y) and torch.equal(ip(x[::2]), y[::2])
    assert torch.equal(ip(x.cpu().numpy()), y)
    for p in (0, 64, 132):
        assert torch.equal(ip(x[p]), y[p:p + 1])
    bad = x.clone()
    bad[5, 0] = float("nan")
    yb = ip(bad)
    keep = torch.arange(133, device="cuda") != 5
    assert torch.equal(yb[keep], y[keep])
    if d > 1 or m > 1:
        assert torch.isnan(yb[5]).all()


@pytest.mark.parametrize("d,m,d_out", [(1, 20, 1), (2, 40, 4), (5, 60, 2), (5, 60, 4), (6, 160, 1),
                                       (6, 160, 4), (40, 80, 2)])
@pytest.mark.parametrize("family", ["leja", "gh"])
def test_jacobian_of_small_plans(gpu, family, d, m, d_out):
    """Both register passes on the same plan (n_jt_blocks = 0 selects the one over jac_unit): the sums
    are the same up to order, at most 400 terms: 400 * 2^-53 * sum |terms|, which 1e-11 of max |J|
    covers; the same NaN at node coordinates."""
    import ctypes

    from smolyax_amd import _native as N
    from smolyax_amd import nodes as SN
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator

    k = np.log((2 + np.arange(d)) / np.log(2))
    gen = SN.Leja(dim=d) if family == "leja" else SN.GaussHermite(dim=d)
    t = OI.find_approximate_threshold(k, m, family == "leja")
    a = np.random.default_rng(d + m).standard_normal((d_out, d)) / (np.arange(d) + 1.0)
    ip = SmolyakBarycentricInterpolator(d_out=d_out, node_gen=gen, k=k, t=t,
                                        f=lambda x: np.cos(a @ np.asarray(x) + 0.3))
    if ip._nplan is None or not ip._newton_fp64_ok:
        pytest.skip("no FP64 Newton form of this plan")
    x = torch.rand((67, d), dtype=torch.float64, device="cuda") * 2 - 1
    x[3, 0] = float(gen[0](1)[1])
    x[4, d - 1] = float(gen[d - 1](1)[0])
    J = ip.gradient(x)
    q = N.NewtonDesc()
    ctypes.pointer(q)[0] = ip._ndesc
    q.n_jt_blocks = 0
    plan, own = ctypes.c_void_p(), ip._nplan
    N.check(N.fn["sbi_newton_plan_create"](ctypes.byref(q), ctypes.byref(plan)), "plan")
    try:
        ip._nplan = plan
        J0 = ip.gradient(x)
    finally:
        ip._nplan = own
        N.fn["sbi_newton_plan_destroy"](plan)
    one_pass = ip._nlayout.n_jac_red == 0 and ip._nlayout.n_vjp_ent * (d_out + 1) <= 800
    print(f"{family} d={d} m={m}: {ip._nlayout.n_vjp_ent} entries, small {one_pass}", flush=True)
    assert torch.equal(J.isnan(), J0.isnan()) and J.isnan().any()
    diff = (J - J0).nan_to_num().abs().max()
    assert float(diff) <= 1e-11 * float(J0.nan_to_num().abs().max())
    if one_pass:
        assert float(diff) == 0.0
