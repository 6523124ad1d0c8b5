"""GPU: the kernels of the combination technique, called as such.

On nested plans evaluate(x, "fp64") takes the Newton form, so these kernels (the path of non-nested
nodes, of values that are not finite and of nested sequences in another order) are called directly on
layouts that only nested plans have: blocks of four and more active dims, streamed sizes outside 2..4,
odd degrees.  Against the exact interpolant, within 4 times the FP64 oracle's own distance from it,
as for every kernel of the technique."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import indices as OI
from oracle import nodes as ON
from oracle import smolyak as OS

pytestmark = pytest.mark.gpu


def pair(d, m, d_out, kind="leja", kscale=1.0, f=None):
    from smolyax_amd import nodes as SN
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator

    k = kscale * np.log((2 + np.arange(d)) / np.log(2))
    ong, sng = (ON.leja(dim=d), SN.Leja(dim=d)) if kind == "leja" else \
        (ON.gauss_hermite(dim=d), SN.GaussHermite(dim=d))
    t = OI.find_approximate_threshold(k, m, ong.is_nested)
    a = np.random.default_rng(d + m).standard_normal((d_out, d)) / (np.arange(d) + 1.0)
    f = f or (lambda x: np.cos(a @ np.asarray(x) + 0.2))
    ref = OS.Interpolant(d_out=d_out, node_gen=ong, k=k, t=t, f=f)
    return ref, SmolyakBarycentricInterpolator(d_out=d_out, node_gen=sng, k=k, t=t, f=f), ong


def walk(ip, plan, x):
    """sbi_bary_eval_f64."""
    from smolyax_amd import _native as N

    xt = torch.as_tensor(x, device="cuda")
    y = torch.full((len(x), ip.d_out), float("nan"), dtype=torch.float64, device="cuda")
    N.check(N.fn["sbi_bary_eval_f64"](plan, xt.data_ptr(), len(x), xt.stride(0), y.data_ptr(),
                                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "eval")
    return y.cpu().numpy()


def few(ip, x, ws=True):
    """sbi_bary_eval_few_f64."""
    from smolyax_amd import _native as N

    xt = torch.as_tensor(x, device="cuda")
    y = torch.full((len(x), ip.d_out), float("nan"), dtype=torch.float64, device="cuda")
    nb = N.fn["sbi_bary_eval_few_workspace"](ip._plan, len(x)) if ws else 0
    W = torch.empty(max(nb, 8), dtype=torch.uint8, device="cuda")
    N.check(N.fn["sbi_bary_eval_few_f64"](ip._plan, xt.data_ptr(), len(x), xt.stride(0), y.data_ptr(),
                                          W.data_ptr(), nb,
                                          ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
            "few")
    return y.cpu().numpy()


def near_exact(y, ref, x):
    ye = ref(x, dtype=np.longdouble).astype(np.float64)
    scale = np.max(np.abs(ye))
    e, eo = np.max(np.abs(y - ye)) / scale, np.max(np.abs(ref(x) - ye)) / scale
    print(f"  {e:.1e} from exact, FP64 oracle {eo:.1e}", flush=True)
    assert e <= max(4.0 * eo, 1e-14)


def points(d, n, seed, ong):
    x = np.random.default_rng(seed).uniform(-1, 1, (n, d))
    x[: min(n, 3), 0] = ong[0](4)[: min(n, 3)]
    return x


@pytest.mark.parametrize("d,m,kscale", [(8, 3000, 0.3), (2, 40, 1.0), (12, 600, 0.2), (6, 200, 1.0)])
def test_record_program_on_nested_layouts(gpu, d, m, kscale):
    from smolyax_amd import _native as N

    ref, ip, ong = pair(d, m, 1, kscale=kscale)
    assert ip._prog is not None and ip._desc.n_pseg > 0
    x = points(d, 131, m, ong)
    print(f"d={d} m={m}: {ip._prog.n_records} records", flush=True)
    y = walk(ip, ip._plan, x)
    near_exact(y, ref, x)
    q = N.BaryDesc()  # the per-block kernel: the same tables without the program
    ctypes.pointer(q)[0] = ip._desc
    q.pseg = None
    plan = ctypes.c_void_p()
    N.check(N.fn["sbi_bary_plan_create"](ctypes.byref(q), ctypes.byref(plan)), "plan")
    try:
        near_exact(walk(ip, plan, x), ref, x)
    finally:
        N.fn["sbi_plan_destroy"](plan)
    assert np.array_equal(walk(ip, ip._plan, x[70:71])[0], y[70])


@pytest.mark.parametrize("d,m,d_out", [(4, 60, 5), (8, 500, 16), (6, 300, 33), (20, 900, 40)])
def test_barycentric_gemm_on_nested_layouts(gpu, d, m, d_out):
    ref, ip, ong = pair(d, m, d_out)
    x = points(d, 150, m, ong)
    xt = torch.as_tensor(x, device="cuda")
    y = ip._eval_bary_gemm(xt)
    near_exact(y[:40].cpu().numpy(), ref, x[:40])
    ip._memory_limit = 64 * 8 * ip.layout.k_raw / 1024**3  # chunks of 64 points
    assert ip._point_chunk(ip.layout.k_raw, 8, 150) == 64
    assert torch.equal(ip._eval_bary_gemm(xt), y)
    assert torch.equal(ip._eval_bary_gemm(xt[149:150])[0], y[149])


@pytest.mark.parametrize("d,m,P", [(5, 300, 65), (40, 2000, 130)])
def test_share_kernel_takes_16_outputs(gpu, monkeypatch, d, m, P):
    """evaluate() sends 16 outputs to the dense contraction, so set_f builds no shares for them; the
    entry point takes them."""
    from smolyax_amd import packing

    assert pair(d, m, 16, kind="gh")[1]._desc.n_share == 0
    monkeypatch.setattr(packing, "SHARE_MAX_OUT", 16)
    ref, ip, ong = pair(d, m, 16, kind="gh")
    assert ip._desc.n_share > 0
    x = points(d, P, m, ong)
    y = few(ip, x)
    near_exact(y[:32], ref, x[:32])
    assert np.array_equal(few(ip, x, ws=False), y)
    assert np.array_equal(few(ip, x[P - 1:])[0], y[P - 1])


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_values_that_are_not_finite_in_one_of_three_outputs(gpu, value):
    """A nested plan with such a value keeps the technique, and gets its shares for it: output 1 is
    what the walk over blocks gives, the others are finite and near it (1e-12 of max |y|: a sum of at
    most 1000 entries, each rounded a few times)."""
    d = 4
    f = lambda x: np.array([np.sum(x), value if np.asarray(x)[1] == 1.0 else 1.0 + x[0], np.cos(x[2])])
    _, ip, ong = pair(d, 60, 3, f=f)
    assert not ip._fp64_newton and ip._desc.n_share > 0
    x = points(d, 70, 3, ong)
    y = ip.evaluate(x, "fp64").cpu().numpy()
    yw = walk(ip, ip._plan, x)
    assert np.array_equal(y, few(ip, x), equal_nan=True)
    assert np.array_equal(np.isnan(y), np.isnan(yw)) and np.array_equal(np.isinf(y), np.isinf(yw))
    assert np.isfinite(y[:, [0, 2]]).all()
    ok = np.isfinite(yw)
    assert np.max(np.abs(y[ok] - yw[ok])) <= 1e-12 * np.max(np.abs(yw[ok]))
