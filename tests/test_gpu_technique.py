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
