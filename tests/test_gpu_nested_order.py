"""GPU: "fp64" on nested sequences of the user's own.  A Newton form is only as stable as the order of
its nodes, so on a sequence whose order spoils it the combination technique has to serve the call.

One dim, f = cos(3 x + o): with 60 or 129 nodes on [-1, 1] the interpolant is f itself far below
FP64, and only the block of the highest degree counts: sum_m F_m l_m(x) with l_m a product of n
differences, n products and a weight of n products, so |error| <= (4 n + 4) 2^-53 sum_m |l_m(x)| for
|F| <= 1 (Newton on these nodes: 2e-4 and 2e-2)."""

import numpy as np
import pytest
import torch

from smolyax_amd import nodes as SN

pytestmark = pytest.mark.gpu


class Sequence1D(SN.Generator1D):
    def __init__(self, seq):
        super().__init__(is_nested=True)
        self.seq = np.asarray(seq, dtype=np.float64)

    def __call__(self, n):
        return self.seq[: n + 1]

    def scale(self, x):
        return x

    scale_back = scale

    def get_random(self, n=1):
        return np.random.uniform(-1, 1, n)

    def get_quadrature_weights(self, n):
        return np.full(n + 1, 1.0 / (n + 1))


def ascending(n):
    return -np.cos(np.pi * (2 * np.arange(n) + 1) / (2 * n))


def level_order(levels):
    """Clenshaw-Curtis nodes: 0, then the ends, then the new nodes of each level from left to right."""
    seq = [0.0, -1.0, 1.0]
    for lv in range(2, levels + 1):
        m = 2**lv
        seq += [-np.cos(np.pi * i / m) for i in range(1, m, 2)]
    return seq


@pytest.mark.parametrize("seq,newton", [(ascending(60), False), (level_order(7), False),
                                        (SN.Leja1D()(59), True)])
@pytest.mark.parametrize("d_out", [1, 3, 17])
def test_fp64_on_other_nested_sequences(gpu, seq, newton, d_out):
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator

    n = len(seq)
    f = lambda x: np.cos(3.0 * float(np.asarray(x)[0]) + np.arange(d_out))
    ip = SmolyakBarycentricInterpolator(d_out=d_out, node_gen=SN.Generator([Sequence1D(seq)]),
                                        k=[1.0], t=n - 0.5, f=f)
    assert ip.n_f_evals == n
    rng = np.random.default_rng(n)
    x = np.concatenate([rng.uniform(-1, 1, 100), -np.cos(np.pi * rng.random(100)), seq[:3]])
    y = ip.evaluate(x[:, None], "fp64").cpu().numpy()
    D = x[:, None] - np.asarray(seq)[None, :]
    dev = np.zeros(len(x))
    for m in range(n):
        ratio = np.delete(D, m, 1) / (seq[m] - np.delete(np.asarray(seq), m))
        dev += np.abs(np.prod(ratio, axis=1))
    bound = (4 * n + 4) * 2.0**-53 * dev
    err = np.abs(y - np.cos(3.0 * x[:, None] + np.arange(d_out))).max(axis=1)
    print(f"n={n} d_out={d_out}: error {err.max():.1e}, bound {bound.max():.1e}, "
          f"Newton {ip._fp64_newton}", flush=True)
    assert (err <= bound + 2.0**-53).all()
    assert ip._fp64_newton == newton
    # the same through the default call, and one point alone
    assert torch.equal(ip(x[5:6, None])[0], torch.as_tensor(y[5], device="cuda"))
