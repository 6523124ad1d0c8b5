"""GPU: the workspaces that spread small FP64 batches over more workgroups stay within memory_limit and
a server's HBM budget; without them the same bits."""

import numpy as np
import pytest
import torch

from oracle import indices as OI

pytestmark = pytest.mark.gpu


def build(kind, d, m, d_out):
    from smolyax_amd import nodes as SN
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator

    k = np.log((2 + np.arange(d)) / np.log(2))
    gen = SN.Leja(dim=d) if kind == "leja" else SN.GaussHermite(dim=d)
    t = OI.find_approximate_threshold(k, m, kind == "leja")
    a = np.random.default_rng(d + m).standard_normal((d_out, d)) / (np.arange(d) + 1.0)
    return SmolyakBarycentricInterpolator(d_out=d_out, node_gen=gen, k=k, t=t,
                                          f=lambda x: np.cos(a @ np.asarray(x) + 0.3))


@pytest.mark.parametrize("kind,d,m,d_out,P", [("gh", 40, 3000, 10, 500), ("gh", 20, 6000, 17, 64),
                                              ("leja", 40, 3000, 33, 64)])
def test_memory_limit(gpu, kind, d, m, d_out, P):
    ip = build(kind, d, m, d_out)
    x = torch.rand((P, d), dtype=torch.float64, device="cuda")
    want = ip.evaluate(x, "fp64")  # (and whatever the path keeps)
    ws = ip.scratch_bytes("fp64", P)
    rows = 0 if kind == "gh" and d_out < 16 else \
        ip.layout.k_raw if kind == "gh" else ip._nlayout.basis_n
    room = rows * P * 8 + 4096  # the basis matrix, no more
    print(f"{kind} d_out={d_out} P={P}: workspace {ws}, basis {rows * P * 8}", flush=True)
    assert ws > 8192
    out = P * d_out * 8

    def peak():
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        y = ip.evaluate(x, "fp64")
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        return torch.cuda.max_memory_allocated() - base

    assert peak() >= rows * P * 8 + out + ws
    ip._memory_limit = room / 1024**3
    assert ip.scratch_bytes("fp64", P) == 0
    assert peak() <= room + out + 2048  # (allocations round up to 512 bytes)


def test_server_budget(gpu):
    from smolyax_amd import serving

    ips = {"a": build("gh", 40, 3000, 10), "b": build("leja", 40, 3000, 33)}
    xs = [(n, torch.rand((200, ips[n].d_in), dtype=torch.float64, device="cuda")) for n in "abababab"]
    want = [ips[n].evaluate(x, "fp64") for n, x in xs]
    most = max(serving.Server(ips, precision="fp64").footprint(n, 200) for n in "ab")
    ws = max(ip.scratch_bytes("fp64", 200) for ip in ips.values())
    for budget, spread in ((most, False), (1 << 30, True)):
        srv = serving.Server(ips, precision="fp64", n_streams=4, hbm_budget_bytes=budget,
                             max_batch_points=200)
        reqs = [srv.submit(n, x) for n, x in xs]
        held = 0
        while srv.step():
            assert srv.reserved <= srv.budget
            held = max(held, max(s.reserved for s in srv.slots))
        assert (held > most) == spread, (held, most, ws)
        for r, y in zip(reqs, want):
            assert torch.equal(r.y, y)
