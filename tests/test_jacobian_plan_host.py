"""Host tables of the Jacobian's register pass (CPU): which singular coordinates the plan lists."""

import numpy as np
import torch

from oracle import indices as OI


def test_any_number_of_singular_coordinates(monkeypatch):
    """A Gauss-Hermite dim of degree 260 has 34 061 of them, more than the 15 bits of a table dim's
    record.  The records only need those of dims that one unit writes; set_f takes every plan."""
    from smolyax_amd import newton as NW
    from smolyax_amd import nodes as SN
    from smolyax_amd.interpolation import SmolyakBarycentricInterpolator as SBI

    d = 30
    k = np.log((2 + np.arange(d)) / np.log(2))
    t = OI.find_approximate_threshold(k, 200, True)
    nf = NW.NewtonForm(k, t, SN.Leja(dim=d), 1)
    nf.set_values(np.arange(len(nf.nus), dtype=np.float64)[:, None])
    L = NW.build_newton_layout(nf)
    split = set(L.jt_red[: 3 * L.n_jt_red: 3].tolist())
    whole = [j for j in L.tab_dim[: L.n_tab_dims].tolist() if j not in split]
    assert split and whole
    count = np.zeros(d, dtype=np.int64)
    for j in L.tab_dim[: L.n_tab_dims]:
        count[j] = 34061 if j in split else 1 + j % 3
    off = np.concatenate([[0], np.cumsum(count)]).astype(np.int32)

    ip = SBI.__new__(SBI)
    ip._d_in, ip._d_out, ip._device = d, 1, torch.device("cpu")
    ip._nform, ip._nlayout, ip._plan, ip._nplan = nf, L, None, None
    monkeypatch.setattr(ip, "_singular_coordinates",
                        lambda: (off, np.linspace(-2.0, 2.0, off[-1])), raising=False)
    ip._upload_newton()
    rec = ip._ndev["jt_dim"].numpy().reshape(-1, 4)
    for (j, row, deg, first), j2, row2, km in zip(rec.tolist(), L.tab_dim, L.tab_row, L.tab_kmax):
        assert (j, row, deg & 0xFFFF) == (j2, row2, km)
        if j in split:
            assert deg >> 16 == 0
        else:
            assert (deg >> 16, first) == (count[j], off[j])


def test_every_group_of_dims_has_its_own_jobs():
    """Jobs of the Jacobian contraction (d_out > 8): every group of 8 dims, with rows or without, is one
    job or several parts; no job writes the groups of others one after another."""
    from smolyax_amd import newton as NW
    from smolyax_amd import nodes as SN

    d, d_out = 203, 9
    k = np.log((2 + np.arange(d)) / np.log(2))
    t = OI.find_approximate_threshold(k, 300, True)
    nf = NW.NewtonForm(k, t, SN.Leja(dim=d), d_out)
    nf.set_values(np.ones((len(nf.nus), d_out)))
    L = NW.build_newton_layout(nf)
    off = L.jac_row_off
    groups = {}
    for a, b, z0, slot in L.jac_job.reshape(-1, 4).tolist():
        assert z0 % 8 == 0 and off[z0] <= a <= b <= off[min(z0 + 8, d)]
        groups.setdefault(z0, []).append((a, b, slot))
    assert sorted(groups) == list(range(0, d, 8))
    assert any(off[z] == off[min(z + 8, d)] for z in groups)  # (groups without rows are there)
    for z0, jobs in groups.items():
        assert jobs[0][0] == off[z0] and jobs[-1][1] == off[min(z0 + 8, d)]
        assert all(p[1] == q[0] for p, q in zip(jobs[:-1], jobs[1:]))
        assert (len(jobs) == 1) == (jobs[0][2] < 0)
