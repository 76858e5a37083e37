"""Mass action by products of powers in the generated one-lane kernel (host
build, tests/lane_host) against the FP64 oracle: networks on both sides of the
size from which products are used, rows that keep the log form beside rows
that do not (a fractional coefficient, a coefficient above 4), and activities
far outside the range an unscaled product could hold.

Bar: the bench options end within ~1e-10 of the root (a residual of 1e-14
relative to the first), 1e-8 as in test_lane_host.py.
"""
import numpy as np
import pytest

from pfchem import workloads
import gpu_util as G
import lane_util as LU


def _compare(wl, tmp_path, f32):
    ref, rec, nfail = G.run_oracle(wl)
    assert nfail == 0
    exe = LU.build_host(wl.net, wl.opt, str(tmp_path))
    got = LU.run_host(exe, wl.state, wl.dt, f32=f32)
    n = wl.state.ncell
    assert np.all(got["status"][0, :n] == 0)
    for f, e in G.compare(ref, got, n, net=wl.net).items():
        assert e <= 1e-8, (f, e)


@pytest.mark.parametrize("naq,ncplx", [(8, 16), (9, 16), (16, 40)])
def test_sizes(naq, ncplx, tmp_path):
    _compare(workloads.random_network_workload(ncell=128, naq=naq, ncplx=ncplx, nmnrl=3,
                                               seed=20261207), tmp_path, naq == 9)


def _reseat(wl):
    """state of the (changed) network at the workload's free molalities"""
    n = wl.state.ncell
    st = wl.state
    m0 = st["pri_molal"][:, :n]
    sec, tot, gp, gc = workloads._equilibrate_gamma(wl.net, m0)
    assert (tot > 0).all()
    for k, v in (("sec_molal", sec), ("pri_act_coef", gp), ("sec_act_coef", gc),
                 ("total", 0.7 * tot + 0.3 * np.roll(tot, 1, axis=1))):
        st[k][:, :n] = v * (st["den_kg"][0, :n] * 1e-3 if k == "total" else 1.0)
    return wl


def test_log_rows_beside_product_rows(tmp_path):
    wl = workloads.random_network_workload(ncell=64, naq=10, ncplx=20, nmnrl=2, seed=20261208)
    net = wl.net
    old = net.eqcplx_stoich[3][0]
    net.eqcplx_stoich[3][0] = float(np.copysign(0.5, old))
    net.eqcplx_logK[3] += (net.eqcplx_stoich[3][0] - old) * net._xref[net.eqcplx_species[3][0]]
    # five of a species instead: log K moves with it
    j = net.eqcplx_species[7][0]
    old = net.eqcplx_stoich[7][0]
    net.eqcplx_stoich[7][0] = 5.0
    net.eqcplx_logK[7] += (5.0 - old) * net._xref[j]
    _compare(_reseat(wl), tmp_path, False)


def test_activities_out_of_product_range(tmp_path):
    """one primary at 1e-60 in the complexes with coefficients up to 3: the
    bare powers leave the FP64 range (1e-180 and, divided, 1e+180 twice)"""
    wl = workloads.random_network_workload(ncell=64, naq=9, ncplx=18, nmnrl=1, seed=20261209)
    net, st, n = wl.net, wl.state, wl.state.ncell
    j = 4
    shift = -60.0 - net._xref[j]
    for k, (sp, nu) in enumerate(zip(net.eqcplx_species, net.eqcplx_stoich)):
        net.eqcplx_logK[k] += sum(v for s, v in zip(sp, nu) if s == j) * shift
    for m, (sp, nu) in enumerate(zip(net.kinmnrl_species, net.kinmnrl_stoich)):
        net.kinmnrl_logK[m] += sum(v for s, v in zip(sp, nu) if s == j) * shift
    st["pri_molal"][j, :n] *= 10.0 ** shift
    sec, tot, gp, gc = workloads._equilibrate_gamma(net, st["pri_molal"][:, :n])
    ok = (tot > 1e-40).all(axis=0)
    assert ok.sum() >= 16
    wl.state = st.subset(np.flatnonzero(ok))
    assert np.all(wl.state["pri_molal"][j] < 1e-58)
    _compare(_reseat(wl), tmp_path, False)


@pytest.mark.parametrize("naq", [8, 9])
def test_inactive_mineral_with_overflowing_saturation(naq, tmp_path, monkeypatch):
    """a mineral without surface area takes no part, also where its Q/K leaves
    the FP64 range: the step is the one with a small Q/K, bit for bit, and no
    further cell is handed over (FP32 pass alone and FP64)"""
    wl = workloads.random_network_workload(ncell=64, naq=naq, ncplx=16, nmnrl=3, seed=20261213)
    wl.state["mnrl_area"][1, :] = 0.0
    monkeypatch.setenv("PFCHEM_HOST_NO_RESCUE", "1")
    out = []
    for logk in (0.0, -400.0):  # Q/K = Q 1e400
        wl.net.kinmnrl_logK[1] = logk
        exe = LU.build_host(wl.net, wl.opt, str(tmp_path))
        out.append([LU.run_host(exe, wl.state, wl.dt, f32=f32) for f32 in (False, True)])
    for small, large in zip(*out):
        assert (small["status"][0] == 0).mean() > 0.9
        for f in ("status", "num_iterations", "pri_molal", "total", "sec_molal", "mnrl_volfrac",
                  "mnrl_rate"):
            assert np.array_equal(small[f], large[f]), f
