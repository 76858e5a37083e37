"""The generated one-lane SomDec step (host build, tests/lane_host) against the
FP64 oracle over the sandbox's options: inhibition, pool-normalized Monod and
thresholds, the temperature and moisture responses, the ELM scalars,
decomposition rates, networks without nitrate, smoothing, the linear
formulation, both forms of the NH4+ / NO3- split, and tracking species that
start empty (1e-20).

Bar: that of test_gpu_somdec.py (the oracle's own spread under a ten-fold
change of its convergence tolerances) on the cells that take the oracle's
sub-steps.  Cells handed over to the team kernel are left as they were.
"""
import numpy as np
import pytest

from pfchem import workloads

import gpu_util as G
import lane_util as LU
import somdec_util as SU
from test_gpu_somdec import CONC_TOL, FIELDS, _oracle_band

NCELL = 512


def _compare(wl, ref, band, got, label, handed):
    n = wl.state.ncell
    st = got["status"][0, :n]
    done = st == 0
    assert np.all(done | (st == 16)), label
    print(label, "handed over", int((~done).sum()))
    assert (~done).mean() <= handed, label
    same = done & (ref["num_sub_steps"][0, :n] == got["num_sub_steps"][0, :n])
    assert (done & ~same).sum() <= 1, label
    for f in FIELDS:
        err = np.abs(got[f][:, :n] - ref[f][:, :n])
        over = (err > CONC_TOL * np.abs(ref[f][:, :n]) + band[f])[:, same]
        print(label, f, float((err / np.maximum(np.abs(ref[f][:, :n]), 1e-300))[:, same].max()))
        assert not over.any(), (label, f)
        # a cell handed over is untouched
        assert np.array_equal(got[f][:, :n][:, ~done], wl.state[f][:, :n][:, ~done])


@pytest.mark.parametrize("which", ("elm-cn",) + SU.OPTION_CASES)
def test_somdec_options(which, tmp_path):
    wl = workloads.somdec_workload(NCELL) if which == "elm-cn" else SU.option_workload(which, NCELL)
    ref, rec, nfail = G.run_oracle(wl)
    assert nfail == 0
    band = _oracle_band(wl, ref)
    # the options change something: pools move
    assert (np.abs(ref["immobile"] - wl.state["immobile"]) > 1e-9 * wl.state["immobile"]).any()
    exe = LU.build_host(wl.net, wl.opt, str(tmp_path))
    for f32 in (False, True):
        got = LU.run_host(exe, wl.state, wl.dt, f32=f32)
        _compare(wl, ref, band, got, which + ("/mixed" if f32 else "/fp64"), 0.05)


def test_unused_entries_of_the_descriptor(tmp_path):
    """the per-reaction tables are as wide as the largest number of terms, and
    a response's parameter is read by its own function only: whatever a caller
    leaves in the unused entries, the kernel compiles and steps the same"""
    wl = SU.option_workload("inhibition", 64)
    exe = LU.build_host(wl.net, wl.opt, str(tmp_path))
    want = LU.run_host(exe, wl.state, wl.dt)
    a = wl.net.somdec.arrays
    for name, count in (("monod_half_saturation", "n_monod"), ("monod_threshold", "n_monod"),
                        ("inhibition_constant", "n_inhibition"),
                        ("inhibition_constant2", "n_inhibition"),
                        ("downstream_stoich", "n_downstream_pools")):
        for r in range(wl.net.somdec.nrxn):
            a[name][r, a[count][r]:] = (np.nan, np.inf, -np.inf)[r % 3]
    a["Ea"][:], a["Q10"][:], a["Ox_half_saturation"][:] = np.nan, np.inf, np.nan
    exe = LU.build_host(wl.net, wl.opt, str(tmp_path))
    got = LU.run_host(exe, wl.state, wl.dt)
    for f in ("status",) + FIELDS:
        assert np.array_equal(got[f], want[f]), f
