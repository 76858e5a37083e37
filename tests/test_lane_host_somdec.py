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


def _cascade(nlit, nsom):
    """litter pools of variable C:N onto a chain of SOM pools"""
    from pfchem import somdec as SD
    from pfchem.network import ReactionNetwork
    prim = ["CO2(aq)", "NH4+", "NO3-", "N2O(aq)", "H+"]
    imm = ["SOM%d" % i for i in range(nsom)]
    imm += [n % i for i in range(nlit) for n in ("Lit%dC", "Lit%dN")]
    mon = [SD.Monod("NH4+", 1e-6), SD.Monod("NO3-", 1e-6)]
    rx = [SD.Reaction("Lit%d" % i, [("SOM%d" % (i % nsom), 0.5)], rate_constant=1e-6, monod=mon)
          for i in range(nlit)]
    rx += [SD.Reaction("SOM%d" % i, [("SOM%d" % (i + 1), 0.5)] if i + 1 < nsom else [],
                       rate_constant=1e-7) for i in range(nsom)]
    pools = [SD.Pool("SOM%d" % i, 12.0) for i in range(nsom)]
    pools += [SD.Pool("Lit%d" % i) for i in range(nlit)]
    return ReactionNetwork(primary_species_names=prim, primary_spec_Z=np.zeros(5),
                           primary_spec_a0=np.zeros(5), immobile_names=imm,
                           somdec=SD.build_somdec(pools, rx, prim, imm))


@pytest.mark.parametrize("nlit,nsom,takes", [(3, 4, True), (6, 9, False), (7, 11, False)])
def test_large_networks_keep_the_team_kernel(nlit, nsom, takes):
    """networks whose unrolled elimination would take the first step long to
    compile (389 and 528 pattern entries; 115 for the ELM-CN cascade's size)"""
    from pfchem import abi, lib
    want = abi.PFCHEM_OK if takes else abi.PFCHEM_ERR_UNSUPPORTED
    assert lib.prepare_kernels(_cascade(nlit, nsom), workloads.somdec_options()) == want
