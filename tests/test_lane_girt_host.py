"""The generated residual and Jacobian block, compiled for the host, against
the FP64 oracle at the bars of test_gpu_residual.py.  The water activity of
the state is an input of the block, whatever use_activity_h2o says (that
option is about updating it)."""
import dataclasses

import numpy as np
import pytest

import lane_util as LU
import pin_util as PU
from test_gpu_residual import DT, _case, _oracle


@pytest.mark.parametrize("which,act_h2o", [("calcite", False), ("calcite", True),
                                           ("random15", False)])
def test_residual_reads_the_water_activity(which, act_h2o, tmp_path):
    wl, st, fixed, fimm = _case(which, 65)
    n, net = st.ncell, wl.net
    rng = np.random.default_rng(3)
    net.eqcplxh2ostoich = rng.integers(-2, 3, net.neqcplx).astype(float)
    net.kinmnrlh2ostoich = rng.integers(-2, 3, net.nkinmnrl).astype(float)
    st["ln_act_h2o"][0, :n] = rng.uniform(-0.2, -0.01, n)
    wl = dataclasses.replace(wl, opt=dataclasses.replace(wl.opt, use_activity_h2o=act_h2o))
    r_ref, j_ref, t_ref, s_ref, acc = _oracle(wl, st, fixed, fimm, np.arange(n), DT)
    exe = LU.build_host_girt(net, wl.opt, str(tmp_path))
    res, jac, got = LU.run_host_girt(exe, net, st, fixed, fimm, DT)
    np.testing.assert_allclose(got["sec_molal"][:, :n], s_ref, rtol=1e-13)
    np.testing.assert_allclose(got["total"][:, :n], t_ref, rtol=1e-13)
    assert np.all(np.abs(res - r_ref) <= 1e-9 * np.maximum(np.abs(r_ref), 1e-12 * acc))
    scale = np.abs(j_ref).max(axis=1, keepdims=True)
    assert (np.abs(jac - j_ref) / np.where(scale > 0, scale, 1.0)).max() <= 1e-11


OPTIONS = {
    "decay": lambda: PU.decay_workload(64)[0],
    "non-isothermal": lambda: PU.nonisothermal_workload(64),
    "temkin+scale": lambda: PU.mineral_options_workload(64, kinmnrl_Temkin_const=2.0,
                                                        kinmnrl_min_scale_factor=1.5),
    "power": lambda: PU.mineral_options_workload(64, kinmnrl_affinity_power=1.7),
    "limiter": lambda: PU.mineral_options_workload(64, kinmnrl_rate_limiter=3.0,
                                                   kinmnrl_affinity_threshold=2.0,
                                                   kinmnrl_irreversible=1),
}


@pytest.mark.parametrize("which", OPTIONS)
def test_residual_options(which, tmp_path, monkeypatch):
    """the options of the networks the one-lane kernel takes: decay, log K and
    rates at the cell's temperature, the mineral rate options; a dry cell"""
    import ctypes as C
    import oracle_lib as O
    wl = OPTIONS[which]()
    st, net, n = wl.state, wl.net, wl.state.ncell
    st["saturation"][0, 3] = 0.0
    naq, rng = net.naqcomp, np.random.default_rng(1)
    fixed = st["total"][:naq] * (1.0 + 1e-3 * rng.standard_normal((naq, st.ld)))
    fimm = st["immobile"][:net.nimmobile] * 1.001 if net.nimmobile else None
    gather = O.CellCtx.gather

    def at_temperature(self, state, cell):  # log K of the cell's temperature
        gather(self, state, cell)
        O.lib().orc_update_temp_dependent_coefs(C.byref(self.n), C.byref(self.o), C.byref(self.c))
        return self

    monkeypatch.setattr(O.CellCtx, "gather", at_temperature)
    r_ref, j_ref, t_ref, s_ref, acc = _oracle(wl, st, fixed, fimm, np.arange(n), DT)
    exe = LU.build_host_girt(net, wl.opt, str(tmp_path))
    res, jac, got = LU.run_host_girt(exe, net, st, fixed, fimm, DT)
    assert np.all(np.abs(res - r_ref) <= 1e-9 * np.maximum(np.abs(r_ref), 1e-12 * acc))
    scale = np.abs(j_ref).max(axis=1, keepdims=True)
    assert (np.abs(jac - j_ref) / np.where(scale > 0, scale, 1.0)).max() <= 1e-11
    np.testing.assert_allclose(got["total"][:, :n], t_ref, rtol=1e-13)
    np.testing.assert_allclose(got["sec_molal"][:, :n], s_ref, rtol=1e-13)
