"""The generated residual and Jacobian block, compiled for the host, against
the FP64 oracle at the bars of test_gpu_residual.py.  The water activity of
the state is an input of the block, whatever use_activity_h2o says (that
option is about updating it)."""
import dataclasses

import numpy as np
import pytest

import lane_util as LU
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
