"""The residual and Jacobian block, one cell per lane, around the edges of its
64-cell workgroups, against the oracle at the bars of test_gpu_residual.py."""
import numpy as np
import pytest

from test_gpu_residual import DT, _case, _oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which,ncell", [("calcite", 1), ("calcite", 63), ("random15", 1),
                                         ("random15", 65), ("random15", 129)])
@pytest.mark.parametrize("jacobian", [True, False])
def test_residual_lane_edges(which, ncell, jacobian):
    import torch
    from pfchem.lib import Context, DeviceState
    wl, st, fixed, fimm = _case(which, ncell)
    r_ref, j_ref, t_ref, s_ref, acc = _oracle(wl, st, fixed, fimm, np.arange(ncell), DT)
    ds = DeviceState(st)
    res, jac = Context(wl.net, wl.opt).residual(
        ds, torch.from_numpy(np.ascontiguousarray(fixed)).cuda(), None, DT, jacobian=jacobian)
    torch.cuda.synchronize()
    got = ds.to_host()
    d = np.abs(res.cpu().numpy()[:, :ncell] - r_ref)
    # terms that cancel leave the rounding of the largest: 1e-12 of the
    # accumulation rate, relative 1e-9 above that
    assert np.all(d <= 1e-9 * np.maximum(np.abs(r_ref), 1e-12 * acc))
    if jacobian:
        j = jac.cpu().numpy().reshape(j_ref.shape[0], j_ref.shape[1], -1)[:, :, :ncell]
        scale = np.abs(j_ref).max(axis=1, keepdims=True)
        assert (np.abs(j - j_ref) / np.where(scale > 0, scale, 1.0)).max() <= 1e-11
    else:
        assert jac is None
    np.testing.assert_allclose(got["total"][:, :ncell], t_ref, rtol=1e-13)
    np.testing.assert_allclose(got["sec_molal"][:, :ncell], s_ref, rtol=1e-13)
