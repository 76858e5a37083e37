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


@pytest.mark.parametrize("ncplx,one_lane", [(160, True), (161, False)])
def test_residual_on_both_sides_of_the_size_line(ncplx, one_lane):
    """networks of many complexes keep the team kernel, whose first call
    compiles nothing (the module of the smaller one takes seconds)"""
    import time
    import torch
    from pfchem import workloads
    from pfchem.lib import Context, DeviceState
    wl = workloads.random_network_workload(ncell=70, naq=16, ncplx=ncplx, nmnrl=5)
    st = wl.state
    fixed = st["total"][:16] * 1.001
    r_ref, j_ref, t_ref, s_ref, acc = _oracle(wl, st, fixed, None, np.arange(70), DT)
    ctx = Context(wl.net, wl.opt)
    ds, fx = DeviceState(st), torch.from_numpy(np.ascontiguousarray(fixed)).cuda()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    res, jac = ctx.residual(ds, fx, None, DT)
    torch.cuda.synchronize()
    first = time.perf_counter() - t0
    print("first call %.2f s" % first, flush=True)
    assert one_lane or first < 2.0
    assert np.all(np.abs(res.cpu().numpy() - r_ref) <= 1e-9 * np.maximum(np.abs(r_ref), 1e-12 * acc))
    j = jac.cpu().numpy().reshape(j_ref.shape)
    scale = np.abs(j_ref).max(axis=1, keepdims=True)
    assert (np.abs(j - j_ref) / np.where(scale > 0, scale, 1.0)).max() <= 1e-11
    got = ds.to_host()
    np.testing.assert_allclose(got["total"], t_ref, rtol=1e-13)
    np.testing.assert_allclose(got["sec_molal"], s_ref, rtol=1e-13)
