"""The streaming LAG activity kernel at cell counts around its blocks, against
the oracle's RActivityCoefficients."""
import numpy as np
import pytest

from pfchem import abi, workloads

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncell,ld,naq,ncplx", [(1, 1, 15, 60), (255, 256, 15, 60),
                                                (257, 300, 8, 32), (300, 300, 17, 13)])
def test_lag_activity_matches_oracle(ncell, ld, naq, ncplx):
    import torch
    from pfchem.lib import Context, DeviceState
    wl = workloads.random_network_workload(ncell=ncell, ld=ld, naq=naq, ncplx=ncplx)
    ds = DeviceState(wl.state)
    Context(wl.net, wl.opt).update_activity(ds)
    torch.cuda.synchronize()
    got = ds.to_host()
    cx = O.CellCtx(wl.net, wl.opt)
    for c in range(0, ncell, 16):
        cc = cx.gather(wl.state, c)
        cc.activity()
        # a sum of naq + ncplx terms, a square root and a power: 1e-13
        np.testing.assert_allclose(got["pri_act_coef"][:, c], cc.get("pri_act_coef", naq),
                                   rtol=1e-13)
        np.testing.assert_allclose(got["sec_act_coef"][:, c], cc.get("sec_act_coef", ncplx),
                                   rtol=1e-13)
    for f in ("pri_act_coef", "sec_act_coef"):
        assert np.array_equal(got[f][:, ncell:], wl.state[f][:, ncell:])
