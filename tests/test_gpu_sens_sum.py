"""The reduced gradient is the sum of the converged cells' gradients, at cell
counts below, at and beside the number of slices of its first launch, and
the same on every call."""
import numpy as np
import pytest

from test_gpu_sens import _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncell", [1, 63, 64, 65, 777])
def test_gradient_is_the_sum_of_the_cells(ncell):
    from pfchem.lib import Context, DeviceState
    wl, wv, ws = _setup("random15", ncell)
    ctx = Context(wl.net, wl.opt)
    ds = DeviceState(wl.state)
    g, f, st, gc = ctx.adjoint(ds, wl.dt, wv, ws, per_cell=True)
    gc = gc.cpu().numpy()[:, :ncell][:, st.cpu().numpy()[:ncell] == 0]
    # ncell additions in another order: ncell roundings of the summed sizes
    bound = ncell * 2.3e-16 * np.abs(gc).sum(axis=1) + 1e-300
    assert np.all(np.abs(gc.sum(axis=1) - g) <= bound)
    again = ctx.adjoint(DeviceState(wl.state), wl.dt, wv, ws)[0]
    assert np.array_equal(again, g)
