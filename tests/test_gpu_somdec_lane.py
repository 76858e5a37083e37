"""The one-lane SomDec step (the default of networks without complexes,
minerals and an oxygen response) at cell counts around its wavefront and
workgroup edges, against the FP64 oracle through the bars of
test_gpu_somdec.py, and its hand-over to the team kernel."""
import numpy as np
import pytest

from pfchem import abi, workloads

import gpu_util as G
from test_gpu_somdec import FIELDS, VARIANTS, _check, _oracle_band

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncell,ld", [(1, 1), (63, 64), (65, 65), (257, 300), (4099, 4099)])
def test_somdec_lane_edges(ncell, ld):
    wl = workloads.somdec_workload(ncell, ld=ld)
    ref, rec, nfail = G.run_oracle(wl)
    assert nfail == 0
    band = _oracle_band(wl, ref)
    for variant in VARIANTS:
        got, _ = G.run_gpu(wl, variant)
        _check(wl, ref, rec, band, got, "somdec-lane/%d/%s" % (ncell, abi.KERNEL_NAMES[variant]))
        for f in FIELDS:  # rows beyond the cells stay as they were
            assert np.array_equal(got[f][:, ncell:], wl.state[f][:, ncell:])


@pytest.mark.parametrize("variant", VARIANTS)
def test_somdec_lane_and_team_agree(variant):
    """Same cells through the two kernels.  Both end at |step| or residual
    below the options' tolerances, so they differ where rounding moves that
    end by an iteration; the oracle's band bounds it, and nearly every cell
    takes the same sub-steps."""
    wl = workloads.somdec_workload(20001)
    lane, ctx = G.run_gpu(wl, variant)
    assert ctx.get_launch(variant)["lanes_per_cell"] == 16  # the hand-over pass's shape
    team, _ = G.run_gpu(wl, variant, lanes=16, block=128)
    one, _ = G.run_gpu(wl, variant, lanes=1, block=256)
    assert np.all(lane["status"] == 0) and np.all(team["status"] == 0)
    same = lane["num_sub_steps"] == team["num_sub_steps"]
    assert (~same).sum() <= 20
    assert (lane["num_iterations"] != team["num_iterations"]).mean() < 0.01
    for f in FIELDS:
        assert np.array_equal(lane[f], one[f]), f  # asked for by shape: the same kernel
        scale = np.abs(team[f]).max(axis=1, keepdims=True)
        err = (np.abs(lane[f] - team[f]) / scale)[:, same[0]]
        # the iteration ends at 1e-8 relative change: one iteration more or
        # less moves an entry by at most that much of its row's range
        assert err.max() <= 1e-8, f


def _one_lane(ctx, wl, variant):
    """whether a step of this context ran the one-lane kernel (its pass is
    what pfchem_set_pass_timing times)"""
    import torch
    from pfchem.lib import DeviceState, PfchemError
    ctx.set_pass_timing(True)
    ctx.step(DeviceState(wl.state), wl.dt, variant)
    torch.cuda.synchronize()
    try:
        return ctx.pass_time() > 0.0
    except PfchemError:
        return False
    finally:
        ctx.set_pass_timing(False)


@pytest.mark.parametrize("variant", VARIANTS)
def test_reported_shape_restores_the_default(variant):
    """reading and setting a shape changes no kernel, and the shape of a fresh
    context brings its kernel back"""
    from pfchem.lib import Context
    wl = workloads.somdec_workload(300)
    ctx = Context(wl.net, wl.opt)
    start = ctx.get_launch(variant)
    put = lambda l: ctx.set_launch(variant, l["lanes_per_cell"], l["block_size"],
                                   l["blocks_per_cu"], l["rows_per_lane"])
    assert _one_lane(ctx, wl, variant)
    put(start)
    assert ctx.get_launch(variant) == start and _one_lane(ctx, wl, variant)
    for shape in ((8, 128, 4, 2), (16, 128, 4, 1), (1, 256, 1, 1)):
        ctx.set_launch(variant, *shape)
        assert _one_lane(ctx, wl, variant) == (shape[0] == 1)
        kept = ctx.get_launch(variant)
        put(kept)
        assert ctx.get_launch(variant) == kept
        assert _one_lane(ctx, wl, variant) == (shape[0] == 1)
    put(start)
    assert _one_lane(ctx, wl, variant)


@pytest.mark.parametrize("variant", VARIANTS)
def test_tuning_keeps_the_one_lane_step(variant, tmp_path):
    """the tuner starts from the default kernel, leaves the state as given and
    ends on a shape that still runs it (the teams are several times slower
    here); so does a context that applies its cache"""
    import torch
    from pfchem.lib import Context, DeviceState
    wl = workloads.somdec_workload(60000)
    ctx = Context(wl.net, wl.opt)
    ds = DeviceState(wl.state)
    cache = str(tmp_path / "tune.json")
    ctx.autotune(ds, wl.dt, variant, cache_path=cache, quick=True)
    torch.cuda.synchronize()
    back = ds.to_host()
    for f in FIELDS:
        assert np.array_equal(back[f], wl.state[f]), f
    small = workloads.somdec_workload(300)
    assert _one_lane(ctx, small, variant)
    other = Context(wl.net, wl.opt)
    other.autotune(ds, wl.dt, variant, cache_path=cache)  # the cached choice
    assert _one_lane(other, small, variant)


@pytest.mark.parametrize("which", ["inhibition", "pool-monod", "responses", "scalars",
                                   "no-smoothing", "trackers"])
def test_somdec_options_on_the_device(which):
    """networks that reach the sandbox's other options, through the device
    build of the kernel and its hand-over (test_lane_host_somdec.py runs every
    option through the host build): the oracle's band on the cells that take
    its sub-steps, which all but a few do"""
    import somdec_util as SU
    wl = SU.option_workload(which, 2049)
    n = wl.state.ncell
    ref, rec, nfail = G.run_oracle(wl)
    assert nfail == 0
    band = _oracle_band(wl, ref)
    for variant in VARIANTS:
        print("case", which, abi.KERNEL_NAMES[variant], flush=True)
        got, ctx = G.run_gpu(wl, variant)
        assert np.all(got["status"] == 0)
        same = got["num_sub_steps"][0] == ref["num_sub_steps"][0]
        assert (~same).sum() <= max(2, n // 1000)
        for f in FIELDS:
            err = np.abs(got[f] - ref[f])
            assert not (err > 1e-8 * np.abs(ref[f]) + band[f])[:, same].any(), f
