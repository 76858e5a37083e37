"""Calls captured into a graph and replayed, between the program's own eager
calls: a SomDec step, which runs the team kernel inside a capture whatever ran
before it, and the residual and Jacobian block, whose one-lane module is used
inside a capture once an eager call has loaded it."""
import numpy as np
import pytest

from pfchem import abi, workloads

from test_gpu_residual import DT, _case

pytestmark = pytest.mark.gpu

OUT = ("pri_molal", "total", "immobile", "num_iterations", "num_sub_steps", "status")


def _load(ds, host):
    import torch
    for f, t in ds.t.items():
        t.copy_(torch.from_numpy(host.arrays[f]))


def _outputs(ds):
    import torch
    torch.cuda.synchronize()
    got = ds.to_host()
    return {f: got[f].copy() for f in OUT}


@pytest.mark.parametrize("variant", [abi.KERNEL_BATCHED_FP64, abi.KERNEL_BATCHED_MIXED])
@pytest.mark.parametrize("warm", [False, True], ids=["first-call", "after-eager-calls"])
def test_somdec_step(variant, warm):
    import torch
    from pfchem.lib import Context, DeviceState
    wl = workloads.somdec_workload(1200)
    every = wl.state
    wl.state = every.subset(np.arange(300))
    hosts = [every.subset(np.arange(k, k + 300)) for k in (300, 600, 900)]
    team = Context(wl.net, wl.opt)
    team.set_launch(variant, 16, 128, 4, 1)
    want = []
    for h in hosts:
        ds = DeviceState(h)
        team.step(ds, wl.dt, variant)
        want.append(_outputs(ds))
    ctx = Context(wl.net, wl.opt)
    ds = DeviceState(wl.state)
    if warm:
        ctx.step(ds, wl.dt, variant)
        torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ctx.step(ds, wl.dt, variant)
    eager = DeviceState(wl.state)
    for k, (h, w) in enumerate(zip(hosts, want)):
        _load(ds, h)
        g.replay()
        got = _outputs(ds)
        for f in OUT:
            assert np.array_equal(got[f], w[f]), f
        # a larger eager step between the replays regrows the context's lists
        ctx.step(DeviceState(every.subset(np.arange(400 * (k + 1)))), wl.dt, variant)
        ctx.step(eager, wl.dt, variant)
        torch.cuda.synchronize()


@pytest.mark.parametrize("warm", [False, True], ids=["first-call", "after-eager-calls"])
def test_residual(warm):
    import torch
    from pfchem.lib import Context, DeviceState
    wl, st, fixed, fimm = _case("random15", 130)
    fx = torch.from_numpy(np.ascontiguousarray(fixed)).cuda()
    ctx = Context(wl.net, wl.opt)
    if warm:
        ctx.residual(DeviceState(st), fx, None, DT)
    ds = DeviceState(st)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        res, jac = ctx.residual(ds, fx, None, DT)
    for k in range(3):
        ds.t["pri_molal"].mul_(1.0 + 0.01 * k)
        g.replay()
        torch.cuda.synchronize()
        other = Context(wl.net, wl.opt)
        r, j = other.residual(ds, fx, None, DT)
        torch.cuda.synchronize()
        # the first capture holds the team kernel, the eager call is one-lane
        for a, b in ((res, r), (jac, j)):
            assert float((a - b).abs().max()) <= 1e-9 * float(b.abs().max())
