"""The team kernels read their state descriptor from a 256-slot device ring
filled by stream-ordered copies from pinned host memory; an event recorded
after each launch guards a slot's reuse.  More launches than slots, queued
without synchronizing and alternating between two streams, must each see
their own descriptor: every result equals the same state stepped alone.
The one-lane kernel's steps use the context's hand-over lists and status
scratch: the steps of one stream share a set, a few streams have one each, and
steps that share a set must not interleave on the device, nor steps that do
not wait for each other.  Each launch's work cursors belong to its descriptor
slot."""
import numpy as np
import pytest

from pfchem import abi, workloads
from pfchem.lib import Context, DeviceState

pytestmark = pytest.mark.gpu


def test_more_launches_than_descriptor_slots():
    import torch
    wl = workloads.calcite_workload(ncell=96)
    ctx = Context(wl.net, wl.opt)
    assert ctx.try_set_launch(abi.KERNEL_BATCHED_FP64, 4, 128, 4, 1)
    n = wl.state.ncell
    rng = np.random.default_rng(5)
    hosts = []
    for _ in range(300):
        h = wl.state.copy()
        h["total"][:, :n] *= 1.0 + 0.05 * rng.random((1, n))
        hosts.append(h)
    print("case ring: 300 launches on two streams", flush=True)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    devs = [DeviceState(h) for h in hosts]
    torch.cuda.synchronize()
    for i, d in enumerate(devs):
        ctx.step(d, wl.dt, abi.KERNEL_BATCHED_FP64, stream=streams[i % 2])
    torch.cuda.synchronize()
    for i in list(range(0, 300, 13)) + [299]:
        alone = DeviceState(hosts[i])
        ctx.step(alone, wl.dt, abi.KERNEL_BATCHED_FP64)
        torch.cuda.synchronize()
        a, b = alone.to_host(), devs[i].to_host()
        assert np.all(b["status"][0, :n] == 0), i
        for f in ("pri_molal", "total", "mnrl_volfrac"):
            np.testing.assert_array_equal(b[f][:, :n], a[f][:, :n], err_msg="launch %d %s" % (i, f))


def test_one_lane_steps_on_two_streams_share_the_hand_over_list():
    """mixed one-lane steps alternate between two streams, half of them with
    no status array (the context's status scratch): the FP32 pass, the
    hand-over list and the FP64 passes of one step must not interleave with
    another step's on the device; each launch's answer equals the same state
    stepped alone"""
    import torch
    wl = workloads.random_network_workload(ncell=512, spread=0.5, wmax=1.0)
    ctx = Context(wl.net, wl.opt)
    assert ctx.get_launch(abi.KERNEL_BATCHED_MIXED)["lanes_per_cell"] == 1
    n = wl.state.ncell
    rng = np.random.default_rng(11)
    hosts = []
    for _ in range(40):
        h = wl.state.copy()
        h["total"][:, :n] *= 1.0 + 0.05 * rng.random((1, n))
        hosts.append(h)
    print("case one-lane: 40 mixed launches on two streams", flush=True)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    devs = [DeviceState(h) for h in hosts]
    for i in range(1, 40, 2):
        devs[i].t.pop("status", None)  # these use the context's status scratch
    torch.cuda.synchronize()
    for i, d in enumerate(devs):
        ctx.step(d, wl.dt, abi.KERNEL_BATCHED_MIXED, stream=streams[i % 2])
    torch.cuda.synchronize()
    for i in range(40):
        alone = DeviceState(hosts[i])
        ctx.step(alone, wl.dt, abi.KERNEL_BATCHED_MIXED)
        torch.cuda.synchronize()
        a, b = alone.to_host(), devs[i].to_host()
        assert np.all(a["status"][0, :n] == 0), i
        for f in ("pri_molal", "total", "sec_molal", "mnrl_volfrac"):
            np.testing.assert_array_equal(b[f][:, :n], a[f][:, :n], err_msg="launch %d %s" % (i, f))


@pytest.mark.parametrize("nstream", [3, 7])
def test_one_lane_steps_on_many_streams(nstream):
    """more streams than sets of lists, cells growing from step to step (the
    lists are regrown in between), half the steps without a status array: each
    answer equals the same cells stepped alone"""
    import torch
    wl = workloads.random_network_workload(ncell=700, spread=0.5, wmax=1.0)
    ctx = Context(wl.net, wl.opt)
    streams = [torch.cuda.Stream() for _ in range(nstream)]
    sizes = [40 + 33 * i for i in range(20)]
    hosts = [wl.state.subset(np.arange(n)) for n in sizes]
    devs = [DeviceState(h) for h in hosts]
    for d in devs[::2]:
        d.t.pop("status", None)
    torch.cuda.synchronize()
    print("case one-lane: 20 growing launches on %d streams" % nstream, flush=True)
    for i, d in enumerate(devs):
        ctx.step(d, wl.dt, abi.KERNEL_BATCHED_MIXED, stream=streams[(i * 5) % nstream])
    torch.cuda.synchronize()
    alone = DeviceState(wl.state)
    Context(wl.net, wl.opt).step(alone, wl.dt, abi.KERNEL_BATCHED_MIXED)
    torch.cuda.synchronize()
    want = alone.to_host()
    for n, d in zip(sizes, devs):
        got = d.to_host()
        for f in ("pri_molal", "total", "sec_molal", "mnrl_volfrac", "num_iterations"):
            np.testing.assert_array_equal(got[f][:, :n], want[f][:, :n], err_msg="%d %s" % (n, f))


@pytest.mark.parametrize("which", ["somdec", "calcite"])
def test_steps_on_two_streams_do_not_wait_for_each_other(which):
    """a step queued on one stream behind a long kernel does not hold back the
    step of another stream (several are tried: two streams may share one of the
    device's few hardware queues)"""
    import torch
    wl = workloads.somdec_workload(64) if which == "somdec" else workloads.calcite_workload(64)
    ctx = Context(wl.net, wl.opt)
    a, b = DeviceState(wl.state), DeviceState(wl.state)
    streams = [torch.cuda.Stream() for _ in range(5)]
    for s in streams:  # module and lists exist
        ctx.step(a, wl.dt, abi.KERNEL_BATCHED_FP64, stream=s)
    torch.cuda.synchronize()
    e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    e0.record()
    torch.cuda._sleep(1000000)
    e1.record()
    torch.cuda.synchronize()
    cycles = int(1000000 * 200.0 / max(e0.elapsed_time(e1), 1e-3))  # 200 ms
    overtook = 0
    for other in streams[1:]:
        done = torch.cuda.Event()
        with torch.cuda.stream(streams[0]):
            torch.cuda._sleep(cycles)
        ctx.step(a, wl.dt, abi.KERNEL_BATCHED_FP64, stream=streams[0])
        ctx.step(b, wl.dt, abi.KERNEL_BATCHED_FP64, stream=other)
        done.record(other)
        done.synchronize()
        overtook += not streams[0].query()
        torch.cuda.synchronize()
    print("case two streams: %d of 4 finished while the other waited" % overtook, flush=True)
    assert overtook > 0
