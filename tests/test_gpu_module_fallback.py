"""A network whose run-time module does not compile keeps the team kernels: the
SomDec step and the residual and Jacobian block ran without a module before
they had one.  The compilation is made to fail from outside, by an option the
run-time compiler takes from its environment, in a process of its own (the
compiler reads that environment once)."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.gpu
def test_failed_modules_leave_the_team_kernels():
    env = dict(os.environ, HIPRTC_COMPILE_OPTIONS_APPEND="-DNet=0x")
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], env=env, timeout=110,
                       capture_output=True, text=True, cwd=HERE)
    assert r.returncode == 0 and "teams agree" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


def main():
    sys.path.insert(0, HERE)
    import conftest  # noqa: F401  (import paths)
    import numpy as np
    import torch
    from pfchem import abi, workloads
    from pfchem.lib import Context, DeviceState
    import gpu_util as G
    from test_gpu_residual import DT, _case
    wl = workloads.somdec_workload(300)
    for variant in (abi.KERNEL_BATCHED_FP64, abi.KERNEL_BATCHED_MIXED):
        got, ctx = G.run_gpu(wl, variant)
        team, _ = G.run_gpu(wl, variant, lanes=16, block=128)
        assert np.all(got["status"] == 0)
        for f in ("num_sub_steps", "num_iterations", "pri_molal", "total", "immobile"):
            assert np.array_equal(got[f], team[f]), f
        again, _ = G.run_gpu(wl, variant, ctx=ctx)
        assert np.array_equal(again["pri_molal"], got["pri_molal"])
        assert not ctx.try_set_launch(variant, 1, 256, 0, 1)  # refused: there is no kernel
    wl, st, fixed, fimm = _case("calcite", 300)
    ctx = Context(wl.net, wl.opt)
    fx = torch.from_numpy(np.ascontiguousarray(fixed)).cuda()
    res, jac = ctx.residual(DeviceState(st), fx, None, DT)
    again, _ = ctx.residual(DeviceState(st), fx, None, DT, jacobian=False)
    torch.cuda.synchronize()
    assert torch.equal(res, again) and bool(torch.isfinite(jac).all())
    assert float(jac.abs().max()) > 0.0
    print("teams agree", flush=True)


if __name__ == "__main__":
    main()
