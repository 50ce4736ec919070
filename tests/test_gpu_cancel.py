"""ucg_cancel reaches a running solve whatever other handles exist.  A process has a few hardware
queues, and streams share them: a cancel that needed a stream of its own waited behind the solve it
was to stop on some of the handles."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
HANDLES = 20


def test_cancel_reaches_every_handle(tables):
    import torch
    from uclchem_amd import gpu, workloads
    params = workloads.static_cloud_grid(64)[27:28]     # runs for seconds: 2.5e5 steps
    dev = torch.device("cuda:0")
    dp = torch.tensor(params, device=dev)
    dy = torch.zeros((1, tables.neq), dtype=torch.float64, device=dev)
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    stats = torch.zeros((1, 8), dtype=torch.int32, device=dev)
    stream = torch.cuda.current_stream(dev)
    nets = [gpu.Network(tables) for _ in range(HANDLES)]
    late = []
    for k, net in enumerate(nets):
        net.solve_device(dp, dy, status, stats, stream=stream.cuda_stream)
        time.sleep(0.15)
        t0 = time.time()
        net.cancel()
        torch.cuda.synchronize()
        wait = time.time() - t0
        print(f"[cancel] handle {k}: {1e3 * wait:.1f} ms, status {status.item()}, {stats[0, 0].item()} steps", flush=True)
        if status.item() != net.CANCELLED or wait > 0.5:     # 16 steps take under a millisecond
            late.append((k, wait, status.item()))
    assert not late, late
    again = nets[0].solve(workloads.static_cloud_point(1e2))
    assert np.all(again["status"] == 0)
