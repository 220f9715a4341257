"""A frame load and its allocation-free backward inside a captured graph: every
replay, with other positions and with eager work of the caller between, gives
what the eager calls give. Bars as for the eager variants: dL/dx bit for bit,
FP64 parameter gradients (atomics in any order) to 1e-12 relative."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from beads_amd import workloads as W
from beads_amd.capi import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reuse", [False, True])
def test_replays_match_eager_calls(reuse):
    w = W.polymer_solvent(n_chains=40, beads_per_chain=20, n_solvent=3000, seed=3, jitter=0.03)
    n_p = 2 * w.n_types * w.n_types + 2 * int(w.bond_k.shape[0])
    gen = torch.Generator(device="cuda").manual_seed(1)
    frames = [torch.tensor(w.positions, device="cuda") + 0.2 * k * torch.randn(
        (w.n, 3), generator=gen, device="cuda") for k in range(5)]
    grads = [torch.randn((w.n, 3), generator=gen, device="cuda") for _ in frames]
    x, g, gx = (torch.empty_like(frames[0]) for _ in range(3))
    gp = torch.empty(n_p, dtype=torch.float64, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with Engine(w) as e, Engine(w) as eager:
        e.set_stream(stream.cuda_stream)

        def step(engine):
            engine.frame_load_async(x.data_ptr(), reuse_list=reuse)
            engine.frame_backward_noalloc(g.data_ptr(), 0.25, gx.data_ptr(), gp.data_ptr())

        x.copy_(frames[0])
        g.copy_(grads[0])
        torch.cuda.synchronize()
        step(e)
        e.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            step(e)
        for k in (1, 2, 0, 4, 3, 1):
            x.copy_(frames[k])
            g.copy_(grads[k])
            gx.fill_(float("nan"))
            gp.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            got_x, got_p = gx.cpu().numpy(), gp.cpu().numpy()
            eager.frame_load(x.data_ptr(), reuse_list=False)
            eager.frame_backward_noalloc(g.data_ptr(), 0.25, gx.data_ptr(), gp.data_ptr())
            eager.synchronize()
            e.synchronize()
            np.testing.assert_array_equal(got_x, gx.cpu().numpy())
            want = gp.cpu().numpy()
            np.testing.assert_allclose(got_p, want, rtol=1e-12, atol=1e-12 * np.abs(want).max())
