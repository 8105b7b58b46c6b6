"""The split of P^T that an APOLLO workspace keeps from step to step.

Bound on g_low, u = 2^-24: the accumulator's rounding of at most six products to an element
(fp32 G in three terms), 6 (K + 2) u sum |g||p|.
"""
import ctypes

import numpy as np
import pytest
import torch

U = 2.0 ** -24


def _step(L, nat, dtype, p, g, pt, ws, v, rank, fresh):
    t = nat.ApolloTensor()
    t.param, t.grad, t.rows, t.cols = p.data_ptr(), g.data_ptr(), p.shape[0], p.shape[1]
    t.proj_t, t.rank, t.v_fp32, t.workspace = pt.data_ptr(), rank, v.data_ptr(), ws.data_ptr()
    rc = L.a8_apollo_step(nat.dtype_code(dtype), 0, ctypes.byref(t), 1, fresh, 0.001, 0.0, 0, 1e-6, -40.0, 0, 2048,
                          8, 0, 0, 32, 1, 1.0, 0, 0, 0.01, 0.0, 1e-3, 1e-3, 0, 0, 1.0, 0.0, 0, 0,
                          torch.cuda.current_stream().cuda_stream)
    nat.check(rc, "a8_apollo_step")


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rank", [((384, 256), 256), ((256, 400), 256), ((300, 290), 64)])
@pytest.mark.parametrize("order", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
def test_one_split_serves_every_gradient_type(shape, rank, order):
    """proj_fresh says that P^T changed, and nothing else: one workspace takes bf16 and fp32
    gradients in turn with the split made at the first call."""
    print(f"[apollo split] {shape} r={rank} {order}", flush=True)
    from adafactor8bit import _native as nat
    L = nat.lib()
    gen = torch.Generator().manual_seed(5)
    right = shape[0] >= shape[1]
    pt = (torch.randn((shape[1], rank) if right else (rank, shape[0]), generator=gen) / rank ** 0.5).cuda()
    ws = torch.full((int(L.a8_apollo_workspace_floats(*shape, rank, 1)),), float("nan"), device="cuda")
    low = (shape[0], rank) if right else (rank, shape[1])
    v = torch.zeros(low, device="cuda")
    P = pt.double().cpu().numpy()
    for i, dt in enumerate(order + order):
        g = torch.randn(shape, generator=gen).to(dt)
        p = torch.zeros(shape, dtype=dt, device="cuda")
        gd = g.cuda()
        _step(L, nat, dt, p, gd, pt, ws, v, rank, int(i == 0))
        torch.cuda.synchronize()
        a, b = (g.double().numpy(), P) if right else (P, g.double().numpy())
        got = ws[:low[0] * low[1]].reshape(low).double().cpu().numpy()
        assert np.all(np.abs(got - a @ b) <= 6 * (min(shape) + 2) * U * (np.abs(a) @ np.abs(b))), (i, dt)
