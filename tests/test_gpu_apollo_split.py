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


def _project(shape, rank, g, pt):
    """g_low and its float64 value, from bf16 g and P^T as given."""
    from adafactor8bit import _native as nat
    L = nat.lib()
    right = shape[0] >= shape[1]
    low = (shape[0], rank) if right else (rank, shape[1])
    ws = torch.full((int(L.a8_apollo_workspace_floats(*shape, rank, 1)),), float("nan"), device="cuda")
    v, p = torch.zeros(low, device="cuda"), torch.zeros(shape, dtype=torch.bfloat16, device="cuda")
    _step(L, nat, torch.bfloat16, p, g, pt, ws, v, rank, 1)
    torch.cuda.synchronize()
    a, b = (g.double(), pt.double()) if right else (pt.double(), g.double())
    return ws[:low[0] * low[1]].view(low).double(), a @ b, a.abs() @ b.abs()


KINDS = ["normal", "zeros", "heavy", "one-signed", "log-uniform", "first slab"]


def _draw(shape, kind, gen):
    g = torch.randn(shape, device="cuda", generator=gen)
    if kind == "zeros":
        g *= torch.rand(shape, device="cuda", generator=gen) >= 0.05
    elif kind == "heavy":
        g = g ** 3
    elif kind == "one-signed":
        g = g.abs()
    elif kind == "log-uniform":
        g = torch.sign(g) * torch.exp2(40.0 * torch.rand(shape, device="cuda", generator=gen) - 40.0)
    elif kind == "first slab":   # products of single elements: P's own rounding shows
        t = g if shape[0] >= shape[1] else g.t()
        t[:, 32:] = 0.0
        t[:, :32] *= torch.eye(32, device="cuda")[torch.arange(t.shape[0], device="cuda") % 32]
    return (g * 1e-3).to(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [32, 47, 64, 256, 2048, 8192])
@pytest.mark.parametrize("left", [False, True])
@pytest.mark.parametrize("kind", KINDS)
def test_two_fp16_terms_err_no_more_than_three_bf16_terms(K, left, kind):
    """g_low's rms error against 64 bits, of its rms: the fp16 tiles against the bf16 ones, which
    the same P^T times 2^20 (an exact factor, out of the fp16 split's range) takes.  Channels of a
    single product show P's own rounding: at most half a unit of fp32, 2^-24 of their rms."""
    print(f"[apollo split error] K={K} left={left} {kind}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(K)
    shape = (512, K) if K <= 512 else (K, K)
    if left:
        shape = (K, max(512, K + 1))
    pt = torch.randn((K, 256) if not left else (256, K), device="cuda", generator=gen) / 16.0
    g = _draw(shape, kind, gen)
    err = []
    for f in (1.0, 2.0 ** 20):
        low, ref, _ = _project(shape, 256, g, pt * f)
        err.append(float((low - ref).square().mean().sqrt() / ref.square().mean().sqrt()))
    print(f"  {err[0]:.3g} {err[1]:.3g}", flush=True)
    assert err[0] <= (2.0 ** -24 if kind == "first slab" else err[1]), err


@pytest.mark.gpu
@pytest.mark.parametrize("power", [-60, -12, -5, -4, 0, 1, 2, 3, 20, 60])
@pytest.mark.parametrize("shape", [(300, 256), (256, 300)])
def test_projection_matrix_of_any_size(shape, power):
    """P^T times a power of two, in and out of the fp16 split's range and at both ends of it;
    an element far above the others.  Bound: three terms, and below 2^-2 of the scaled
    range 2^-25, which is 2^-35 of the largest element at least."""
    print(f"[apollo split range] {shape} 2^{power}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(9)
    g = _draw(shape, "normal", gen)
    for spike in (False, True):
        pt = torch.randn((256, 256), device="cuda", generator=gen) / 16.0
        if spike:
            pt[17, 100] = 2.0 ** 12
        low, ref, mag = _project(shape, 256, g, pt * 2.0 ** power)
        floor = 2.0 ** -35 * float(pt.abs().max()) * 2.0 ** power * float(g.double().abs().max()) * 256
        assert torch.all((low - ref).abs() <= 3 * 258 * U * mag + floor), (spike, float(((low - ref).abs() / mag).max()))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(512, 384), (384, 640)])
def test_split_depends_on_the_projection_alone(shape):
    """A run whose P^T the device drew, and fresh optimizers, capturable and default, that load it
    from a checkpoint: the next steps have the same bits.  The gradient holds one element per
    channel, so that every term of P's split shows in g_low."""
    print(f"[apollo split history] {shape}", flush=True)
    from adafactor8bit import Adafactor8Bit
    from test_gpu_apollo import C4_KW, _ws
    kw = dict(C4_KW, apollo_update_proj_gap=3)
    gen = torch.Generator(device="cuda").manual_seed(11)
    pa = torch.nn.Parameter(torch.zeros(shape, dtype=torch.bfloat16, device="cuda"))
    oa = Adafactor8Bit([pa], **dict(kw, capturable=True))
    for _ in range(5):   # the projection is drawn anew at step 4
        pa.grad = _draw(shape, "normal", gen)
        oa.step()
    runs = [(pa, oa)]
    for capturable in (True, False):
        p = torch.nn.Parameter(pa.detach().clone())
        o = Adafactor8Bit([p], **dict(kw, capturable=capturable))
        o.load_state_dict(oa.state_dict())
        runs.append((p, o))
    g = _draw(shape, "first slab", gen)
    for p, o in runs:
        p.grad = g
        o.step()
    torch.cuda.synchronize()
    n = max(shape) * 256
    for p, o in runs[1:]:
        assert torch.equal(torch.from_numpy(_ws(oa, pa)[:n]), torch.from_numpy(_ws(o, p)[:n]))
        assert torch.equal(pa, p)
