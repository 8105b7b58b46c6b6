"""g_low and the channel norms of APOLLO's bf16 projection kernels against 64 bits.

Wide tiles (ranks that are a multiple of 256) hold both operands as scaled fp16: G from a
scale that two slabs of each channel suggest, P^T as two terms.  The inputs below take every
way through that: the usual one, channels that are zero where the scale looks, values far
above it, values that are not finite, and the ends of the exponent range.  Narrow tiles are
taken at both heights and at every split of the reduction over their waves.  The low-rank
second moment is decoded through a table or directly, by its block size.

Bounds, u = 2^-24: the accumulator's rounding of T K products, T terms of P^T, is at most
T (K + 2) u sum |g||p|; the fp16 split adds one unit of an element's 24th bit (2 u |p|), and
values below the fp16 range 2^-28 of their channel's largest and 2^-35 of P^T's.  A channel's
squares: 16-term fp32 sums (16 u), their sum in 64 bits, and the norm rounded and squared (3 u).
"""
import numpy as np
import pytest
import torch

from test_gpu_apollo import C4_KW, _ws

U = 2.0 ** -24


def _low(shape, rank, g):
    from adafactor8bit import Adafactor8Bit
    p = torch.nn.Parameter(torch.zeros(shape, dtype=torch.bfloat16, device="cuda"))
    opt = Adafactor8Bit([p], **dict(C4_KW, apollo_rank=rank))
    p.grad = g.cuda()
    opt.step()
    torch.cuda.synchronize()
    pt = opt.state[p]["apollo_proj_matrix_T"].double().cpu().numpy()
    G = np.where(np.isfinite(g.double().numpy()), g.double().numpy(), 0.0)
    right = shape[0] >= shape[1]
    out = (shape[0], rank) if right else (rank, shape[1])
    ws = _ws(opt, p)
    n = out[0] * out[1]
    return right, G, pt, ws[:n].reshape(out).astype(np.float64), ws[2 * n:2 * n + max(shape)].astype(np.float64)


def _gradient(shape, kind, seed):
    gen = torch.Generator().manual_seed(seed)
    g = torch.randn(shape, generator=gen)
    ch, k = (0, 1) if shape[0] >= shape[1] else (1, 0)
    at = torch.arange(shape[ch])
    t = g if ch == 0 else g.t()      # channels first
    if kind == "zeros":              # some channels, and the first slab of others
        t[at % 7 == 0] = 0.0
        t[at % 5 == 1, :32] = 0.0
        t[at % 5 == 1, shape[k] // 64 * 32:shape[k] // 64 * 32 + 32] = 0.0
        t[at % 11 == 3] = 0.0        # zero but for one element, off the looked-at slabs where K allows it
        t[at % 11 == 3, 101] = 1.0
    elif kind == "outliers":
        t[at, (40 + 3 * at) % shape[k]] *= 2.0 ** 20
    elif kind == "nonfinite":
        t[at[::3], (7 * at[::3]) % shape[k]] = float("inf")
        t[at[1::3], (5 * at[1::3]) % shape[k]] = float("nan")
    elif kind == "tiny":
        t *= 2.0 ** -120
    elif kind == "spread":
        t *= torch.exp2((at % 81 - 40).float())[:, None]
    return g.to(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "zeros", "outliers", "nonfinite", "tiny", "spread"])
@pytest.mark.parametrize("shape,rank", [((256, 256), 256), ((513, 264), 256), ((768, 544), 512), ((300, 290), 256),
                                        ((288, 512), 256), ((264, 1001), 256), ((544, 700), 512)])
def test_wide_tiles_against_64_bits(shape, rank, kind):
    print(f"[apollo wide] {shape} r={rank} {kind}", flush=True)
    right, G, pt, low, nsq = _low(shape, rank, _gradient(shape, kind, 21))
    a, b = (G, pt) if right else (pt, G)
    K = min(shape)
    top = np.abs(G).max(axis=1, keepdims=True) if right else np.abs(G).max(axis=0, keepdims=True)
    sp = np.abs(pt).sum(axis=0, keepdims=True) if right else np.abs(pt).sum(axis=1, keepdims=True)
    sg = np.abs(G).sum(axis=1, keepdims=True) if right else np.abs(G).sum(axis=0, keepdims=True)
    bound = (2 * (K + 2) + 2) * U * (np.abs(a) @ np.abs(b)) + 2.0 ** -28 * top * sp + 2.0 ** -35 * np.abs(pt).max() * sg
    err = np.abs(low - a @ b)
    assert np.all(err <= bound + 1e-44), float((err / (bound + 1e-44)).max())
    if kind != "tiny":               # its squares are below the fp32 range
        exact = (G * G).sum(axis=1 if right else 0)
        assert np.all(np.abs(nsq - exact) <= 19 * U * exact)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [200, 49250])    # 32 rows to a tile, and 96 where there are enough of them
@pytest.mark.parametrize("cols,rank", [(72, 32), (136, 32), (135, 64), (154, 65), (153, 33), (130, 130)])
def test_narrow_tiles_against_64_bits(rows, cols, rank):
    for shape in ((rows, cols), (cols, rows)):
        print(f"[apollo narrow] {shape} r={rank}", flush=True)
        right, G, pt, low, nsq = _low(shape, rank, _gradient(shape, "plain", 22))
        a, b = (G, pt) if right else (pt, G)
        err = np.abs(low - a @ b)
        bound = 3 * (cols + 2) * U * (np.abs(a) @ np.abs(b))
        assert np.all(err <= bound), float((err / bound).max())
        exact = (G * G).sum(axis=1 if right else 0)
        assert np.all(np.abs(nsq - exact) <= 19 * U * exact)


@pytest.mark.gpu
@pytest.mark.parametrize("quant,top", [("al8", 255), ("al16", 65535)])
@pytest.mark.parametrize("block", [256, 512, 1024, 2048])
def test_low_rank_second_moment_decode(quant, top, block):
    """The second step's V from the first one's codes, in units of 2048 elements and a part of one:
    the block's range to fp32 rounding of its logarithms (below 64: 2^-18, twice), the codes to a tie."""
    print(f"[apollo v] {quant} {block}", flush=True)
    from adafactor8bit import Adafactor8Bit
    shape, rank = (1001, 40), 37
    gen = torch.Generator().manual_seed(block)
    p = torch.nn.Parameter(torch.zeros(shape, device="cuda"))
    opt = Adafactor8Bit([p], **dict(C4_KW, apollo_rank=rank, block_size=block, v_quant_type=quant))
    v = None
    for _ in range(2):
        p.grad = (torch.randn(shape, generator=gen) * 1e-3).cuda()
        opt.step()
        torch.cuda.synchronize()
        st = opt.state[p]
        q = st["v_low_q"].cpu().numpy().reshape(-1).view(np.uint8 if top == 255 else np.uint16).astype(np.float64)
        sc, lo = (st[k].cpu().numpy().astype(np.float32).repeat(block) for k in ("v_low_scale", "v_low_min_log"))
        n = shape[0] * rank
        if v is None:
            x = (q.astype(np.float32) - np.float32(1)) * sc / np.float32(top - 1) + lo
            v = np.where(q == 0, 0.0, np.exp2(x.astype(np.float64)).astype(np.float32))[:n].astype(np.float64)
    g = _ws(opt, p)[:n]
    w = np.float64(np.float32(1.0 - 0.999))
    v = np.pad(v + w * ((g * g).astype(np.float32) - v.astype(np.float32)), (0, q.size - n))
    logs = np.log2(np.where(v > 0, v, 1.0)).reshape(-1, block)
    nz = (v > 0).reshape(-1, block)
    least = np.maximum(np.where(nz, logs, np.inf).min(1), 2 * np.log2(1e-6))
    most = np.where(nz, logs, -np.inf).max(1)
    assert np.abs(lo[::block] - least).max() <= 2.0 ** -17
    assert np.abs(sc[::block] - (most - least)).max() <= 2.0 ** -17
    want = np.clip(np.rint((logs - lo[::block, None]) / sc[::block, None] * (top - 1)) + 1, 1, top)
    off = np.abs(q - np.where(nz, want, 0).reshape(-1))
    assert off.max() <= 1 and (off > 0).mean() <= (1e-4 if top == 255 else 0.02)


@pytest.mark.gpu
@pytest.mark.parametrize("capturable", [False, True])
@pytest.mark.parametrize("order", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
def test_projection_split_follows_the_dtype(order, capturable):
    """A parameter that changes between bf16 and fp32 has P^T split anew: the two kernels read
    different forms of it.  Bound: the accumulator's, six products to an element at most."""
    print(f"[apollo dtype] {order} {capturable}", flush=True)
    from adafactor8bit import Adafactor8Bit
    p = torch.nn.Parameter(torch.zeros((384, 256), device="cuda", dtype=order[0]))
    opt = Adafactor8Bit([p], **dict(C4_KW, capturable=capturable))
    for t, dt in enumerate(order + order):
        p.grad = None
        p.data = p.data.to(dt)
        g = torch.randn((384, 256), generator=torch.Generator().manual_seed(t)).to(dt)
        p.grad = g.cuda()
        opt.step()
        torch.cuda.synchronize()
        pt = opt.state[p]["apollo_proj_matrix_T"].double().cpu().numpy()
        G = g.double().numpy()
        low = _ws(opt, p)[:384 * 256].reshape(384, 256).astype(np.float64)
        assert np.all(np.abs(low - G @ pt) <= 6 * 258 * U * (np.abs(G) @ np.abs(pt)))


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rank", [((300, 2048), 256), ((515, 1000), 512)])
@pytest.mark.parametrize("slab", [0, 1, 2, 17, 30, -1])
@pytest.mark.parametrize("kind", ["large", "inf", "late"])
def test_wide_tiles_leave_fp16_at_any_slab(shape, rank, slab, kind):
    """One channel of a tile has an element that its fp16 scale does not hold in one slab: from
    there on the tile takes the three bf16 terms.  late: the channel is zero until then.  Bound:
    three terms' roundings, and the fp16 slabs' floor (above)."""
    print(f"[apollo leave fp16] {shape} r={rank} slab {slab} {kind}", flush=True)
    K = shape[1]
    at = (slab if slab >= 0 else (K - 1) // 32) * 32 + (5 if slab >= 0 else 0)
    g = torch.randn(shape, generator=torch.Generator().manual_seed(31))
    if kind == "late":
        g[7, :at] = 0.0
        g[7, K // 64 * 32:K // 64 * 32 + 32] = 0.0
    g[7, at] = {"large": 2.0 ** 14, "inf": float("inf"), "late": 1.0}[kind]
    for t in (g, g.t().contiguous()):
        right, G, pt, low, nsq = _low(tuple(t.shape), rank, t.to(torch.bfloat16))
        a, b = (G, pt) if right else (pt, G)
        ax = 1 if right else 0
        top, sp = np.abs(G).max(axis=ax, keepdims=True), np.abs(pt).sum(axis=1 - ax, keepdims=True)
        bound = 3 * (K + 2) * U * (np.abs(a) @ np.abs(b)) + 2.0 ** -28 * top * sp
        err = np.abs(low - a @ b)
        assert np.all(err <= bound), float((err / bound).max())
        exact = (G * G).sum(axis=ax)
        assert np.all(np.abs(nsq - exact) <= 19 * U * exact)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(32000, 2048), (2048, 32000)])
@pytest.mark.parametrize("value", [2.0 ** 17, float("inf")])
def test_values_off_the_fp16_scale_cost_no_second_projection(shape, value):
    """One element per tile that its channel's fp16 scale does not hold (GRAD x 2^17), or that is
    not finite, in a random slab: the tile goes on from there, so the step takes at most the
    share of it that three terms take more than two (half of a third, measured 8%); multiplying
    the tile twice took 35% more.  The least of five interleaved times each."""
    print(f"[apollo off scale] {shape} {value}", flush=True)
    from adafactor8bit import Adafactor8Bit
    gen = torch.Generator(device="cuda").manual_seed(3)
    ps = [torch.nn.Parameter(torch.zeros(shape, dtype=torch.bfloat16, device="cuda")) for _ in range(4)]
    opt = Adafactor8Bit(ps, **C4_KW)
    plain = [torch.randn(shape, device="cuda", generator=gen).mul_(1e-3).to(torch.bfloat16) for _ in ps]
    odd = [g.clone() for g in plain]
    for g in odd:
        t = g if shape[0] >= shape[1] else g.t()
        at = torch.arange(0, max(shape), 256, device="cuda")
        t[at, torch.randint(64, min(shape), at.shape, device="cuda", generator=gen)] = 1e-3 * value
    best = {}
    for rep in range(6):
        for name, gs in (("plain", plain), ("odd", odd)):
            for p, g in zip(ps, gs):
                p.grad = g
            opt.step()
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(4):
                opt.step()
            b.record()
            torch.cuda.synchronize()
            if rep:
                best[name] = min(best.get(name, 1e9), a.elapsed_time(b))
    print(best, flush=True)
    assert best["odd"] <= 1.22 * best["plain"], best


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["zeros", "outliers", "nonfinite", "tiny", "spread"])
@pytest.mark.parametrize("cols,rank", [(154, 32), (154, 65), (135, 64), (130, 130)])
def test_narrow_tiles_of_uneven_gradients(cols, rank, kind):
    """The narrow tiles' exact split, shared by one, two and four waves, on gradients of every kind."""
    for shape in ((200, cols), (cols, 200)):
        print(f"[apollo narrow] {shape} r={rank} {kind}", flush=True)
        right, G, pt, low, nsq = _low(shape, rank, _gradient(shape, kind, 23))
        a, b = (G, pt) if right else (pt, G)
        err = np.abs(low - a @ b)
        assert np.all(err <= 3 * (cols + 2) * U * (np.abs(a) @ np.abs(b)) + 1e-44)
        if kind != "tiny":
            exact = (G * G).sum(axis=1 if right else 0)
            assert np.all(np.abs(nsq - exact) <= 19 * U * exact)
