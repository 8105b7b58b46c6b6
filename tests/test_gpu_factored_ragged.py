"""Factored Adafactor and CAME on matrices whose rows start anywhere: column counts at the
edges of the 4-column windows, of a wave's 256 columns and of the 1024-column tiles, and fewer
than four columns; without momentum, with fp32 and with coded momentum (blocks straddling rows,
an odd number of nibbles), against the exact-reduction oracle.

Tolerances: the codes of one step from a zero state are the oracle's except on ties of a sum
rounded once on either side (at most one code of a vector, by one step); parameters rtol 1e-5 plus
1e-4 of the largest displacement (the bar of test_gpu_factored_shapes).  Stochastic rounding: a
step's bf16 parameters are sr_round_bf16 of the fp32 step's values but for elements whose fp32
value differs in its last bits (at most 1%, by one bf16 step).
"""
import numpy as np
import pytest
import torch

from inputs import make_grad, make_param

SHAPES = [(5, 1), (130, 2), (70, 3), (64, 4), (33, 5), (40, 255), (300, 257), (35, 1021), (66, 1022), (31, 1023),
          (64, 1025), (97, 1030), (2, 40, 131)]
ADAFACTOR = dict(beta1=None, beta2=None, beta2_decay=-0.8, beta3=None, factored=True, relative_step=False, lr=1e-2,
                 block_size=128, v_quant_type="al8", d=1.0, min_8bit_size=64)
CAME = dict(beta1=0.9, beta2=0.999, beta2_decay=None, beta3=0.9999, factored=True, relative_step=False,
            scale_parameter=False, scale_weight_decay=False, d=1.0, eps_came=1e-16, lr=1e-3, block_size=256,
            m_block_size=32, v_quant_type="al8", min_8bit_size=64)
CASES = {"plain": ADAFACTOR, "fp32_m": dict(CAME, m_quant_type="fp32"), "uf8": dict(CAME, m_quant_type="uf8"),
         "uf4": dict(CAME, m_quant_type="uf4"), "d4_fira": dict(CAME, m_quant_type="d4", enable_fira_for_adafactor=True)}


def _grad(s, i, t):
    g = make_grad(s, i, t, 17)
    g.view(-1)[::7] = 0.0
    return g


@pytest.mark.gpu
@pytest.mark.parametrize("case", sorted(CASES))
def test_ragged_columns_match_oracle(case):
    import oracle.fallback as F
    from adafactor8bit import Adafactor8Bit
    kw = CASES[case]
    pc = [torch.nn.Parameter(make_param(s, i, 17)) for i, s in enumerate(SHAPES)]
    p0 = [p.detach().clone() for p in pc]
    pg = [torch.nn.Parameter(p.detach().clone().cuda()) for p in pc]
    oc, og = F.OracleOptimizer(pc, **kw), Adafactor8Bit(pg, **kw)
    old = F.set_exact_reductions(True)
    try:
        for t in (1, 2):
            for i, (a, b) in enumerate(zip(pc, pg)):
                a.grad = _grad(SHAPES[i], i, t)
                b.grad = a.grad.cuda()
            oc.step()
            og.step()
            torch.cuda.synchronize()
            for i, (a, b) in enumerate(zip(pc, pg)):
                for k, v in oc.state[id(a)].items():
                    if not (torch.is_tensor(v) and k.endswith("_q")):
                        continue
                    x = og.state[b][k].cpu().numpy().reshape(-1).astype(np.int64)
                    y = v.numpy().reshape(-1).astype(np.int64)
                    far = (x != y).sum()
                    assert far <= 1 + 1e-3 * y.size, (case, t, SHAPES[i], k, int(far))
                ref, mine = a.detach().numpy(), b.detach().cpu().numpy()
                disp = float(np.abs(ref - p0[i].numpy()).max())
                close = np.abs(mine - ref) <= 1e-5 * np.abs(ref) + 1e-8 + 1e-4 * disp
                assert (~close).mean() <= 1e-3, (case, t, SHAPES[i], float((~close).mean()))
                np.testing.assert_allclose(mine, ref, rtol=2e-3, atol=1e-8 + 2e-2 * disp, err_msg=f"{case} {SHAPES[i]}")
    finally:
        F.set_exact_reductions(old)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["plain", "uf8"])
def test_ragged_columns_stochastic_rounding(case):
    from adafactor8bit import Adafactor8Bit
    from oracle.sr import sr_round_bf16
    kw = dict(CASES[case], scale_parameter=False)
    p16 = [torch.nn.Parameter(make_param(s, i, 18).to(torch.bfloat16).cuda()) for i, s in enumerate(SHAPES)]
    p32 = [torch.nn.Parameter(p.detach().float()) for p in p16]
    o16, o32 = Adafactor8Bit(p16, **dict(kw, stochastic_round_writeback=True)), Adafactor8Bit(p32, **kw)
    for i, (a, b) in enumerate(zip(p16, p32)):
        a.grad = _grad(SHAPES[i], i, 1).to(torch.bfloat16).cuda()
        b.grad = a.grad.float()
    o16.step()
    o32.step()
    for i, (a, b) in enumerate(zip(p16, p32)):
        want = sr_round_bf16(b.detach().cpu().numpy().reshape(-1), seed=int(o16.state[a]["sr_seed"]), step=1)
        got = a.detach().cpu().view(torch.int16).numpy().reshape(-1).astype(np.int64) & 0xFFFF
        want = np.asarray(want).astype(np.int64) & 0xFFFF
        assert (got != want).sum() <= 1 + 0.01 * got.size, (case, SHAPES[i])
        assert np.abs(got - want).max() <= 1, (case, SHAPES[i])


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["plain", "fp32_m", "uf8"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float64])
def test_ragged_columns_of_every_type(case, dtype):
    """fp16, bf16 (rounded to nearest) and fp64 parameters, gradients with infinities and NaN: the
    step of the fp32 twin (same values, non-finite gradients zero).  fp16 and bf16: to half a unit
    of the type and fp32's 1e-5 of the update, rounded once; fp64: its gradient is that of the
    twin exactly, its arithmetic fp32 but for the last addition."""
    from adafactor8bit import Adafactor8Bit
    kw = dict(CASES[case], scale_parameter=False)
    eps = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float64: 2.0 ** -24}[dtype]
    pa = [torch.nn.Parameter(make_param(s, i, 19).to(torch.bfloat16).to(dtype).cuda()) for i, s in enumerate(SHAPES)]
    pb = [torch.nn.Parameter(p.detach().float()) for p in pa]
    start = [p.detach().clone() for p in pb]
    oa, ob = Adafactor8Bit(pa, **kw), Adafactor8Bit(pb, **kw)
    for i, (a, b) in enumerate(zip(pa, pb)):
        g = (_grad(SHAPES[i], i, 1) * 16.0).to(torch.bfloat16).float().cuda()
        f = g.view(-1)
        f[3::11], f[4::13], f[1::17] = float("inf"), float("nan"), -float("inf")
        a.grad = g.to(dtype)
        b.grad = torch.nan_to_num(g, nan=0.0, posinf=0.0, neginf=0.0)
    oa.step()
    ob.step()
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(pa, pb)):
        x, y = a.detach().double(), b.detach().double()
        assert torch.isfinite(x).all()
        tol = eps * y.abs() + 1e-5 * (y - start[i].double()).abs() + (6e-8 if dtype == torch.float16 else 0.0)
        assert torch.all((x - y).abs() <= tol), (case, dtype, SHAPES[i], float(((x - y).abs() - tol).max()))
        for k, v in ob.state[b].items():
            if torch.is_tensor(v) and v.dtype == torch.uint8:
                assert torch.equal(v, oa.state[a][k]), (case, dtype, SHAPES[i], k)
