"""A matrix's factored step does not depend on what else its group holds.

Groups above 2^28 elements take statistics tiles of 256 rows, smaller ones of 32, so a small
matrix is stepped alone and beside one of 272 M elements.  The order of the sums over rows
(the column statistics, sum p^2) shows in a column of 1, 2^-24 and 254 times 2^-54: summed
row by row the small ones are lost, and the sum is the tie between 1 and 1 + 2^-23; added up
in groups first they lift it above the tie.
"""
import pytest
import torch

BIG = (16640, 16384)
KW = dict(block_size=256, m_block_size=256, factored=True, relative_step=False, lr=1e-3, d=1.0, eps=(1e-30, 1e-3))
ALGO = {"adafactor": dict(beta1=None, beta2=None, beta2_decay=-0.8, beta3=None, scale_parameter=True),
        "came": dict(beta1=0.9, beta2=0.999, beta3=0.9999, beta2_decay=None, eps_came=1e-16, scale_parameter=True)}
_big = {}


def _run(shape, fill, dtype, beside, steps, **kw):
    from adafactor8bit import Adafactor8Bit
    p = torch.nn.Parameter(fill(shape, 0).to("cuda", dtype))
    ps = [p]
    if beside:
        if dtype not in _big:
            _big.clear()
            _big[dtype] = (torch.ones(BIG, device="cuda", dtype=dtype), torch.full(BIG, 1e-3, device="cuda", dtype=dtype))
        ps.append(torch.nn.Parameter(_big[dtype][0]))
        ps[1].grad = _big[dtype][1]
    opt = Adafactor8Bit(ps, **dict(KW, **kw))
    for t in range(1, steps + 1):
        p.grad = fill(shape, t).to("cuda", dtype)
        opt.step()
    torch.cuda.synchronize()
    return p.detach(), opt.state[p]


def _same(a, b):
    assert torch.equal(a[0], b[0]), "parameter"
    for k, v in a[1].items():
        if torch.is_tensor(v):
            assert torch.equal(v, b[1][k]), k


def _lift(shape, t):
    x = torch.full(shape, 2.0 ** -27)
    x[0], x[1] = 1.0, 2.0 ** -12
    if t == 0:
        x[:, 1:] = 0.0   # sum p^2 in one lane
    return x


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [32, 40, 256, 257, 1300])
def test_sums_over_rows_keep_their_order_in_any_group(rows):
    print(f"[factored group order] {rows}", flush=True)
    kw = dict(ALGO["adafactor"], v_quant_type="fp32")
    _same(*[_run((rows, 160), _lift, torch.float32, beside, 1, **kw) for beside in (False, True)])


@pytest.mark.gpu
@pytest.mark.parametrize("algo", sorted(ALGO))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(33, 2050), (513, 1283), (2, 300, 257), (1025, 300), (2305, 64), (33000, 36), (270000, 4)])
def test_a_matrix_steps_the_same_in_a_small_and_a_large_group(algo, dtype, shape):
    print(f"[factored group] {algo} {dtype} {shape}", flush=True)
    gen = torch.Generator().manual_seed(4)
    data = {t: torch.randn(shape, generator=gen) * (0.02 if t == 0 else 1e-3) for t in range(3)}
    kw = dict(ALGO[algo], stochastic_round_writeback=dtype == torch.bfloat16)
    torch.manual_seed(0)
    runs = []
    for beside in (False, True):
        torch.manual_seed(0)
        runs.append(_run(shape, lambda s, t: data[t], dtype, beside, 2, **kw))
    _same(*runs)
