"""Factored steps of matrices whose rows hold 4 GB and more: the tiles address a row by 32-bit
byte offsets, so these take element loads and flat update units.  One step
against 64 bits in the first and the last columns (rtol 1e-5)."""
import pytest
import torch

COLS = (1 << 30) + 1003


@pytest.mark.gpu
@pytest.mark.parametrize("beta1", [None, 0.9])
def test_rows_of_four_gigabytes(beta1):
    print(f"[factored wide rows] {beta1}", flush=True)
    from adafactor8bit import Adafactor8Bit
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of device memory")
    g = torch.empty((2, COLS), device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(6)
    step = 1 << 26
    rows = torch.zeros(2, dtype=torch.float64, device="cuda")
    for a in range(0, COLS, step):
        x = torch.randn((2, min(step, COLS - a)), device="cuda", generator=gen)
        x[1] *= 3.0
        g[:, a:a + step] = x
        rows += x.double().square().sum(1)
    p = torch.nn.Parameter(torch.zeros((2, COLS), device="cuda"))
    p.grad = g
    opt = Adafactor8Bit([p], lr=1e-3, beta1=beta1, beta2=None, beta2_decay=-0.8, beta3=None, factored=True, d=0.0,
                        relative_step=False, scale_parameter=False, v_quant_type="fp32", m_quant_type="fp32")
    opt.step()
    torch.cuda.synchronize()
    row = rows / COLS
    for lo in (0, COLS // 2, (1 << 30) - 1024, COLS - 64):
        x = g[:, lo:lo + 64].double()
        col = x.square().mean(0)
        u = (x if beta1 is None else 0.1 * x) / (row / row.mean()).sqrt()[:, None] / col.sqrt()
        torch.testing.assert_close(p.detach()[:, lo:lo + 64].double(), -1e-3 * u, rtol=1e-5, atol=1e-9)
