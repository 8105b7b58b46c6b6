"""The norms of a narrow projection's matrix do not depend on what else its group holds.

Groups of at least 512 right-side tiles take tiles of 96 rows, others of 32, so a matrix is
stepped alone and beside one of 49,664 rows.  The order in which ||G||^2 is summed shows in a
first row whose square lies half a unit of fp32 above one, and two rows of 2^-53 of it: added
to it one by one they are lost, together they lift the sum.
"""
import numpy as np
import pytest
import torch


def _rows():
    """A first row (bf16 values) of sum of squares x + half a unit, with a root that tells x from x + a unit."""
    for b in range(1, 128):
        x = np.float32(1.0 + (b / 128.0) ** 2)
        if np.sqrt(x) != np.sqrt(np.nextafter(x, np.float32(2.0))) and int(x.view(np.uint32)) % 2 == 0:
            return b / 128.0
    raise AssertionError


def _gradient(shape):
    g = torch.zeros(shape, dtype=torch.bfloat16)
    g[0, :2] = torch.tensor([1.0, _rows()])
    g[0, 8] = 2.0 ** -12   # (eight elements are squared and added in fp32)
    g[64, :2] = 2.0 ** -27
    g[96, :2] = 2.0 ** -27
    return g.cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("scale_type", ["tensor", "channel"])
@pytest.mark.parametrize("shape", [(128, 64), (131, 70)])
def test_norms_are_summed_in_the_same_order_in_any_group(shape, scale_type):
    print(f"[apollo group order] {shape} {scale_type}", flush=True)
    from adafactor8bit import Adafactor8Bit
    from test_gpu_apollo import C4_KW
    big = (49664, 64)
    runs = []
    for beside in (False, True):
        ps = [torch.nn.Parameter(torch.full(s, 0.01, dtype=torch.bfloat16, device="cuda"))
              for s in ([shape, big] if beside else [shape])]
        opt = Adafactor8Bit(ps, **dict(C4_KW, apollo_rank=32, apollo_scale_type=scale_type, scale_parameter=True))
        ps[0].grad = _gradient(shape)
        if beside:
            ps[1].grad = torch.full_like(ps[1], 1e-3)
        opt.step()
        torch.cuda.synchronize()
        runs.append((ps[0].detach(), opt.state[ps[0]]))
    (pa, sa), (pb, sb) = runs
    for k, v in sa.items():
        if torch.is_tensor(v):
            assert torch.equal(v, sb[k]), k
    assert torch.equal(pa, pb)
