"""The AL codecs' powers and logarithms are correctly rounded: decoding every code of many
block ranges, and encoding, agree with float64 arithmetic rounded once (adafactor8bit
optimizer.py:299-353).  The ranges include those the fast division and exponent do not cover
(tiny, huge and infinite scales)."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _decode_ref(levels, s, lm):
    c1 = np.arange(levels, dtype=np.float32) - np.float32(1)
    with np.errstate(all="ignore"):
        arg = (c1 * s).astype(np.float32) / np.float32(levels - 2) + lm
        out = np.exp2(arg.astype(np.float64)).astype(np.float32)
    out[0] = 0.0
    return np.where(np.isinf(out), np.float32(np.nan), out)   # the EMA's 0 * (0 - inf) + inf


@pytest.mark.parametrize("block", [256, 128])
def test_step_decodes_every_code_exactly(block):
    """beta2 = 1 keeps V: the fp32 V' that the NORM pass writes is the decoded code."""
    from adafactor8bit import adafactor8bit_cuda as mod  # noqa: F401  (loads the library)
    from adafactor8bit import _native as nat
    rng = np.random.default_rng(5)
    scales = np.concatenate([10.0 ** rng.uniform(-3, 2.3, 500), [1e-12, 1e-25, 1.0, 254.0, 3e5, np.inf, 0.0]])
    mins = np.concatenate([rng.uniform(-140, 100, 500), [-20.0, -20.0, -149.0, -126.0, -1e5, -3.0, -7.0]])
    nb = len(scales) * (256 // block)
    codes = np.tile(np.arange(256, dtype=np.uint8), len(scales))
    q = torch.from_numpy(codes).cuda()
    s = torch.from_numpy(np.repeat(scales.astype(np.float32), 256 // block)).cuda()
    lm = torch.from_numpy(np.repeat(mins.astype(np.float32), 256 // block)).cuda()
    n = codes.size
    g = torch.zeros(n, device="cuda")
    vbuf = torch.empty(n, device="cuda")
    nb_f = torch.zeros(1, device="cuda")
    L = nat.lib()
    parts = torch.empty(int(L.a8_norm_parts_1d(n, block, block)), dtype=torch.float64, device="cuda")
    nat.check(L.a8_fused_update_1d(nat.MODE_NORM, 0, nat.F32, None, g.data_ptr(), None, None, q.data_ptr(),
                                   s.data_ptr(), lm.data_ptr(), vbuf.data_ptr(), nb_f.data_ptr(), parts.data_ptr(),
                                   None, None, None, 0, 1, 0.0, 0.0, 1e-8, 1, -126.0, 0.0, 1e-16, n, block, block,
                                   8, 0, 0.0, 8, 0, 0.0, 1.0, 0, nat.stream_of(g.device)))
    got = vbuf.cpu().numpy().reshape(len(scales), 256)
    for i, (a, b) in enumerate(zip(scales.astype(np.float32), mins.astype(np.float32))):
        want = _decode_ref(256, a, b)
        np.testing.assert_array_equal(got[i], want, err_msg=f"scale {a} min_log {b}")


@pytest.mark.parametrize("bits", [8, 16])
def test_encode_ranges_are_rounded_logarithms(bits):
    """The block range of a re-encoded tensor: log2 of its extremes, rounded once -- subnormal,
    huge and near-one values included."""
    from adafactor8bit import _native as nat
    rng = np.random.default_rng(6)
    bs, nb = 128, 4000
    lo = np.exp2(rng.uniform(-126, 120, nb)).astype(np.float32)
    hi = (lo * np.exp2(rng.uniform(0.001, 7, nb)).astype(np.float32)).astype(np.float32)
    lo[:300] = np.float32(1) + np.arange(300, dtype=np.float32) * np.float32(2 ** -23)
    hi[:300] = lo[:300] * np.float32(1.0001)
    lo[300:310] = np.float32(1.2e-38)
    x = np.repeat(lo[:, None], bs, 1)
    x[:, 1] = hi
    x[:, 2] = 0.0
    t = torch.from_numpy(x.reshape(-1).copy()).cuda()
    q = torch.empty(x.size, dtype=torch.uint8 if bits == 8 else torch.int16, device="cuda")
    s, lm = torch.empty(nb, device="cuda"), torch.empty(nb, device="cuda")
    nat.check(nat.lib().a8_al_encode(q.data_ptr(), s.data_ptr(), lm.data_ptr(), t.data_ptr(), x.size, bs, bits, -126.0,
                                     nat.stream_of(t.device)))
    llo = np.log2(lo.astype(np.float64)).astype(np.float32)
    lhi = np.log2(hi.astype(np.float64)).astype(np.float32)
    llo = np.maximum(llo, np.float32(-126.0))
    llo = np.where(llo >= lhi, lhi - np.float32(1), llo)
    np.testing.assert_array_equal(lm.cpu().numpy(), llo)
    np.testing.assert_array_equal(s.cpu().numpy(), np.maximum(lhi - llo, np.float32(1e-12)))
    assert math.isfinite(float(s.max()))
