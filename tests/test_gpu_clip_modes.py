"""SUM / APPLYC of the quantised 1-D step give the bits of NORM / APPLY (which pass V' through
v_buf): every momentum codec, both V codecs, unit and general block sizes, ragged ends."""
import pytest
import torch

from inputs import make_grad, make_param

pytestmark = pytest.mark.gpu

# (numel, B_V, B_M, v_bits, (m_bits, m_mode) or None, momentum_only)
FORMS = [(1, 128, 32, 8, (8, 0), 0), (2047, 256, 64, 8, (8, 0), 1), (2049, 2048, 256, 8, (4, 0), 0),
         (70001, 2048, 2048, 16, (8, 0), 0), (40007, 512, 128, 8, (8, 1), 0), (40007, 1024, 32, 16, (4, 1), 1),
         (50003, 384, 96, 8, (8, 0), 0), (262147, 131072, 32, 8, (4, 0), 0), (30001, 512, 512, 8, None, 0)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", FORMS, ids=[f"n{f[0]}_bv{f[1]}_bm{f[2]}_v{f[3]}_m{f[4]}_{f[5]}" for f in FORMS])
def test_sum_applyc_equal_norm_apply(form, dtype):
    from adafactor8bit import _native as nat
    from adafactor8bit import _state as S
    n, bv, bm, vbits, mc, mo = form
    dev = torch.device("cuda", 0)
    S.ensure_qmap(dev)
    L = nat.lib()
    gen = torch.Generator().manual_seed(3)
    nv, nm = -(-n // bv), -(-n // bm)
    sr = int(dtype == torch.bfloat16)
    p0 = make_param((n,), 0, 3).to(dtype).cuda()
    g = (make_grad((n,), 0, 1, 3) * 3).to(dtype).cuda()
    vq0 = torch.randint(0, 256 if vbits == 8 else 32768, (nv * bv,), generator=gen)
    vq0[n:] = 0
    vq0 = vq0.to(torch.uint8 if vbits == 8 else torch.int16).cuda()
    vs0, vl0 = torch.full((nv,), 9.0, device=dev), torch.full((nv,), -26.0, device=dev)
    mbits, mmode = mc if mc else (8, 0)
    mq0 = torch.randint(0, 256, (nm * bm * mbits // 8,), generator=gen).to(torch.uint8).cuda()
    ms0 = torch.full((nm,), 1e-3, device=dev)

    def run(norm, apply, vbuf):
        p, vq, vs, vl, mq, ms = (x.clone() for x in (p0, vq0, vs0, vl0, mq0, ms0))
        acc = torch.zeros(1, device=dev)
        parts = torch.empty(int(L.a8_norm_parts_1d(n, bv, bm if mc else bv)), dtype=torch.float64, device=dev)
        for mode in (norm, apply):
            nat.check(L.a8_fused_update_1d(
                mode, sr, nat.dtype_code(dtype), p.data_ptr(), g.data_ptr(), mq.data_ptr() if mc else None,
                ms.data_ptr() if mc else None, vq.data_ptr(), vs.data_ptr(), vl.data_ptr(), nat.ptr(vbuf),
                acc.data_ptr(), parts.data_ptr(), None, None, None, 5, 7, 0.9, 0.001, 1e-8, int(not mo), -126.0,
                0.0, 1e-16, n, bv, bm if mc else bv, mbits, mmode, 0.01, vbits, mo, 1e-3, 0.999, 1,
                nat.stream_of(dev)))
        return [x.cpu() for x in (p, vq, vs, vl, mq, ms, acc)]

    a = run(nat.MODE_NORM, nat.MODE_APPLY, torch.empty(n, device=dev))
    b = run(nat.MODE_SUM, nat.MODE_APPLYC, None)
    for name, x, y in zip(("p", "v_q", "v_scale", "v_min_log", "m_q", "m_scale", "norm"), a, b):
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8)), name
    if n > 1000:
        assert not torch.equal(a[0].float(), p0.cpu().float())


@pytest.mark.parametrize("kernel_rule", [False, True])
@pytest.mark.parametrize("form", FORMS, ids=[f"n{f[0]}_bv{f[1]}_bm{f[2]}_v{f[3]}_m{f[4]}_{f[5]}" for f in FORMS])
def test_modes_without_v_buf_under_either_rule(form, kernel_rule):
    """SUM, MSUM (momentum codes, momentum-only) and APPLYC against NORM, MNORM and APPLY, under the
    CPU quantiser's rule and the reference kernels'."""
    from adafactor8bit import _native as nat
    from adafactor8bit import _state as S
    n, bv, bm, vbits, mc, _ = form
    mo = int(mc is not None)
    dev = torch.device("cuda", 0)
    S.ensure_qmap(dev)
    L = nat.lib()
    gen = torch.Generator().manual_seed(4)
    nv, nm = -(-n // bv), -(-n // bm)
    p0 = make_param((n,), 0, 4).cuda()
    g = (make_grad((n,), 0, 1, 4) * 3).cuda()
    vq0 = torch.randint(0, 256 if vbits == 8 else 32768, (nv * bv,), generator=gen)
    vq0[n:] = 0
    vq0 = vq0.to(torch.uint8 if vbits == 8 else torch.int16).cuda()
    mbits, mmode = mc if mc else (8, 0)
    mq0 = torch.randint(0, 256, (nm * bm * mbits // 8,), generator=gen).to(torch.uint8).cuda()
    vb = vbits | (nat.AL_KERNEL_RULE if kernel_rule else 0)

    def run(modes, vbuf):
        p, vq, mq = p0.clone(), vq0.clone(), mq0.clone()
        vs, vl = torch.full((nv,), 9.0, device=dev), torch.full((nv,), -26.0, device=dev)
        ms = torch.full((nm,), 1e-3, device=dev)
        acc = torch.zeros(2, device=dev)   # sum of U^2 | sum of M'^2
        parts = torch.empty(int(L.a8_norm_parts_1d(n, bv, bm if mc else bv)), dtype=torch.float64, device=dev)
        for mode in modes:
            m_sum = mode in (nat.MODE_MNORM, nat.MODE_MSUM)
            nat.check(L.a8_fused_update_1d(
                mode, 0, nat.F32, p.data_ptr(), g.data_ptr(), mq.data_ptr() if mc else None,
                ms.data_ptr() if mc else None, vq.data_ptr(), vs.data_ptr(), vl.data_ptr(), nat.ptr(vbuf),
                acc.data_ptr() + (4 if m_sum else 0), parts.data_ptr(), None, acc.data_ptr() if m_sum else None, None,
                5, 7, 0.9, 0.001, 1e-8, int(not mo), -126.0, 0.0, 1e-16, n, bv, bm if mc else bv, mbits, mmode, 0.01,
                vb, mo, 1e-3, 0.999, 1, nat.stream_of(dev)))
        return [x.cpu() for x in (p, vq, vs, vl, mq, ms, acc)]

    with_m = lambda *m: m if mc else (m[0], m[2])
    a = run(with_m(nat.MODE_NORM, nat.MODE_MNORM, nat.MODE_APPLY), torch.empty(n, device=dev))
    b = run(with_m(nat.MODE_SUM, nat.MODE_MSUM, nat.MODE_APPLYC), None)
    for name, x, y in zip(("p", "v_q", "v_scale", "v_min_log", "m_q", "m_scale", "norms"), a, b):
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8)), name
    assert a[6][0] > 0 and (a[6][1] > 0) == bool(mc)
