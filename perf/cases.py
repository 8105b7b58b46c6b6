"""Performance cases: whole optimizer steps through ``Adafactor8Bit``.

One pass is one ``opt.step()`` (or one replay of a captured ``step()``) in the middle of a
training run: parameters, gradients and a quantised state of some tens of steps are in HBM, as
they are when a program's backward pass has just ended.  The four optimizers are those the
project quotes state sizes and step targets for (AdamW, Adafactor, CAME, APOLLO), with the
model shapes of ``bench.py`` and of the tests; ragged sizes stand for everything that is not a
multiple of the tiles.

A case is a dict of plain values:
  algo     adamw | adafactor | came | apollo
  shapes   parameter shapes, "22@5632x2048 45@2048" = 22 matrices and 45 vectors
  dtype    fp32 | bf16 (bf16 steps write back with stochastic rounding)
  vq, cq, mq   codecs of the second moment, the CAME confidence and the momentum
  bv, bm   block sizes of the second moment and the momentum
  d, fira, wd, rank, variant   RMS clip, Fira limiter, weight decay, APOLLO rank and low-rank form
  mode     "eager": opt.step(); "graph": a replay of one captured step (capturable=True)

Parameters, gradients and each kind of state live in one flat buffer each, the tensors being
256-byte aligned views of it, as in a program that shards or checkpoints them in one piece.  So
a pass returns everything it writes in a few tensors.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "adafactor-8bit_amd")

GRAD = 1e-3      # gradient scale of the headline workload
STEP0 = 40       # steps already taken by the state that prepare() makes
DT = {"fp32": torch.float32, "bf16": torch.bfloat16}

_BASE = dict(dtype="fp32", vq="al8", cq="al8", mq="uf8", bv=2048, bm=256, d=0.0, fira=False, wd=0.0, rank=0,
             variant="", mode="eager")


def _case(**kw):
    return dict(_BASE, **kw)


def _llama(hidden, ffn, kv, vocab, layers):
    """Shapes of a Llama-like model, as bench.py builds them (embedding, head, per layer q, o / k, v /
    gate, up / down and two norm vectors, a last norm vector)."""
    return (f"2@{vocab}x{hidden} {2 * layers}@{hidden}x{hidden} {2 * layers}@{kv}x{hidden} "
            f"{2 * layers}@{ffn}x{hidden} {layers}@{hidden}x{ffn} {2 * layers + 1}@{hidden}")


_TINYLLAMA = _llama(2048, 5632, 256, 32000, 22)   # 1.1 B parameters, 201 tensors


def listed():
    return [
        # The smallest step: a matrix and its bias, where launches and latency are all there is.
        _case(name="adamw_small", algo="adamw", shapes="1@1000x300 1@300", mode="graph"),
        # One matrix of a layer (the 16.8 M-parameter configuration of the CPU baseline).
        _case(name="adamw_matrix", algo="adamw", shapes="1@4096x4096", mode="graph"),
        # The headline: a whole 1.1 B-parameter model in fp32.
        _case(name="adamw_1.1b", algo="adamw", shapes=_TINYLLAMA),
        # bf16 training with stochastic rounding and weight decay: one large decoder layer.
        _case(name="adamw_bf16_layer", algo="adamw", dtype="bf16", bv=256, wd=0.01,
              shapes="2@4096x4096 2@1024x4096 2@14336x4096 1@4096x14336 2@4096"),
        # One rank's flat shard of the 1.1 B-parameter model, with an update clip and the norm-growth limiter.
        _case(name="adamw_shard_clip", algo="adamw", shapes="1@137506048", d=1.0, fira=True, mode="graph"),
        # Factored Adafactor on the whole model (row / column second moment, RMS scaling and clip).
        _case(name="adafactor_1.1b", algo="adafactor", shapes=_TINYLLAMA, bv=256, d=1.0),
        # Ragged matrices, a stack of experts among them, in bf16: rows and columns off every tile.
        _case(name="adafactor_ragged", algo="adafactor", dtype="bf16", bv=256, d=1.0, mode="graph",
              shapes="1@3x1100x2050 1@2304x2081 1@4160x1283 1@515x7777 3@1283"),
        # CAME with 16-bit statistics codes and the limiter on the whole model.
        _case(name="came_1.1b", algo="came", shapes=_TINYLLAMA, vq="al16", cq="al16", d=1.0, fira=True),
        # CAME on one layer in bf16.
        _case(name="came_bf16_layer", algo="came", dtype="bf16", d=1.0,
              shapes="2@2048x2048 2@256x2048 2@5632x2048 1@2048x5632 2@2048"),
        # APOLLO at rank 256 on the whole model in bf16.
        _case(name="apollo_1.1b_bf16", algo="apollo", dtype="bf16", rank=256, fira=True, shapes=_TINYLLAMA),
        # APOLLO in fp32 (the published setting), a model of four layers.
        _case(name="apollo_fp32", algo="apollo", rank=256, fira=True, shapes=_llama(2048, 5632, 256, 32000, 4)),
        # APOLLO at a low rank on uneven matrices, both projection sides, replayed from a graph.
        _case(name="apollo_rank64_ragged", algo="apollo", dtype="bf16", rank=64, fira=True, mode="graph",
              shapes="1@1100x2050 1@2304x2080 1@4160x1283 1@515x7777 3@1283"),
    ]


def draw(rng):
    """One more case: any optimizer, 1e4 to 2e8 parameters, even and odd dimensions, either dtype, the codecs,
    block sizes and options above."""
    algo = rng.choice(["adamw", "adamw", "adafactor", "came", "apollo"])
    total = int(10.0 ** rng.uniform(4.0, 8.3))
    rank = rng.choice([16, 32, 64, 128, 256]) if algo == "apollo" else 0
    toks, left = [], total
    if algo == "adamw" and rng.random() < 0.3:
        toks.append(f"1@{max(4096, total)}")
        left = 0
    for _ in range(rng.randint(1, 6)):
        if left < 10000 and toks:
            break
        n = max(10000, int(left * rng.uniform(0.3, 1.0)))
        side = math.sqrt(n) * 2.0 ** rng.uniform(-1.5, 1.5)
        rows = max(32, rank, int(side))
        cols = max(32, rank, n // max(rows, 1))
        if rng.random() < 0.5:
            rows, cols = -(-rows // 64) * 64, -(-cols // 64) * 64
        toks.append(f"1@{rows}x{cols}")
        left -= rows * cols
    if rng.random() < 0.6:
        toks.append(f"{rng.randint(1, 5)}@{rng.randint(16, 4095)}")
    case = _case(algo=algo, shapes=" ".join(toks), dtype=rng.choice(["fp32", "bf16"]),
                 vq=rng.choice(["al8", "al8", "al16"]), mq=rng.choice(["uf8", "uf8", "uf4"]),
                 bv=rng.choice([256, 512, 2048, 2048]), bm=rng.choice([64, 128, 256]),
                 wd=rng.choice([0.0, 0.01]), mode=rng.choice(["eager", "graph"]), rank=rank)
    case["cq"] = case["vq"]
    if algo == "adamw":
        case["d"], case["fira"] = rng.choice([(0.0, False), (0.0, False), (1.0, False), (1.0, True)])
    elif algo == "apollo":
        case["fira"] = True
        case["variant"] = rng.choice(["", "", "factorize"])
    else:
        case["d"], case["fira"] = 1.0, rng.choice([False, True])
    return case


# ------------------------------------------------------------------ options and shapes
def _shapes(case):
    out = []
    for tok in case["shapes"].split():
        n, s = tok.split("@")
        out += [tuple(int(x) for x in s.split("x"))] * int(n)
    return out


def _options(case):
    """Constructor options: the presets' values, as bench.py passes them."""
    kw = dict(block_size=case["bv"], m_block_size=case["bm"], v_quant_type=case["vq"], m_quant_type=case["mq"],
              weight_decay=case["wd"], d=case["d"], stochastic_round_writeback=case["dtype"] == "bf16",
              relative_step=False, beta3=None, capturable=case["mode"] == "graph")
    algo = case["algo"]
    if algo == "adafactor":
        kw.update(beta1=None, beta2=None, beta2_decay=-0.8, factored=True, lr=1e-3,
                  enable_fira_for_adafactor=case["fira"])
        return kw
    kw.update(beta1=0.9, beta2=0.999, beta2_decay=None, factored=False, scale_parameter=False,
              scale_weight_decay=False, lr=1e-4)
    if algo == "adamw":
        kw.update(eps=(1e-8, 1e-3), enable_fira_for_adafactor=case["fira"])
    elif algo == "came":
        kw.update(beta3=0.9999, factored=True, eps_came=1e-16, c_quant_type=case["cq"],
                  enable_fira_for_adafactor=case["fira"])
    else:
        kw.update(eps=(1e-6, 1e-3), apollo_eps=1e-6, apollo_rank=case["rank"], apollo_update_proj_gap=200,
                  apollo_scale_type="channel", apollo_cache_proj=True, enable_fira_for_apollo=case["fira"], lr=1e-3,
                  apollo_factorize=case["variant"] == "factorize")
    return kw


def _route(case, shape):
    if len(shape) >= 2 and case["algo"] in ("adafactor", "came"):
        return "factored"
    return "apollo" if len(shape) >= 2 and case["algo"] == "apollo" else "full"


# ------------------------------------------------------------------ inputs and state
class _Flat:
    """One flat buffer per name; tensors are laid out in it at 256-byte boundaries."""

    def __init__(self):
        self.plan, self.size, self.dtype, self.buf = [], {}, {}, {}

    def add(self, name, owner, key, numel, dtype):
        at = self.size.get(name, 0)
        self.plan.append((name, owner, key, at, numel))
        unit = 256 // torch.empty((), dtype=dtype).element_size()
        self.size[name] = at + -(-numel // unit) * unit
        self.dtype[name] = dtype

    def alloc(self, dev):
        for name, n in self.size.items():
            self.buf[name] = torch.zeros(n, dtype=self.dtype[name], device=dev)
        return {(o, k): self.buf[name][at:at + n] for name, o, k, at, n in self.plan}


def _ceil(a, b):
    return -(-a // b)


def _fill_al(q, scale, min_log, n, centre, spread, gen):
    """Codes of a second moment in mid-training: log-values spread around `centre` (log2), 0.5% never touched."""
    top = 255 if q.dtype == torch.uint8 else 65535
    step = 4 << 20
    for a in range(0, n, step):
        b = min(n, a + step)
        x = torch.randn(b - a, device=q.device, generator=gen).mul_(0.15).add_(0.6).mul_(top).round_().clamp_(1, top)
        x[::199] = 0
        q[a:b] = (x if top == 255 else torch.where(x > 32767, x - 65536, x)).to(q.dtype)
    scale.copy_(spread * (1.0 + 0.25 * torch.rand(scale.shape, device=q.device, generator=gen)))
    min_log.copy_(centre - 0.6 * scale)


def _fill_m(q, scale, n, size, bits, gen):
    """Momentum codes: normal values, a block's largest near its scale; past the end the code of zero."""
    q.fill_(128 if bits == 8 else 0x88)
    step = 4 << 20
    for a in range(0, n, step):
        b = min(n, a + step)
        if bits == 8:
            q[a:b] = torch.randn(b - a, device=q.device, generator=gen).mul_(40.0).add_(128.0).round_().clamp_(0, 255).to(q.dtype)
        else:
            x = torch.randn(b - a + (b - a) % 2, device=q.device, generator=gen).mul_(2.5).add_(8.0).round_().clamp_(0, 15)
            x[b - a:] = 8.0
            q[a // 2:a // 2 + x.numel() // 2] = (x[0::2] * 16.0 + x[1::2]).to(q.dtype)
    scale.copy_(size * (0.7 + 0.6 * torch.rand(scale.shape, device=q.device, generator=gen)))


def _low(case, shape):
    R, C = shape[0], math.prod(shape[1:])
    return (R, case["rank"]) if R >= C else (case["rank"], C)


def _slots(case, shape):
    """(slot, kind, elements, codec) of a parameter's state: kind "v" (log-space codes) or "m" (momentum codes)."""
    n = math.prod(shape)
    coded = n >= 4096
    route, out = _route(case, shape), []
    v, c = (case["vq"], case["cq"]) if coded else ("fp32", "fp32")
    m = case["mq"] if coded else "fp32"
    if route == "factored":
        rows, cols = n // shape[-1], n // shape[-2]
        out += [("row_var", "v", rows, v), ("col_var", "v", cols, v)]
        if case["algo"] == "came":
            out += [("conf_row", "v", rows, c), ("conf_col", "v", cols, c)]
    elif route == "apollo":
        n = math.prod(_low(case, shape))
        if case["variant"] == "factorize":
            out += [("row_var_low", "v", _low(case, shape)[0], "fp32"), ("col_var_low", "v", _low(case, shape)[1], "fp32")]
        else:
            out.append(("v_low", "v", n, v))
        out.append(("m_low", "m", n, m))
        return out
    else:
        out.append(("variance", "v", n, v))
    if case["algo"] != "adafactor":
        out.append(("m", "m", n, m))
    return out


def _inputs(case, seed):
    """Flat buffers, the views of each parameter, its gradient and its state, all from the seed."""
    dev = torch.device("cuda", 0)
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed))
    shapes, dt = _shapes(case), DT[case["dtype"]]
    flat = _Flat()
    for i, s in enumerate(shapes):
        n = math.prod(s)
        flat.add("p", i, "p", n, dt)
        flat.add("grad", i, "g", n, dt)
        for slot, kind, k, codec in _slots(case, s):
            if codec == "fp32":
                flat.add(slot, i, slot, k, torch.float32)
            elif kind == "v":
                nb = _ceil(k, case["bv"])
                flat.add(slot + "_q", i, slot + "_q", nb * case["bv"], torch.uint8 if codec == "al8" else torch.int16)
                flat.add(slot + "_scale", i, slot + "_scale", nb, torch.float32)
                flat.add(slot + "_min_log", i, slot + "_min_log", nb, torch.float32)
            else:
                nb = _ceil(k, case["bm"])
                flat.add(slot + "_q", i, slot + "_q", nb * case["bm"] // (2 if codec == "uf4" else 1), torch.uint8)
                flat.add(slot + "_scale", i, slot + "_scale", nb, torch.float32)
        if case["fira"] and (len(s) >= 2 and case["algo"] != "adamw"):
            flat.add("fira", i, "fira", 1, torch.float32)
        if _route(case, s) == "apollo":
            flat.add("proj", i, "proj", case["rank"] * min(s[0], n // s[0]), torch.float32)
    view = flat.alloc(dev)
    for i, s in enumerate(shapes):
        n = math.prod(s)
        p, g = view[i, "p"], view[i, "g"]
        step = 16 << 20
        for a in range(0, n, step):
            b = min(n, a + step)
            x = torch.randn(b - a, device=dev, generator=gen)
            p[a:b] = x.mul_(0.02) if len(s) >= 2 or n > 4096 else x.mul_(0.02).add_(1.0)
            x = torch.randn(b - a, device=dev, generator=gen).mul_(GRAD)
            g[a:b] = x.mul_(torch.rand(b - a, device=dev, generator=gen) >= 0.05)
        lg = 2.0 * math.log2(GRAD)
        for slot, kind, k, codec in _slots(case, s):
            size, centre, spread = GRAD, lg, 9.0
            if slot in ("row_var", "col_var"):
                spread = 3.0
            elif slot.startswith("conf"):
                centre, spread = -3.0, 3.0
            elif slot.endswith("low"):   # a projected gradient's element sums min(R, C) products
                centre = lg + math.log2(min(s[0], n // s[0]) / case["rank"])
                size = 2.0 ** (0.5 * centre)
            if slot == "m" and (case["algo"] == "came"):
                size = 1.0   # CAME's momentum is of the normalised update
            if codec == "fp32":
                x = view[i, slot]
                if kind == "v":
                    x.copy_(torch.exp2(centre + torch.randn(k, device=dev, generator=gen)))
                else:
                    x.copy_(torch.randn(k, device=dev, generator=gen).mul_(0.3 * size))
            elif kind == "v":
                _fill_al(view[i, slot + "_q"], view[i, slot + "_scale"], view[i, slot + "_min_log"], k, centre, spread, gen)
            else:
                _fill_m(view[i, slot + "_q"], view[i, slot + "_scale"], k, size, 4 if codec == "uf4" else 8, gen)
        if (i, "proj") in view:
            x = view[i, "proj"]
            x.copy_(torch.randn(x.numel(), device=dev, generator=gen).div_(math.sqrt(case["rank"])))
        if (i, "fira") in view:   # a little below this step's norm: the limiter acts on some tensors
            view[i, "fira"].fill_(math.sqrt(n) * (GRAD if case["algo"] == "apollo" else 1.0) * (0.5 + 0.1 * (i % 7)))
    return shapes, flat, view


def _state(case, i, shape, view):
    """The optimizer's state entry of parameter i: the stored format's keys over the flat buffers' views."""
    n = math.prod(shape)
    coded = n >= 4096
    st = {"step": STEP0, "is_quantized": coded, "block_size": case["bv"], "v_quant_type": case["vq"],
          "c_quant_type": case["cq"] if case["algo"] == "came" else case["vq"]}
    if case["dtype"] == "bf16":
        st["sr_seed"] = 11 + i
    route = _route(case, shape)
    lead = list(shape[:-2])
    for slot, kind, k, codec in _slots(case, shape):
        if slot in ("row_var", "conf_row"):
            full = lead + [shape[-2], 1]
        elif slot in ("col_var", "conf_col"):
            full = lead + [1, shape[-1]]
        elif slot.endswith("_low"):
            full = {"row_var_low": (k, 1), "col_var_low": (1, k), "v_low": (k,), "m_low": _low(case, shape)}[slot]
        else:
            full = shape
        if codec == "fp32":
            st[slot] = view[i, slot].view(tuple(full))
            continue
        st[slot + "_q"], st[slot + "_scale"] = view[i, slot + "_q"], view[i, slot + "_scale"]
        if kind == "v":
            st[slot + "_min_log"] = view[i, slot + "_min_log"]
            st[slot + "_shape"], st[slot + "_pad"] = tuple(full), _ceil(k, case["bv"]) * case["bv"] - k
        else:
            st["m_block_size"] = case["bm"]
    if case["algo"] != "adafactor":
        st["m_quant_type"] = case["mq"]
    if route == "apollo":
        st.update(apollo_seed=1000 + i, current_proj_seed=900 + i, apollo_rank=case["rank"],
                  apollo_factorize=case["variant"] == "factorize", beta3=None, apollo_update_proj_gap=200,
                  last_proj_step=1)
        right = shape[0] >= n // shape[0]
        st["apollo_proj_matrix_T"] = view[i, "proj"].view((-1, case["rank"]) if right else (case["rank"], -1))
        if (i, "fira") in view:
            st["scaled_grad_norm_prev"] = view[i, "fira"].view(())
    elif (i, "fira") in view:
        st["fira_prev_norm"] = view[i, "fira"].view(())
    return st


def prepare(case, seed):
    if _PKG not in sys.path:
        sys.path.insert(0, _PKG)
    from adafactor8bit import Adafactor8Bit
    shapes, flat, view = _inputs(case, seed)
    params = []
    for i, s in enumerate(shapes):
        p = torch.nn.Parameter(view[i, "p"].view(s))
        p.grad = view[i, "g"].view(s)
        params.append(p)
    opt = Adafactor8Bit(params, **_options(case))
    for i, p in enumerate(params):
        opt.state[p].update(_state(case, i, shapes[i], view))
    state = {"opt": opt, "graph": None, "out": {k: v for k, v in flat.buf.items() if k not in ("grad", "proj")}}
    if case["mode"] == "graph":
        # capture as a training program does: one eager step, then a captured one; the state is put back after
        kept = {k: v.clone() for k, v in state["out"].items()}
        opt.step()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
            opt.step()
        torch.cuda.current_stream().wait_stream(side)
        for k, v in kept.items():
            state["out"][k].copy_(v)
        for i, p in enumerate(params):   # the limiter's norms that the step keeps in a buffer of its own
            t = opt.state[p].get("fira_prev_norm")
            if torch.is_tensor(t) and (i, "fira") not in view:
                t.zero_()
        torch.cuda.synchronize()
        state["graph"] = graph
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        state["opt"].step()
    return state["out"]


def work(case):
    """Bytes: gradient read, parameter and state read and written, APOLLO's projection read; the projection's flops."""
    nbytes = flops = 0.0
    pb = 2 if case["dtype"] == "bf16" else 4
    for s in _shapes(case):
        n = math.prod(s)
        nbytes += 3.0 * pb * n
        for slot, kind, k, codec in _slots(case, s):
            per = {"fp32": 8.0, "al8": 2.0, "uf8": 2.0, "uf4": 1.0, "al16": 4.0}[codec]
            meta = 0.0 if codec == "fp32" else 16.0 * _ceil(k, case["bv"]) if kind == "v" else 8.0 * _ceil(k, case["bm"])
            nbytes += per * k + meta
        if _route(case, s) == "apollo":
            nbytes += 4.0 * case["rank"] * min(s[0], n // s[0])
            flops += 2.0 * n * case["rank"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what one pass differs from exact() over the listed and forty drawn cases.  fp32: parameters
    1.3e-7, block ranges 2e-7 (APOLLO's, whose values are projected sums, 1.3e-6, an element 2e-5); bf16: a rounding
    step is 2^-7 of a value.  Codes are whole numbers with ties: AL16's step is an fp32 rounding error wide, and a
    factored matrix has few codes, so that one of them is a larger share."""
    algo = case["algo"]
    if "al16" in (case["vq"], case["cq"]):
        differ = 0.01
    else:
        differ = 4e-3 if algo in ("adafactor", "came") else 4e-4
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.04, "differ": differ}
    rel, most = {"adamw": (1e-6, 2e-6), "adafactor": (1e-6, 4e-6), "came": (1e-6, 4e-6), "apollo": (6e-6, 8e-5)}[algo]
    return {"rel": rel, "max": most, "differ": differ}


# ------------------------------------------------------------------ the same step in 64 bits
def _dec_v(view, i, slot, k, codec, bv):
    if codec == "fp32":
        return view[i, slot].double()
    q = view[i, slot + "_q"][:k].to(torch.float64)
    top = 254.0
    if codec == "al16":
        q, top = torch.where(q < 0, q + 65536.0, q), 65534.0
    at = torch.arange(k, device=q.device) // bv
    x = torch.exp2((q - 1.0) * view[i, slot + "_scale"].double()[at] / top + view[i, slot + "_min_log"].double()[at])
    return torch.where(q == 0, torch.zeros_like(x), x)


def _dec_m(view, i, slot, k, codec, bm):
    if codec == "fp32":
        return view[i, slot].double()
    q = view[i, slot + "_q"]
    if codec == "uf4":
        q = torch.stack((q >> 4, q & 15), dim=-1).reshape(-1)
    zero = 8.0 if codec == "uf4" else 128.0
    at = torch.arange(k, device=q.device) // bm
    return (q[:k].to(torch.float64) - zero) * (view[i, slot + "_scale"].double()[at] / zero)


def _put_v(out, at, slot, v, codec, bv, floor=-126.0):
    """The new block ranges of a log-space slot (its codes are whole numbers with ties: left out)."""
    if codec == "fp32":
        out[slot][at[slot]] = v.reshape(-1)
        return
    x = torch.nn.functional.pad(v.reshape(-1), (0, -v.numel() % bv)).view(-1, bv)
    logs = torch.log2(x.clamp(min=1e-38))
    hi = logs.amax(1)
    lo = torch.where(x == 0, torch.full_like(logs, math.inf), logs).amin(1).clamp(min=floor)
    lo = torch.where(lo >= hi, hi - 1.0, lo)
    out[slot + "_scale"][at[slot + "_scale"]] = (hi - lo).clamp(min=1e-12)
    out[slot + "_min_log"][at[slot + "_min_log"]] = lo


def _put_m(out, at, slot, m, codec, bm):
    if codec == "fp32":
        out[slot][at[slot]] = m.reshape(-1)
        return
    x = torch.nn.functional.pad(m.reshape(-1), (0, -m.numel() % bm)).view(-1, bm)
    out[slot + "_scale"][at[slot + "_scale"]] = x.abs().amax(1).clamp(min=1e-12)


def _limit(norm, prev, margin=0.01):
    """Fira's norm-growth limiter: (scale, the norm to keep)."""
    if prev is None or float(prev) < 1e-6:
        return 1.0, norm
    lim = max(norm / (float(prev) + 1e-8), 1.0 + margin) / (1.0 + margin)
    return 1.0 / lim, norm / lim


def exact(case, seed):
    """One step from the same inputs in float64, written from the optimizers' formulas."""
    shapes, flat, view = _inputs(case, seed)
    kw = _options(case)
    dev = view[0, "p"].device
    out, where = {}, {}
    for name, owner, key, a, n in flat.plan:
        where.setdefault(owner, {})[key] = slice(a, a + n)
    for name, buf in flat.buf.items():
        if name in ("grad", "proj"):
            continue
        out[name] = torch.zeros(buf.numel(), dtype=torch.float64, device=dev) if buf.is_floating_point() else None
    t = STEP0 + (2 if case["mode"] == "graph" else 1)   # a captured program has taken one step more
    bv, bm, d, lr, wd = case["bv"], case["bm"], case["d"], kw["lr"], case["wd"]
    w2 = t ** -0.8 if case["algo"] == "adafactor" else 1e-3
    eps1 = kw.get("eps", (1e-30, 1e-3))[0]
    for i, s in enumerate(shapes):
        n, at = math.prod(s), where[i]
        p, g = view[i, "p"].double(), view[i, "g"].double()
        slots = {slot: (k, codec) for slot, kind, k, codec in _slots(case, s)}
        dec = {slot: (_dec_v if kind == "v" else _dec_m)(view, i, slot, k, codec, bv if kind == "v" else bm)
               for slot, kind, k, codec in _slots(case, s)}
        prev = view.get((i, "fira"))
        adam = case["algo"] in ("adamw", "apollo")
        bc1, bc2 = 1.0 - 0.9 ** t, 1.0 - 0.999 ** t
        alpha = rho = lr
        if case["algo"] == "adafactor":
            alpha = rho * max(float(p.norm()) / math.sqrt(n), 1e-3)
        if adam:
            alpha = lr * math.sqrt(bc2) / bc1
        if wd and _route(case, s) != "apollo":
            p *= 1.0 - (alpha if kw.get("scale_weight_decay", True) else rho) * wd
        if _route(case, s) == "apollo":
            p = _exact_apollo(case, kw, s, view, i, out, at, p.view(s[0], -1), g.view(s[0], -1), dec, slots, t, prev)
        elif _route(case, s) == "factored":
            p = _exact_factored(case, s, out, at, p, g.view(s), dec, slots, w2, alpha, eps1, prev)
        else:
            v = dec["variance"]
            v = v + w2 * (g * g + (0.0 if adam else eps1) - v)
            _put_v(out, at, "variance", v, slots["variance"][1], bv)
            inv = 1.0 / (v.sqrt() + eps1 * math.sqrt(bc2)) if adam else \
                v.clamp(min=max(eps1 * eps1, 1.17549435e-38)).rsqrt()
            if adam:
                m = 0.9 * dec["m"] + 0.1 * g
                _put_m(out, at, "m", m, slots["m"][1], bm)
                u, clip = m * inv, True
            else:
                u, clip = g * inv, True
                if "m" in dec:   # momentum of the clipped, normalised gradient
                    u = u / max(1.0, float(u.norm()) / math.sqrt(n) / d) if d else u
                    u = 0.9 * dec["m"] + 0.1 * u
                    _put_m(out, at, "m", u, slots["m"][1], bm)
                    clip = False
            norm = float(u.norm())
            scale = _limit(norm, None)[0] if case["fira"] else 1.0
            p = p - alpha * scale / (max(1.0, norm / (math.sqrt(n) * d)) if clip and d else 1.0) * u
        out["p"][at["p"]] = p.reshape(-1)
    return out


def _exact_factored(case, s, out, at, p, g, dec, slots, w2, alpha, eps1, prev):
    n, bv, d = g.numel(), case["bv"], case["d"]
    lead = s[:-2]
    rs, cs = lead + (s[-2], 1), lead + (1, s[-1])
    sq = g * g
    row = dec["row_var"].view(rs)
    col = dec["col_var"].view(cs)
    row = row + w2 * (sq.mean(-1, keepdim=True) + eps1 - row)
    col = col + w2 * (sq.mean(-2, keepdim=True) + eps1 - col)
    _put_v(out, at, "row_var", row, slots["row_var"][1], bv)
    _put_v(out, at, "col_var", col, slots["col_var"][1], bv)
    u = g * (row / row.mean(-2, keepdim=True).clamp(min=eps1)).rsqrt() * col.rsqrt()
    clip = True
    if "conf_row" in slots:
        u = u / max(1.0, float(u.norm()) / math.sqrt(n) / d) if d else u
        m = 0.9 * dec["m"].view(s) + 0.1 * u
        _put_m(out, at, "m", m, slots["m"][1], case["bm"])
        res = (u - m) ** 2 + 1e-16
        cr, cc = dec["conf_row"].view(rs), dec["conf_col"].view(cs)
        cr = cr + 1e-4 * (res.mean(-1, keepdim=True) - cr)
        cc = cc + 1e-4 * (res.mean(-2, keepdim=True) - cc)
        _put_v(out, at, "conf_row", cr, slots["conf_row"][1], bv)
        _put_v(out, at, "conf_col", cc, slots["conf_col"][1], bv)
        u = m * (cr / cr.mean(-2, keepdim=True).clamp(min=eps1)).rsqrt() * cc.rsqrt()
        clip = False
    norm, scale = float(u.norm()), 1.0
    if case["fira"]:
        scale, keep = _limit(norm, prev)
        out["fira"][at["fira"]] = keep
    return p - (alpha * scale / (max(1.0, norm / (math.sqrt(n) * d)) if clip and d else 1.0) * u).reshape(-1)


def _exact_apollo(case, kw, s, view, i, out, at, p, g, dec, slots, t, prev):
    R, C = g.shape
    right, rank, eps = R >= C, case["rank"], kw["apollo_eps"]
    proj = view[i, "proj"].double().view((C, rank) if right else (rank, R))
    low = g @ proj if right else proj @ g
    m = 0.9 * dec["m_low"].view(low.shape) + 0.1 * low
    _put_m(out, at, "m_low", m, slots["m_low"][1], case["bm"])
    if case["variant"] == "factorize":
        row, col = dec["row_var_low"].view(-1, 1), dec["col_var_low"].view(1, -1)
        sq = low * low
        row = row + 1e-3 * (sq.mean(-1, keepdim=True) + 1.17549435e-38 - row)
        col = col + 1e-3 * (sq.mean(-2, keepdim=True) + 1.17549435e-38 - col)
        _put_v(out, at, "row_var_low", row, "fp32", 0)
        _put_v(out, at, "col_var_low", col, "fp32", 0)
        v = row * col / row.mean().clamp(min=eps)
    else:
        v = dec["v_low"].view(low.shape)
        v = v + 1e-3 * (low * low - v)
        _put_v(out, at, "v_low", v, slots["v_low"][1], case["bv"], floor=math.log2(eps * eps))
    u = m / (v.sqrt() + eps)
    dim = -1 if right else -2
    f = u.norm(dim=dim, keepdim=True) / (low.norm(dim=dim, keepdim=True) + 1e-8)
    if case["fira"]:
        norm = float(((g * g).sum(dim, keepdim=True) * f * f).sum().sqrt())
        scale, keep = _limit(norm, prev)
        out["fira"][at["fira"]] = keep
        f = f * scale
    if case["wd"]:
        p = p * (1.0 - kw["lr"] * case["wd"])
    return p - kw["lr"] * math.sqrt(1.0 - 0.999 ** t) / (1.0 - 0.9 ** t) * (g * f)
