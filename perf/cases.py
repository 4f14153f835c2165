"""Performance cases of the quantization framework: the calls its users make, through the public
entry points, over the range of sizes and options that those calls take.

Four kinds of work:
  layer      quantize_layer on the matrices that share one input, with a new Hessian each time (the
             factorisation is part of the pass; the matrices after the first reuse it, as in the
             model pipeline). Options: bits, group, act-order, MSE grid, high-precision skeleton,
             asymmetric target, repair on or off, host or device memory.
  capture    a calibration Hessian: one accumulation per forward batch, then the 1/N normalisation.
  container  a quantized matrix packed into the cdclq-v1 byte streams and expanded again.
  evaluate   round-to-nearest, the proxy loss and the held-out output error of a quantized matrix.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "cdcl-gptq_amd"))
import cdclq  # noqa: E402

DEV = "cuda:0"


# ------------------------------------------------------------------------------------- the cases
def _layer(name, d_outs, n, **opts):
    c = dict(kind="layer", d_outs=d_outs, n=n, bits=4, group=128, act_order=True, mse_grid=False,
             skeleton_pct=0.0, repair=True, asym=False, host=False)
    c.update(opts)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest call: a toy model's projection through the host-memory entry point, where
        # launches, copies and allocations count
        _layer("layer_toy_host", "256", 256, group=32, bits=3, host=True),
        # a single 2048 x 2048 linear at the reference's default group: the usual small layer
        _layer("layer_2048", "2048", 2048),
        # sizes that no tile divides: rows, columns and the last group are all ragged
        _layer("layer_ragged", "1001", 1350, bits=3),
        # gate and up of a 1.1B-shaped decoder layer, INT3, one shared factorisation
        _layer("layer_gate_up_int3", "5632+5632", 2048, bits=3),
        # INT2 g64 with the searched clip grid and 5% of the column groups kept at 8 bits (the
        # column order then depends on the weights)
        _layer("layer_int2_skeleton", "2048", 5632, bits=2, group=64, mse_grid=True, skeleton_pct=5.0),
        # q, k and v of an 8B-shaped decoder layer on one shared input
        _layer("layer_qkv", "4096+1024+1024", 4096),
        # the asymmetric target (calibration on the quantized model's inputs)
        _layer("layer_asym", "4096", 4096, bits=3, asym=True),
        # plain GPTQ, one grid per row, natural column order: the fast, repair-free setting
        _layer("layer_gptq_per_row", "4096", 4096, group=0, act_order=False, repair=False),
        # the largest matrix of an 8B-shaped decoder layer: a 14336-wide factorisation
        _layer("layer_down", "4096", 14336),
        # the capture hooks over 8 forward batches of 2 x 2048 tokens, tokens weighted
        dict(name="capture_4096", kind="capture", n=4096, t=4096, batches=8, weighted=True),
        # the container of a gate projection, expanded to bf16 (`cdclq dequant`)
        dict(name="container_gate", kind="container", d_out=14336, n=4096, bits=4, group=128, skeleton=0,
             dtype="BF16"),
        # held-out evaluation of one quantized matrix
        dict(name="evaluate_2048", kind="evaluate", d_out=2048, n=2048, t=4096, bits=4, group=128, mse_grid=False),
    ]


def _cost(c):
    """Rough cost in f32 operations, to keep a drawn case below the largest listed one."""
    if c["kind"] == "layer":
        n = c["n"]
        rows = sum(_d_outs(c))
        per_row = 2 + (6 if c["asym"] else 0) + (44 if c["repair"] else 0) + (8 if c["mse_grid"] else 0)
        return (2.0 * n ** 3 + rows * n * n * per_row) * (1 if n % 4 == 0 else 4)
    if c["kind"] == "capture":
        return 2.0 * c["n"] ** 2 * (c["t"] + 256) * c["batches"] * (1 if c["n"] % 4 == 0 else 4)
    if c["kind"] == "container":
        return 500.0 * c["d_out"] * c["n"]
    return 10.0 * c["d_out"] * c["n"] * (c["n"] + c["t"])


def _size(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm: whole tiles, multiples of 8, or any
    number."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    step = rng.choice([128, 64, 8, 1])
    return max(lo, min(hi, max(step, v // step * step)))


def _draw(rng):
    kind = rng.choice(["layer"] * 6 + ["capture", "capture", "container", "evaluate"])
    if kind == "layer":
        n = _size(rng, 64, 8192)
        rows = [str(_size(rng, 32, 8192)) for _ in range(rng.choice([1, 1, 2, 3]))]
        repair = rng.random() < 0.8
        group = rng.choice([128, 128, 64, 32] + ([] if repair else [0]))
        bits = rng.choice([2, 3, 4, 4, 8])
        skel = rng.random() < 0.2 and 0 < group < n and bits < 8
        return _layer("", "+".join(rows), n, bits=bits, group=group, act_order=rng.random() < 0.75,
                      mse_grid=rng.random() < 0.2, skeleton_pct=5.0 if skel else 0.0, repair=repair,
                      asym=rng.random() < 0.2, host=rng.random() < 0.2)
    if kind == "capture":
        return dict(kind="capture", n=_size(rng, 64, 8192), t=_size(rng, 16, 8192), batches=rng.randint(1, 8),
                    weighted=rng.random() < 0.5)
    if kind == "container":
        return dict(kind="container", d_out=_size(rng, 32, 16384), n=_size(rng, 64, 16384),
                    bits=rng.choice([2, 3, 4, 8]), group=rng.choice([32, 64, 128, 0]),
                    skeleton=rng.choice([0, 0, 1]), dtype=rng.choice(["BF16", "F16", "F32"]))
    return dict(kind="evaluate", d_out=_size(rng, 32, 4096), n=_size(rng, 64, 4096), t=_size(rng, 64, 8192),
                bits=rng.choice([2, 3, 4, 8]), group=rng.choice([32, 64, 128]), mse_grid=rng.random() < 0.3)


def draw(rng):
    most = {}
    for c in listed():
        most[c["kind"]] = max(most.get(c["kind"], 0.0), _cost(c))
    top = max(most.values())
    while True:
        c = _draw(rng)
        if _cost(c) <= top / 4:
            return c


# ----------------------------------------------------------------------------------- the inputs
class _Buf:
    """A torch tensor handed to the C ABI (the binding's functions take objects with a .ptr)."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


_context = None


def _ctx():
    """The program's one context (stream, workspace and factor cache)."""
    global _context
    if _context is None:
        _context = cdclq.Context(0)
    return _context


def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + salt) % (1 << 62))


def _d_outs(case):
    return [int(v) for v in case["d_outs"].split("+")]


def _tokens(seed, salt, t, n):
    """Activations of t tokens: unit normal channels, a few directions that all channels share, and
    1% of outlier channels."""
    g = _gen(seed, salt)
    x = torch.randn(t, n, device=DEV, generator=g)
    for _ in range(3):
        a = torch.randn(t, 1, device=DEV, generator=g)
        b = torch.randn(1, n, device=DEV, generator=g)
        x.addcmul_(a, b, value=0.3)
    k = max(1, n // 100)
    big = torch.randperm(n, device=DEV, generator=_gen(seed, salt + 1))[:k]  # the channels of a model input
    x[:, big] *= 20.0
    return x


def _weights(seed, salt, d_out, n):
    return torch.randn(d_out, n, device=DEV, generator=_gen(seed, salt)) * 0.02


def _wait():
    torch.cuda.synchronize()


def _hessian(x, y=None):
    """(X^T Y) / T as the capture produces it, f32."""
    t, n = x.shape
    y = x if y is None else y
    acc = torch.zeros(n, n, dtype=torch.float64, device=DEV)
    h = torch.empty(n, n, device=DEV)
    _wait()
    ctx, L = _ctx(), cdclq.lib()
    ctx.check(L.cdclq_hessian_accumulate_device(ctx.ptr, x.data_ptr(), y.data_ptr(), None, t, n, acc.data_ptr()))
    ctx.check(L.cdclq_hessian_finalize_device(ctx.ptr, acc.data_ptr(), n, t, h.data_ptr()))
    return h


def _config(case):
    return cdclq.Config(bits=case["bits"], group=case["group"], act_order=case["act_order"],
                        mse_grid=case["mse_grid"], skeleton_pct=case["skeleton_pct"],
                        method=cdclq.Method.Cdcl if case["repair"] else cdclq.Method.Gptq)


def _num_groups(group, n):
    return 1 if group == 0 or group >= n else (n + group - 1) // group


def _prepare_layer(case, seed):
    n, cfg = case["n"], _config(case)
    t = (max(2048, n + n // 4) + 63) // 64 * 64
    x = _tokens(seed, 1, t, n)
    m = None
    if case["asym"]:
        xq = x + 0.05 * torch.randn(t, n, device=DEV, generator=_gen(seed, 5))
        h, m = _hessian(xq), _hessian(x, xq)
        del xq
    else:
        h = _hessian(x)
    del x
    ng = _num_groups(case["group"], n)
    mats = []
    for i, d_out in enumerate(_d_outs(case)):
        w = _weights(seed, 10 + i, d_out, n)
        if case["host"]:
            mats.append(dict(d_out=d_out, w=w.cpu().numpy()))
            continue
        mats.append(dict(d_out=d_out, w=_Buf(w), codes=_Buf(torch.empty(d_out, n, dtype=torch.uint8, device=DEV)),
                         scales=_Buf(torch.empty(d_out, ng, device=DEV)),
                         zeros=_Buf(torch.empty(d_out, ng, device=DEV))))
    if case["host"]:
        h, m = h.cpu().numpy(), None if m is None else m.cpu().numpy()
    else:
        h, m = _Buf(h), None if m is None else _Buf(m)
    _wait()
    return dict(kind="layer", host=case["host"], n=n, cfg=cfg, h=h, m=m, mats=mats)


def _capture_batch(case, seed, b):
    x = _tokens(seed, 100 + 10 * b, case["t"], case["n"])
    w = None
    if case["weighted"]:
        w = 0.5 + torch.rand(case["t"], device=DEV, generator=_gen(seed, 105 + 10 * b))
    return x, w


def _prepare_capture(case, seed):
    n = case["n"]
    batches = [_capture_batch(case, seed, b) for b in range(case["batches"])]
    acc = torch.empty(n, n, dtype=torch.float64, device=DEV)
    h = torch.empty(n, n, device=DEV)
    _wait()
    return dict(kind="capture", n=n, t=case["t"], batches=batches, acc=acc, h=h)


def _quantized(case, seed):
    """Codes, scales and zeros of a quantized matrix, its column order and its group widths."""
    d_out, n, bits = case["d_out"], case["n"], case["bits"]
    group = n if case["group"] == 0 or case["group"] >= n else case["group"]
    ng = (n + group - 1) // group
    gbits = np.full(ng, bits, np.uint8)
    if case["skeleton"] and ng > 1:
        gbits[:max(1, ng // 20)] = 8
    width = torch.from_numpy(np.repeat(gbits.astype(np.int64), group)[:n]).to(DEV)
    g = _gen(seed, 1)
    u = torch.rand(d_out, n, device=DEV, generator=g)
    codes = (u * torch.pow(2.0, width.float())).to(torch.uint8)
    scales = (0.002 + 0.01 * torch.rand(d_out, ng, device=DEV, generator=g)).half().float()
    zeros = torch.floor(torch.rand(d_out, ng, device=DEV, generator=g) * 2.0 ** bits)
    perm = torch.randperm(n, device=DEV, generator=g)
    return group, gbits, codes, scales, zeros, perm


def _prepare_container(case, seed):
    d_out, n = case["d_out"], case["n"]
    group, gbits, codes, scales, zeros, perm = _quantized(case, seed)
    ng = gbits.size
    rb = cdclq.row_bytes(n, group, gbits)
    i32 = perm.to(torch.int32)
    dt = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[case["dtype"]]
    s = dict(kind="container", d_out=d_out, n=n, group=group, gbits=gbits, dtype=cdclq._DTYPE_CODE[case["dtype"]],
             codes=codes, scales=scales, zeros=zeros, perm=i32,
             qweight=torch.empty(d_out, rb, dtype=torch.uint8, device=DEV),
             s16=torch.empty(d_out, ng, dtype=torch.float16, device=DEV),
             qzeros=torch.empty(d_out, ng, dtype=torch.uint8, device=DEV),
             perm32=torch.empty(n, dtype=torch.int32, device=DEV),
             out=torch.empty(d_out, n, dtype=dt, device=DEV))
    _wait()
    return s


def _rounded(w, bits):
    """A quantized stand-in of w: rounded on one grid per row."""
    step = w.abs().amax(dim=1, keepdim=True) / 2.0 ** (bits - 1)
    return torch.round(w / step) * step


def _plain_hessian(x):
    x = x.double()
    return ((x.t().contiguous() @ x) / x.shape[0]).float()


def _prepare_evaluate(case, seed):
    d_out, n = case["d_out"], case["n"]
    w = _weights(seed, 1, d_out, n)
    x = _tokens(seed, 2, case["t"], n)
    s = dict(kind="evaluate", d_out=d_out, n=n, t=case["t"], w=w, x=x, w_hat=_rounded(w, case["bits"]),
             h=_plain_hessian(x),
             rtn=torch.empty(d_out, n, device=DEV),
             cfg=cdclq.Config(bits=case["bits"], group=case["group"], mse_grid=case["mse_grid"]))
    _wait()
    return s


def prepare(case, seed):
    return {"layer": _prepare_layer, "capture": _prepare_capture, "container": _prepare_container,
            "evaluate": _prepare_evaluate}[case["kind"]](case, seed)


# -------------------------------------------------------------------------------------- one pass
def _run_layer(s):
    ctx, out = _ctx(), []
    n = s["n"]
    cache = cdclq.PrepCache(ctx=ctx)  # a new, empty cache: this Hessian has not been factored
    cache.claim()
    for m in s["mats"]:
        if s["host"]:
            q, st = cdclq.quantize_layer(m["w"], m["d_out"], n, s["h"], s["m"], "input", s["cfg"], cache)
            codes, scales, zeros, perm, gbits = q.codes, q.scales, q.zeros, q.perm, q.gbits
        else:
            perm, gbits, st = cdclq.quantize_layer_device(ctx, m["w"], m["d_out"], n, s["h"], s["m"], "input",
                                                          s["cfg"], m["codes"], m["scales"], m["zeros"])
            codes, scales, zeros = m["codes"].t, m["scales"].t, m["zeros"].t
        out.append(dict(codes=codes, scales=scales, zeros=zeros, perm=perm.astype(np.int64), gbits=gbits,
                        loss_gptq=st.loss_gptq, loss_final=st.loss_final, code_updates=st.code_updates))
    return out


def _run_capture(s):
    ctx, L = _ctx(), cdclq.lib()
    n, t = s["n"], s["t"]
    acc = s["acc"]
    ctx.check(L.cdclq_memset_device(ctx.ptr, acc.data_ptr(), 0, n * n * 8))
    for x, w in s["batches"]:
        ctx.check(L.cdclq_hessian_accumulate_device(ctx.ptr, x.data_ptr(), x.data_ptr(),
                                                    None if w is None else w.data_ptr(), t, n, acc.data_ptr()))
    ctx.check(L.cdclq_hessian_finalize_device(ctx.ptr, acc.data_ptr(), n, t * len(s["batches"]), s["h"].data_ptr()))
    return s["h"]


def _run_container(s):
    ctx, L = _ctx(), cdclq.lib()
    gb = s["gbits"]
    ctx.check(L.cdclq_pack_layer_device(ctx.ptr, s["d_out"], s["n"], s["group"], gb.ctypes.data, gb.size,
                                        s["codes"].data_ptr(), s["scales"].data_ptr(), s["zeros"].data_ptr(),
                                        s["perm"].data_ptr(), s["qweight"].data_ptr(), s["qweight"].numel(),
                                        s["s16"].data_ptr(), s["qzeros"].data_ptr(), s["perm32"].data_ptr()))
    ctx.check(L.cdclq_dequantize_packed_device(ctx.ptr, s["d_out"], s["n"], s["group"], gb.ctypes.data, gb.size,
                                               s["qweight"].data_ptr(), s["qweight"].numel(), s["s16"].data_ptr(),
                                               s["qzeros"].data_ptr(), s["perm32"].data_ptr(), s["dtype"],
                                               s["out"].data_ptr()))
    return dict(qweight=s["qweight"], scales=s["s16"], qzeros=s["qzeros"], perm=s["perm32"], weight=s["out"])


def _run_evaluate(s):
    ctx, L = _ctx(), cdclq.lib()
    cfg = s["cfg"]._c()
    d_out, n = s["d_out"], s["n"]
    ctx.check(L.cdclq_rtn_layer_device(ctx.ptr, s["w"].data_ptr(), d_out, n, ctypes.byref(cfg), s["rtn"].data_ptr()))
    proxy, rel = ctypes.c_double(), ctypes.c_double()
    ctx.check(L.cdclq_proxy_loss_device(ctx.ptr, s["w"].data_ptr(), s["w_hat"].data_ptr(), d_out, n,
                                        s["h"].data_ptr(), ctypes.byref(proxy)))
    ctx.check(L.cdclq_rel_err_device(ctx.ptr, s["w"].data_ptr(), s["w_hat"].data_ptr(), s["x"].data_ptr(),
                                     s["x"].data_ptr(), d_out, n, s["t"], ctypes.byref(rel)))
    return dict(rtn=s["rtn"], proxy_loss=proxy.value, rel_err=rel.value)


def run(state):
    return {"layer": _run_layer, "capture": _run_capture, "container": _run_container,
            "evaluate": _run_evaluate}[state["kind"]](state)


# ---------------------------------------------------------------------- necessary work, tolerance
def work(case):
    if case["kind"] == "layer":
        n, ng = case["n"], _num_groups(case["group"], case["n"])
        byts, flops = 4.0 * n * n * (2 if case["asym"] else 1) + 4 * n, float(n) ** 3  # n^3/3 + 2n^3/3 (f64)
        if case["skeleton_pct"] > 0:
            flops *= len(_d_outs(case))  # the column order depends on the weights: no shared factorisation
        for d in _d_outs(case):
            byts += d * n * 5.0 + 8.0 * d * ng
            flops += float(d) * n * n  # phase 1: each column's error over the columns after it
            if case["asym"]:
                flops += 4.0 * d * n * n  # W M, and two triangular products
            if case["repair"]:
                # 10 passes of refit and descent and the last refit, each step on the gradient the
                # step before left: 21 products E H when no row chunk converges early
                flops += 21 * 2.0 * d * n * n
        return {"bytes": byts, "flops": flops}
    if case["kind"] == "capture":
        n, t, b = case["n"], case["t"], case["batches"]
        return {"bytes": 4.0 * t * n * b + (4.0 * t * b if case["weighted"] else 0) + 4.0 * n * n,
                "flops": float(n) * (n + 1) * t * b}
    if case["kind"] == "container":
        d, n, ng = case["d_out"], case["n"], _num_groups(case["group"], case["n"])
        out = {"F32": 4, "F16": 2, "BF16": 2}[case["dtype"]]
        # codes in, the container out and in again, the weight out
        return {"bytes": d * n * (1 + 2 * case["bits"] / 8.0 + out) + d * ng * (8 + 2 * 3.0) + 12.0 * n, "flops": 0}
    d, n, t = case["d_out"], case["n"], case["t"]
    return {"bytes": 4.0 * (3 * d * n + n * n + t * n), "flops": 2.0 * d * n * n + 4.0 * d * n * t}


def tolerance(case):
    # Quantized layers, Hessians and containers reproduce the reference engine's results bit for
    # bit: an engine that differs in one code is another engine. The evaluation's two figures are
    # f32 products summed in f64.
    return {"rel": 1e-6} if case["kind"] == "evaluate" else "exact"


def exact(case, seed):
    """What run() returns, in 64-bit arithmetic, where that is a computed number: the captured
    Hessian, the expanded weights, the two error figures."""
    if case["kind"] == "capture":
        h = torch.zeros(case["n"], case["n"], dtype=torch.float64, device=DEV)
        for b in range(case["batches"]):
            x, w = _capture_batch(case, seed, b)
            x = x.double()
            h.addmm_(x.t().contiguous(), x if w is None else x * w.double()[:, None])
        return h / (case["t"] * case["batches"])
    if case["kind"] == "container":
        group, _, codes, scales, zeros, perm = _quantized(case, seed)
        gi = torch.arange(case["n"], device=DEV) // group
        out = torch.empty(case["d_out"], case["n"], dtype=torch.float64, device=DEV)
        out[:, perm] = scales.double()[:, gi] * (codes.double() - zeros.double()[:, gi])
        return dict(qweight=None, scales=scales.double(), qzeros=None, perm=None, weight=out)
    if case["kind"] == "evaluate":
        w = _weights(seed, 1, case["d_out"], case["n"]).double()
        w_hat = _rounded(w.float(), case["bits"]).double()
        x = _tokens(seed, 2, case["t"], case["n"]).double()
        e = w - w_hat
        h = _plain_hessian(x).double()
        proxy = ((e @ h) * e).sum()
        o, d = w @ x.t().contiguous(), e @ x.t().contiguous()
        return dict(rtn=None, proxy_loss=float(proxy), rel_err=float(d.square().sum() / o.square().sum()))
    return None
