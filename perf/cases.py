"""The calls whose speed this repository is judged by, through its public entry points.

`listed()` gives the named cases, `draw(rng)` one more of the same ranges; `prepare` makes what a training or scoring
program holds before the call, `run` is one pass, `exact` the same results in 64-bit torch arithmetic, `work` the bytes
and operations the pass cannot do without, `tolerance` how far another correct implementation may be off.

Values follow the benchmark configurations: hidden states after an RMS norm, weights N(0, 0.02^2) in fp32, a Zipf
unigram prior as the head's bias, Zipf tokens, a pointer candidate on about 60% of the rows.
"""
import math

import torch

from memarch_amd import chunk_ce as _chunk
from memarch_amd import fused_ops, induct, swiglu

_DT = {"bf16": torch.bfloat16, "fp32": torch.float32, "fp16": torch.float16}
_DEV = "cuda"


def listed():
    return [
        # a small model's step, as unit runs and sweeps of small models make it: launches and host time count
        dict(name="mix_tiny", op="mix_biased", n=250, d=256, v=4003, v_real=4003, h="bf16", w="fp32"),
        # one 1024-token text per micro-batch (gradient accumulation) on the 131072-id vocabulary
        dict(name="mix_text_v131k", op="mix_biased", n=1024, d=2048, v=131072, v_real=131072, h="bf16", w="fp32"),
        # the loss head's own call shape, 16 texts of 1024 tokens at d = 1024: the bias folded into w (K = d + 16)
        dict(name="mix_folded_16k", op="mix_folded", n=16384, d=1024, v=50304, v_real=50304, h="bf16", w="fp32"),
        # the headline step: 32 texts of 1024 tokens, d = 2048, padded vocabulary
        dict(name="mix_32k", op="mix_biased", n=32768, d=2048, v=50304, v_real=50257, h="bf16", w="fp32"),
        # plain cross-entropy without autocast (fp32 hidden states), unpadded vocabulary, ragged rows, ignored targets
        dict(name="ce_ragged_fp32", op="ce", n=2999, d=768, v=50257, v_real=50257, h="fp32", w="fp32"),
        # cross-entropy with the phrase/pointer bias of three candidate ids per row
        dict(name="sparse_8k", op="sparse", n=8192, d=1024, v=50304, v_real=50304, h="bf16", w="fp32", kc=3),
        # (logsumexp, target logit) with upstream gradients on both, as the short-range and auxiliary losses use it
        dict(name="chunk_4k", op="chunk", n=4096, d=2048, v=50304, v_real=50304, h="bf16", w="fp32"),
        # validation loss of four texts, fp32 tensors, forward only
        dict(name="eval_4k_fp32", op="rows_mix", n=4096, d=512, v=50257, v_real=50257, h="fp32", w="fp32"),
        # scoring a short continuation with bf16 weights: the head's weights have to be read once
        dict(name="score_64", op="rows_ce", n=64, d=2048, v=50304, v_real=50257, h="bf16", w="bf16"),
        # pointer candidates of a training batch: token, pair and triple locks
        dict(name="induct_32x1024", op="induct", b=32, t=1024, v=50257, locks=3, longest=True),
        # pointer candidates of long texts (needle-in-a-book evaluation)
        dict(name="induct_4x16384", op="induct", b=4, t=16384, v=50257, locks=3, longest=True),
        # the feed-forward gate of a d = 2048 model, forward and backward
        dict(name="swiglu_8k", op="swiglu", rows=8192, hidden=8192, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["mix_biased", "mix_biased", "mix_folded", "mix_folded", "ce", "sparse", "chunk", "rows_mix",
                     "rows_ce", "induct", "induct", "swiglu"])
    if op == "induct":
        t = _log(rng, 32, 32768)
        return dict(op=op, b=_log(rng, 1, max(1, min(64, (1 << 19) // t))), t=t, v=rng.choice([300, 50257, 131072]),
                    locks=rng.choice([2, 3, 3]), longest=rng.random() < 0.7)
    if op == "swiglu":
        hidden = _log(rng, 64, 8192)
        hidden = hidden if rng.random() < 0.3 else max(64, hidden // 64 * 64)
        return dict(op=op, rows=_log(rng, 16, min(32768, (1 << 27) // hidden)), hidden=hidden,
                    dtype=rng.choice(["bf16", "bf16", "fp32", "fp16"]))
    d = _log(rng, 128, 2048)
    d = max(128, d // 64 * 64) if rng.random() < 0.7 else d
    v = rng.choice([50304, 50257, 131072, _log(rng, 1000, 131072)])
    n = _log(rng, 16 if op.startswith("rows") else 64, 32768)
    n = n // 256 * 256 if n > 512 and rng.random() < 0.4 else n
    n = max(16, min(n, 32768 * 2048 * 50304 // (d * v)))
    case = dict(op=op, n=n, d=d, v=v, v_real=50257 if v == 50304 and op == "mix_biased" else v,
                h=rng.choice(["bf16", "bf16", "bf16", "fp32"]), w=rng.choice(["fp32", "fp32", "fp32", "bf16"]))
    if op == "sparse":
        case["kc"] = rng.choice([2, 3, 3, 32])
    return case


# ------------------------------------------------------------------------------------------------------ inputs


def _zipf(g, shape, v, s):
    """Ids with p(id) ~ (id + 1)^-s."""
    cdf = torch.arange(1, v + 1, dtype=torch.float64, device=_DEV).pow_(-s).cumsum(0)
    u = torch.rand(shape, generator=g, dtype=torch.float64, device=_DEV) * cdf[-1]
    return torch.searchsorted(cdf, u).clamp_(max=v - 1)


def _tokens(g, b, t, v):
    """Zipf texts in which a third of the positions continue copies of earlier spans of 8 tokens."""
    x = _zipf(g, (b, t), v, 1.05)
    if t < 32:
        return x
    blk = t // 8
    src = (torch.rand(b, blk, generator=g, device=_DEV) * torch.arange(blk, device=_DEV)).long()
    copy = torch.rand(b, blk, generator=g, device=_DEV) < 0.33
    src = torch.where(copy, src, torch.arange(blk, device=_DEV).expand(b, blk))
    spans = x[:, :blk * 8].reshape(b, blk, 8)
    x[:, :blk * 8] = spans.gather(1, src[..., None].expand(b, blk, 8)).reshape(b, blk * 8)
    return x


def prepare(case, seed):
    g = torch.Generator(device=_DEV).manual_seed(seed)
    op = case["op"]
    if op == "induct":
        x = _tokens(g, case["b"], case["t"], case["v"])
        bucket = torch.randint(0, 8, (case["v"],), generator=g, device=_DEV) if case["longest"] else None
        return dict(case=case, x=x, bucket=bucket)
    if op == "swiglu":
        r, hd, dt = case["rows"], case["hidden"], _DT[case["dtype"]]
        gu = torch.randn(r, 2 * hd, generator=g, device=_DEV).to(dt).requires_grad_()
        go = torch.randn(r, hd, generator=g, device=_DEV).to(dt)
        return dict(case=case, gu=gu, go=go)
    n, d, v, v_real = case["n"], case["d"], case["v"], case["v_real"]
    hdt, wdt = _DT[case["h"]], _DT[case["w"]]
    h = torch.randn(n, d, generator=g, device=_DEV)
    h = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-7)
    w = torch.randn(v, d, generator=g, device=_DEV) * 0.02
    w[v_real:] = 0
    p = torch.arange(1, v_real + 1, dtype=torch.float64, device=_DEV).pow_(-1.1)
    bias = torch.zeros(v, device=_DEV)
    bias[:v_real] = (p / p.sum()).log().float()
    y = _zipf(g, (n,), v_real, 1.1)
    s = dict(case=case, y=y, go=torch.full((), 1.0 / n, device=_DEV))
    if op.startswith("mix") or op == "rows_mix":
        has = torch.rand(n, generator=g, device=_DEV) < 0.6
        s["hit"] = ((torch.rand(n, generator=g, device=_DEV) < 0.3) & has).float()
        s["gate"] = torch.sigmoid(torch.randn(n, generator=g, device=_DEV)) * has
    if op == "mix_folded":
        # the caller's layout: h = [h, 1, 0 x 15], w = [W, bias, 0 x 15]
        h = torch.cat([h, torch.ones(n, 1, device=_DEV), torch.zeros(n, 15, device=_DEV)], 1)
        w = torch.cat([w, bias[:, None], torch.zeros(v, 15, device=_DEV)], 1)
    elif op in ("mix_biased", "chunk", "rows_mix"):
        s["bias"] = bias
    if op == "ce":
        y[torch.rand(n, generator=g, device=_DEV) < 0.05] = -100
    if op == "sparse":
        s["cand"] = _zipf(g, (n, case["kc"]), v, 1.1)
        s["b"] = torch.randn(n, case["kc"], generator=g, device=_DEV)
    if op == "chunk":
        s["g_lse"] = torch.rand(n, generator=g, device=_DEV) / n
        s["g_ly"] = -torch.rand(n, generator=g, device=_DEV) / n
    s["h"], s["w"] = h.to(hdt), w.to(wdt)
    if not op.startswith("rows"):
        for k in ("h", "w", "bias", "gate", "b"):
            if k in s:
                s[k].requires_grad_()
    return s


# -------------------------------------------------------------------------------------------------------- one pass


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "induct":
        return induct.induct_raw(s["x"], locks=case["locks"], longest=case["longest"], bucket=s["bucket"])
    if op == "swiglu":
        out = swiglu.swiglu(s["gu"])
        (dgu,) = torch.autograd.grad(out, [s["gu"]], s["go"])
        return out, dgu
    if op == "rows_mix":
        return fused_ops.forward_rows(s["h"], s["w"], s["y"], s["gate"], s["hit"], bias=s["bias"])
    if op == "rows_ce":
        return fused_ops.forward_rows(s["h"], s["w"], s["y"], None, None, v_real=case["v_real"])
    if op == "chunk":
        lse, ly = _chunk.chunk_ce(s["h"], s["w"], s["bias"], s["y"])
        grads = torch.autograd.grad([lse, ly], [s["h"], s["w"], s["bias"]], [s["g_lse"], s["g_ly"]])
        return (lse, ly) + grads
    if op == "mix_biased":
        loss = fused_ops.linear_ce_mix_biased(s["h"], s["w"], s["bias"], s["y"], s["gate"], s["hit"],
                                              v_real=case["v_real"])
        wrt = ("h", "w", "bias", "gate")
    elif op == "mix_folded":
        loss = fused_ops.linear_ce_mix(s["h"], s["w"], s["y"], s["gate"], s["hit"])
        wrt = ("h", "w", "gate")
    elif op == "sparse":
        loss = fused_ops.linear_ce_sparse(s["h"], s["w"], s["y"], s["cand"], s["b"])
        wrt = ("h", "w", "b")
    else:
        loss = fused_ops.linear_ce(s["h"], s["w"], s["y"])
        wrt = ("h", "w")
    return (loss,) + torch.autograd.grad(loss, [s[k] for k in wrt], s["go"])


# ---------------------------------------------------------------------------------------------- what it has to do


def work(case):
    op = case["op"]
    if op == "induct":
        pos = case["b"] * case["t"]
        return dict(bytes=pos * (8 + case["locks"] * 9 + 8), flops=0)   # tokens in; cand, on, bk out
    if op == "swiglu":
        size = torch.finfo(_DT[case["dtype"]]).bits // 8
        el = case["rows"] * case["hidden"]
        return dict(bytes=8 * el * size, flops=20 * el)   # gu twice, out, go, dgu
    n, v, k = case["n"], case["v"], case["d"] + (16 if op == "mix_folded" else 0)
    hb, wb = (torch.finfo(_DT[case[x]]).bits // 8 for x in ("h", "w"))
    if op.startswith("rows"):
        return dict(bytes=n * k * hb + v * k * wb + 32 * n, flops=2 * n * v * k)
    return dict(bytes=2 * (n * k * hb + v * k * wb) + 40 * n + 8 * v, flops=6 * n * v * k)


def tolerance(case):
    op = case["op"]
    if op == "induct":
        return "exact"
    if op == "swiglu":
        return {"rel": {"fp32": 2e-6, "fp16": 1.5e-3, "bf16": 1e-2}[case["dtype"]]}
    if op.startswith("rows"):
        return {"rel": 1e-5, "max": 1e-3}   # fp32 sums of the same bf16 products: up to 2e-6 against exact
    # the logits' gradient is held in bf16 between the products: 2-3e-3 against exact; single elements of it may
    # round the other way
    return {"rel": 1e-2, "max": 0.4}


# ------------------------------------------------------------------------------------------------------- in 64 bits


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    if op == "induct":
        return None
    if op == "swiglu":
        gu, go = s["gu"].detach().double(), s["go"].double()
        a, u = gu.chunk(2, -1)
        sg = torch.sigmoid(a)
        return a * sg * u, torch.cat([go * u * (sg + a * sg * (1 - sg)), go * a * sg], -1)
    # the products are of bf16 operands
    h = s["h"].detach().to(torch.bfloat16).double()
    w = s["w"].detach().to(torch.bfloat16).double()
    y = s["y"]
    n, v, v_real = case["n"], case["v"], case["v_real"]
    bias = s["bias"].detach().double() if "bias" in s else None
    go = 1.0 / n
    train = not op.startswith("rows")
    dh, dw = (torch.zeros_like(h), torch.zeros_like(w)) if train else (None, None)
    db = torch.zeros(v, dtype=torch.float64, device=_DEV)
    rows = {k: torch.zeros(n, dtype=torch.float64, device=_DEV) for k in ("loss", "lse", "ly", "wgt", "dgr")}
    dcand = torch.zeros(s["cand"].shape, dtype=torch.float64, device=_DEV) if op == "sparse" else None
    step = max(1, (1 << 27) // v)
    for i in range(0, n, step):
        j = min(n, i + step)
        x = h[i:j] @ w.t()
        if bias is not None:
            x += bias
        if v_real < v:
            x[:, v_real:] = -math.inf
        if op == "sparse":
            x.scatter_add_(1, s["cand"][i:j], s["b"][i:j].detach().double())
        lse = torch.logsumexp(x, 1)
        ok = (y[i:j] >= 0) & (y[i:j] < v_real)
        yc = y[i:j].clamp(0, v - 1)[:, None]
        ly = x.gather(1, yc)[:, 0]
        rows["lse"][i:j], rows["ly"][i:j] = lse, ly
        if "gate" in s:
            gt, hit = s["gate"][i:j].detach().double(), s["hit"][i:j].double()
            py = (ly - lse).exp()
            pr = (1 - gt) * py + gt * hit
            rows["loss"][i:j] = -pr.clamp(min=1e-30).log()
            keep = pr >= 1e-30
            wgt = torch.where(keep, (1 - gt) * py / pr, 0.0)
            rows["dgr"][i:j] = torch.where(keep, (py - hit) / pr, 0.0)
        else:
            rows["loss"][i:j] = torch.where(ok, lse - ly, 0.0)
            wgt = ok.double()
        rows["wgt"][i:j] = wgt
        if not train:
            continue
        gl, gy = (s["g_lse"][i:j].double(), s["g_ly"][i:j].double()) if op == "chunk" else (go * wgt, -go * wgt)
        grad = (x - lse[:, None]).exp_().mul_(gl[:, None])
        grad.scatter_add_(1, yc, (gy * ok)[:, None])
        dh[i:j] = grad @ w
        dw.addmm_(grad.t(), h[i:j])
        db += grad.sum(0)
        if op == "sparse":
            dcand[i:j] = grad.gather(1, s["cand"][i:j])
        del x, grad
    loss = rows["loss"].sum()
    if op.startswith("rows"):
        return dict(loss_sum=loss, loss_rows=rows["loss"], lse=rows["lse"], wgt=rows["wgt"], dgr=rows["dgr"])
    if op == "chunk":
        return rows["lse"], rows["ly"], dh, dw, db
    if op == "mix_biased":
        return loss, dh, dw, db, go * rows["dgr"]
    if op == "mix_folded":
        return loss, dh, dw, go * rows["dgr"]
    if op == "sparse":
        return loss, dh, dw, dcand
    return loss, dh, dw
