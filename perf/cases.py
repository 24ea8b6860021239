"""The work that fine-tuning has this framework do, as cases that can be timed.

A case is one pass of one layer's operator over a batch that is resident on
the GPU, forward and backward unless it says otherwise, through the C ABI's
Python binding (attention, q/k prologue, LoRA linear) or the torch helpers
(the language-model losses), with descriptors, buffers and workspaces made
once, as a training loop keeps them.

  attn       fused attention: causal, sliding window, right padding, or an
             additive mask tensor (left padding); fp32 and bf16
  prologue   a layer's q and k heads through RMSNorm and RoPE, as one batch
  lm_head    streaming cross-entropy from hidden states and the LM head
  dense_ce   cross-entropy of given logits
  lora       LoRA-augmented linear layer

Inputs are normal values of the sizes the layers see (unit q, k, v; output
gradients of 0.1; labels with a tenth ignored, as prompt tokens are).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mobilefinetuner_amd import capi
from mobilefinetuner_amd import lm_loss as L

NEG = -1e10  # the reference's additive mask value
EPS = 1e-6
DT = {"f32": torch.float32, "bf16": torch.bfloat16}
CODE = {"f32": capi.MFT_F32, "bf16": capi.MFT_BF16}
NORM = {"none": capi.MFT_NORM_NONE, "gemma": capi.MFT_NORM_GEMMA, "affine": capi.MFT_NORM_AFFINE}


# --------------------------------------------------------------------- cases
def _attn(dtype, B, Hq, Hkv, S, D, mask="causal", window=0, shortest=0, grad=True, bshd=False):
    return dict(kind="attn", dtype=dtype, B=B, Hq=Hq, Hkv=Hkv, S=S, D=D, mask=mask, window=window,
                shortest=shortest or S, grad=grad, bshd=bshd)


def _prologue(dtype, B, Hq, Hkv, S, D, norm, theta):
    return dict(kind="prologue", dtype=dtype, B=B, Hq=Hq, Hkv=Hkv, S=S, D=D, norm=norm, theta=theta)


def _lm_head(dtype, B, S, H, V):
    return dict(kind="lm_head", dtype=dtype, B=B, S=S, H=H, V=V)


def _dense_ce(dtype, B, S, V):
    return dict(kind="dense_ce", dtype=dtype, B=B, S=S, V=V)


def _lora(w, N, n_in, n_out, r, w_out_in, bias):
    return dict(kind="lora", w=w, N=N, n_in=n_in, n_out=n_out, r=r, w_out_in=w_out_in, bias=bias)


def listed():
    return [
        # GPT-2 small on short sequences in fp32: the smallest step, four launches of a few microseconds
        dict(_attn("f32", 4, 12, 12, 128, 64), name="attn_gpt2_short"),
        # GPT-2 medium in fp32 on a batch whose length fills no tile
        dict(_attn("f32", 4, 16, 16, 487, 64), name="attn_gpt2_ragged"),
        # Qwen2.5-0.5B evaluation (perplexity): forward alone, nothing kept for a backward
        dict(_attn("bf16", 2, 14, 2, 2048, 64, grad=False), name="attn_qwen_eval"),
        # Gemma-3-1B's global layers at the longest context
        dict(_attn("bf16", 1, 4, 1, 4096, 256), name="attn_gemma_long"),
        # Gemma-3's sliding layers on a right-padded batch, q, k, v as the projections leave them ([B,S,H,D])
        dict(_attn("bf16", 3, 4, 1, 1000, 256, "window_pad", 512, 390, bshd=True), name="attn_gemma_sliding"),
        # Qwen2.5-0.5B on a left-padded batch: the base and padding masks come as tensors
        dict(_attn("bf16", 4, 14, 2, 512, 64, "leftpad", shortest=200), name="attn_qwen_leftpad"),
        # Gemma-3-1B's q/k RMSNorm and RoPE at the longest context
        dict(_prologue("bf16", 1, 4, 1, 4096, 256, "gemma", 1e6), name="prologue_gemma"),
        # Gemma-3-1B's LM head and loss over 4096 positions: the largest call of a step
        dict(_lm_head("bf16", 1, 4096, 1152, 262144), name="lm_head_gemma"),
        # GPT-2 small's LM head and loss in fp32, with a vocabulary of odd size
        dict(_lm_head("f32", 4, 128, 768, 50257), name="lm_head_gpt2"),
        # the loss of logits that GPT-2 has written out, rows of an odd number of values
        dict(_dense_ce("f32", 4, 512, 50257), name="dense_ce_gpt2"),
        # Gemma-3-1B's gate projection with LoRA on a frozen bf16 weight, as the injector stores it
        dict(_lora("bf16", 4096, 1152, 6912, 8, True, False), name="lora_gemma_gate"),
        # GPT-2 small's fused q/k/v projection with LoRA on its fp32 weight, on a short batch
        dict(_lora("f32", 509, 768, 2304, 8, False, True), name="lora_gpt2_qkv"),
    ]


def _log(rng, lo, hi):
    """A whole number, spread over its logarithm; half of them odd."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, n | 1) if rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(["attn"] * 6 + ["prologue", "lm_head", "lm_head", "dense_ce", "lora", "lora"])
    heads = rng.choice([(12, 12, 64), (16, 16, 64), (14, 2, 64), (8, 4, 128), (4, 1, 256)])
    Hq, Hkv, D = heads
    if kind == "attn":
        dtype = rng.choice(["f32", "bf16", "bf16"])
        mask = rng.choice(["causal", "causal", "causal", "pad", "window", "window_pad", "leftpad"])
        S = _log(rng, 32, 1024 if mask == "leftpad" else 4096)
        B = min(8, max(1, rng.randrange(1024, 8193) // S))
        window = _log(rng, 16, 1024) if "window" in mask else 0
        shortest = rng.randrange(max(1, S // 4), S + 1) if "pad" in mask else 0
        return _attn(dtype, B, Hq, Hkv, S, D, mask, window, shortest, rng.random() < 0.75, rng.random() < 0.4)
    if kind == "prologue":
        S = _log(rng, 64, 4096)
        B = min(8, max(1, rng.randrange(1024, 8193) // S))
        norm, theta = rng.choice([("gemma", 1e6), ("gemma", 1e4), ("affine", 1e6), ("none", 1e6)])
        return _prologue(rng.choice(["f32", "bf16", "bf16"]), B, Hq, Hkv, S, D, norm, theta)
    if kind == "lm_head":
        dtype = rng.choice(["f32", "bf16", "bf16"])
        S = _log(rng, 64, 2048)
        B = max(1, rng.randrange(128, 4097) // S) if dtype == "bf16" else max(1, rng.randrange(128, 1025) // S)
        return _lm_head(dtype, B, S, rng.choice([640, 768, 896, 1024, 1152]),
                        _log(rng, 8192, 262144 if dtype == "bf16" else 65536))
    if kind == "dense_ce":
        V = _log(rng, 8192, 262144)
        N = _log(rng, 64, max(65, min(4096, (3 << 26) // V)))
        return _dense_ce(rng.choice(["f32", "bf16"]), 1, N, V)
    n_in, n_out = rng.choice([(640, 1024), (640, 2048), (768, 768), (768, 2304), (768, 3072), (896, 896), (896, 4864),
                              (1024, 1152), (1152, 1024), (1152, 6912), (2048, 640), (3072, 768), (6912, 1152)])
    return _lora(rng.choice(["f32", "bf16", "bf16"]), _log(rng, 32, 4096), n_in, n_out, rng.choice([4, 8, 16, 32]),
                 rng.random() < 0.7, rng.random() < 0.4)


# ------------------------------------------------------------------- prepare
def _lengths(c):
    """Valid keys of each sequence, from S down to the shortest."""
    B, S, short = c["B"], c["S"], c["shortest"]
    return [S if B == 1 and "pad" not in c["mask"] else short if B == 1 else S - (S - short) * b // (B - 1)
            for b in range(B)]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _attn_inputs(c, seed):
    g = _gen(seed)
    B, Hq, Hkv, S, D = (c[n] for n in ("B", "Hq", "Hkv", "S", "D"))

    def rand(H, sigma=1.0):
        if c["bshd"]:
            return (sigma * torch.randn(B, S, H, D, device="cuda", generator=g)).to(DT[c["dtype"]]).transpose(1, 2)
        return (sigma * torch.randn(B, H, S, D, device="cuda", generator=g)).to(DT[c["dtype"]])

    q, k, v, dO = rand(Hq), rand(Hkv), rand(Hkv), rand(Hq, 0.1)
    # padding positions carry no loss, so no gradient comes back from them
    for b, n in enumerate(_lengths(c)):
        if c["mask"] == "leftpad":
            dO[b, :, : S - n] = 0
        elif "pad" in c["mask"]:
            dO[b, :, n:] = 0
    return q, k, v, dO


def _masks(c):
    """The base mask [S, S] and the padding mask [B, S], as the model graphs build them."""
    S = c["S"]
    i = torch.arange(S, device="cuda")
    hidden = i[None, :] > i[:, None]
    if c["window"]:
        hidden |= i[:, None] - i[None, :] >= c["window"]
    n = torch.tensor(_lengths(c), device="cuda")[:, None]
    off = i[None, :] < S - n if c["mask"] == "leftpad" else (i[None, :] >= n) & ("pad" in c["mask"])
    return hidden.float() * NEG, off.float() * NEG


def _strides(t):
    return (t.stride(0), t.stride(1), t.stride(2))


def _prepare_attn(c, seed):
    q, k, v, dO = _attn_inputs(c, seed)
    B, Hq, Hkv, S, D = (c[n] for n in ("B", "Hq", "Hkv", "S", "D"))
    o = torch.empty_like(q)
    dq, dk, dv = (torch.empty_like(t, dtype=torch.float32) for t in (q, k, v))
    ops = dict(q=q, k=k, v=v, o=o, dO=dO, dq=dq, dk=dk, dv=dv)
    masks, keep, kv_len = [], [], None
    if c["mask"] == "leftpad":
        base, pad = (m.contiguous() for m in _masks(c))
        masks = [(base.data_ptr(), (0, 0, S, 1)), (pad.data_ptr(), (S, 0, 0, 1))]
        keep = [base, pad]
    elif "pad" in c["mask"]:
        kv_len = torch.tensor(_lengths(c), dtype=torch.int32, device="cuda")
    d = capi.desc(B, Hq, Hkv, S, D, 1.0 / math.sqrt(D), not masks, CODE[c["dtype"]], c["window"],
                  None if kv_len is None else kv_len.data_ptr(),
                  {n: _strides(t) for n, t in ops.items()} if c["bshd"] else None, masks)
    lse = torch.empty(B, Hq, S, *([2] if masks else []), device="cuda")
    f, b = capi.workspace_size(d)
    fws = torch.empty(max(f, 1), dtype=torch.uint8, device="cuda")
    bws = torch.empty(max(b, 1), dtype=torch.uint8, device="cuda")
    p = {n: t.data_ptr() for n, t in ops.items()}
    return dict(c=c, d=d, ops=ops, p=p, lse=lse, plse=lse.data_ptr(), fws=fws, bws=bws,
                pf=fws.data_ptr() if f else None, pb=bws.data_ptr(), keep=(keep, kv_len))


def _prologue_inputs(c, seed):
    g = _gen(seed)
    B, S, D = c["B"], c["S"], c["D"]
    out = []
    for H in (c["Hq"], c["Hkv"]):
        x = torch.randn(B, S, H, D, device="cuda", generator=g).to(DT[c["dtype"]]).transpose(1, 2)
        w = None if c["norm"] == "none" else 0.3 * torch.randn(D, device="cuda", generator=g)
        dy = 0.1 * torch.randn(B, H, S, D, device="cuda", generator=g)  # the attention's dq or dk
        out.append((x, w, dy))
    return out


def _prepare_prologue(c, seed):
    ins = _prologue_inputs(c, seed)
    B, S, D = c["B"], c["S"], c["D"]
    ds, ys, dxs, dws = [], [], [], []
    for x, w, _ in ins:
        H = x.shape[1]
        ds.append(capi.prologue_desc(B, H, S, D, CODE[c["dtype"]], NORM[c["norm"]], EPS, c["theta"],
                                     dict(x=_strides(x))))
        ys.append(torch.empty(B, H, S, D, dtype=x.dtype, device="cuda"))
        dxs.append(torch.empty(B, H, S, D, device="cuda"))
        dws.append(None if w is None else torch.empty(D, device="cuda"))
    n = capi.prologue_workspace_size_n(ds)
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")

    def ptr(ts):
        return [0 if t is None else t.data_ptr() for t in ts]

    xs, wts, dys = zip(*ins)
    return dict(c=c, ds=ds, keep=ins, ys=ys, dxs=dxs, dws=dws, ws=ws, pw=ws.data_ptr() if n else None,
                px=ptr(xs), pwt=ptr(wts), pdy=ptr(dys), py=ptr(ys), pdx=ptr(dxs), pdw=ptr(dws))


def _labels(c, g):
    B, S, V = c["B"], c["S"], c["V"]
    y = torch.randint(0, V, (B, S), device="cuda", generator=g, dtype=torch.int32)
    off = torch.rand(B, S, device="cuda", generator=g) < 0.1
    off[:, -1] = False  # at least one position of each sequence is scored
    return torch.where(off, torch.full_like(y, -100), y)


def _prepare_lm_head(c, seed):
    g = _gen(seed)
    h = (0.5 * torch.randn(c["B"], c["S"], c["H"], device="cuda", generator=g)).to(DT[c["dtype"]])
    w = (0.05 * torch.randn(c["V"], c["H"], device="cuda", generator=g)).to(DT[c["dtype"]])
    return dict(c=c, hidden=h, weight=w, labels=_labels(c, g), one=torch.ones(1, device="cuda"))


def _prepare_dense_ce(c, seed):
    g = _gen(seed)
    z = (2.0 * torch.randn(c["B"], c["S"], c["V"], device="cuda", generator=g)).to(DT[c["dtype"]])
    return dict(c=c, logits=z, labels=_labels(c, g), one=torch.ones(1, device="cuda"))


def _lora_inputs(c, seed):
    g = _gen(seed)
    N, I, O, r = c["N"], c["n_in"], c["n_out"], c["r"]

    def rand(sigma, *shape):
        return sigma * torch.randn(*shape, device="cuda", generator=g)

    # W and the adapters in the injector's layout ([out, in], A [r, in], B [out, r]) or in GPT-2's ([in, out])
    W = rand(0.03, *((O, I) if c["w_out_in"] else (I, O))).to(DT[c["w"]])
    A = rand(0.02, *((r, I) if c["w_out_in"] else (I, r)))
    B = rand(0.02, *((O, r) if c["w_out_in"] else (r, O)))
    return dict(x=rand(1.0, N, I), W=W, A=A, B=B, bias=rand(0.1, O) if c["bias"] else None, dy=rand(0.1, N, O))


def _prepare_lora(c, seed):
    t = _lora_inputs(c, seed)
    N, I, O, r = c["N"], c["n_in"], c["n_out"], c["r"]
    t.update(y=torch.empty(N, O, device="cuda"), u=torch.empty(N, r, device="cuda"), dx=torch.empty(N, I, device="cuda"),
             gA=torch.empty_like(t["A"]), gB=torch.empty_like(t["B"]))
    p = {n: None if v is None else v.data_ptr() for n, v in t.items()}
    d = capi.lora_desc(N, I, O, CODE[c["w"]], c["w_out_in"],
                       [dict(A=p["A"], B=p["B"], grad_A=p["gA"], grad_B=p["gB"], scale=2.0, rank=r, col0=0, cols=O,
                             a_transposed=c["w_out_in"], b_transposed=c["w_out_in"])])
    ws = torch.empty(max(capi.lora_workspace_size(d)), dtype=torch.uint8, device="cuda")
    return dict(c=c, d=d, t=t, p=p, ws=ws, pws=ws.data_ptr())


def prepare(case, seed):
    s = globals()["_prepare_" + case["kind"]](case, seed)
    s["stream"] = torch.cuda.current_stream().cuda_stream
    return s


# ----------------------------------------------------------------------- run
def _run_attn(s):
    p, st = s["p"], s["stream"]
    grad = s["c"]["grad"]
    capi.attn_fwd(s["d"], p["q"], p["k"], p["v"], p["o"], s["plse"] if grad else None, s["pf"], st)
    if not grad:
        return {"o": s["ops"]["o"]}
    capi.attn_bwd(s["d"], p["q"], p["k"], p["v"], p["o"], p["dO"], s["plse"], p["dq"], p["dk"], p["dv"], s["pb"], st)
    return {"lse": s["lse"], **{n: s["ops"][n] for n in ("o", "dq", "dk", "dv")}}


def _run_prologue(s):
    st = s["stream"]
    capi.prologue_fwd_n(s["ds"], s["px"], s["pwt"], s["py"], st)
    capi.prologue_bwd_n(s["ds"], s["px"], s["pwt"], s["pdy"], s["pdx"], s["pdw"], s["pw"], st)
    return {"y": s["ys"], "dx": s["dxs"], "dw": s["dws"]}


def _run_lm_head(s):
    h, w, y = s["hidden"], s["weight"], s["labels"]
    loss, lse = L.streaming_lm_cross_entropy(h, w, y, check_labels=False)
    gh, gw = L.streaming_lm_cross_entropy_backward(h, w, y, lse, s["one"])
    return {"loss": loss, "lse": lse, "grad_hidden": gh, "grad_weight": gw}


def _run_dense_ce(s):
    z, y = s["logits"], s["labels"]
    loss, lse = L.lm_cross_entropy(z, y, check_labels=False)
    return {"loss": loss, "lse": lse, "grad": L.lm_cross_entropy_backward(z, y, lse, s["one"])}


def _run_lora(s):
    p, st = s["p"], s["stream"]
    capi.lora_fwd(s["d"], p["x"], p["W"], p["bias"], p["y"], p["u"], s["pws"], st)
    capi.lora_bwd(s["d"], p["x"], p["W"], p["dy"], p["u"], p["dx"], s["pws"], st)
    return {n: s["t"][n] for n in ("y", "dx", "gA", "gB")}


def run(state):
    return globals()["_run_" + state["c"]["kind"]](state)


# ---------------------------------------------------------------------- work
def _pairs(c):
    """Visible (query, key) pairs of the batch, per query head."""
    S, w = c["S"], c["window"] or c["S"]
    i = np.arange(S)
    total = 0
    for n in _lengths(c):
        lo = np.maximum(0, i - w + 1)
        hi = i
        if c["mask"] == "leftpad":
            lo = np.maximum(lo, S - n)
        elif "pad" in c["mask"]:
            hi = np.minimum(i, n - 1)
        total += int(np.maximum(0, hi - lo + 1).sum())
    return total


def work(case):
    c, kind = case, case["kind"]
    if kind == "attn":
        e = 2 if c["dtype"] == "bf16" else 4
        nq, nk = c["B"] * c["Hq"] * c["S"] * c["D"], c["B"] * c["Hkv"] * c["S"] * c["D"]
        unit = 2.0 * c["D"] * c["Hq"] * _pairs(c)  # one product over the visible pairs
        if not c["grad"]:
            return {"bytes": e * (2 * nq + 2 * nk), "flops": 2 * unit}
        # q, k, v, dO in; o, lse, dq, dk, dv out; two products forward and five backward
        return {"bytes": e * (3 * nq + 2 * nk) + 4 * (nq + 2 * nk) + 4 * nq // c["D"], "flops": 7 * unit}
    if kind == "prologue":
        e = 2 if c["dtype"] == "bf16" else 4
        n = c["B"] * (c["Hq"] + c["Hkv"]) * c["S"] * c["D"]
        return {"bytes": n * (2 * e + 8), "flops": 20.0 * n}
    if kind == "lm_head":
        e = 2 if c["dtype"] == "bf16" else 4
        N, H, V = c["B"] * c["S"], c["H"], c["V"]
        # logits forward and again backward (they are never kept), grad_hidden, grad_weight
        return {"bytes": (e + 4) * (N * H + V * H), "flops": 8.0 * N * V * H}
    if kind == "dense_ce":
        e = 2 if c["dtype"] == "bf16" else 4
        n = c["B"] * c["S"] * c["V"]
        return {"bytes": (e + 4) * n, "flops": 10.0 * n}
    N, I, O, r = c["N"], c["n_in"], c["n_out"], c["r"]
    e = 2 if c["w"] == "bf16" else 4
    # x, W, A, B, dy in; y, dx, grad_A, grad_B out; W's products both ways, u and its update, g, grad_A, grad_B, dx's update
    return {"bytes": 4 * (2 * N * I + 2 * N * O) + e * I * O + 8 * r * (I + O),
            "flops": 4.0 * N * I * O + 6.0 * N * r * (I + O)}


def tolerance(case):
    c, kind = case, case["kind"]
    if kind == "lora":
        return {"rel": 1e-2} if c["w"] == "bf16" else {"rel": 1e-5}
    return {"rel": 1e-2} if c["dtype"] == "bf16" else {"rel": 1e-5}


# --------------------------------------------------------------------- exact
def _exact_attn(c, seed):
    q, k, v, dO = (t.double() for t in _attn_inputs(c, seed))
    S, r = c["S"], c["Hq"] // c["Hkv"]
    scale = 1.0 / math.sqrt(c["D"])
    base, pad = (m.double() for m in _masks(c))
    o, dq = torch.empty_like(q), torch.empty_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    lse = torch.empty(*q.shape[:3], *([2] if c["mask"] == "leftpad" else []), dtype=torch.float64, device="cuda")
    for b in range(c["B"]):
        m = base + pad[b][None, :]
        off = m < 0.5 * NEG  # adding -1e10 in single precision leaves nothing of the score
        for h in range(c["Hq"]):
            x = torch.where(off, m, scale * (q[b, h] @ k[b, h // r].T))
            top = x.max(dim=1, keepdim=True).values
            P = (x - top).exp_()
            total = P.sum(dim=1, keepdim=True)
            P /= total
            if c["mask"] == "leftpad":
                lse[b, h] = torch.cat([top, total.log()], dim=1)
            else:
                lse[b, h] = torch.where(off.all(dim=1), math.inf, (top + total.log())[:, 0])
            o[b, h] = P @ v[b, h // r]
            dP = dO[b, h] @ v[b, h // r].T
            dS = P * (dP - (dO[b, h] * o[b, h]).sum(dim=1, keepdim=True))
            dv[b, h // r] += P.T @ dO[b, h]
            dq[b, h] = scale * (dS @ k[b, h // r])
            dk[b, h // r] += scale * (dS.T @ q[b, h])
    return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv} if c["grad"] else {"o": o}


def _exact_prologue(c, seed):
    S, D = c["S"], c["D"]
    # the rotation's frequencies and angles are single-precision numbers by definition
    f = np.float32(1) / np.power(np.float32(c["theta"]), np.arange(0, D, 2, dtype=np.float32) / np.float32(D))
    ang = torch.from_numpy(np.arange(S, dtype=np.float32)[:, None] * f[None, :].astype(np.float32)).cuda().double()
    cos, sin = ang.cos(), ang.sin()
    ys, dxs, dws = [], [], []
    for x, w, dy in _prologue_inputs(c, seed):
        x, dy = x.double(), dy.double()
        if w is not None:
            gain = w.double() + (1.0 if c["norm"] == "gemma" else 0.0)
            inv = 1.0 / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + float(np.float32(EPS)))
            n = x * inv
            z = n * gain
        else:
            z = x
        a, b = z[..., : D // 2], z[..., D // 2:]
        ys.append(torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1))
        a, b = dy[..., : D // 2], dy[..., D // 2:]
        dz = torch.cat([a * cos + b * sin, b * cos - a * sin], dim=-1)
        if w is None:
            dxs.append(dz)
            dws.append(None)
            continue
        dn = dz * gain
        dxs.append(inv * (dn - n * (dn * n).mean(dim=-1, keepdim=True)))
        dws.append((dz * n).sum(dim=(0, 1, 2)))
    return {"y": ys, "dx": dxs, "dw": dws}


def _targets(c, labels):
    """Scored positions and their targets: position s is scored against labels[:, s + 1]."""
    t = torch.full_like(labels, -100)
    t[:, :-1] = labels[:, 1:]
    t = t.reshape(-1).long()
    return t, t >= 0


def _exact_lm_head(c, seed):
    s = _prepare_lm_head(c, seed)
    N, H, V = c["B"] * c["S"], c["H"], c["V"]
    h, w = s["hidden"].double().reshape(N, H), s["weight"]
    t, on = _targets(c, s["labels"])
    step, top, total = 8192, torch.full((N,), -math.inf, dtype=torch.float64, device="cuda"), torch.zeros(
        N, dtype=torch.float64, device="cuda")
    at = torch.zeros_like(total)
    for v in range(0, V, step):
        z = h @ w[v: v + step].double().T
        m = torch.maximum(top, z.max(dim=1).values)
        total = total * (top - m).exp() + (z - m[:, None]).exp().sum(dim=1)
        top = m
        here = on & (t >= v) & (t < v + step)
        at[here] = z[here, t[here] - v]
    lse = top + total.log()
    loss = (lse - at)[on].mean().reshape(1)
    gh, gw = torch.zeros_like(h), torch.empty(V, H, dtype=torch.float64, device="cuda")
    for v in range(0, V, step):
        wc = w[v: v + step].double()
        g = (h @ wc.T - lse[:, None]).exp_()
        here = on & (t >= v) & (t < v + step)
        g[here, t[here] - v] -= 1.0
        g *= on[:, None] / on.sum()
        gh += g @ wc
        gw[v: v + step] = g.T @ h
    lse = torch.where(on, lse, 0.0)
    return {"loss": loss, "lse": lse.reshape(c["B"], c["S"]), "grad_hidden": gh.reshape(c["B"], c["S"], H),
            "grad_weight": gw}


def _exact_dense_ce(c, seed):
    s = _prepare_dense_ce(c, seed)
    z = s["logits"].double().reshape(-1, c["V"])
    t, on = _targets(c, s["labels"])
    lse = torch.logsumexp(z, dim=1)
    rows = torch.nonzero(on)[:, 0]
    loss = (lse[rows] - z[rows, t[rows]]).mean().reshape(1)
    g = (z - lse[:, None]).exp_()
    g[rows, t[rows]] -= 1.0
    g *= on[:, None] / on.sum()
    return {"loss": loss, "lse": torch.where(on, lse, 0.0).reshape(c["B"], c["S"]),
            "grad": g.reshape(c["B"], c["S"], c["V"])}


def _exact_lora(c, seed):
    t = {n: None if v is None else v.double() for n, v in _lora_inputs(c, seed).items()}
    W, A, B = (t[n].T if c["w_out_in"] else t[n] for n in ("W", "A", "B"))
    u = t["x"] @ A
    y = t["x"] @ W + 2.0 * (u @ B)
    if t["bias"] is not None:
        y = y + t["bias"]
    g = 2.0 * (t["dy"] @ B.T)
    gA, gB = t["x"].T @ g, 2.0 * (u.T @ t["dy"])
    return {"y": y, "dx": t["dy"] @ W.T + g @ A.T, "gA": gA.T if c["w_out_in"] else gA,
            "gB": gB.T if c["w_out_in"] else gB}


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)
