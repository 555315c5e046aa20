"""The work that a program built on ugk has it do, as cases to time and to check.

A case is a dict of plain values; its "kind" names the path it takes through the public entry points:

  layernorm  one LayerNorm, forward and backward (the per-op entry points)
  block      one transformer block's layer kernels around the caller's GEMMs and attention, forward and
             backward, over buffers cut from one flat activation array as the step driver lays them out
  encoder    token + position embedding, forward (gather) and backward (scatter-add)
  head       softmax + cross-entropy over the vocabulary and its gradient
  posterior  the Bayes-by-Backprop parameter update: "fused" (one pass), "drawn" (op by op, eps from
             Philox) or "given" (op by op, eps in memory, with the KL total a program logs)
  step       bayes_materialize and the GPT-2 layer-kernel driver, forward and backward (or forward alone,
             as an evaluation runs it)

"exact" selects the modes whose results equal the CPU's bit for bit. Backward outputs accumulate, as in
gradient accumulation; nothing is cleared between passes.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "uncertain-gpt_amd"))

import ugk  # noqa: E402

SEED, STEP = 0x5EED, 3  # of the Philox draws
SP, KLW = 0.1, 1e-6  # prior scale, weight of the KL gradient
LR, BETA1, BETA2, AEPS, WD = 3e-4, 0.9, 0.999, 1e-8, 0.0
MAX_T = 1024  # positions a model's wpe holds


def listed():
    return [
        # one LayerNorm of the character-level model (4 x 64 tokens): a call of a few microseconds
        {"name": "ln_text8", "kind": "layernorm", "B": 4, "T": 64, "C": 384, "exact": False},
        # one LayerNorm of GPT-2-124M over a large batch
        {"name": "ln_gpt2", "kind": "layernorm", "B": 16, "T": 1024, "C": 768, "exact": False},
        # one LayerNorm of a model several times wider, over sequences of odd length
        {"name": "ln_wide", "kind": "layernorm", "B": 4, "T": 1023, "C": 4096, "exact": False},
        # one block of GPT-2-124M over a batch whose odd token count leaves half of the flat buffer's
        # arrays off a 16-byte boundary
        {"name": "block_ragged", "kind": "block", "B": 15, "T": 1023, "C": 768, "exact": False},
        # the embedding of GPT-2-124M with tokens as text has them: a few very frequent, most rare
        {"name": "encoder_zipf", "kind": "encoder", "B": 16, "T": 1024, "C": 768, "V": 50257, "law": "zipf",
         "exact": False},
        # the embedding of the character-level model at its large batch: 27 tokens, hundreds of rows each
        {"name": "encoder_text8", "kind": "encoder", "B": 128, "T": 64, "C": 384, "V": 27, "law": "zipf",
         "exact": False},
        # the head of GPT-2-124M
        {"name": "head_gpt2", "kind": "head", "B": 8, "T": 1024, "V": 50257, "exact": False},
        # the head of a model with a large vocabulary
        {"name": "head_long", "kind": "head", "B": 2, "T": 1024, "V": 100003, "exact": False},
        # the update of the character-level model (11,061,531 parameters) op by op with eps in memory, the
        # form whose results a CPU run can be compared with
        {"name": "posterior_text8", "kind": "posterior", "form": "given", "n": 11061531, "exact": False},
        # the update of GPT-2-124M in the one-pass form a training run takes
        {"name": "posterior_gpt2", "kind": "posterior", "form": "fused", "n": 124439808, "exact": False},
        # the layer kernels of a training step of the character-level model: many launches of little work
        {"name": "step_text8", "kind": "step", "L": 6, "C": 384, "NH": 6, "V": 27, "B": 4, "T": 64, "train": True,
         "exact": False},
        # the layer kernels of a training step of GPT-2-124M
        {"name": "step_gpt2", "kind": "step", "L": 12, "C": 768, "NH": 12, "V": 50257, "B": 8, "T": 1024,
         "train": True, "exact": False},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _channels(rng, lo, hi):
    """A width: mostly a multiple of 64, now and then of 4, seldom any number."""
    c, r = _log_int(rng, lo, hi), rng.random()
    step = 64 if r < 0.7 else 4 if r < 0.9 else 1
    return max(step, c // step * step)


def _batch(rng, rows_lo, rows_hi):
    """B sequences of T tokens, T odd about half of the time."""
    rows = _log_int(rng, rows_lo, rows_hi)
    B = _log_int(rng, 1, max(1, min(16, rows // 32)))
    return B, max(1, min(1024, rows // B - rng.randrange(2)))


def draw(rng):
    kind = rng.choice(("layernorm", "layernorm", "block", "encoder", "encoder", "head", "head", "posterior", "step"))
    exact = rng.random() < 0.2
    if kind == "layernorm":
        C = _channels(rng, 64, 8192)
        B, T = _batch(rng, 64, min(16384, (1 << (22 if exact else 24)) // C))
        return {"kind": kind, "B": B, "T": T, "C": C, "exact": exact}
    if kind == "block":
        C = 64 * _log_int(rng, 2, 25)
        B, T = _batch(rng, 64, min(16384, (1 << 23) // C))
        return {"kind": kind, "B": B, "T": T, "C": C, "exact": exact}
    if kind == "encoder":
        C = _channels(rng, 64, 1600)
        B, T = _batch(rng, 64, 16384)
        return {"kind": kind, "B": B, "T": T, "C": C, "V": _log_int(rng, 27, 50257),
                "law": rng.choice(("uniform", "zipf")), "exact": exact}
    if kind == "head":
        V = _log_int(rng, 27, 200000)
        B, T = _batch(rng, 64, min(8192, (1 << (26 if exact else 28)) // V))
        return {"kind": kind, "B": B, "T": T, "V": V, "exact": exact}
    if kind == "posterior":
        form = rng.choice(("given", "drawn", "fused"))
        return {"kind": kind, "form": form, "n": _log_int(rng, 10000, 100000000 if form == "fused" else 40000000),
                "exact": exact}
    # an evaluation (forward alone) takes sequences of any length; a training step an even token count
    C, L, train = 64 * _log_int(rng, 2, 12), rng.randint(2, 12), rng.random() < 0.6
    B, T = _batch(rng, 64, min(8192, (1 << (22 if exact else 25)) // (C * L)))
    if train and B * T % 2:
        T += 1
    return {"kind": kind, "L": L, "C": C, "NH": C // 64, "V": _log_int(rng, 27, 50257), "B": B, "T": T, "train": train,
            "exact": exact}


# ---- inputs ---------------------------------------------------------------------

class _Rand:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def n(self, *shape, scale=1.0, mean=0.0):
        t = torch.randn(*shape, generator=self.g, device="cuda")
        if scale != 1.0:
            t.mul_(scale)
        return t.add_(mean) if mean else t

    def ids(self, n, V, law="uniform"):
        """Token ids: uniform, or Zipf(1.1) over the vocabulary."""
        if law == "uniform":
            return torch.randint(0, V, (n,), generator=self.g, device="cuda", dtype=torch.int32)
        w = torch.arange(1, V + 1, device="cuda", dtype=torch.float64).pow_(-1.1)
        cdf = torch.cumsum(w, 0)
        u = torch.rand(n, generator=self.g, device="cuda", dtype=torch.float64) * cdf[-1]
        return torch.searchsorted(cdf, u).clamp_(max=V - 1).to(torch.int32)


def _empty(*shape):
    return torch.empty(*shape, device="cuda")


def _zeros(*shape):
    return torch.zeros(*shape, device="cuda")


def _set_modes(exact):
    for f in (ugk.set_gelu_exact, ugk.set_philox_exact, ugk.set_kl_exact, ugk.set_softmax_exact,
              ugk.set_layernorm_exact, ugk.set_encoder_exact):
        f(exact)


def _param_layout(c):
    """Offsets of the flat parameter buffer's parts that the layer kernels use."""
    C, V, L = c["C"], c["V"], c["L"]
    block = {"lng": 0, "lnb": C, "ln2g": 2 * C + 4 * C * C + 4 * C, "ln2b": 3 * C + 4 * C * C + 4 * C}
    stride = 12 * C * C + 13 * C
    blk0 = V * C + MAX_T * C
    end = blk0 + L * stride
    return {"wte": 0, "wpe": V * C, "blk0": blk0, "stride": stride, "block": block, "flng": end, "flnb": end + C}


def _block_layout(BT, C):
    """Offsets and sizes of one block's arrays in the flat activation buffer, and the block's size."""
    at, o = {}, 0
    for name, size in (("lno", BT * C), ("lnm", BT), ("lnr", BT), ("qkv", 3 * BT * C), ("atty", BT * C),
                       ("apr", BT * C), ("resa", BT * C), ("ln2o", BT * C), ("ln2m", BT), ("ln2r", BT),
                       ("fch", 4 * BT * C), ("gelu", 4 * BT * C), ("mlpo", BT * C), ("res1", BT * C)):
        at[name] = (o, size)
        o += size
    return at, o


def _config(c):
    return ugk.Config(B=c["B"], T=c["T"], C=c["C"], V=c["V"], NH=c["NH"], maxT=MAX_T, L=c["L"])


def prepare(case, seed):
    r, c, kind = _Rand(seed), case, case["kind"]
    _set_modes(c["exact"])
    if kind == "posterior":
        n = c["n"]
        s = {"mu": r.n(n, scale=0.02), "rho": r.n(n, scale=0.1, mean=-5.0), "dw": r.n(n, scale=0.01), "w": _zeros(n)}
        for k in ("mu", "rho"):
            s["m_" + k] = r.n(n, scale=0.01)
            s["v_" + k] = r.n(n, scale=1e-4).abs_()
            if c["form"] != "fused":
                s["d" + k] = _zeros(n)
        if c["form"] == "given":
            s["eps"] = r.n(n)
        return {"case": c, **s}
    B, T = c["B"], c["T"]
    BT = B * T
    if kind == "head":
        V = c["V"]
        return {"case": c, "logits": r.n(BT * V, scale=3.0), "targets": r.ids(BT, V), "losses": _empty(BT),
                "probs": _empty(BT * V), "dlogits": _empty(BT * V)}
    C = c["C"]
    if kind == "layernorm":
        return {"case": c, "inp": r.n(BT * C), "weight": r.n(C, scale=0.1, mean=1.0), "bias": r.n(C, scale=0.1),
                "dout": r.n(BT * C), "out": _empty(BT * C), "mean": _empty(BT), "rstd": _empty(BT),
                "dinp": _zeros(BT * C), "dweight": _zeros(C), "dbias": _zeros(C)}
    if kind == "encoder":
        V = c["V"]
        return {"case": c, "inp": r.ids(BT, V, c["law"]), "wte": r.n(V * C, scale=0.02), "wpe": r.n(T * C, scale=0.01),
                "dout": r.n(BT * C), "out": _empty(BT * C), "dwte": _zeros(V * C), "dwpe": _zeros(T * C)}
    if kind == "block":
        at, size = _block_layout(BT, C)
        acts = r.n(BT * C + size)  # the incoming stream, then the block
        grads = _zeros(BT * C + size)
        a = {k: acts[BT * C + o:BT * C + o + m] for k, (o, m) in at.items()}
        g = {k: grads[BT * C + o:BT * C + o + m] for k, (o, m) in at.items()}
        a["in"], g["in"] = acts[:BT * C], grads[:BT * C]
        for k in ("res1", "gelu", "ln2o"):  # the gradients that the caller's ops and the layer above left
            g[k].copy_(r.n(g[k].numel()))
        return {"case": c, "a": a, "g": g, "weight": r.n(C, scale=0.1, mean=1.0), "bias": r.n(C, scale=0.1),
                "dweight": _zeros(C), "dbias": _zeros(C)}
    cfg, lay = _config(c), _param_layout(c)
    n, na, L = ugk.param_count(cfg), ugk.act_count(cfg), c["L"]
    s = {"case": c, "cfg": cfg, "n": n, "mu": r.n(n, scale=0.02), "rho": r.n(n, scale=0.1, mean=-5.0), "eps": r.n(n),
         "w": _empty(n), "inp": r.ids(BT, c["V"], "zipf"), "acts": r.n(na)}
    for l in range(L):
        for k in ("lng", "ln2g"):
            o = lay["blk0"] + l * lay["stride"] + lay["block"][k]
            s["mu"][o:o + C] += 1.0
    s["mu"][lay["flng"]:lay["flng"] + C] += 1.0
    at, stride = _block_layout(BT, C)
    blk0, end = BT * C, BT * C + L * stride

    def blocks(buf, k):
        o, m = at[k]
        return buf[blk0:end].view(L, stride)[:, o:o + m]

    acts = s["acts"]
    out = {"w": s["w"], "enc": acts[:BT * C], "flo": acts[end:end + BT * C], "flm": acts[end + BT * C:][:BT],
           "flr": acts[end + BT * C + BT:][:BT]}
    out.update({k: blocks(acts, k) for k in ("lno", "lnm", "lnr", "resa", "ln2o", "ln2m", "ln2r", "gelu", "res1")})
    if c["train"]:
        # zero but for what the loss and the dense ops between the layer kernels leave
        gacts = s["gacts"] = _zeros(na)
        for k in ("lno", "ln2o", "gelu"):
            v = blocks(gacts, k)
            v.copy_(r.n(*v.shape))
        gacts[end:end + BT * C].copy_(r.n(BT * C))
        s["grads"] = out["grads"] = _zeros(n)
        out["denc"] = gacts[:BT * C]
        out.update({"d" + k: blocks(gacts, k) for k in ("fch", "apr", "mlpo")})
    s["out"] = out
    return s


# ---- one pass -------------------------------------------------------------------

def run(s):
    c = s["case"]
    return _RUN[c["kind"]](s, c)


def _run_layernorm(s, c):
    B, T, C = c["B"], c["T"], c["C"]
    ugk.layernorm_forward(s["out"], s["mean"], s["rstd"], s["inp"], s["weight"], s["bias"], B, T, C)
    ugk.layernorm_backward(s["dinp"], s["dweight"], s["dbias"], s["dout"], s["inp"], s["weight"], s["mean"], s["rstd"],
                           B, T, C)
    return [s[k] for k in ("out", "mean", "rstd", "dinp", "dweight", "dbias")]


def _run_block(s, c):
    B, T, C, a, g = c["B"], c["T"], c["C"], s["a"], s["g"]
    N = B * T * C
    ugk.residual_layernorm_forward(a["resa"], a["ln2o"], a["ln2m"], a["ln2r"], a["in"], a["apr"], s["weight"], s["bias"],
                                   B, T, C)
    ugk.gelu_forward(a["gelu"], a["fch"], 4 * N)
    ugk.residual_forward(a["res1"], a["resa"], a["mlpo"], N)
    ugk.residual_backward(g["resa"], g["mlpo"], g["res1"], N)
    ugk.gelu_backward(g["fch"], a["fch"], g["gelu"], 4 * N)
    ugk.layernorm_residual_backward(g["resa"], s["dweight"], s["dbias"], g["in"], g["apr"], g["ln2o"], a["resa"],
                                    s["weight"], a["ln2m"], a["ln2r"], B, T, C)
    return [a[k] for k in ("resa", "ln2o", "ln2m", "ln2r", "gelu", "res1")] + \
           [g[k] for k in ("resa", "mlpo", "fch", "in", "apr")] + [s["dweight"], s["dbias"]]


def _run_encoder(s, c):
    B, T, C = c["B"], c["T"], c["C"]
    ugk.encoder_forward(s["out"], s["inp"], s["wte"], s["wpe"], B, T, C)
    ugk.encoder_backward(s["dwte"], s["dwpe"], s["dout"], s["inp"], B, T, C)
    return [s["out"], s["dwte"], s["dwpe"]]


def _run_head(s, c):
    B, T, V = c["B"], c["T"], c["V"]
    ugk.softmax_crossentropy(s["losses"], s["probs"], s["logits"], s["targets"], B, T, V)
    ugk.crossentropy_softmax_backward_zeroed(s["dlogits"], s["probs"], s["targets"], B, T, V)
    return [s["losses"], s["probs"], s["dlogits"]]


def _run_posterior(s, c):
    n, form = c["n"], c["form"]
    if form == "fused":
        ugk.bbb_step_fused(s["mu"], s["rho"], s["m_mu"], s["v_mu"], s["m_rho"], s["v_rho"], s["w"], s["dw"], n, SEED,
                           STEP, SP, KLW, 1.0 - BETA1 ** STEP, 1.0 - BETA2 ** STEP, LR, BETA1, BETA2, AEPS, WD)
        return [s[k] for k in ("mu", "rho", "m_mu", "v_mu", "m_rho", "v_rho", "w", "dw")]
    out = [s[k] for k in ("w", "dmu", "drho", "mu", "rho", "m_mu", "v_mu", "m_rho", "v_rho")]
    if form == "drawn":
        ugk.bayes_sample(s["w"], None, s["mu"], s["rho"], n, SEED, STEP)
        ugk.bayes_backward_philox(s["dmu"], s["drho"], s["dw"], s["rho"], n, SEED, STEP)
    else:
        ugk.bayes_materialize(s["w"], s["mu"], s["rho"], s["eps"], n)
        ugk.bayes_backward(s["dmu"], s["drho"], s["dw"], s["eps"], s["rho"], n)
        out.append(ugk.kl_forward(s["mu"], s["rho"], n, SP))
    ugk.kl_backward(s["dmu"], s["drho"], s["mu"], s["rho"], n, SP, KLW)
    for k in ("mu", "rho"):
        ugk.adamw_update(s[k], s["d" + k], s["m_" + k], s["v_" + k], n, STEP, LR, BETA1, BETA2, AEPS, WD)
    return out


def _run_step(s, c):
    ugk.bayes_materialize(s["w"], s["mu"], s["rho"], s["eps"], s["n"])
    ugk.gpt2_layers_forward(s["acts"], s["w"], s["inp"], s["cfg"])
    if c["train"]:
        ugk.gpt2_layers_backward_zeroed(s["grads"], s["gacts"], s["acts"], s["w"], s["inp"], s["cfg"])
    return s["out"]


_RUN = {"layernorm": _run_layernorm, "block": _run_block, "encoder": _run_encoder, "head": _run_head,
        "posterior": _run_posterior, "step": _run_step}


# ---- what a pass cannot do without -------------------------------------------------

def _distinct(n, V, law):
    """The distinct ids that n draws of a law take, on average."""
    if law == "uniform":
        return V * -math.expm1(n * math.log1p(-1.0 / V))
    p = torch.arange(1, V + 1, dtype=torch.float64).pow_(-1.1)
    return float(-torch.expm1(n * torch.log1p(-p / p.sum())).sum())


def work(case):
    """Bytes with each input read once and each output written once (an accumulated output is both), and
    the float operations."""
    c, kind = case, case["kind"]
    if kind == "posterior":
        n = c["n"]
        if c["form"] == "fused":  # dw, mu, rho and the four moments read and written, w written
            return {"bytes": 60 * n, "flops": 100 * n}
        # mu, rho, dmu, drho and the four moments read and written, dw read, w written (eps read)
        return {"bytes": (76 if c["form"] == "given" else 72) * n, "flops": 100 * n}
    BT = c["B"] * c["T"]
    if kind == "head":  # logits read; probs and dlogits written
        N = BT * c["V"]
        return {"bytes": 12 * N + 12 * BT, "flops": 8 * N}
    C = c["C"]
    N = BT * C
    if kind == "layernorm":  # inp, dout read; out written; dinp read and written
        return {"bytes": 20 * N + 8 * BT + 24 * C, "flops": 25 * N}
    if kind == "encoder":
        rows = _distinct(BT, c["V"], c["law"])  # of wte read, and of dwte read and written
        return {"bytes": 8 * N + 12 * rows * C + 12 * c["T"] * C + 4 * BT, "flops": 3 * N}
    if kind == "block":
        # read: in, apr, fch, mlpo, the gradients of res1, gelu, ln2o; written: resa, ln2o, gelu, res1;
        # read and written: the gradients of resa, mlpo, in, apr and fch
        return {"bytes": 4 * N * (1 + 1 + 4 + 1 + 1 + 4 + 1 + 1 + 1 + 4 + 1 + 2 * (1 + 1 + 1 + 1 + 4)) + 8 * BT + 24 * C,
                "flops": 150 * N}
    L, V = c["L"], c["V"]
    n = V * C + MAX_T * C + L * (12 * C * C + 13 * C) + 2 * C + C * V + V
    rows = _distinct(BT, V, "zipf")
    # materialize; wte rows and wpe read, enc and the first LayerNorm's output written; per block apr, fch,
    # mlpo read and resa, ln2o, gelu, res1, the next LayerNorm's output written
    total = 16 * n + 4 * (rows * C + c["T"] * C + 2 * N) + 4 * N * L * (1 + 4 + 1 + 1 + 1 + 4 + 1 + 1)
    if c["train"]:
        # per block: dgelu, fch, dln2o, dlno, resa, res1 read; dfch, dresa, dmlpo, dapr, dres1 written; and
        # the last LayerNorm's dout, the encoder's gradient and its tables' rows
        total += 4 * N * L * (4 + 4 + 1 + 1 + 1 + 1 + 4 + 1 + 1 + 1 + 1) + 8 * N + 8 * (rows * C + c["T"] * C)
    return {"bytes": total, "flops": 150 * N * L}


def tolerance(case):
    """32-bit sums in any order: the results are 3e-8 to 2e-7 (2-norm) from their 64-bit values at every
    size, so two sound orders differ by up to 3e-7. The exact modes promise the CPU's bits; the KL total is a
    64-bit sum in either mode."""
    if not case["exact"]:
        return {"rel": 1e-6, "max": 2e-5}
    return {"rel": 1e-13, "max": 1e-12} if case["kind"] == "posterior" else "exact"


# ---- the same in 64 bits -------------------------------------------------------------

_GELU_K = math.sqrt(2.0 / math.pi)


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.tanh(_GELU_K * (x + 0.044715 * x ** 3)))


def _gelu_grad64(x):
    t = torch.tanh(_GELU_K * (x + 0.044715 * x ** 3))
    return 0.5 * (1.0 + t) + 0.5 * x * (1.0 - t * t) * _GELU_K * (1.0 + 3 * 0.044715 * x * x)


def _ln64(x, w, b):
    m = x.mean(1, keepdim=True)
    r = ((x - m).square().mean(1, keepdim=True) + 1e-5).rsqrt()
    return (x - m) * r * w + b, m.reshape(-1), r.reshape(-1)


def _ln_bwd64(dout, x, w, m, r):
    """dinp, dweight and dbias of a LayerNorm."""
    xh = (x - m[:, None]) * r[:, None]
    dn = dout * w
    dinp = r[:, None] * (dn - dn.mean(1, keepdim=True) - xh * (dn * xh).mean(1, keepdim=True))
    return dinp, (dout * xh).sum(0), dout.sum(0)


def _softplus64(x):
    return torch.where(x > 20.0, x, torch.log1p(torch.exp(x)))


def _philox_normal64(seed, step, n):
    """The stream's normals: Philox4x32-10 words to float uniforms, Box-Muller's cosine branch in 64 bits."""
    mask = 0xFFFFFFFF
    i = torch.arange(n, device="cuda", dtype=torch.int64)
    c0, c1, c2, c3 = i & mask, i >> 32, torch.full_like(i, step), torch.zeros_like(i)
    k0, k1 = seed & mask, seed >> 32

    def mul(a, x):  # high and low words of a 32 x 32 bit product
        hi = (a * (x >> 16) + (a * (x & 0xFFFF) >> 16)) >> 16
        return hi, a * x & mask

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c0)
        h1, l1 = mul(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    u1, u2 = (((x.to(torch.float32) + 0.5) * 2.0 ** -32).double() for x in (c0, c1))
    return torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(2.0 * math.pi * u2)


def _adamw64(p, g, m, v, bc1, bc2):
    m = BETA1 * m + (1.0 - BETA1) * g
    v = BETA2 * v + (1.0 - BETA2) * g * g
    return p - LR * ((m / bc1) / (torch.sqrt(v / bc2) + AEPS) + WD * p), m, v


def exact(case, seed):
    s = prepare(case, seed)
    return _EXACT[case["kind"]](s, case)


def _exact_layernorm(s, c):
    C = c["C"]
    x, dout, w, b = s["inp"].double().view(-1, C), s["dout"].double().view(-1, C), s["weight"].double(), s["bias"].double()
    out, m, r = _ln64(x, w, b)
    dinp, dw, db = _ln_bwd64(dout, x, w, m, r)
    return [out.reshape(-1), m, r, dinp.reshape(-1), dw, db]


def _exact_block(s, c):
    C = c["C"]
    a, g = ({k: v.double() for k, v in s[q].items()} for q in ("a", "g"))
    w, b = s["weight"].double(), s["bias"].double()
    resa = a["in"] + a["apr"]
    ln2o, m, r = _ln64(resa.view(-1, C), w, b)
    gresa = g["resa"] + g["res1"]
    dinp, dw, db = _ln_bwd64(g["ln2o"].view(-1, C), resa.view(-1, C), w, m, r)
    gresa = gresa + dinp.reshape(-1)
    return [resa, ln2o.reshape(-1), m, r, _gelu64(a["fch"]), resa + a["mlpo"], gresa, g["mlpo"] + g["res1"],
            g["fch"] + _gelu_grad64(a["fch"]) * g["gelu"], g["in"] + gresa, g["apr"] + gresa, dw, db]


def _exact_encoder(s, c):
    B, T, C = c["B"], c["T"], c["C"]
    ids, dout = s["inp"].long(), s["dout"].double().view(B * T, C)
    out = s["wte"].double().view(-1, C)[ids].view(B, T, C) + s["wpe"].double().view(T, C)
    dwte = s["dwte"].double().view(-1, C).index_add_(0, ids, dout)
    return [out.reshape(-1), dwte.reshape(-1), dout.view(B, T, C).sum(0).reshape(-1)]


def _exact_head(s, c):
    V, t = c["V"], s["targets"].long()
    p = torch.softmax(s["logits"].double().view(-1, V), 1)
    losses = -torch.log(p.gather(1, t[:, None]))
    d = p / p.shape[0]
    d.scatter_add_(1, t[:, None], torch.full_like(losses, -1.0 / p.shape[0]))
    return [losses.reshape(-1), p.reshape(-1), d.reshape(-1)]


def _exact_posterior(s, c):
    n, form, s = c["n"], c["form"], {k: v.double() for k, v in s.items() if k != "case"}
    mu, rho, dw, sp2 = s["mu"], s["rho"], s["dw"], SP * SP
    bc1, bc2 = 1.0 - BETA1 ** STEP, 1.0 - BETA2 ** STEP
    eps = s["eps"] if form == "given" else _philox_normal64(SEED, STEP, n)
    sigma, sg = _softplus64(rho), torch.sigmoid(rho)
    dmu = dw + KLW * mu / sp2
    drho = dw * eps * sg + KLW * (sigma / sp2 - 1.0 / sigma) * sg
    mu1, m_mu, v_mu = _adamw64(mu, dmu, s["m_mu"], s["v_mu"], bc1, bc2)
    rho1, m_rho, v_rho = _adamw64(rho, drho, s["m_rho"], s["v_rho"], bc1, bc2)
    if form == "fused":
        return [mu1, rho1, m_mu, v_mu, m_rho, v_rho, mu1 + _softplus64(rho1) * _philox_normal64(SEED, STEP + 1, n),
                torch.zeros_like(dw)]
    out = [mu + sigma * eps, dmu, drho, mu1, rho1, m_mu, v_mu, m_rho, v_rho]
    if form == "given":
        out.append(float((torch.log(SP / sigma) + (sigma * sigma + mu * mu) / (2.0 * sp2) - 0.5).sum()))
    return out


def _exact_step(s, c):
    L, C, V, B, T = (c[k] for k in ("L", "C", "V", "B", "T"))
    BT, lay = B * T, _param_layout(c)
    at, stride = _block_layout(BT, C)
    w = s["mu"].double() + _softplus64(s["rho"].double()) * s["eps"].double()

    def p(l, k):
        o = lay["blk0"] + l * lay["stride"] + lay["block"][k]
        return slice(o, o + C)

    def act(buf, l, k):
        o, m = at[k]
        return buf[BT * C + l * stride + o:][:m].double()

    acts, ids = s["acts"], s["inp"].long()
    wte, wpe = w[:V * C].view(V, C), w[lay["wpe"]:lay["wpe"] + T * C].view(T, C)
    out = {k: [] for k in ("lno", "lnm", "lnr", "resa", "ln2o", "ln2m", "ln2r", "gelu", "res1")}
    stream = (wte[ids].view(B, T, C) + wpe).view(BT, C)
    out["w"], out["enc"] = w, stream.reshape(-1)
    for l in range(L):
        o, m, r = _ln64(stream, w[p(l, "lng")], w[p(l, "lnb")])
        out["lno"].append(o), out["lnm"].append(m), out["lnr"].append(r)
        resa = stream + act(acts, l, "apr").view(BT, C)
        o, m, r = _ln64(resa, w[p(l, "ln2g")], w[p(l, "ln2b")])
        out["resa"].append(resa), out["ln2o"].append(o), out["ln2m"].append(m), out["ln2r"].append(r)
        out["gelu"].append(_gelu64(act(acts, l, "fch")))
        stream = resa + act(acts, l, "mlpo").view(BT, C)
        out["res1"].append(stream)
    fw, fb = (slice(lay[k], lay[k] + C) for k in ("flng", "flnb"))
    flo, flm, flr = _ln64(stream, w[fw], w[fb])
    out["flo"], out["flm"], out["flr"] = flo.reshape(-1), flm, flr
    if c["train"]:
        gacts, grads = s["gacts"], torch.zeros_like(w)
        d = {"dfch": [None] * L, "dapr": [None] * L, "dmlpo": [None] * L}
        end = BT * C + L * stride
        g, grads[fw], grads[fb] = _ln_bwd64(gacts[end:end + BT * C].double().view(BT, C), stream, w[fw], flm, flr)
        for l in reversed(range(L)):
            d["dmlpo"][l] = g.reshape(-1)
            d["dfch"][l] = _gelu_grad64(act(acts, l, "fch")) * act(gacts, l, "gelu")
            dx, grads[p(l, "ln2g")], grads[p(l, "ln2b")] = _ln_bwd64(
                act(gacts, l, "ln2o").view(BT, C), out["resa"][l], w[p(l, "ln2g")], out["ln2m"][l], out["ln2r"][l])
            g = g + dx
            d["dapr"][l] = g.reshape(-1)
            x = out["res1"][l - 1] if l else out["enc"].view(BT, C)
            dx, grads[p(l, "lng")], grads[p(l, "lnb")] = _ln_bwd64(
                act(gacts, l, "lno").view(BT, C), x, w[p(l, "lng")], out["lnm"][l], out["lnr"][l])
            g = g + dx
        grads[:V * C].view(V, C).index_add_(0, ids, g)
        grads[lay["wpe"]:lay["wpe"] + T * C] = g.view(B, T, C).sum(0).reshape(-1)
        out.update(d)
        out["grads"], out["denc"] = grads, g.reshape(-1)
    return {k: torch.stack([x.reshape(-1) for x in v]) if isinstance(v, list) else v for k, v in out.items()}


_EXACT = {"layernorm": _exact_layernorm, "block": _exact_block, "encoder": _exact_encoder, "head": _exact_head,
          "posterior": _exact_posterior, "step": _exact_step}
