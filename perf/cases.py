"""The work a user of sparseforge_amd has it do, as timed cases.

Each case is a dict of plain values; "kind" picks one of the package's entry points:

  linear     SparseLinear forward and backward (sparse_modeling.SparseLinear): the training layer
  infer      SparseLinear24 forward (finalize.SparseLinear24): a finalized layer, packed 2:4
  attention  llama.causal_attention forward and backward
  model      LlamaDecoder forward, cross-entropy and every gradient
  probe      one Hutchinson probe of a LlamaDecoder (utils.update_hessian_hutchinson)
  kl         distill.chunked_kl_loss with its gradient
  mask       utils.calculate_model_mask over a stack of layers
  adamw      adamw.AdamW.step over a stack of layers
  bsr        BlockSparseLinear forward and backward (block_sparse.BlockSparseLinear)

Sizes are those of this repository's benchmark and tests (the 7B decoder layer at 8192 tokens, the 1.1B
retraining model at 2 x 2048 tokens, the GPT-2-small MLP in float32, the block-sparse layer) and what lies
between and below them; draw() spreads them over the whole range, odd and ragged sizes among them.
"""
from __future__ import annotations

import math

import torch
from torch import nn

from sparseforge_amd.adamw import AdamW
from sparseforge_amd.block_sparse import BlockSparseLinear
from sparseforge_amd.distill import chunked_kl_loss
from sparseforge_amd.finalize import SparseLinear24
from sparseforge_amd.llama import LlamaDecoder, LlamaShape, causal_attention, rotary_tables
from sparseforge_amd.sparse_modeling import SparseLinear, SparseLinearConfig
from sparseforge_amd.utils import calculate_model_mask, update_hessian_hutchinson

DEV = "cuda"
DT = {"bf16": torch.bfloat16, "f32": torch.float32}
MASK_STEP = 5000  # mid-training: the mask update is due, the hardening under way


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the widest linear of a LLaMA-2-7B layer in the last phase of training (hard 2:4 mask, SLoRB rank 64),
        # one batch of 8192 tokens: the benchmark's headline layer, and the largest matrix work there is
        {"name": "train 7B gate hard", "kind": "linear", "tokens": 8192, "fin": 4096, "fout": 11008, "rank": 64,
         "bias": False, "dtype": "bf16", "hx": 0.0},
        # an attention projection of the 1.1B retraining model while its mask hardens, a 2 x 2048 micro-batch
        {"name": "train 1.1B q hardening", "kind": "linear", "tokens": 4096, "fin": 2048, "fout": 2048, "rank": 64,
         "bias": False, "dtype": "bf16", "hx": 0.5},
        # the GPT-2-small MLP in float32 under its soft mask, with bias, eight sequences of ragged length
        {"name": "train GPT-2 f32 ragged", "kind": "linear", "tokens": 8 * 1021, "fin": 768, "fout": 3072, "rank": 16,
         "bias": True, "dtype": "f32", "hx": 1.0},
        # a finalized 7B projection decoding for a few users: the smallest call, one token each
        {"name": "decode 7B q", "kind": "infer", "tokens": 4, "fin": 4096, "fout": 4096, "rank": 64, "bias": False},
        # a finalized 7B MLP projection over a batch of prompts of odd total length
        {"name": "prefill 7B down", "kind": "infer", "tokens": 1537, "fin": 11008, "fout": 4096, "rank": 64,
         "bias": False},
        # the attention of one layer of the 1.1B retraining model, a micro-batch of 2 x 2048 tokens
        {"name": "attention 1.1B", "kind": "attention", "batch": 2, "seq": 2048, "heads": 32, "dim": 64,
         "dtype": "bf16"},
        # a whole training pass (logits, loss, every gradient) of a two-layer model of the 1.1B width
        {"name": "model 2 layers", "kind": "model", "batch": 1, "seq": 2048, "hidden": 2048, "ffn": 5632, "heads": 32,
         "layers": 2, "vocab": 32000, "rank": 64, "hx": 0.8},
        # the Hutchinson probe that every retraining step takes, on one layer of that width
        {"name": "probe 1 layer", "kind": "probe", "batch": 1, "seq": 1024, "hidden": 2048, "ffn": 5632, "heads": 32,
         "layers": 1, "vocab": 8192, "rank": 64, "hx": 0.8},
        # the distillation loss of a micro-batch against its teacher, LLaMA vocabulary
        {"name": "kl 4096 x 32000", "kind": "kl", "rows": 4096, "vocab": 32000, "dtype": "bf16"},
        # the periodic mask update over four decoder layers of the 1.1B model
        {"name": "mask update 4 layers", "kind": "mask", "layers": 4, "hidden": 2048, "ffn": 5632, "dtype": "bf16"},
        # the optimizer step over the same four layers
        {"name": "adamw 4 layers", "kind": "adamw", "layers": 4, "hidden": 2048, "ffn": 5632, "dtype": "f32"},
        # a block-sparse MLP projection at half density, forward and both gradients
        {"name": "block sparse 0.5", "kind": "bsr", "tokens": 8192, "fin": 4096, "fout": 11008, "density": 0.5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, m):
    return max(m, _log(rng, lo, hi) // m * m)


def draw(rng):
    kind = rng.choices(["linear", "infer", "attention", "model", "probe", "kl", "mask", "adamw", "bsr"],
                       [30, 16, 12, 5, 5, 10, 8, 7, 7])[0]
    if kind == "linear":
        f32 = rng.random() < 0.25
        top = 4096 if f32 else 11008
        while True:
            c = {"kind": kind, "tokens": _log(rng, 16, 8192), "fin": _mult(rng, 256, top, 64),
                 "fout": _mult(rng, 256, top, 8), "rank": rng.choice([0, 16, 32, 64]), "bias": rng.random() < 0.4,
                 "dtype": "f32" if f32 else "bf16", "hx": rng.choice([1.0, 0.5, 0.25, 0.0, 0.0])}
            if c["tokens"] * c["fin"] * c["fout"] <= (8192 * 768 * 3072 * 2 if f32 else 8192 * 4096 * 11008):
                return c
    if kind == "infer":
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "fin": _mult(rng, 512, 11008, 64),
                "fout": _mult(rng, 512, 11008, 32), "rank": rng.choice([0, 64]), "bias": rng.random() < 0.3}
    if kind == "attention":
        seq = _log(rng, 64, 2048)
        dim = rng.choice([64, 64, 128])
        heads = rng.choice([8, 12, 16, 32]) if dim == 64 else rng.choice([8, 16, 32])
        batch = max(1, min(8, int(2 * (2048 / seq) * rng.random()) or 1))
        while batch * heads * seq * seq > 2 * 32 * 2048 * 2048:
            batch = max(1, batch // 2)
        return {"kind": kind, "batch": batch, "seq": seq, "heads": heads, "dim": dim,
                "dtype": "f32" if seq <= 1024 and rng.random() < 0.15 else "bf16"}
    if kind in ("model", "probe"):
        hidden = rng.choice([512, 1024, 2048])
        return {"kind": kind, "batch": rng.choice([1, 2]), "seq": _log(rng, 128, 1024), "hidden": hidden,
                "ffn": _mult(rng, 2 * hidden, 3 * hidden, 64), "heads": hidden // 64,
                "layers": 2 if kind == "model" else 1, "vocab": _mult(rng, 2048, 32000 if kind == "model" else 8192, 8),
                "rank": 64, "hx": rng.choice([0.8, 0.3, 0.0])}
    if kind == "kl":
        vocab = rng.choice([32000, 50257, 50304, 128256, _log(rng, 2000, 130000)])
        dtype = rng.choice(["bf16", "bf16", "f32"])
        return {"kind": kind, "rows": _log(rng, 64, max(128, min(8192, 4096 * 32000 // vocab))), "vocab": vocab,
                "dtype": dtype}
    if kind in ("mask", "adamw"):
        hidden = _mult(rng, 256, 2048, 64)
        return {"kind": kind, "layers": rng.choice([1, 2, 3, 4]), "hidden": hidden,
                "ffn": _mult(rng, 2 * hidden, int(2.75 * hidden), 8), "dtype": rng.choice(["bf16", "f32"])}
    return {"kind": kind, "tokens": _log(rng, 64, 8192), "fin": _mult(rng, 512, 4096, 64),
            "fout": _mult(rng, 512, 11008, 64), "density": round(rng.uniform(0.1, 0.6), 3)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, shape, std, dtype):
    return (torch.randn(shape, generator=g, device=DEV) * std).to(dtype)


def _soft_mask(g, fout, fin, dtype):
    """A soft mask in [0, 1] whose groups of four have four distinct values (no ties for the projection)."""
    order = torch.rand(fout, fin // 4, 4, generator=g, device=DEV).argsort(-1).float()
    u = torch.rand(fout, fin // 4, 4, generator=g, device=DEV)
    return ((order + 0.1 + 0.7 * u) / 4).reshape(fout, fin).to(dtype)


def _config(case, **kw):
    cfg = SparseLinearConfig(mask_type="unstructured", hard_mask_type="nm_2_4", mask_metric="hessian_ratio",
                             sparsity_ratio=0.5, beta=0.98, mask_update_period_before=30, mask_update_period_after=10,
                             mask_update_switch_step=2000, mask_lr=0.1, sparsity_warmup_steps=500,
                             mask_penalty_lr=0.1, mask_penalty_mode="nm_2_4", mask_hardening_start=2000,
                             mask_hardening_duration=15000, SLoRB_init_type="sum", trainable_projection=True, **kw)
    cfg.enable_hutchinson = True
    return cfg


def _linear_tensors(case, seed):
    """What a linear case is made of: every tensor from the seed, as the layer holds it."""
    g = _gen(seed)
    dt = DT[case.get("dtype", "bf16")]
    fin, fout, r = case["fin"], case["fout"], case["rank"]
    t = {"W": _randn(g, (fout, fin), 0.02, dt), "M": _soft_mask(g, fout, fin, dt),
         "b": _randn(g, (fout,), 0.02, dt) if case["bias"] else None,
         "P": _randn(g, (r, fin), 0.02, dt) if r else None, "S": _randn(g, (fout, r), 0.02, dt) if r else None,
         "x": _randn(g, (case["tokens"], fin), 1.0, dt)}
    if case["kind"] == "linear":
        t["gy"] = _randn(g, (case["tokens"], fout), 1.0, dt)
    return t


def _build_linear(case, t):
    fin, fout, r = case["fin"], case["fout"], case["rank"]
    lin = SparseLinear(fin, fout, sparselinear_config=_config(case, SLoRB=r > 0, SLoRB_k=fin // r if r else 64),
                       bias=case["bias"], device=DEV, dtype=t["W"].dtype)
    with torch.no_grad():
        lin.weight.copy_(t["W"])
        lin.mask.copy_(t["M"])
        if t["b"] is not None:
            lin.bias.copy_(t["b"])
        if r:
            lin.x_proj.copy_(t["P"])
            lin.SLoRB_Weight.copy_(t["S"])
    lin.hardening_x = float(case.get("hx", 0.0))
    return lin


def _model(case, seed):
    shape = LlamaShape(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["ffn"],
                       num_hidden_layers=case["layers"], num_attention_heads=case["heads"])
    g = _gen(seed)
    m = LlamaDecoder(shape, _config(case, SLoRB=True), case["rank"], DEV, torch.bfloat16)
    m.init_random(g)
    with torch.no_grad():
        for mod in m.modules():
            if isinstance(mod, SparseLinear):
                mod.mask.copy_(_soft_mask(g, mod.out_features, mod.in_features, torch.bfloat16))
                mod.hardening_x = float(case["hx"])
    seq = torch.randint(0, case["vocab"], (case["batch"], case["seq"] + 1), generator=g, device=DEV)
    return m, seq[:, :-1].contiguous(), seq[:, 1:].contiguous(), g


def _stack_shapes(case):
    h, f = case["hidden"], case["ffn"]
    return [(h, h)] * 4 + [(h, f)] * 2 + [(f, h)]


def prepare(case, seed):
    kind = case["kind"]
    torch.manual_seed(seed)  # the mask update draws its threshold sample from torch's default generator
    if kind == "linear":
        t = _linear_tensors(case, seed)
        lin = _build_linear(case, t)
        x = t["x"].requires_grad_(True)
        params = [("dx", x), ("dW", lin.weight)]
        if case["bias"]:
            params.append(("db", lin.bias))
        if case["rank"]:
            params += [("dP", lin.x_proj), ("dS", lin.SLoRB_Weight)]
        return {"case": case, "lin": lin, "x": x, "gy": t["gy"], "params": params}
    if kind == "infer":
        t = _linear_tensors(case, seed)
        return {"case": case, "lin": SparseLinear24.from_sparse_linear(_build_linear(case, t)), "x": t["x"]}
    if kind == "attention":
        g, dt = _gen(seed), DT[case["dtype"]]
        shape = (case["batch"], case["seq"], case["heads"], case["dim"])
        q, k, v = (_randn(g, shape, 1.0, dt).requires_grad_(True) for _ in range(3))
        go = _randn(g, (shape[0], shape[1], shape[2] * shape[3]), 1.0, dt)
        cos, sin = rotary_tables(case["seq"], case["dim"], 10000.0, DEV)
        return {"case": case, "qkv": (q, k, v), "go": go, "cos": cos, "sin": sin}
    if kind in ("model", "probe"):
        m, idx, tgt, g = _model(case, seed)
        s = {"case": case, "model": m, "idx": idx, "tgt": tgt}
        if kind == "probe":
            s["probes"] = [(torch.randint(0, 2, mod.weight.shape, generator=g, device=DEV) * 2 - 1).to(torch.bfloat16)
                           for mod in m.modules() if isinstance(mod, SparseLinear)]
            s["H"] = [mod.hessian_diag for mod in m.modules() if isinstance(mod, SparseLinear)]
        else:
            s["params"] = [(n, p) for n, p in m.named_parameters() if p.requires_grad]
        return s
    if kind == "kl":
        g, dt = _gen(seed), DT[case["dtype"]]
        t = _randn(g, (case["rows"], case["vocab"]), 2.0, dt)
        s = (t.float() + torch.randn(t.shape, generator=g, device=DEV)).to(dt).requires_grad_(True)
        return {"case": case, "student": s, "teacher": t}
    if kind == "mask":
        g, dt = _gen(seed), DT[case["dtype"]]
        mods = nn.ModuleList()
        for _ in range(case["layers"]):
            for fin, fout in _stack_shapes(case):
                lin = SparseLinear(fin, fout, sparselinear_config=_config(case), bias=False, device=DEV, dtype=dt)
                with torch.no_grad():
                    lin.weight.copy_(torch.randn(fout, fin, generator=g, device=DEV) * 0.02)
                    lin.hessian_diag.copy_(torch.rand(fout, fin, generator=g, device=DEV) * 1e-3 + 1e-6)
                    lin.mask.copy_(torch.rand(fout, fin, generator=g, device=DEV))
                mods.append(lin)
        return {"case": case, "model": mods}
    if kind == "adamw":
        ps, st = _adamw_tensors(case, seed)
        params = [nn.Parameter(p) for p, _, _ in ps]
        opt = AdamW(params, lr=1e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.1)
        for p, (_, grad, mask), (m, v) in zip(params, ps, st):
            p.grad, p.mask = grad, mask
            opt.state[p] = {"step": 10, "exp_avg": m, "exp_avg_sq": v}
        return {"case": case, "opt": opt, "params": params}
    g = _gen(seed)
    W, keep, x, gy = _bsr_tensors(case, g)
    mask = keep.repeat_interleave(16, 0).repeat_interleave(16, 1).to(W.dtype)
    lin = BlockSparseLinear.from_dense(W, mask, trainable=True)
    return {"case": case, "lin": lin, "x": x.requires_grad_(True), "gy": gy}


def _adamw_tensors(case, seed):
    g, dt = _gen(seed), DT[case["dtype"]]
    ps, st = [], []
    for _ in range(case["layers"]):
        for fin, fout in _stack_shapes(case):
            mask = torch.rand(fout, fin, generator=g, device=DEV).to(dt)
            ps.append((_randn(g, (fout, fin), 0.02, dt), _randn(g, (fout, fin), 1e-3, dt), mask))
            st.append((_randn(g, (fout, fin), 1e-3, dt),
                       (torch.rand(fout, fin, generator=g, device=DEV) * 1e-6 + 1e-8).to(dt)))
        for n in (case["hidden"], case["hidden"]):  # the two norms
            ps.append((torch.ones(n, device=DEV, dtype=dt), _randn(g, (n,), 1e-3, dt), None))
            st.append((_randn(g, (n,), 1e-3, dt),
                       (torch.rand(n, generator=g, device=DEV) * 1e-6 + 1e-8).to(dt)))
    return ps, st


def _bsr_tensors(case, g):
    fin, fout = case["fin"], case["fout"]
    W = _randn(g, (fout, fin), 0.02, torch.bfloat16)
    n = (fout // 16) * (fin // 16)
    keep = torch.zeros(n, dtype=torch.bool, device=DEV)
    keep[torch.randperm(n, generator=g, device=DEV)[:max(1, round(n * case["density"]))]] = True
    keep = keep.view(fout // 16, fin // 16)
    return (W, keep, _randn(g, (case["tokens"], fin), 1.0, torch.bfloat16),
            _randn(g, (case["tokens"], fout), 1.0, torch.bfloat16))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["case"]["kind"]
    if kind == "linear":
        y = s["lin"](s["x"])
        grads = torch.autograd.grad(y, [p for _, p in s["params"]], s["gy"])
        return {"y": y, **{n: g for (n, _), g in zip(s["params"], grads)}}
    if kind == "infer":
        return {"y": s["lin"](s["x"])}
    if kind == "attention":
        o = causal_attention(*s["qkv"], s["cos"], s["sin"])
        dq, dk, dv = torch.autograd.grad(o, s["qkv"], s["go"])
        return {"o": o, "dq": dq, "dk": dk, "dv": dv}
    if kind == "model":
        logits, loss, _ = s["model"](s["idx"], s["tgt"])
        grads = torch.autograd.grad(loss, [p for _, p in s["params"]])
        return {"logits": logits, "loss": loss, "grads": {n: g for (n, _), g in zip(s["params"], grads)}}
    if kind == "probe":
        _, loss, _ = s["model"](s["idx"], s["tgt"])
        update_hessian_hutchinson(s["model"], loss, probes=s["probes"])
        return {"H%d" % i: h for i, h in enumerate(s["H"])}
    if kind == "kl":
        loss = chunked_kl_loss(s["student"], s["teacher"])
        grad, = torch.autograd.grad(loss, s["student"])
        return {"loss": loss, "grad": grad}
    if kind == "mask":
        calculate_model_mask(s["model"], MASK_STEP, lambda_mid=0.5)
        return {"masks": [m.mask for m in s["model"]], "flips": [m.weight.flipped_mask for m in s["model"]]}
    if kind == "adamw":
        s["opt"].step(decay=1e-4)
        st = [s["opt"].state[p] for p in s["params"]]
        if len(s["params"]) <= 20:
            return {"p": s["params"], "m": [t["exp_avg"] for t in st], "v": [t["exp_avg_sq"] for t in st]}
        return {"p": s["params"], "m": [t["exp_avg"] for t in st[:14]], "v": [t["exp_avg_sq"] for t in st[14:28]]}
    y = s["lin"](s["x"])
    gx, gb = torch.autograd.grad(y, [s["x"], s["lin"].sparse_blocks], s["gy"])
    return {"y": y, "dx": gx, "dblocks": gb}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    es = 4 if case.get("dtype") == "f32" else 2
    if kind == "linear":
        T, i, o, r = case["tokens"], case["fin"], case["fout"], case["rank"]
        # x, gy, y, dx; W, mask, dW; P, S and their gradients
        return {"bytes": es * (2 * T * (i + o) + 3 * i * o + 2 * r * (i + o)), "flops": 6.0 * T * (i * o + r * (i + o))}
    if kind == "infer":
        T, i, o, r = case["tokens"], case["fin"], case["fout"], case["rank"]
        return {"bytes": 2 * (T * (i + o) + r * (i + o)) + i * o * 9 / 8, "flops": 2.0 * T * (i * o / 2 + r * (i + o))}
    if kind == "attention":
        n = case["batch"] * case["seq"] * case["heads"] * case["dim"]
        # q, k, v, o, go, dq, dk, dv; seven products over the causal half
        return {"bytes": 8 * es * n, "flops": 7 * 2.0 * n * case["seq"] / 2}
    if kind in ("model", "probe"):
        T, h, f, L, V = case["batch"] * case["seq"], case["hidden"], case["ffn"], case["layers"], case["vocab"]
        w = L * (4 * h * h + 3 * h * f)
        fl = 6.0 * T * (w + V * h) + L * 7 * 2.0 * T * h * case["seq"] / 2
        if kind == "probe":  # forward, first-order gradients, then their derivatives (twice the gradients' work)
            return {"bytes": 2 * (6 * w + 2 * V * h) + 2 * T * V, "flops": 2.0 * fl}
        return {"bytes": 2 * (3 * w + 4 * V * h) + 4 * T * V, "flops": fl}
    if kind == "kl":
        n = case["rows"] * case["vocab"]
        return {"bytes": 3 * es * n, "flops": 12.0 * n}
    if kind in ("mask", "adamw"):
        n = case["layers"] * sum(i * o for i, o in _stack_shapes(case))
        # mask: W, H, mask read, mask written; adamw: p, m, v read and written, gradient and mask read
        return {"bytes": es * n * (4 if kind == "mask" else 8), "flops": 20.0 * n}
    T, i, o, d = case["tokens"], case["fin"], case["fout"], case["density"]
    return {"bytes": 2 * (2 * T * (i + o) + 2 * d * i * o), "flops": 6.0 * T * i * o * d}


def tolerance(case):
    kind = case["kind"]
    f32 = case.get("dtype") == "f32"
    if kind == "linear":
        return {"rel": 1e-5} if f32 else {"rel": 1e-2, "max": 0.1}
    if kind == "infer" or kind == "bsr":
        return {"rel": 1e-2, "max": 0.1}
    if kind == "attention":
        return {"rel": 2e-5} if f32 else {"rel": 2e-2, "max": 0.5}
    if kind in ("model", "probe"):  # bf16 roundings of one layer travel through all that follow
        return {"rel": 3e-2, "max": 0.99}
    if kind == "kl":
        return {"rel": 1e-5} if f32 else {"rel": 1e-2, "max": 0.1}
    if kind == "mask":  # float32: a changed order of the statistics' sums; bf16: a rare neighbouring value
        return {"rel": 1e-5, "max": 1e-2} if f32 else {"rel": 1e-4, "max": 2e-2}
    return {"rel": 1e-6, "max": 1e-4} if f32 else {"rel": 5e-3, "max": 5e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _effective(M, hx):
    """The effective mask of a soft mask M at hardening_x = hx, the top two of every four columns being kept."""
    M = M.double()
    if hx >= 1.0:
        return M
    g = M.view(M.shape[0], -1, 4)
    hard = torch.zeros_like(g).scatter_(-1, g.topk(2, dim=-1).indices, 1.0).view_as(M)
    return hx * M + (1.0 - hx) * hard


class _StraightThrough(torch.autograd.Function):
    """x (W.E)^T whose weight gradient does not see E (differentiable twice)."""

    @staticmethod
    def forward(ctx, x, W, E):
        ctx.save_for_backward(x, W, E)
        return x @ (W * E).t()

    @staticmethod
    def backward(ctx, gy):
        x, W, E = ctx.saved_tensors
        return gy @ (W * E), gy.flatten(0, -2).t() @ x.flatten(0, -2), None


def _rotated(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def _attend(q, k, v, cos, sin):
    B, S, H, D = q.shape
    q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    s = _rotated(q, cos, sin) @ _rotated(k, cos, sin).transpose(-1, -2) * D ** -0.5
    s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    return (s.softmax(-1) @ v).transpose(1, 2).reshape(B, S, H * D)


def _rms(x, w, eps):
    return w * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _exact_model(case, seed):
    m, idx, tgt, g = _model(case, seed)
    W = {n: p.detach().double().requires_grad_(p.requires_grad) for n, p in m.named_parameters()}
    E = {n[:-5]: _effective(p.detach(), case["hx"]) for n, p in m.named_parameters() if n.endswith(".mask")}
    cos, sin = (t.double() for t in rotary_tables(case["seq"], case["hidden"] // case["heads"], 10000.0, DEV))

    def lin(x, name):
        z = (x @ W[name + ".x_proj"].t()) @ W[name + ".SLoRB_Weight"].t()
        return _StraightThrough.apply(x, W[name + ".weight"], E[name]) + z

    h = W["embed_tokens.weight"][idx]
    B, S, _ = h.shape
    for i in range(case["layers"]):
        p = "layers.%d." % i
        n = _rms(h, W[p + "input_layernorm.weight"], 1e-5)
        q, k, v = (lin(n, p + "self_attn.%s_proj" % c).view(B, S, case["heads"], -1) for c in "qkv")
        h = h + lin(_attend(q, k, v, cos, sin), p + "self_attn.o_proj")
        n = _rms(h, W[p + "post_attention_layernorm.weight"], 1e-5)
        gate = lin(n, p + "mlp.gate_proj")
        h = h + lin(gate * torch.sigmoid(gate) * lin(n, p + "mlp.up_proj"), p + "mlp.down_proj")
    logits = _rms(h, W["norm.weight"], 1e-5) @ W["lm_head.weight"].t()
    loss = nn.functional.cross_entropy(logits.flatten(0, 1), tgt.flatten())
    return m, W, logits, loss, g


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "infer"):
        t = {n: None if v is None else v.double() for n, v in _linear_tensors(case, seed).items()}
        WE = t["W"] * _effective(t["M"], float(case.get("hx", 0.0)))
        y = t["x"] @ WE.t()
        if case["rank"]:
            z = t["x"] @ t["P"].t()
            y += z @ t["S"].t()
        if case["bias"]:
            y += t["b"]
        if kind == "infer":
            return {"y": y}
        out = {"y": y, "dx": t["gy"] @ WE, "dW": t["gy"].t() @ t["x"]}
        if case["bias"]:
            out["db"] = t["gy"].sum(0)
        if case["rank"]:
            dz = t["gy"] @ t["S"]
            out["dx"] += dz @ t["P"]
            out["dP"], out["dS"] = dz.t() @ t["x"], t["gy"].t() @ z
        return out
    if kind == "attention":
        s = prepare(case, seed)
        q, k, v = (t.detach().double().requires_grad_(True) for t in s["qkv"])
        o = _attend(q, k, v, s["cos"].double(), s["sin"].double())
        return {"o": o, **dict(zip(("dq", "dk", "dv"), torch.autograd.grad(o, (q, k, v), s["go"].double())))}
    if kind == "model":
        _, W, logits, loss, _ = _exact_model(case, seed)
        names = [n for n, p in W.items() if p.requires_grad]
        grads = torch.autograd.grad(loss, [W[n] for n in names])
        return {"logits": logits, "loss": loss, "grads": dict(zip(names, grads))}
    if kind == "probe":
        m, W, _, loss, g = _exact_model(case, seed)
        names = [n + ".weight" for n, mod in m.named_modules() if isinstance(mod, SparseLinear)]
        vs = [(torch.randint(0, 2, W[n].shape, generator=g, device=DEV) * 2 - 1).double() for n in names]
        grads = torch.autograd.grad(loss, [W[n] for n in names], create_graph=True)
        dot = sum((a * v).sum() for a, v in zip(grads, vs))
        hv = torch.autograd.grad(dot, [W[n] for n in names])
        return {"H%d" % i: 0.02 * (h * v).clamp(min=0) for i, (h, v) in enumerate(zip(hv, vs))}
    if kind == "kl":
        st = prepare(case, seed)
        a = st["student"].detach().double().requires_grad_(True)
        q = (a.clamp(-100, 100) / 2).log_softmax(-1)
        p = (st["teacher"].double().clamp(-100, 100) / 2).log_softmax(-1)
        loss = (p.exp() * (p - q)).sum() * 4 / case["rows"]
        return {"loss": loss, "grad": torch.autograd.grad(loss, a)[0]}
    if kind == "mask":
        return None  # the threshold comes from a random sample of the scores, drawn by the library itself
    if kind == "adamw":
        ps, st = _adamw_tensors(case, seed)
        out = {"p": [], "m": [], "v": []}
        for (p, grad, mask), (m, v) in zip(ps, st):
            p, grad, m, v = (t.double() for t in (p, grad, m, v))
            p = p * (1 - 1e-4 * 0.1)
            if mask is not None:
                grad = grad + 1e-4 * p * (1 - mask.double())
            m, v = 0.9 * m + 0.1 * grad, 0.95 * v + 0.05 * grad * grad
            p = p - 1e-4 / (1 - 0.9 ** 11) * m / (v.sqrt() / math.sqrt(1 - 0.95 ** 11) + 1e-8)
            for name, t in (("p", p), ("m", m), ("v", v)):
                out[name].append(t)
        if len(ps) > 20:
            out["m"], out["v"] = out["m"][:14], out["v"][14:28]
        return out
    W, keep, x, gy = _bsr_tensors(case, _gen(seed))
    x, gy = x.double(), gy.double()
    WE = W.double() * keep.repeat_interleave(16, 0).repeat_interleave(16, 1)
    dW = (gy.t() @ x).view(keep.shape[0], 16, keep.shape[1], 16).transpose(1, 2)
    return {"y": x @ WE.t(), "dx": gy @ WE, "dblocks": dW[keep]}
