"""Performance cases of sparton_amd: the work its users have it do, through its public entry points.

A case is a dict of plain values. `listed()` gives the named ones, `draw(rng)` one more of the same
ranges, `prepare(case, seed)` the inputs and modules a program holds before the call, `run(state)` one
pass, `work(case)` the bytes and operations such a pass cannot do without, `exact(case, seed)` the
same outputs in 64 bits from plain torch, and `tolerance(case)` how far another correct
implementation may be from them.

Kinds:
  encode     SpartonHead without gradients: hidden states -> reps (indexing documents, serving queries)
  train      SpartonHead forward and backward; with `autocast` over fp32 parameters and hidden states
  loss       the SPLADE training loss and its gradients on query and document reps
  transform  SpartonMLMTransform forward and backward

Where gradients are taken, the head's inputs lie on a grid that makes every logit exact in fp32
whatever the order of its sum, so the position of every maximum, which decides where the gradients
go, is the same for every correct implementation.
"""
import math

import torch
from torch import nn

from sparton_amd import SpartonHead
from sparton_amd.loss import splade_training_loss
from sparton_amd.transform import SpartonMLMTransform

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    head = dict(autocast=False, precision="highest", bias=True, density=1.0, mask="int64")
    return [
        # One short query against the BERT-base vocabulary: the smallest serving call.
        dict(head, name="encode-query", kind="encode", B=1, S=16, D=768, V=30522, dtype="bf16", len_lo=6, len_hi=16),
        # A batch of documents being indexed, at a wider model and an odd batch and length.
        dict(head, name="encode-docs", kind="encode", B=61, S=181, D=1024, V=30522, dtype="fp16", len_lo=24, len_hi=181, mask="bool"),
        # The smallest training call: two short rows in fp32, matmul precision 'high' as the reference sets it.
        dict(head, name="train-fp32-tiny", kind="train", B=2, S=32, D=768, V=30522, dtype="fp32", precision="high", len_lo=8, len_hi=32),
        # fp32 training without autocast at torch's default precision.
        dict(head, name="train-fp32", kind="train", B=8, S=128, D=768, V=30522, dtype="fp32", len_lo=16, len_hi=128),
        # The BERT-base SPLADE head, the headline workload.
        dict(head, name="train-bert", kind="train", B=32, S=256, D=768, V=30522, dtype="bf16", len_lo=32, len_hi=256, density=0.05),
        # Mixed precision as training scripts run it: fp32 parameters under bf16 autocast, and a dense
        # gradient, since the regularisers reach every active term.
        dict(head, name="train-autocast", kind="train", B=16, S=256, D=768, V=30522, dtype="bf16", autocast=True, len_lo=32, len_hi=256),
        # Long documents in fp16.
        dict(head, name="train-longdoc", kind="train", B=8, S=512, D=768, V=30522, dtype="fp16", len_lo=288, len_hi=512, density=0.05),
        # The multilingual vocabulary (XLM-RoBERTa base).
        dict(head, name="train-xlmr", kind="train", B=32, S=256, D=768, V=250002, dtype="bf16", len_lo=16, len_hi=256, density=0.05),
        # A decoder-only backbone's head without bias: the largest call.
        dict(head, name="train-llm", kind="train", B=16, S=512, D=4096, V=128256, dtype="bf16", bias=False, len_lo=128, len_hi=512, density=0.05),
        # The loss on the head's reps: a small batch, and a large one with a hard negative per query.
        dict(name="loss-small", kind="loss", Bq=32, Bd=32, V=30522, dtype="bf16"),
        dict(name="loss-large", kind="loss", Bq=256, Bd=512, V=30522, dtype="fp16"),
        # The MLM transform in front of the head, at the headline workload's rows.
        dict(name="transform", kind="transform", M=8192, D=768, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["encode", "train", "train", "loss", "transform"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if kind == "loss":
        Bq = _log(rng, 4, 512)
        return dict(kind=kind, Bq=Bq, Bd=Bq * rng.choice([1, 1, 2]) + rng.choice([0, rng.randrange(8)]),
                    V=rng.choice([30522, _log(rng, 3000, 60000)]), dtype=dtype)
    if kind == "transform":
        return dict(kind=kind, M=_log(rng, 64, 32768), D=rng.choice([384, 768, 768, 1000, 1024]), dtype=dtype)
    D = rng.choice([384, 768, 768, 772, 1024])
    V = rng.choice([30522, 30522, 50265, _log(rng, 5000, 250002)])
    autocast = kind == "train" and dtype != "fp32" and rng.random() < 0.4
    density = 0.05 if kind == "train" and rng.random() < 0.5 else 1.0
    # The budget keeps a drawn call well under the largest listed one's cost.
    budget = 1.0e11 if dtype == "fp32" else (4.0e11 if density == 1.0 and kind == "train" else 1.5e12)
    S = _log(rng, 8, 512)
    B = max(1, min(_log(rng, 1, 256), int(budget / (2.0 * S * D * V))))
    return dict(kind=kind, B=B, S=S, D=D, V=V, dtype=dtype, autocast=autocast,
                precision=rng.choice(["highest", "high"]) if dtype == "fp32" else "highest",
                bias=rng.random() < 0.8, density=density, mask=rng.choice(["int64", "bool"]),
                len_lo=max(1, S // 8), len_hi=S)


# ---- inputs -------------------------------------------------------------------------

def _grid(x, step, top):
    return (x / step).round_().mul_(step).clamp_(-top, top)


def _head_inputs(case, seed):
    """(hidden, weight, bias or None, mask, grad or None) of a head case, in float32 (mask aside)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, S, D, V = case["B"], case["S"], case["D"], case["V"]
    rand = lambda f, *n: f(*n, generator=g, device="cuda")
    # hidden ~ N(0, 1) and weight ~ N(0, 0.02), or half of each for wide models: what a LayerNorm and a trained
    # decoder give. The grid's steps leave eight bits per value (nine for fp32 hidden states), and logits that fp32
    # holds with bits to spare. fp32 encoding, which hands out no positions, takes the values as they are drawn.
    scale = 0.5 if D > 2048 else 1.0
    wide = case["dtype"] == "fp32"
    hidden, weight = rand(torch.randn, B, S, D) * scale, rand(torch.randn, V, D) * (0.02 * scale)
    if not (wide and case["kind"] == "encode"):
        hidden = _grid(hidden, scale / (128 if wide else 32), 4.0 * scale)
        weight = _grid(weight, scale / 2048, 0.125 * scale)
    bias = _grid(rand(torch.randn, V) * 0.1 - 0.5, 1.0 / 256, 1.0) if case["bias"] else None
    lengths = torch.randint(case["len_lo"], case["len_hi"] + 1, (B,), generator=g, device="cuda")
    if B > 1:
        lengths[0] = case["len_hi"]  # batches are padded to their longest row
    mask = torch.arange(S, device="cuda")[None, :] < lengths[:, None]
    mask = mask if case["mask"] == "bool" else mask.to(torch.int64)
    grad = None
    if case["kind"] == "train":
        grad = rand(torch.rand, B, V)
        if case["density"] < 1.0:
            grad = grad * (rand(torch.rand, B, V) < case["density"])
    return hidden, weight, bias, mask, grad


def _loss_inputs(case, seed):
    """Sparse reps as a trained encoder gives them: about 1% of a query's terms and 2% of a document's are active,
    and each query's own document (row i) shares a few of its terms."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    def reps(B, density):
        keep = torch.rand(B, case["V"], generator=g, device="cuda") < density
        return torch.rand(B, case["V"], generator=g, device="cuda") * 2.0 * keep
    q, d = reps(case["Bq"], 0.01), reps(case["Bd"], 0.02)
    shared = q * (torch.rand(q.shape, generator=g, device="cuda") < 0.03)
    d[: case["Bq"]] = torch.maximum(d[: case["Bq"]], shared)
    dt = DTYPES[case["dtype"]]
    return q.to(dt), d.to(dt)


LOSS_STEP = 20000    # past the regularisers' warm-up
FP16_SCALE = 1024.0  # fp16 training scales its loss


def _transform_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    M, D, dt = case["M"], case["D"], DTYPES[case["dtype"]]
    rand = lambda *n: torch.randn(*n, generator=g, device="cuda")
    x, w, dy = rand(M, D).to(dt), (rand(D, D) * 0.04).to(dt), (rand(M, D) * 0.01).to(dt)
    vecs = (rand(D) * 0.02, 1.0 + rand(D) * 0.1, rand(D) * 0.1)
    return x, w, dy, tuple(v.to(dt) for v in vecs)


def prepare(case, seed):
    if case["kind"] == "loss":
        q, d = _loss_inputs(case, seed)
        return dict(case=case, q=q.requires_grad_(), d=d.requires_grad_())
    if case["kind"] == "transform":
        x, w, dy, (b, gamma, beta) = _transform_inputs(case, seed)
        D = case["D"]
        with torch.device("cuda"):
            dense, norm = nn.utils.skip_init(nn.Linear, D, D), nn.LayerNorm(D, eps=1e-12)
        dense, norm = dense.to(device="cuda", dtype=x.dtype), norm.to(device="cuda", dtype=x.dtype)
        with torch.no_grad():
            dense.weight.copy_(w)
            dense.bias.copy_(b)
            norm.weight.copy_(gamma)
            norm.bias.copy_(beta)
        return dict(case=case, module=SpartonMLMTransform(dense, norm), x=x.requires_grad_(), dy=dy)
    hidden, weight, bias, mask, grad = _head_inputs(case, seed)
    dt = DTYPES[case["dtype"]]
    held = torch.float32 if case["autocast"] else dt  # what the program keeps parameters and hidden states in
    with torch.device("meta"):
        head = SpartonHead(case["V"], case["D"], use_bias=case["bias"])
    head.weight = nn.Parameter(weight.to(held))
    if case["bias"]:
        head.bias = nn.Parameter(bias.to(held))
    state = dict(case=case, head=head, hidden=hidden.to(held), mask=mask)
    if case["kind"] == "train":
        state["hidden"].requires_grad_()
        state["grad"] = grad.to(dt)
    return state


# ---- one pass -----------------------------------------------------------------------

def run(state):
    case = state["case"]
    if case["kind"] == "loss":
        q, d = state["q"], state["d"]
        q.grad = d.grad = None
        out = splade_training_loss(q, d, LOSS_STEP)
        (out.total * FP16_SCALE if case["dtype"] == "fp16" else out.total).backward()
        return [t.detach() for t in out] + [q.grad, d.grad]
    if case["kind"] == "transform":
        module, x = state["module"], state["x"]
        module.zero_grad(set_to_none=True)
        x.grad = None
        y = module(x)
        y.backward(state["dy"])
        return [y.detach(), x.grad] + [p.grad for p in module.parameters()]
    head, hidden, mask = state["head"], state["hidden"], state["mask"]
    torch.set_float32_matmul_precision(case["precision"])
    if case["kind"] == "encode":
        with torch.no_grad():
            return head(hidden, mask)
    head.zero_grad(set_to_none=True)
    hidden.grad = None
    if case["autocast"]:
        with torch.autocast("cuda", dtype=DTYPES[case["dtype"]]):
            reps = head(hidden, mask)
    else:
        reps = head(hidden, mask)
    reps.backward(state["grad"])
    return [reps.detach(), hidden.grad] + [p.grad for p in head.parameters()]


# ---- what a pass cannot do without ------------------------------------------------------

def work(case):
    """Each input read once and each output written once; multiply-adds count two."""
    e = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "loss":
        Bq, Bd, V = case["Bq"], case["Bd"], case["V"]
        # scores, and their two gradients; reps in, gradients out
        return dict(bytes=2 * (Bq + Bd) * V * e, flops=6.0 * Bq * Bd * V)
    if case["kind"] == "transform":
        M, D = case["M"], case["D"]
        # x, weight, dy and the vectors in; y, dx and the parameters' gradients out
        return dict(bytes=(4 * M * D + 2 * D * D + 6 * D) * e, flops=6.0 * M * D * D)
    B, S, D, V = case["B"], case["S"], case["D"], case["V"]
    held = 4 if case["autocast"] else e
    tokens = B * (case["len_lo"] + case["len_hi"]) / 2.0  # expected unmasked positions
    n_bias = V if case["bias"] else 0
    bytes_ = (tokens * D + V * D + n_bias) * held + B * S * (1 if case["mask"] == "bool" else 8) + B * V * e
    flops = 2.0 * tokens * D * V
    if case["kind"] == "train":
        bytes_ += B * V * e + (B * S * D + V * D + n_bias) * held  # upstream gradient in; three gradients out
        flops += 4.0 * case["density"] * B * V * D                 # one row of W and one of H per active term
    return dict(bytes=bytes_, flops=flops)


def tolerance(case):
    """About four times what the path showed against exact() over these ranges."""
    dtype = case["dtype"]
    if case["kind"] == "transform":
        return {"rel": {"fp32": 3e-6, "fp16": 1.4e-3, "bf16": 1.1e-2}[dtype]}
    if case["kind"] == "loss":
        return {"rel": {"fp32": 3e-6, "fp16": 1e-3, "bf16": 7e-3}[dtype]}
    return {"rel": {"fp32": 1.2e-5, "fp16": 1e-3, "bf16": 7e-3}[dtype]}


# ---- the same in 64 bits ------------------------------------------------------------------

def _exact_head(case, seed):
    hidden, weight, bias, mask, grad = _head_inputs(case, seed)
    dt, f64 = DTYPES[case["dtype"]], torch.float64
    B, S, D, V = case["B"], case["S"], case["D"], case["V"]
    h, m = hidden.to(dt).to(f64), mask.to(f64)
    rows = torch.arange(B, device="cuda")[:, None]
    reps = torch.empty(B, V, dtype=f64, device="cuda")
    if case["kind"] == "train":
        g = grad.to(dt).to(f64)
        dh, dw = torch.zeros_like(h), torch.empty(V, D, dtype=f64, device="cuda")
        db = torch.empty(V, dtype=f64, device="cuda")
    step = max(64, min(V, int(2.0e8 / (B * max(S, D)))))
    for v0 in range(0, V, step):
        v1 = min(V, v0 + step)
        w = weight[v0:v1].to(dt).to(f64)
        x = (h.reshape(B * S, D) @ w.t()).reshape(B, S, v1 - v0)
        if bias is not None:
            x += bias[v0:v1].to(dt).to(f64)
        x *= m[:, :, None]
        top = x.amax(dim=1)
        at = torch.argmax((x == top[:, None, :]).to(torch.uint8), dim=1)  # the lowest position of a tie
        top = top.clamp_min(0.0)
        reps[:, v0:v1] = torch.log1p(top)
        if case["kind"] != "train":
            continue
        gp = torch.where(top > 0, g[:, v0:v1] / (1.0 + top), torch.zeros_like(top))
        db[v0:v1] = gp.sum(0)
        for b in range(B):
            if b == 0:
                dw[v0:v1] = gp[b][:, None] * h[b][at[b]]
            else:
                dw[v0:v1] += gp[b][:, None] * h[b][at[b]]
            dh[b].index_add_(0, at[b], gp[b][:, None] * w)
    if case["kind"] != "train":
        return reps
    return [reps, dh, dw] + ([db] if bias is not None else [])


def _exact_loss(case, seed):
    q, d = (t.double().requires_grad_() for t in _loss_inputs(case, seed))
    s = q @ d.t()
    ce = torch.nn.functional.cross_entropy(s, torch.arange(case["Bq"], device="cuda"))
    l1 = [x.abs().sum(1).mean() for x in (q, d)]
    fl = [(x.sum(0) ** 2).mean() for x in (q, d)]
    total = ce + 1e-4 * (l1[0] + l1[1]) + 1e-4 * (fl[0] + fl[1])
    (total * FP16_SCALE if case["dtype"] == "fp16" else total).backward()
    return [t.detach() for t in (total, ce, *l1, *fl)] + [q.grad, d.grad]


def _exact_transform(case, seed):
    x, w, dy, vecs = _transform_inputs(case, seed)
    x, w, b, gamma, beta = (t.double().requires_grad_() for t in (x, w, *vecs))
    z = torch.nn.functional.gelu(x @ w.t() + b)
    y = torch.nn.functional.layer_norm(z, (case["D"],), gamma, beta, 1e-12)
    y.backward(dy.double())
    return [y.detach(), x.grad, w.grad, b.grad, gamma.grad, beta.grad]


def exact(case, seed):
    return {"loss": _exact_loss, "transform": _exact_transform}.get(case["kind"], _exact_head)(case, seed)
