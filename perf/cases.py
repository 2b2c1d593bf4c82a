"""The calls whose time matters, from the smallest to the benchmark's own sizes.

A case names one family of calls and its sizes:

* ``objective``: draft and teacher logits given as [N, V] tensors, ``ce_kl_loss`` then
  ``ce_kl_backward`` (metrics and dl);
* ``head``: the fused head step of training, hidden states in, metrics, dh and dl out, without a
  Markov head, with dense Markov logits, or with the factored Markov head (whose two gradients
  are formed too); the teacher given row by row, or as every position's logits with the rows to
  read; optionally final_norm around it, or the masked rows skipped;
* ``linear`` / ``teacher``: the LM head alone (logits), or as the teacher's producer, which also
  forms each row's log-sum-exp;
* ``fp8``: the teacher head in block-scaled e4m3, with the log-sum-exp;
* ``norm``: final_norm forward and backward.

Inputs follow the distributions of ``nanospec_amd.synthetic``.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from nanospec_amd import head, objective, ops
from nanospec_amd.config import Objective

VOCAB = 248_320
HIDDEN = 5_120
RANK = 256          # the Markov head's default rank
EPS = 1e-6
BF16 = torch.bfloat16


def _case(name, kind, n, v=VOCAB, d=HIDDEN, k=8, gamma=4.0, dtype="bf16", markov="none", teacher="rows",
          norm=False, ragged=False, skip=False, steps=1):
    c = {"kind": kind, "n": n, "v": v, "d": d, "k": k, "gamma": gamma, "dtype": dtype, "markov": markov,
         "teacher": teacher, "norm": norm, "ragged": ragged, "skip": skip, "steps": steps}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # A unit test's or a small model's objective: launches and latency.
        _case("objective_small", "objective", 64, v=8192, d=0),
        # One sequence of the default objective (32 anchors x 7 slots) with a tokenizer's odd
        # vocabulary, logits kept in fp32.
        _case("objective_odd_fp32", "objective", 224, v=50_001, d=0, k=7, dtype="fp32", ragged=True),
        # The benchmark's bandwidth case: 512 anchors x 8 slots, supervision of unequal length.
        _case("objective_bulk", "objective", 4096, d=0, ragged=True),
        # Logits of one block of draft slots, as a drafting step asks for them.
        _case("linear_block", "linear", 7, k=7),
        # The plumbing size: the whole fused step on a small model.
        _case("head_small", "head", 64, v=8192, d=256, markov="dense"),
        # One sequence per step at the default objective (32 anchors x 7 slots): factored Markov
        # head with its gradients, teacher logits gathered from every position, final_norm.
        _case("head_one_sequence", "head", 224, k=7, markov="factored", teacher="gathered", norm=True,
              ragged=True),
        # A micro-batch that fills no tile evenly, the plain head, gradients accumulated.
        _case("head_ragged_batch", "head", 1001, k=7, ragged=True, steps=4),
        # Supervision of unequal length with the masked rows skipped.
        _case("head_skip_masked", "head", 2048, gamma=2.0, markov="dense", ragged=True, skip=True),
        # The benchmark's headline: 512 anchors x 8 slots, dense Markov logits.
        _case("head_bulk", "head", 4096, markov="dense"),
        # Teacher logits of one sequence's slots from the block-scaled fp8 head.
        _case("fp8_one_sequence", "fp8", 224, k=7),
        # ... and of the benchmark's batch.
        _case("fp8_bulk", "fp8", 4096),
        # final_norm around the head for eight sequences.
        _case("norm_batch", "norm", 1792, v=0, k=7),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["objective", "objective", "linear", "teacher", "head", "head", "head", "head", "fp8", "fp8",
                       "norm"])
    k = rng.choice([4, 7, 8])
    gamma = rng.choice([0.0, 2.0, 4.0])
    ragged = rng.random() < 0.5
    if kind == "norm":
        return _case(None, kind, max(1, int(_log_uniform(rng, 8, 16384))), v=0,
                     d=rng.choice([256, 1024, 2048, 4096, HIDDEN]))
    n = k * max(1, int(_log_uniform(rng, 1, 3584 / k)))
    if kind == "objective":
        v = int(_log_uniform(rng, 4096, VOCAB))
        if rng.random() < 0.6:
            v = max(8, v // 8 * 8)
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return _case(None, kind, n, v=v, d=0, k=k, gamma=gamma, dtype=dtype, ragged=ragged,
                     steps=rng.choice([1, 4]))
    step = 128 if kind == "fp8" else 64
    d = rng.choice([256, 1024, 2048, HIDDEN, step * rng.randint(2, HIDDEN // step)])
    v = VOCAB if rng.random() < 0.5 else int(_log_uniform(rng, 4096, VOCAB))
    v = v // 128 * 128 if kind == "fp8" else v // 8 * 8
    if kind != "head":
        return _case(None, kind, n, v=v, d=d, k=k)
    markov = rng.choice(["none", "dense", "factored"])
    skip = ragged and markov != "factored" and rng.random() < 0.4
    return _case(None, kind, n, v=v, d=d, k=k, gamma=gamma, markov=markov,
                 teacher="rows" if skip else rng.choice(["rows", "rows", "gathered", "fp32", "lse"]),
                 norm=rng.random() < 0.4, ragged=ragged, skip=skip, steps=rng.choice([1, 1, 4]))


# ---- inputs -----------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, scale, dtype):
    """scale * N(0, 1) in `dtype`, drawn in fp32 a few rows at a time."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    rows = max(1, (1 << 28) // max(1, shape[1]))
    for i in range(0, shape[0], rows):
        part = out[i:i + rows]
        part.copy_(scale * torch.randn(part.shape, generator=g, device="cuda"))
    return out


def _slots(g, c):
    """weights, target ids and validity of N / K blocks: prefix-valid lengths when ragged."""
    nb, k = c["n"] // c["k"], c["k"]
    labels = torch.randint(0, c["v"], (nb, k), generator=g, device="cuda")
    if c["ragged"]:
        lengths = torch.randint(0 if nb > 1 else 1, k + 1, (nb, 1), generator=g, device="cuda")
    else:
        lengths = torch.full((nb, 1), k, device="cuda")
    slot = torch.arange(k, device="cuda")
    valid = slot < lengths
    w = valid.float()
    if c["gamma"] > 0:
        w = w * torch.exp(-slot.float() / c["gamma"])
    return SimpleNamespace(weights=w, target_ids=labels, valid=valid)


def _logits(g, n, v, scale, peak, dtype, at=None):
    out = _normal(g, (n, v), scale, dtype)
    if at is None:
        at = torch.randint(0, v, (n,), generator=g, device="cuda")
    row = torch.arange(n, device="cuda")
    out[row, at] = (out[row, at].float() + peak).to(dtype)
    return out, at


def _fp8_weight(g, v, d):
    """N(0, 0.02) weights as e4m3 codes with one fp32 scale per 128 x 128 block (amax / 448)."""
    w = _normal(g, (v, d), 0.02, torch.float32)
    codes = torch.empty((v, d), dtype=torch.float8_e4m3fn, device="cuda")
    scale = torch.empty((v // 128, d // 128), device="cuda")
    for i in range(0, v, 8192):
        blocks = w[i:i + 8192].view(-1, 128, d // 128, 128)
        s = blocks.abs().amax(dim=(1, 3)) / 448.0
        scale[i // 128:i // 128 + s.shape[0]] = s
        q = (blocks / s[:, None, :, None]).clamp(-448, 448)
        codes[i:i + 8192] = q.view(-1, d).to(torch.float8_e4m3fn)
    return codes, scale


def prepare(case, seed):
    c, g = case, _gen(seed)
    n, v, d, kind = c["n"], c["v"], c["d"], c["kind"]
    s = SimpleNamespace(case=c)
    s.o = Objective(block_size=c["k"], gamma=c["gamma"])
    if kind == "objective":
        dtype = torch.float32 if c["dtype"] == "fp32" else BF16
        s.z, peak = _logits(g, n, v, 2.0, 6.0, dtype)
        other = torch.randint(0, v, (n,), generator=g, device="cuda")
        same = torch.rand(n, generator=g, device="cuda") < 0.6
        s.u, _ = _logits(g, n, v, 3.0, 8.0, dtype, torch.where(same, peak, other))
        s.slots = _slots(g, c)
        shape = (n // c["k"], c["k"], v)
        s.z, s.u = s.z.view(shape), s.u.view(shape)
        return s
    if kind == "norm":
        s.x = _normal(g, (n, d), 1.0, BF16)
        s.weight = (1.0 + 0.1 * torch.randn(d, generator=g, device="cuda")).to(BF16)
        s.dy = _normal(g, (n, d), 0.01, BF16)
        s.weight_grad = torch.empty(d, dtype=BF16, device="cuda")
        return s
    if kind == "fp8":
        s.x = _normal(g, (n, d), 1.0, BF16)
        s.codes, s.scale = _fp8_weight(g, v, d)
        return s
    s.x = _normal(g, (n, d), 1.0, BF16)
    s.w = _normal(g, (v, d), 0.02, BF16)
    if kind in ("linear", "teacher"):
        return s
    s.slots = _slots(g, c)
    if c["norm"]:
        s.norm_weight = (1.0 + 0.1 * torch.randn(d, generator=g, device="cuda")).to(BF16)
        s.norm_grad = torch.empty(d, dtype=BF16, device="cuda")
    else:
        x = s.x.float()
        s.x = (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)).to(BF16)
    s.markov = s.factors = None
    if c["markov"] == "dense":
        s.markov = _normal(g, (n, v), 0.5, BF16)
    elif c["markov"] == "factored":
        prev = torch.randint(0, v, (n,), generator=g, device="cuda")
        w1 = _normal(g, (v, RANK), 1.0, BF16)
        w2 = _normal(g, (v, RANK), 0.05, BF16)
        s.factors = head.MarkovFactors(prev, w1, w2)
        s.grads = (torch.empty_like(w1), torch.empty_like(w2))
    rows = n
    if c["teacher"] == "gathered":   # the logits of a longer sequence's positions, some read often
        rows = n + n // 2 + 1
    u, _ = _logits(g, rows, v, 3.0, 8.0, torch.float32 if c["teacher"] == "fp32" else BF16)
    s.u, s.rows, s.lse = u, None, None
    if c["teacher"] == "gathered":
        s.rows = torch.randint(0, rows, (n,), generator=g, device="cuda")
    elif c["teacher"] == "lse":      # the producer's log-sum-exp of each row
        s.lse = torch.cat([torch.logsumexp(p.double(), -1).float() for p in u.split(64)])
    s.target = u if s.rows is None and s.lse is None else head.TeacherLogits(u, s.rows, s.lse)
    s.shape = (n // c["k"], c["k"])
    return s


# ---- one pass ---------------------------------------------------------------------------------


def _metrics(m):
    return [m.ce, m.kl, m.numerator, m.denominator, m.accept_len_sum, m.accept_len_total]


def run(s):
    c = s.case
    kind = c["kind"]
    if kind == "objective":
        m, saved = objective.ce_kl_loss(s.z, s.u, s.slots, s.o)
        return {"metrics": _metrics(m), "dl": objective.ce_kl_backward(saved, c["steps"])}
    if kind == "linear":
        return {"logits": ops.linear(s.x, s.w)}
    if kind == "teacher":
        t = head.teacher_logits(s.x, s.w)
        return {"logits": t.logits, "lse": t.lse}
    if kind == "fp8":
        t = ops.fp8_teacher_logits(s.x, s.codes, s.scale)
        return {"logits": t.logits, "lse": t.lse}
    if kind == "norm":
        y, saved = ops.rms_norm(s.x, s.weight, EPS)
        return {"y": y, "dx": ops.rms_norm_backward(s.dy, saved, s.weight, s.weight_grad), "dw": s.weight_grad}
    hidden, final_norm = s.x, None
    if c["norm"]:
        hidden, saved = ops.rms_norm(s.x, s.norm_weight, EPS)
        final_norm = (saved, s.norm_weight, s.norm_grad)
    grads = None
    if s.factors is not None:
        grads = s.grads
        grads[0].zero_()   # a step's gradient of the embedding starts from zero
    m, dh, dl = head.head_step(hidden.view(s.shape + (c["d"],)), s.w, s.target, s.slots, s.o,
                               markov_logits=s.markov, markov=s.factors, markov_grads=grads,
                               final_norm=final_norm, accumulation_steps=c["steps"],
                               skip_masked_rows=c["skip"])
    out = {"metrics": _metrics(m), "dh": dh, "dl": dl}
    if grads is not None:
        out["w1_grad"], out["w2_grad"] = grads
    if c["norm"]:
        out["norm_grad"] = s.norm_grad
    return out


# ---- what a pass cannot do without ------------------------------------------------------------


def work(case):
    c = case
    n, v, d, kind = c["n"], c["v"], c["d"], c["kind"]
    if kind == "objective":
        return {"bytes": 3 * n * v * (4 if c["dtype"] == "fp32" else 2), "flops": 20 * n * v}
    if kind == "norm":
        return {"bytes": 2 * 5 * n * d, "flops": 20 * n * d}
    if kind == "fp8":
        return {"bytes": v * d + 2 * n * d + 2 * n * v, "flops": 2 * n * v * d}
    if kind in ("linear", "teacher"):
        return {"bytes": 2 * (v * d + n * d + n * v), "flops": 2 * n * v * d}
    kept = n
    if c["ragged"] and c["skip"]:
        kept = n // 2
    size = 4 if c["teacher"] == "fp32" else 2
    nbytes = 2 * v * d + 4 * n * d + size * n * v + 2 * n * v + (4 * n * d if c["norm"] else 0)
    flops = 2 * n * v * d + 2 * kept * v * d
    if c["markov"] == "dense":
        nbytes += 2 * n * v
    elif c["markov"] == "factored":
        nbytes += 2 * v * RANK * 3
        flops += 6 * n * v * RANK
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "objective" and case["dtype"] == "fp32":
        return {"rel": 4e-6}
    # one rounding to bf16 is 1.7e-3 in the 2-norm; dh carries those of dl as well
    return {"rel": 8e-3, "max": 0.1}


# ---- the same in 64 bits ----------------------------------------------------------------------


def _objective64(z, u, labels, w, o, inv_acc):
    """Per row CE, KL, accept rate and dl of fp64 logits (rows, V)."""
    logp, logt = torch.log_softmax(z, -1), torch.log_softmax(u, -1)
    p, t = logp.exp(), logt.exp()
    ce = -logp.gather(1, labels[:, None])[:, 0]
    kl = (t * (logt - logp)).sum(-1)
    acc = torch.minimum(p, t).sum(-1)
    dl = (o.ce + o.kl) * p - o.kl * t
    dl.scatter_add_(1, labels[:, None], torch.full_like(ce, -o.ce)[:, None])
    return ce, kl, acc, dl * (w * inv_acc)[:, None]


def _metrics64(ce, kl, acc, slots, o):
    w = slots.weights.double().reshape(-1)
    valid = slots.valid.double()
    den = w.sum()
    dc = den.clamp_min(1e-6)
    a = (acc.view(valid.shape) * valid).cumprod(-1)
    block = slots.valid.any(-1).double()
    ces, kls = (w * ce).sum(), (w * kl).sum()
    return [ces / dc, kls / dc, o.ce * ces + o.kl * kls, den, ((1.0 + a.sum(-1)) * block).sum(), block.sum()]


def _norm64(x, weight):
    inv = (x.pow(2).mean(-1, keepdim=True) + EPS).rsqrt()
    return x * inv * weight, inv


def _norm_backward64(dy, x, inv, weight):
    dz = dy * weight
    dx = dz * inv - x * inv.pow(3) * (dz * x).mean(-1, keepdim=True)
    return dx, (dy * x * inv).sum(0)


def _mm64(a, b, chunk=8192):
    """a [n, d] (fp64) times b [v, d]^T, b converted a slice at a time."""
    out = torch.empty((a.shape[0], b.shape[0]), dtype=torch.float64, device=a.device)
    for i in range(0, b.shape[0], chunk):
        out[:, i:i + chunk] = a @ b[i:i + chunk].double().t()
    return out


def _quantised64(x):
    """Activations through 1 x 128 e4m3 blocks, dequantised: the head's own definition."""
    blocks = x.float().view(x.shape[0], -1, 128)
    # the quotients correctly rounded (torch divides by a host scalar through its reciprocal)
    s = (blocks.abs().amax(-1, keepdim=True).double() / 448.0).float()
    q = (blocks.double() / s.clamp_min(torch.finfo(torch.float32).tiny).double()).float()
    q = q.clamp(-448, 448).to(torch.float8_e4m3fn)
    return (q.float().double() * s.double()).view(x.shape)


def _fp8_mm64(x, codes, scale, chunk=8192):
    out = torch.empty((x.shape[0], codes.shape[0]), dtype=torch.float64, device=x.device)
    d = codes.shape[1]
    for i in range(0, codes.shape[0], chunk):
        w = codes[i:i + chunk].float().double().view(-1, 128, d // 128, 128)
        w = w * scale[i // 128:i // 128 + w.shape[0]].double()[:, None, :, None]
        out[:, i:i + chunk] = x @ w.view(-1, d).t()
    return out


def exact(case, seed):
    c = case
    n, v, d, kind = c["n"], c["v"], c["d"], c["kind"]
    s = prepare(c, seed)
    if kind == "norm":
        x, w, dy = s.x.double(), s.weight.double(), s.dy.double()
        y, inv = _norm64(x, w)
        dx, dw = _norm_backward64(dy, x, inv, w)
        return {"y": y, "dx": dx, "dw": dw}
    if kind == "linear":
        return {"logits": _mm64(s.x.double(), s.w)}
    if kind in ("teacher", "fp8"):
        z = _mm64(s.x.double(), s.w) if kind == "teacher" else _fp8_mm64(_quantised64(s.x), s.codes, s.scale)
        # the log-sum-exp is that of the rounded logits, which are the tensor it goes with
        lse = torch.cat([torch.logsumexp(p.to(BF16).double(), -1) for p in z.split(64)])
        return {"logits": z, "lse": lse}
    w = s.slots.weights.double().reshape(-1)
    labels = s.slots.target_ids.reshape(-1)
    dl = torch.empty((n, v), dtype=torch.float64, device="cuda")
    ce, kl, acc = (torch.empty(n, dtype=torch.float64, device="cuda") for _ in range(3))
    step = max(1, (1 << 27) // v)
    if kind == "objective":
        z2, u2 = s.z.view(n, v), s.u.view(n, v)
        for i in range(0, n, step):
            j = slice(i, min(n, i + step))
            ce[j], kl[j], acc[j], dl[j] = _objective64(z2[j].double(), u2[j].double(), labels[j], w[j], s.o,
                                                       1.0 / c["steps"])
        return {"metrics": _metrics64(ce, kl, acc, s.slots, s.o), "dl": dl.view(s.z.shape)}
    x64, inv = s.x.double(), None
    hidden = x64
    if c["norm"]:
        # the head reads the norm's bf16 output, whose definition rounds the normalised row first
        _, inv = _norm64(x64, s.norm_weight.double())
        hidden = ((x64 * inv).to(BF16).double() * s.norm_weight.double()).to(BF16).double()
    for i in range(0, n, step):
        j = slice(i, min(n, i + step))
        z = _mm64(hidden[j], s.w)
        if s.markov is not None:
            z += s.markov[j].double()
        if s.factors is not None:
            z += _mm64(s.factors.w1[s.factors.previous[j]].double(), s.factors.w2)
        u = s.u[s.rows[j]] if s.rows is not None else s.u[j]
        ce[j], kl[j], acc[j], dl[j] = _objective64(z, u.double(), labels[j], w[j], s.o, 1.0 / c["steps"])
        del z, u
    dh = torch.zeros((n, d), dtype=torch.float64, device="cuda")
    for i in range(0, v, 8192):
        dh += dl[:, i:i + 8192] @ s.w[i:i + 8192].double()
    out = {"metrics": _metrics64(ce, kl, acc, s.slots, s.o), "dl": dl.view(s.shape + (v,))}
    if s.factors is not None:
        f = s.factors
        dprev = torch.zeros((n, RANK), dtype=torch.float64, device="cuda")
        w2_grad = torch.empty((v, RANK), dtype=torch.float64, device="cuda")
        e = f.w1[f.previous].double()
        for i in range(0, v, 8192):
            dprev += dl[:, i:i + 8192] @ f.w2[i:i + 8192].double()
            w2_grad[i:i + 8192] = dl[:, i:i + 8192].t() @ e
        out["w1_grad"] = torch.zeros((v, RANK), dtype=torch.float64, device="cuda").index_add_(0, f.previous, dprev)
        out["w2_grad"] = w2_grad
    if c["norm"]:
        dh, out["norm_grad"] = _norm_backward64(dh, x64, inv, s.norm_weight.double())
    out["dh"] = dh.view(s.shape + (d,))
    return out
