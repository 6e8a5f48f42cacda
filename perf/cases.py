"""The LM-head work a trainer asks of this package, as timed and compared cases.

A case is one call (or one forward and backward) of a micro-batch through octopus_amd.head_op:

  score    the logprob and entropy columns of the scored rows, no gradient (compute_logp)
  train    the fused GRPO step, loss.backward() included (fused_grpo_head)
  bound    the same step behind the head's columns, the objective a separate op (grpo_bound_head: the route of a
           bound model whose trainer computes its own GRPO loss)
  later    the columns, a loss of the caller's own (policy gradient plus a KL penalty), its backward (fused_head)
  tree     label pairs of a prefix tree built on the device, then the fused step over them (fused_grpo_tree_head)
  columns  the columns of logits that exist already, and their gradient (head_columns)

N packed rows, `scored` of them (a share; the unscored ones first: the shared prompt), hidden width d, vocabulary V.
Hidden rows have RMS 1, weights N(0, 0.02), targets Zipf(1.1); a row leans towards its target's weight so that the
target's logit is 2 .. 18, which makes its probability anything from 1e-5 to nearly 1, as on sampled text. Advantages
are one normal number per sequence, behaviour logprobs the model's own plus N(0, 0.01).
"""

import math

import torch

from octopus_amd import head_op
from octopus_amd.rl.prefix_tree import TreeMeta

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": torch.bfloat16}
CAP = 30.0  # the soft-cap: z' = 30 tanh(z / 30)
EPS_LO, EPS_HI, REJECT = 0.2, 0.28, 5.0
KL = 0.05


def _case(kind, N, d, V, dtype="bf16", scored=1.0, T=1.0, softcap=False, seqs=1, name=None):
    c = {"kind": kind, "N": N, "d": d, "V": V, "dtype": dtype, "scored": scored, "T": T, "softcap": softcap,
         "seqs": seqs}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one short turn's tokens scored while an episode is assembled: the smallest call, the weight read once
        _case("score", 57, 2560, 151936, name="score-turn"),
        # the 512-row fp32 configuration of the workloads: a small model checked in full precision
        _case("score", 512, 1024, 32000, "f32", name="score-fp32"),
        # the behaviour logprobs of an ordinary micro-batch with a masked prompt, tempered sampling, an odd row count
        _case("score", 8191, 4096, 128256, scored=0.75, T=0.7, seqs=6, name="score-batch"),
        # a gradient step on one short turn
        _case("train", 300, 2560, 151936, scored=0.75, name="train-turn"),
        # an ordinary micro-batch through a bound model, the trainer's own GRPO loss on the columns
        _case("bound", 4000, 2560, 151936, scored=0.75, seqs=4, name="train-bound"),
        # the packed prefix-tree micro-batch the benchmark runs: the largest
        _case("train", 32768, 2560, 151936, scored=0.75, seqs=12, name="train-packed"),
        # a frozen fp8 head (adapters train): the gradient of the hidden rows alone
        _case("train", 16384, 2560, 151936, "fp8", scored=0.875, seqs=4, name="train-fp8"),
        # a loss the head cannot know ahead (KL to a reference policy), the larger width and its temperature
        _case("later", 8192, 4096, 128256, scored=0.4375, T=0.7, seqs=3, name="train-kl"),
        # eight completions of one prompt as a prefix tree, pairs deduplicated on the device
        _case("tree", 4608, 2560, 151936, scored=0.8, seqs=8, name="train-tree"),
        # a soft-capped model trained in f16, ragged rows and width
        _case("train", 1501, 2304, 64000, "f16", scored=0.9, softcap=True, seqs=3, name="train-softcap-f16"),
        # a small model trained in full precision
        _case("later", 512, 1024, 32000, "f32", scored=0.75, name="train-fp32"),
        # one 2,048-row chunk of logits that another module produced
        _case("columns", 2048, 0, 151936, seqs=2, name="columns-chunk"),
    ]


def draw(rng):
    def spread(lo, hi):  # even over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["score", "score", "score", "train", "train", "train", "bound", "later", "later", "tree",
                       "columns"])
    dtype = {"score": ["bf16", "bf16", "bf16", "f16", "fp8", "f32"],
             "train": ["bf16", "bf16", "bf16", "f16", "fp8"], "bound": ["bf16", "bf16", "f16", "fp8"],
             "later": ["bf16", "bf16", "f16", "f32"], "tree": ["bf16", "bf16", "f16"],
             "columns": ["bf16", "f16", "f32"]}[kind]
    dtype = rng.choice(dtype)
    T = rng.choice([1.0, 1.0, 0.7])
    softcap = rng.random() < 0.2
    scored = rng.choice([1.0, 0.9, 0.75, 0.5])
    if kind == "columns":
        V = rng.choice([32000, 50257, 128256, 151936, 248320])
        return _case(kind, spread(1, 4096 if dtype != "f32" else 2048), 0, V, dtype, T=T)
    if dtype == "f32":
        return _case(kind, spread(1, 1536), rng.choice([512, 1024]), rng.choice([8000, 32000]), dtype, scored, T,
                     softcap)
    d = rng.choice([1024, 1536, 2048, 2304, 2560, 2880, 4096])
    V = rng.choice([32000, 50257, 64000, 128256, 151936, 151936, 248320])
    # rows such that no case costs more than train-packed's work (half of it for the routes that do more per row)
    most = 24576 * 2560 * 151936 / (d * V) * (1.0 if kind in ("score", "train") else 0.5)
    if kind == "tree":
        return _case(kind, spread(64, min(16384, most)), d, V, dtype, rng.choice([0.9, 0.7]), T, softcap,
                     rng.choice([2, 4, 8, 16]))
    return _case(kind, spread(1, min(32768, most)), d, V, dtype, scored, T, softcap, rng.choice([1, 3, 8]))


# ---- inputs ------------------------------------------------------------------------------------------------------


def _dev():
    return torch.device("cuda")


def _zipf(n, V, g):
    """n targets, P(rank k) proportional to k^-1.1, the ranks spread over the vocabulary by a permutation."""
    cdf = torch.cumsum(torch.arange(1, V + 1, dtype=torch.float64, device=_dev()).pow(-1.1), 0)
    u = torch.rand(n, generator=g, device=_dev(), dtype=torch.float64) * cdf[-1]
    ranks = torch.searchsorted(cdf, u).clamp_(max=V - 1)
    return torch.randperm(V, generator=g, device=_dev())[ranks]


def _weight(case, g):
    """(weight as the call takes it, its row scale or None, its values in bf16 / f16 / f32)."""
    w = torch.empty(case["V"], case["d"], device=_dev()).normal_(0.0, 0.02, generator=g)
    if case["dtype"] == "fp8":
        scale = (w.abs().amax(dim=1) / 448.0).clamp_(min=1e-12)
        q = (w / scale[:, None]).clamp_(-448, 448).to(torch.float8_e4m3fn)
        return q, scale, (q.float() * scale[:, None]).to(torch.bfloat16)
    w = w.to(DTYPES[case["dtype"]])
    return w, None, w


def _hidden(case, plain_w, labels, g):
    n, d = labels.numel(), case["d"]
    x = torch.randn(n, d, generator=g, device=_dev())
    x /= x.norm(dim=1, keepdim=True)
    lean = plain_w[labels].float()
    norm = lean.norm(dim=1, keepdim=True)
    z = torch.empty(n, 1, device=_dev()).uniform_(2.0, 18.0, generator=g)
    a = (z / (norm * math.sqrt(d))).clamp_(max=0.95)
    return (math.sqrt(d) * (a * lean / norm + (1 - a * a).sqrt() * x)).to(DTYPES[case["dtype"]])


def _post(case):
    return head_op.Post(1.0 / CAP, CAP, True) if case["softcap"] else head_op.Post()


def _logp(case, rows, plain_w, labels):
    """The rows' logprobs to input precision, 2,048 rows at a time: where the behaviour logprobs start from."""
    out = []
    for h, y in zip(rows.split(2048), labels.split(2048)):
        z = (h @ plain_w.T).float()
        if case["softcap"]:
            z = CAP * torch.tanh(z / CAP)
        z /= case["T"]
        out.append(z.gather(1, y[:, None])[:, 0] - torch.logsumexp(z, 1))
    return torch.cat(out)


def _sequences(n, seqs):
    """The sequence each of n rows belongs to: seqs runs of about equal length."""
    return (torch.arange(n, device=_dev()) * seqs // max(n, 1)).clamp_(max=seqs - 1)


def _tree(case, g):
    """N flat tokens of `seqs` sequences: a prompt they share, runs that pairs of them share, and tails of their own.
    (flat tokens, sequence offsets, tree position of each flat token, tree tokens, scored flat positions)."""
    seqs, N = case["seqs"], case["N"]
    each = max(4, N // seqs)
    prompt = max(1, int(round((1 - case["scored"]) * each)))
    shared = max(1, (each - prompt) // 4)
    tail = max(1, each - prompt - shared)
    f2t, scored, at = [], [], prompt
    for s in range(seqs):
        if s % 2 == 0:
            mid, at = at, at + shared
        own, at = at, at + tail
        f2t.append(torch.cat([torch.arange(prompt), torch.arange(mid, mid + shared), torch.arange(own, own + tail)]))
        scored.append(torch.cat([torch.zeros(prompt, dtype=torch.bool), torch.ones(shared + tail, dtype=torch.bool)]))
    f2t = torch.cat(f2t).to(_dev())
    tokens = _zipf(at, case["V"], g)
    cu = torch.arange(seqs + 1, device=_dev()) * (prompt + shared + tail)
    return tokens[f2t], cu, f2t, at, torch.cat(scored).to(_dev())


def prepare(case, seed):
    g = torch.Generator(device=_dev()).manual_seed(seed)
    kind, N, V = case["kind"], case["N"], case["V"]
    s = {"case": case}
    if kind == "columns":
        s["labels"] = _zipf(N, V, g)
        z = torch.randn(N, V, generator=g, device=_dev())
        z.scatter_(1, s["labels"][:, None], torch.empty(N, 1, device=_dev()).uniform_(2.0, 18.0, generator=g))
        s["logits"] = z.to(DTYPES[case["dtype"]]).requires_grad_(True)
        s["coef"] = torch.randn(N, generator=g, device=_dev()) / N
        return s
    weight, s["w_scale"], plain = _weight(case, g)
    plain = plain.detach()
    s["weight"] = weight if case["dtype"] == "fp8" or kind == "score" else weight.requires_grad_(True)
    if kind == "tree":
        s["flat"], s["cu"], s["f2t"], s["T_tree"], s["scored"] = _tree(case, g)
        nxt = torch.zeros(s["T_tree"], dtype=torch.int64, device=_dev())
        after = torch.cat([s["flat"][1:], s["flat"][:1]])
        nxt.scatter_reduce_(0, s["f2t"], after, "amax")  # the token a tree position's row leans towards
        s["hidden"] = _hidden(case, plain, nxt, g)[None].requires_grad_(True)
        n_tok = s["flat"].numel()
        owner = torch.bucketize(torch.arange(n_tok, device=_dev()), s["cu"][1:], right=True)
        at = torch.nonzero(s["scored"])[:, 0]
        rows, labels = s["hidden"].detach()[0][s["f2t"][at]], after[at]
    else:
        s["labels"] = _zipf(N, V, g)
        s["rows"] = _hidden(case, plain, s["labels"], g).requires_grad_(kind != "score")
        n_tok = N
        s["scored"] = torch.arange(N, device=_dev()) >= N - max(1, int(round(case["scored"] * N)))
        owner = _sequences(N, case["seqs"])
        at = torch.nonzero(s["scored"])[:, 0]
        rows, labels = s["rows"].detach()[at], s["labels"][at]
    if kind == "score":
        return s
    adv = torch.randn(case["seqs"], generator=g, device=_dev())
    s["mask"] = s["scored"].float()
    if kind == "tree":  # the last token of a sequence asks for nothing
        s["mask"][s["cu"][1:] - 1] = 0.0
    s["adv"] = adv[owner].contiguous()
    s["old"] = torch.zeros(n_tok, device=_dev())
    s["old"][at] = _logp(case, rows, plain, labels)
    s["old"] += torch.randn(n_tok, generator=g, device=_dev()) * 0.01
    if kind == "later":
        s["ref"] = s["old"] + torch.randn(n_tok, generator=g, device=_dev()) * 0.1
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------


def _rows_of(s):
    """The keyword arguments that name the scored rows: a compaction of the mask unless every row is scored."""
    if s["case"]["scored"] >= 1.0:
        return {}
    idx, count = head_op.compact_rows(s["scored"])
    return {"idx": idx, "count": count}


def _own_loss(s, logp):
    """Policy gradient with a KL penalty to a reference policy, averaged over the scored tokens."""
    off = s["ref"] - logp
    return (s["mask"] * (KL * (off.exp() - off - 1) - s["adv"] * logp)).sum() / s["mask"].sum()


def run(s):
    c = s["case"]
    kind, T, post = c["kind"], c["T"], _post(c)
    if kind == "columns":
        s["logits"].grad = None
        out = head_op.head_columns(s["logits"], T, s["labels"])
        (s["coef"] * out[:, 0]).sum().backward()
        return {"out": out.detach(), "grad": s["logits"].grad}
    if kind == "score":
        at = _rows_of(s)
        many = {"labels_via_idx": True, "scatter": True} if at else {}
        with torch.no_grad():
            return {"out": head_op.fused_head(s["rows"], s["weight"], s["labels"], T, post, w_scale=s["w_scale"],
                                              **at, **many)}
    x = s["hidden"] if kind == "tree" else s["rows"]
    x.grad = s["weight"].grad = None
    if kind == "tree":
        meta = TreeMeta.on_device(s["flat"], s["cu"], s["f2t"], s["T_tree"], s["scored"])
        loss, out = head_op.fused_grpo_tree_head(x, s["weight"], meta, T, s["adv"], s["mask"], old=s["old"], post=post)
    elif kind == "train":
        at = _rows_of(s)
        many = {"labels_via_idx": True, "scatter": True} if at else {}
        loss, out = head_op.fused_grpo_head(x, s["weight"], s["labels"], T, s["adv"], s["mask"], old=s["old"],
                                            post=post, w_scale=s["w_scale"], **at, **many)
    elif kind == "bound":
        grpo = head_op.GrpoInputs(adv=s["adv"], old=s["old"], prox=None, mask=s["mask"])
        out = head_op.grpo_bound_head(x, s["weight"], s["labels"], T, grpo, post=post, w_scale=s["w_scale"],
                                      **_rows_of(s))
        loss, _ = head_op.grpo_loss(out[:, 0], None, s["old"], s["adv"], s["mask"], EPS_LO, EPS_HI, REJECT)
    else:
        at = _rows_of(s)
        many = {"labels_via_idx": True, "scatter": True} if at else {}
        out = head_op.fused_head(x, s["weight"], s["labels"], T, post, w_scale=s["w_scale"], **at, **many)
        loss = _own_loss(s, out[:, 0])
    loss.backward()
    got = {"loss": loss.detach(), "out": out.detach(), "grad_rows": x.grad}
    if s["weight"].grad is not None:
        got["grad_weight"] = s["weight"].grad
    return got


# ---- what a pass has to do, and how closely ----------------------------------------------------------------------


def work(case):
    """The operands read once, the results written once, and the products' multiply-adds."""
    N, d, V, kind = case["N"], case["d"], case["V"], case["kind"]
    size = 4 if case["dtype"] == "f32" else 2
    if kind == "columns":
        return {"bytes": 2 * N * V * size + 8 * N * 3, "flops": 12 * N * V}
    n = max(1, int(round(case["scored"] * N)))
    if kind == "tree":  # pairs: tails of their own, runs shared by two sequences
        each = max(4, N // case["seqs"])
        prompt = max(1, int(round((1 - case["scored"]) * each)))
        shared = max(1, (each - prompt) // 4)
        n = case["seqs"] * max(1, each - prompt - shared) + shared * ((case["seqs"] + 1) // 2)
    w = V * d * (1 if case["dtype"] == "fp8" else size)
    if kind == "score":
        return {"bytes": w + n * d * size + 8 * N, "flops": 2 * n * d * V}
    both = case["dtype"] != "fp8"
    return {"bytes": w + (w if both else 0) + 2 * n * d * size + 8 * N, "flops": (6 if both else 4) * n * d * V}


def tolerance(case):
    """About four times the distance from 64 bits that the path shows."""
    if case["kind"] == "score":
        return {"rel": 5e-6, "max": 2e-4}  # 32-bit sums, of exact products for 16-bit operands: 2e-7 .. 1.1e-6
    if case["dtype"] == "f32":
        return {"rel": 1.5e-5, "max": 1e-3}  # 32-bit sums throughout: 3.2e-6
    if case["dtype"] == "f16":
        # dz in f16 loses its smallest entries below 2^-24: 4e-3 .. 2.2e-2 of the hidden rows' gradient, by how small
        # the weights are; an implementation that scales dz first loses none
        return {"rel": 2.5e-2}
    return {"rel": 1.2e-2}  # dz and the gradients rounded to bf16: 2.3e-3 .. 3.1e-3


# ---- the same in 64 bits -----------------------------------------------------------------------------------------


def _exact_rows(case, rows, w64, labels, g_of, need_w):
    """(columns [n, 2], grad_rows [n, d] or None, grad_weight or None) of rows against w64; g_of(r0, r1, logp) is
    dL/dlogprob of rows r0 .. r1 (None: no gradient)."""
    cols, grads = [], []
    gw = torch.zeros_like(w64) if need_w else None
    step = max(1, min(2048, (1 << 28) // case["V"]))
    for r0 in range(0, rows.shape[0], step):
        h, y = rows[r0:r0 + step].double(), labels[r0:r0 + step]
        z = h @ w64.T
        slope = 1.0
        if case["softcap"]:
            th = torch.tanh(z / CAP)
            z, slope = CAP * th, 1 - th * th
        z = z / case["T"]
        lse = torch.logsumexp(z, 1, keepdim=True)
        lp = z - lse
        p = lp.exp()
        at = lp.gather(1, y[:, None])
        cols.append(torch.stack([at[:, 0], -(p * lp).sum(1)], 1))
        if g_of is None:
            continue
        gr = g_of(r0, r0 + h.shape[0], at[:, 0])[:, None]
        p.mul_(-gr)
        p.scatter_add_(1, y[:, None], gr)
        p = p * slope / case["T"]
        grads.append(p @ w64)
        if need_w:
            gw += p.T @ h
    return torch.cat(cols), (torch.cat(grads) if grads else None), gw


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "columns":
        z = s["logits"].detach().double() / case["T"]
        lp = z - torch.logsumexp(z, 1, keepdim=True)
        del z
        p = lp.exp()
        at = lp.gather(1, s["labels"][:, None])
        out = torch.stack([at[:, 0], -(p * lp).sum(1)], 1)
        g = s["coef"].double()[:, None]
        p.mul_(-g).scatter_add_(1, s["labels"][:, None], g)
        return {"out": out, "grad": p / case["T"]}
    w64 = s["weight"].detach().double() if s["w_scale"] is None else \
        s["weight"].double() * s["w_scale"].double()[:, None]
    need_w = kind != "score" and s["weight"].requires_grad
    if kind == "tree":
        asks = s["scored"].clone()
        asks[s["cu"][1:] - 1] = False
        at = torch.nonzero(asks)[:, 0]
        src = s["hidden"].detach()[0]
        pos, labels, n_tok = s["f2t"][at], s["flat"][at + 1], s["flat"].numel()
    else:
        at = torch.nonzero(s["scored"])[:, 0]
        src, pos, labels, n_tok = s["rows"].detach(), at, s["labels"][at], case["N"]
    if kind == "score":
        cols, _, _ = _exact_rows(case, src[pos], w64, labels, None, False)
        out = torch.zeros(n_tok, 2, dtype=torch.float64, device=src.device)
        out[at] = cols
        return {"out": out}
    adv, old, mask = (s[k].double()[at] for k in ("adv", "old", "mask"))
    Z = s["mask"].double().sum().clamp(min=1.0)
    losses = []

    def g_of(r0, r1, lp):
        a, m = adv[r0:r1], mask[r0:r1]
        if kind == "later":
            off = s["ref"].double()[at][r0:r1] - lp
            losses.append((m * (KL * (off.exp() - off - 1) - a * lp)).sum() / Z)
            return m * (KL * (1 - off.exp()) - a) / Z
        w = (lp - old[r0:r1]).exp()  # the proximal policy is the model itself: the ratio is 1
        w = torch.where(w > REJECT, torch.zeros_like(w), w)
        losses.append(-(m * w * a).sum() / Z)
        return -m * w * a / Z

    cols, grads, gw = _exact_rows(case, src[pos], w64, labels, g_of, need_w)
    out = torch.zeros(n_tok, 2, dtype=torch.float64, device=src.device)
    out[at] = cols
    gx = torch.zeros(src.shape, dtype=torch.float64, device=src.device)
    gx.index_add_(0, pos, grads)
    got = {"loss": torch.stack(losses).sum(), "out": out, "grad_rows": gx[None] if kind == "tree" else gx}
    if need_w:
        got["grad_weight"] = gw
    return got
