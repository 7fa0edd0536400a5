"""Workloads of the framework's public entry points, for timing and comparing builds.

listed() names them, draw() makes more of the same ranges, prepare() makes
what a program holds before the call (a context with its graph, corpus or
tables, made from the seed), run() is one pass through the entry points and
returns what they compute, work() counts the bytes and operations a pass
cannot do without, and exact() evaluates the tuple and scoring paths in 64
bits (the walker's outputs are integers; concurrent training has no fixed
order of updates, so it has no exact result).
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gdistger-re_amd"))

import distger  # noqa: E402
from distger import ffi  # noqa: E402

FORMS = {"plain": ffi.DG_SGNS_PLAIN_FP32, "fp32": ffi.DG_SGNS_BATCHED_FP32, "bf16": ffi.DG_SGNS_BATCHED_BF16,
         "dsgl": ffi.DG_SGNS_DSGL_FP32, "reuse": ffi.DG_SGNS_NEGREUSE_FP32}


def listed():
    return [
        # a program's first call: CSR, common neighbours and thresholds of a
        # power-law graph at the 2.2M-vertex configuration's mean degree
        {"name": "graph_131k", "kind": "graph", "v": 131072, "degree": 13, "weighted": False, "data": False},
        # the 10,000-vertex configuration: round 1 (5 walks per vertex, at
        # most 80 vertices each), its corpus and visit counts read back
        {"name": "walk_10k", "kind": "walk", "v": 10000, "degree": 5, "rounds": 1, "max_length": 80, "corpus": True},
        # the walk phase of a whole job: round 1 and five more, every round
        # kept for training
        {"name": "walk_run_262k", "kind": "walk", "v": 262144, "degree": 13, "rounds": 6, "max_length": 0,
         "corpus": False},
        # the flagship: walk rounds each trained as they come (BF16, dim 128),
        # six rounds and the embeddings at the end
        {"name": "pipeline_bf16_d128", "kind": "pipeline", "graph": "chung-lu", "v": 65536, "degree": 13, "rounds": 6,
         "form": "bf16", "dim": 128, "window": 10, "negative": 5},
        # training over an appended corpus (10 walks per vertex) in each form:
        # the wide embedding,
        {"name": "train_bf16_d256", "kind": "train", "v": 32768, "degree": 13, "rounds": 6, "form": "bf16",
         "dim": 256, "window": 10, "negative": 5, "iter": 1},
        # the default form,
        {"name": "train_fp32_d128", "kind": "train", "v": 32768, "degree": 13, "rounds": 6, "form": "fp32",
         "dim": 128, "window": 10, "negative": 5, "iter": 1},
        # the reference's CPU trainer,
        {"name": "train_dsgl_d128", "kind": "train", "v": 65536, "degree": 13, "rounds": 6, "form": "dsgl",
         "dim": 128, "window": 10, "negative": 5, "iter": 1},
        # and the reference's GPU trainer
        {"name": "train_plain_d128", "kind": "train", "v": 16384, "degree": 13, "rounds": 6, "form": "plain",
         "dim": 128, "window": 10, "negative": 5, "iter": 1},
        # a training loop over the differentiable interface: 16 minibatches of
        # 65,536 tuples, the tables at the end
        {"name": "sgd_bf16_65536", "kind": "sgd", "rows": 65536, "dim": 128, "n": 65536, "negative": 5, "steps": 16,
         "bf16": True},
        # the smallest ordinary call: one small minibatch forward, its caller's
        # own loss gradient backward, and the gradient rows
        {"name": "adjoint_fp32_512", "kind": "adjoint", "rows": 100003, "dim": 128, "n": 512, "negative": 5,
         "bf16": False},
        # serving: the allocation-free forward on device buffers
        {"name": "serve_131072", "kind": "serve", "rows": 500009, "dim": 128, "n": 131072, "negative": 5},
        # link prediction: scores of held-out pairs and as many non-edges
        {"name": "score_500k", "kind": "score", "rows": 500009, "dim": 128, "n": 500000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["graph", "walk", "walk", "pipeline", "train", "train", "train", "sgd", "adjoint", "serve",
                       "score"])
    if kind == "graph":
        return {"kind": kind, "v": _log(rng, 1000, 131072), "degree": rng.randint(3, 13),
                "weighted": rng.random() < 0.3, "data": rng.random() < 0.2}
    if kind == "walk":
        return {"kind": kind, "v": _log(rng, 1000, 200000), "degree": rng.randint(3, 13), "rounds": rng.randint(1, 6),
                "max_length": rng.choice([0, 0, 20 + rng.randint(3, 60)]), "corpus": rng.random() < 0.5}
    if kind == "pipeline":
        graph = rng.choice(["chung-lu", "rmat"])
        form = rng.choice(["bf16", "bf16", "fp32"])
        return {"kind": kind, "graph": graph, "v": 1 << rng.randint(12, 15) if graph == "rmat" else _log(rng, 4000, 40000),
                "degree": rng.randint(6, 13), "rounds": rng.randint(1, 6), "form": form, "dim": 128,
                "window": rng.randint(5, 10), "negative": rng.randint(4, 7)}
    if kind == "train":
        form = rng.choice(["bf16", "fp32", "dsgl", "plain", "reuse"])
        dim = {"bf16": rng.choice([128, 256]), "fp32": rng.choice([64, 128]), "dsgl": rng.choice([64, 128, 256]),
               "plain": rng.choice([64, 128, 256]), "reuse": rng.choice([64, 128, 256])}[form]
        most = 8192 if form in ("plain", "reuse") else 16384
        return {"kind": kind, "v": _log(rng, 4000, most), "degree": rng.randint(6, 13), "rounds": rng.randint(2, 6),
                "form": form, "dim": dim, "window": rng.randint(5, 10), "negative": rng.choice([3, 5, 5, 7, 10]),
                "iter": rng.randint(1, 2)}
    if kind == "sgd":
        return {"kind": kind, "rows": _log(rng, 5000, 60000), "dim": rng.choice([64, 128, 256]),
                "n": _log(rng, 1000, 60000), "negative": rng.choice([1, 5, 5, 10, 15]), "steps": rng.randint(2, 6),
                "bf16": rng.random() < 0.5}
    if kind == "adjoint":
        return {"kind": kind, "rows": _log(rng, 5000, 200000), "dim": rng.choice([64, 128, 256]),
                "n": _log(rng, 33, 4000), "negative": rng.choice([1, 5, 5, 10, 15]), "bf16": rng.random() < 0.5}
    if kind == "serve":
        return {"kind": kind, "rows": _log(rng, 20000, 400000), "dim": rng.choice([64, 128, 256]),
                "n": _log(rng, 64, 131072), "negative": rng.choice([1, 5, 5, 10, 15])}
    return {"kind": kind, "rows": _log(rng, 20000, 400000), "dim": rng.choice([64, 128, 256]),
            "n": _log(rng, 1000, 500000)}


# ---- inputs ------------------------------------------------------------------

def _edges(case, seed):
    if case.get("graph") == "rmat":
        return distger.gen_rmat(int(math.log2(case["v"])), case["degree"], 0.57, 0.19, 0.19, seed)
    return distger.gen_chung_lu(case["v"], case["v"] * case["degree"], 2.2, 2, seed)


def _split_edges(case, seed):
    """The training edges of a link-prediction split: 80% of the edges, in no order."""
    e = _edges(case, seed)
    return e[np.random.default_rng(seed + 3).permutation(len(e))[: case["v"] * case["degree"] * 4 // 5]]


def _graph_context(case, seed, rmat=False):
    ctx = distger.Context(0)
    mode = ffi.DG_CN_COMPUTE_WEIGHTED if rmat else ffi.DG_CN_COMPUTE
    ctx.graph_from_edges(case["v"], _edges(case, seed), undirected=True, cn_mode=mode)
    return ctx


# Rate of the training cases: the reference's per-walk-file schedule
# (0.01 e^(-0.1 n)) around the twentieth file, on tables as training leaves
# them (rows of norm 2 to 4), i.e. the middle of a job and not its first steps.
ALPHA, SIGMA = 0.0015, 0.25


def _trainer(ctx, case, seed):
    """Trainer parameters, the vocabulary, and tables in the middle of a job."""
    sp = _sgns_params(ctx, case, seed)
    ctx.sgns_init(sp)
    ctx.sgns_set_tables(*_tables({"rows": len(ctx.sgns_vocab()), "dim": case["dim"]}, seed, SIGMA))
    return sp


def _sgns_params(ctx, case, seed):
    return ctx.default_sgns_params(dim=case["dim"], window=case["window"], negative=case["negative"],
                                   form=FORMS[case["form"]], iter=case.get("iter", 1), alpha=ALPHA,
                                   table_size=10_000_000, seed=seed + 2)


def _tables(case, seed, sigma=0.1):
    """Rows N(0, sigma^2)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed + 7)
    t = [torch.randn(case["rows"], case["dim"], device="cuda", generator=g) * sigma for _ in range(2)]
    return [x.cpu().numpy() for x in t]


def _tuples(case, seed):
    """(center, context, negatives) ids, Zipf(1.1) as word frequencies are."""
    count = case["n"] * (case["negative"] + 2) * case.get("steps", 1)
    t = distger.gen_zipf(case["rows"], 1.1, count, seed + 11)
    return t.reshape(case.get("steps", 1), case["n"], case["negative"] + 2)


def _dlogits(case, seed):
    r = np.random.default_rng(seed + 13)
    return r.uniform(-1.0, 1.0, (case["n"], case["negative"] + 1)).astype(np.float32)


def _grad_ids(t):
    """Input and output row of every use in a minibatch."""
    return t[:, 1], np.concatenate([t[:, :1], t[:, 2:]], axis=1).reshape(-1)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "graph":
        s["ctx"] = distger.Context(0)
        s["edges"] = _split_edges(case, seed)
        if case["weighted"] or case["data"]:
            r = np.random.default_rng(seed)
            s["edges"]["data"] = (r.integers(0, 30, len(s["edges"])) if case["data"]
                                  else 1.0 - r.random(len(s["edges"]), dtype=np.float32))
        return s
    if kind == "walk":
        s["ctx"] = _graph_context(case, seed)
        s["wp"] = s["ctx"].default_walk_params(seed=seed + 1, max_length=case["max_length"],
                                               max_rounds=case["rounds"])
        return s
    if kind == "pipeline":
        ctx = s["ctx"] = _graph_context(case, seed, rmat=case["graph"] == "rmat")
        s["wp"] = ctx.default_walk_params(seed=seed + 1)
        s["sp"] = _trainer(ctx, case, seed)
        return s
    if kind == "train":
        ctx = s["ctx"] = _graph_context(case, seed)
        ctx.walk_run(ctx.default_walk_params(seed=seed + 1, max_rounds=case["rounds"]), keep_corpus=True)
        s["sp"] = _trainer(ctx, case, seed)
        return s
    ctx = s["ctx"] = distger.Context(0)
    syn0, syn1 = _tables(case, seed)
    ctx.sgns_tables_create(syn0, syn1)
    if kind == "score":
        r = np.random.default_rng(seed + 17)
        s["src"], s["dst"] = (r.integers(0, case["rows"], case["n"], dtype=np.uint32) for _ in range(2))
        return s
    s["tuples"] = _tuples(case, seed)
    if kind == "adjoint":
        s["dlogits"] = _dlogits(case, seed)
        s["in_rows"], s["out_rows"] = _grad_ids(s["tuples"][0])
    if kind == "serve":
        s["d_tuples"] = torch.from_numpy(s["tuples"][0].view(np.int32)).cuda()
        s["logits"] = torch.zeros(case["n"], case["negative"] + 1, device="cuda")
        s["loss"] = torch.zeros(1, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
    return s


# ---- one pass ----------------------------------------------------------------

def _round(st):
    return {"tokens": int(st.tokens), "steps": int(st.steps), "draws": int(st.draws), "moves": int(st.moves),
            "max_walk_len": int(st.max_walk_len), "re": float(st.re)}


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "graph":
        mode = (ffi.DG_CN_FROM_DATA if case["data"]
                else ffi.DG_CN_COMPUTE_WEIGHTED if case["weighted"] else ffi.DG_CN_COMPUTE)
        ctx.graph_from_edges(case["v"], s["edges"], undirected=True, cn_mode=mode)
        rp, nbr, cn = ctx.graph_csr()
        return {"row_ptr": rp.view(np.int64), "nbr": nbr.view(np.int32), "cn": cn.view(np.int32),
                "thresholds": ctx.graph_thresholds().view(np.int32)}
    if kind == "walk":
        if case["corpus"]:
            ctx.walk_reset()
            out = {"round": _round(ctx.walk_round(s["wp"], 1, 0, case["v"] * s["wp"].init_round))}
            tok, off = ctx.corpus()
            out["tokens"], out["offsets"] = tok.view(np.int32), off.view(np.int64)
        else:
            ctx.train_corpus_clear()
            rounds = [_round(st) for st in ctx.walk_run(s["wp"], keep_corpus=True)]
            out = {k: np.array([r[k] for r in rounds]) for k in rounds[0]}
        out["freq"] = ctx.vertex_freq().view(np.int32)
        return out
    if kind == "pipeline":
        ctx.walk_reset()
        rounds = []
        for r in range(1, case["rounds"] + 1):
            n = case["v"] * (s["wp"].init_round if r == 1 else 1)
            rs, ss = ctx.pipeline_step(s["wp"], r, 0, n, s["sp"], allow_undefined_re=case["graph"] == "rmat")
            rounds.append([int(rs.tokens), int(rs.draws), int(rs.moves), int(ss.words), int(ss.kept)])
        syn0, syn1 = ctx.sgns_tables(case["dim"])
        return {"rounds": np.array(rounds), "syn0": syn0, "syn1": syn1}
    if kind == "train":
        st = ctx.sgns_train(s["sp"], corpus=ffi.DG_CORPUS_TRAIN)
        syn0, syn1 = ctx.sgns_tables(case["dim"])
        return {"words": int(st.words), "kept": int(st.kept), "syn0": syn0, "syn1": syn1}
    K = case.get("negative")
    if kind == "sgd":
        logits, losses = [], []
        for t in s["tuples"]:
            z, loss = ctx.tuples_step(t, K, bf16=case["bf16"], lr=LR, apply=True)
            logits.append(z)
            losses.append(loss)
        syn0, syn1 = ctx.sgns_tables(case["dim"])
        return {"logits": logits, "loss": np.array(losses), "syn0": syn0, "syn1": syn1}
    if kind == "adjoint":
        t = s["tuples"][0]
        logits, loss = ctx.tuples_forward(t, K, bf16=case["bf16"])
        ctx.tuples_backward(t, K, bf16=case["bf16"], dlogits=s["dlogits"])
        return {"logits": logits, "loss": loss, "grad0": ctx.grad_rows(0, s["in_rows"], case["dim"]),
                "grad1": ctx.grad_rows(1, s["out_rows"], case["dim"])}
    if kind == "serve":
        rc = ctx.L.dg_sgns_tuples_forward_noalloc(ctx.h, s["d_tuples"].data_ptr(), case["n"], K,
                                                  s["logits"].data_ptr(), s["loss"].data_ptr())
        if rc != ffi.DG_OK:
            raise distger.DgError(rc, ctx.L.dg_last_error(ctx.h).decode())
        return {"logits": s["logits"], "loss": s["loss"]}
    return {"scores": ctx.sgns_score_pairs(s["src"], s["dst"])}


LR = 5e-5  # of the minibatch loop: hot rows sum tens of thousands of gradients per step


# ---- what a pass cannot do without -----------------------------------------------

WALK = 22  # vertices of a walk with the reference's parameters


def _walks(case):
    return case["v"] * (5 + case["rounds"] - 1)


def work(case):
    kind = case["kind"]
    if kind == "graph":
        m = 2 * case["v"] * case["degree"]
        # edges in, CSR with counts and thresholds out, each neighbour list hashed and probed once
        return {"bytes": 12 * m / 2 + 8 * case["v"] + 12 * m, "flops": 20.0 * m}
    if kind == "walk":
        tok = _walks(case) * WALK
        # per token: one adjacency unit and one row of offsets, the token written once
        return {"bytes": tok * (8 + 16 + 4) + 4 * case["v"], "flops": 60.0 * tok}
    if kind in ("pipeline", "train"):
        words = _walks(case) * WALK * case.get("iter", 1)
        d, k1 = case["dim"], case["negative"] + 1
        ctx_per_word = min(case["window"] + 1, WALK * 0.42)
        bytes_ = 4 * words * (1 + k1) + 16 * case["v"] * d  # ids and draws; both tables read and written
        if kind == "pipeline":
            bytes_ += words * 28
        return {"bytes": bytes_, "flops": 6.0 * d * k1 * ctx_per_word * words}
    if kind == "score":
        return {"bytes": 12 * case["n"] + 8 * case["dim"] * min(case["n"], case["rows"]), "flops": 2.0 * case["dim"] * case["n"]}
    n, k1, d, steps = case["n"], case["negative"] + 1, case["dim"], case.get("steps", 1)
    rows = min(2 * case["rows"], n * (k1 + 1) // 2)  # distinct rows of a Zipf minibatch, about half its ids
    width = 2 if case.get("bf16") else 4
    one = 4 * n * (k1 + 1) + 4 * n * k1 + rows * d * width
    if kind == "serve":
        return {"bytes": one, "flops": 2.0 * n * k1 * d}
    if kind == "adjoint":
        return {"bytes": one + rows * d * 4 + 4 * n * k1, "flops": 6.0 * n * k1 * d}
    return {"bytes": steps * (one + rows * d * 8) + 8 * case["rows"] * d, "flops": 6.0 * n * k1 * d * steps}


# ---- 64 bits -----------------------------------------------------------------------

def _forward64(x0, x1, t):
    """logits, loss, live mask of tuples t (int64, n x (K + 2))."""
    out = torch.cat([t[:, :1], t[:, 2:]], dim=1)
    live = out != out[:, :1]
    live[:, 0] = True
    z = torch.empty(out.shape, dtype=torch.float64, device=t.device)
    for j in range(out.shape[1]):
        z[:, j] = (x0[t[:, 1]] * x1[out[:, j]]).sum(1)
    sign = torch.ones(out.shape[1], dtype=torch.float64, device=t.device)
    sign[0] = -1.0
    loss = torch.where(live, torch.nn.functional.softplus(z * sign, threshold=700.0), torch.zeros_like(z)).sum()
    return out, live, z, loss


def _grads64(x0, x1, t, out, dz):
    g0, g1 = torch.zeros_like(x0), torch.zeros_like(x1)
    c = torch.zeros(len(t), x0.shape[1], dtype=torch.float64, device=t.device)
    for j in range(out.shape[1]):
        g1.index_add_(0, out[:, j], dz[:, j : j + 1] * x0[t[:, 1]])
        c += dz[:, j : j + 1] * x1[out[:, j]]
    g0.index_add_(0, t[:, 1], c)
    return g0, g1


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("sgd", "adjoint", "serve", "score"):
        return None
    x0, x1 = (torch.from_numpy(x).cuda().double() for x in _tables(case, seed))
    if kind == "score":
        r = np.random.default_rng(seed + 17)
        src, dst = (torch.from_numpy(r.integers(0, case["rows"], case["n"], dtype=np.uint32).astype(np.int64)).cuda()
                    for _ in range(2))
        return {"scores": (x0[src] * x0[dst]).sum(1).cpu().numpy()}
    batches = _tuples(case, seed)
    if kind == "serve":
        t = torch.from_numpy(batches[0].astype(np.int64)).cuda()
        _, _, z, loss = _forward64(x0, x1, t)
        return {"logits": z, "loss": loss.reshape(1)}
    if kind == "adjoint":
        t = torch.from_numpy(batches[0].astype(np.int64)).cuda()
        out, live, z, loss = _forward64(x0, x1, t)
        dz = torch.from_numpy(_dlogits(case, seed)).cuda().double() * live
        g0, g1 = _grads64(x0, x1, t, out, dz)
        in_rows, out_rows = (torch.from_numpy(x.astype(np.int64)).cuda() for x in _grad_ids(batches[0]))
        return {"logits": z, "loss": float(loss), "grad0": g0[in_rows], "grad1": g1[out_rows]}
    logits, losses = [], []
    for b in batches:
        t = torch.from_numpy(b.astype(np.int64)).cuda()
        out, live, z, loss = _forward64(x0, x1, t)
        dz = torch.sigmoid(z)
        dz[:, 0] -= 1.0
        g0, g1 = _grads64(x0, x1, t, out, dz * live)
        x0 -= LR * g0
        x1 -= LR * g1
        logits.append(z)
        losses.append(float(loss))
    return {"logits": logits, "loss": np.array(losses), "syn0": x0, "syn1": x1}
