"""The work whose speed is tracked: the package's public entry points at the sizes that its
users give them, with inputs, expected results and tolerances.

``listed()`` names the cases, ``draw(rng)`` picks another one from the same ranges,
``prepare(case, seed)`` makes what a program holds before the call, ``run(state)`` makes one
pass, ``exact(case, seed)`` gives the same results in 64 bits by plain torch, and
``work(case)`` / ``tolerance(case)`` say what a pass needs at least and how close two correct
evaluations are.  Sizes are this repository's own configurations and test shapes.
"""
import contextlib
import io
import math
import tempfile

import numpy as np
import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

from mathbrain import synthetic
from mathbrain.data import WikiTextMMapDataset, corpus_states, preprocess_corpus
from mathbrain.factored_ema import factored_ema_forward
from mathbrain.flash_ema_attention import flash_ema_forward as dense_flash_ema_forward
from mathbrain.layernorm import layer_norm
from mathbrain.model import SlotTransformerLM
from mathbrain.rmsnorm import rms_norm
from mathbrain.swiglu import swiglu_product
from mathbrain.triton_ema_query import compute_query_ema_history
from mathbrain.triton_flash_ema import FlashEMAFunction, flash_ema_forward, precompute_boundaries
from mathbrain.triton_fused_gating import GatedQueryFunction

DEV = "cuda"
VOCAB = 50257


def listed():
    return [
        # The dense entry point at the CPU reference configuration: a small call, forward and
        # backward, no carried state; launches and a nearly idle chip.
        dict(name="dense_small", kind="dense", B=2, T=128, H=4, hd=32, N=16, V=1000),
        # One attention layer of a training step at its usual size, with the state that a
        # 4096-token history leaves, at a freshly initialised module's weight scales.
        dict(name="attention_layer", kind="attention", B=56, T=512, H=8, hd=64, N=64, V=VOCAB, history=4096,
             pad=0.0, precision="bf16", scale="init"),
        # The same layer on long chunks with padded tails and twice the rates: the largest call.
        dict(name="attention_long", kind="attention", B=16, T=4096, H=8, hd=64, N=128, V=VOCAB, history=4096,
             pad=0.1, precision="bf16", scale="small"),
        # The fp32 mode on a small ragged batch (checks and fine-tuning on few sequences).
        dict(name="attention_fp32_ragged", kind="attention", B=3, T=201, H=6, hd=32, N=33, V=5000, history=300,
             pad=0.3, precision="fp32", scale="small"),
        # Evaluation of one long document chunk: both scans and the forward, no gradients.
        dict(name="eval_long_chunk", kind="eval", B=1, T=10001, H=8, hd=64, N=64, V=VOCAB, history=2000,
             precision="bf16", scale="small"),
        # The query-side counter scan with its carried state, as a streaming caller keeps it.
        dict(name="query_scan", kind="scan", B=56, T=2048, N=128, V=VOCAB, history=8192),
        # The query gate of a training step, forward and backward.
        dict(name="query_gating", kind="gating", B=56, T=512, D=512, N=64),
        # The row operations between the matrix products of a training step: RMSNorm, the slot
        # rows' LayerNorm and SwiGLU's product on the bf16 values that autocast gives it.
        dict(name="row_operations", kind="rows", rows=28672, slots=50257, D=512, hidden=1536),
        # The factored (linear-gate) attention, forward and backward with carried state.
        dict(name="factored_layer", kind="factored", B=56, T=512, H=8, hd=64, N=64, V=VOCAB, history=4096),
        # Preprocessing: the state of every position of a corpus.
        dict(name="corpus_states", kind="corpus", T=4000000, N=64, V=VOCAB, median=1500),
        # The data loader: one collated batch of history-expanded chunks.
        dict(name="slot_batch", kind="batch", T=300000, B=56, block=512, N=64, V=VOCAB, median=4000),
        # The whole model, a small training step: logits and every gradient.
        dict(name="model_step", kind="model", B=8, T=512, D=512, layers=2, H=8, N=64, V=VOCAB),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm, odd ones among them."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    most = _cost(next(c for c in listed() if c["name"] == "attention_long"))
    while True:
        kind = rng.choice(["attention", "attention", "attention", "dense", "eval", "scan", "gating", "rows",
                           "factored", "corpus", "batch", "model"])
        if kind == "attention":
            precision = rng.choice(["bf16", "bf16", "fp16", "fp32"])
            c = dict(kind=kind, B=_log(rng, 1, 56), T=_log(rng, 64, 4096), H=rng.choice([1, 2, 3, 4, 6, 8, 12]),
                     hd=rng.choice([32, 64, 64] if precision == "fp32" else [32, 64, 64, 128]),
                     N=rng.choice([16, 33, 64] if precision == "fp32" else [16, 33, 64, 64, 128]),
                     V=rng.choice([5000, VOCAB]), history=rng.choice([0, 300, 4096]), pad=rng.choice([0.0, 0.1, 0.3]),
                     precision=precision, scale="small")
        elif kind == "dense":
            c = dict(kind=kind, B=_log(rng, 1, 4), T=_log(rng, 64, 400), H=rng.choice([2, 4]), hd=rng.choice([32, 64]),
                     N=rng.choice([8, 16]), V=rng.choice([1000, 3000]))
        elif kind == "eval":
            c = dict(kind=kind, B=_log(rng, 1, 4), T=_log(rng, 500, 10001), H=rng.choice([4, 8]), hd=64,
                     N=rng.choice([16, 64]), V=VOCAB, history=rng.choice([0, 2000]), precision="bf16", scale="small")
        elif kind == "scan":
            c = dict(kind=kind, B=_log(rng, 1, 56), T=_log(rng, 100, 8192), N=rng.choice([16, 33, 64, 128]), V=VOCAB,
                     history=rng.choice([0, 1000, 8192]))
        elif kind == "gating":
            c = dict(kind=kind, B=_log(rng, 1, 56), T=_log(rng, 65, 1024), D=rng.choice([128, 256, 512, 768]),
                     N=rng.choice([16, 33, 64, 128]))
        elif kind == "rows":
            D = rng.choice([128, 512, 768])
            c = dict(kind=kind, rows=_log(rng, 200, 32768), slots=_log(rng, 300, 60000), D=D, hidden=3 * D)
        elif kind == "factored":
            c = dict(kind=kind, B=_log(rng, 1, 24), T=_log(rng, 64, 600), H=rng.choice([4, 8]), hd=rng.choice([32, 64]),
                     N=rng.choice([16, 64]), V=rng.choice([5000, VOCAB]), history=rng.choice([300, 4096]))
        elif kind == "corpus":
            c = dict(kind=kind, T=_log(rng, 20000, 8000000), N=rng.choice([16, 64, 128]), V=rng.choice([5000, VOCAB]),
                     median=rng.choice([300, 1500, 4000]))
        elif kind == "batch":
            c = dict(kind=kind, T=_log(rng, 50000, 300000), B=_log(rng, 1, 64), block=rng.choice([128, 512, 1000]),
                     N=rng.choice([16, 64]), V=rng.choice([5000, VOCAB]), median=rng.choice([1500, 4000]))
        else:
            c = dict(kind=kind, B=_log(rng, 1, 8), T=_log(rng, 64, 512), D=rng.choice([128, 256, 512]), layers=2,
                     H=4, N=rng.choice([16, 64]), V=rng.choice([5000, VOCAB]))
        if _cost(c) <= most:
            return c


def _cost(case):
    w = work(case)
    return max(w["flops"] / 50, w["bytes"])


# ---- sizes that follow from the tokens -------------------------------------------------

_distinct = {}


def _slots(n, V):
    """Expected distinct ids of n Zipf(1.1) draws from V."""
    if (n, V) not in _distinct:
        p = np.arange(1, V + 1, dtype=np.float64) ** -1.1
        _distinct[n, V] = float((-np.expm1(n * np.log1p(-p / p.sum()))).sum())
    return _distinct[n, V]


def _width(n, V):
    """A slot list's width: the most distinct ids that a row of n draws is likely to hold."""
    return max(16, min(n, V, int(_slots(n, V) + 3 * math.sqrt(_slots(n, V)) + 8)))


# ---- inputs ------------------------------------------------------------------------------

def _normal(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device=DEV) * std


def _uniform(gen, *shape, bound=1.0):
    return (torch.rand(*shape, generator=gen, device=DEV) * 2 - 1) * bound


def _to_dev(d):
    return {k: v.to(DEV) for k, v in d.items() if k in ("x", "unique", "c_base", "rhos", "counts", "targets")}


def _token_batch(case, seed):
    """A batch as the data loader hands it over, on the GPU: Zipf(1.1) tokens, each row's
    slots (its distinct tokens in order, then those only its history holds, as far as they
    fit; -1 padding) and c_base, the history's counters at the chunk's start.  ``pad``: up to
    that share of a row's tail holds token 0."""
    B, T, V, N, W = (case[k] for k in ("B", "T", "V", "N", "history"))
    g = torch.Generator(DEV).manual_seed(seed)
    p = torch.arange(1, V + 1, device=DEV, dtype=torch.float64) ** -1.1
    cdf = (p / p.sum()).cumsum(0)
    ids = torch.randperm(V, generator=g, device=DEV)
    drawn = torch.rand(B, W + T, generator=g, device=DEV, dtype=torch.float64)
    tokens = ids[torch.searchsorted(cdf, drawn).clamp(max=V - 1)]
    history, x = tokens[:, :W], tokens[:, W:].contiguous()
    tail = (torch.rand(B, 1, generator=g, device=DEV) * case.get("pad", 0.0) * T).long()
    x[torch.arange(T, device=DEV) >= T - tail] = 0
    rhos = synthetic.rhos_from_half_lives(N, 1.0, 4096.0).to(DEV)
    weight = rhos.double() ** torch.arange(W, 0, -1, dtype=torch.float64, device=DEV).unsqueeze(1)
    K = _width(T + W, V)
    rows = []
    for b in range(B):
        own = torch.unique(x[b])
        old = torch.unique(history[b])
        rows.append(torch.cat([own, old[~torch.isin(old, own)]])[:K])
    unique = torch.full((B, K), -1, dtype=torch.int64, device=DEV)
    c_base = torch.zeros(B, K, N, device=DEV)
    for b, r in enumerate(rows):
        unique[b, :len(r)] = r
        if W:
            c_base[b, :len(r)] = ((r.unsqueeze(1) == history[b]).double() @ weight).float()
    return dict(x=x, unique=unique, c_base=c_base, rhos=rhos, tail=tail)


def _attention_inputs(case, seed):
    """A batch of Zipf tokens with its slots and carried state, and the layer's operands.
    scale "small": N(0, 0.02), the configurations' weights; "init": what q_proj, k_proj and
    v_proj give normalised rows and pe_proj holds when a module has just been made."""
    d = _token_batch(case, seed)
    B, T, H, hd, N = (case[k] for k in ("B", "T", "H", "hd", "N"))
    K = d["unique"].shape[1]
    g = torch.Generator(DEV).manual_seed(seed + 1)
    std = 1 / math.sqrt(3) if case["scale"] == "init" else 0.02
    d["Q"] = _normal(g, B, T, H, hd, std=std).transpose(1, 2)  # as q_proj's rows are viewed per head
    d["E_k"] = _normal(g, B, K, H * hd, std=std)
    d["E_v"] = _normal(g, B, K, H * hd, std=std)
    d["W"] = (_uniform(g, N, H * hd, bound=1 / math.sqrt(N)) if case["scale"] == "init"
              else _normal(g, N, H * hd, std=0.02))
    d["dO"] = _normal(g, B, H, T, hd)
    # no loss reads the outputs of the padded tail
    d["dO"] *= (torch.arange(T, device=DEV) < T - d["tail"])[:, None, :, None]
    return d


def _dense_inputs(case, seed):
    B, T, H, hd, N, V = (case[k] for k in ("B", "T", "H", "hd", "N", "V"))
    D = H * hd
    gen = torch.Generator().manual_seed(seed)
    x = synthetic.zipf_tokens((B, T), V, 1.1, gen, torch.randperm(V, generator=gen)).to(DEV)
    g = torch.Generator(DEV).manual_seed(seed)
    pe = torch.nn.Linear(N, D, bias=False, device=DEV)
    with torch.no_grad():
        pe.weight.copy_(_normal(g, D, N, std=0.3))
    return dict(x=x, pe=pe, rhos=synthetic.rhos_from_half_lives(N, 1.0, 1024.0).to(DEV),
                Q=_normal(g, B, T, D), E_k=_normal(g, V, D, std=0.5), E_v=_normal(g, V, D, std=0.5),
                dO=_normal(g, B, T, D))


def _gating_inputs(case, seed):
    B, T, D, N = (case[k] for k in ("B", "T", "D", "N"))
    g = torch.Generator(DEV).manual_seed(seed)
    # counters: mostly small, larger for the slow rates of frequent tokens
    C = _normal(g, B, T, N).abs() * torch.logspace(-1, 1.5, N, device=DEV) * torch.rand(B, T, 1, generator=g, device=DEV)
    return dict(x=_normal(g, B, T, D), C=C, W=_uniform(g, D, N, bound=1 / math.sqrt(N)),
                w=1 + _normal(g, D, std=0.1), b=_normal(g, D, std=0.1), dy=_normal(g, B, T, D))


def _rows_inputs(case, seed):
    D, hidden = case["D"], case["hidden"]
    g = torch.Generator(DEV).manual_seed(seed)
    s = dict(x=_normal(g, case["rows"], D), w=1 + _normal(g, D, std=0.1), dy=_normal(g, case["rows"], D),
             e=_normal(g, case["slots"], D), lw=1 + _normal(g, D, std=0.1), lb=_normal(g, D, std=0.1),
             de=_normal(g, case["slots"], D))
    for k in ("a", "b", "dm"):
        s[k] = _normal(g, case["rows"], hidden).to(torch.bfloat16)
    return s


def _factored_inputs(case, seed):
    d = _token_batch(case, seed)
    D = case["H"] * case["hd"]
    g = torch.Generator(DEV).manual_seed(seed + 1)
    d["Q"] = _normal(g, case["B"], case["T"], D, std=0.02)
    d["E_k"] = _normal(g, case["V"], D, std=0.02)
    d["E_v"] = _normal(g, case["V"], D, std=0.02)
    d["W"] = _normal(g, case["N"], D, std=0.02)
    d["dO"] = _normal(g, case["B"], case["T"], D)
    return d


def _corpus_inputs(case, seed):
    tokens, docs = synthetic.zipf_corpus(case["T"], case["V"], median_len=case["median"], seed=seed)
    return dict(tokens=torch.from_numpy(tokens).to(DEV), docs=torch.from_numpy(docs).to(DEV),
                rhos=synthetic.rhos_from_half_lives(case["N"], 1.0, 2048.0).to(DEV))


def _batch_inputs(case, seed):
    """A preprocessed corpus of Zipf documents and one batch of its chunks.  One document is a
    word list, all distinct, and its last chunk has the longest slot list of the batch."""
    V, block, most = case["V"], case["block"], 2 * case["median"]
    rng = np.random.default_rng(seed)
    listed = _width(most + block, V)
    docs = [rng.permutation(V)[:listed + (1 - listed) % block if listed < V - block else V].tolist()]
    p = np.arange(1, V + 1) ** -1.1
    ids, cdf = rng.permutation(V), np.cumsum(p / p.sum())
    while sum(map(len, docs)) < case["T"]:
        n = max(2, min(most, int(case["median"] * math.exp(0.5 * rng.standard_normal()))))
        docs.append(ids[np.minimum(np.searchsorted(cdf, rng.random(n)), V - 1)].tolist())
    folder = tempfile.TemporaryDirectory()
    with contextlib.redirect_stdout(io.StringIO()):  # both print what they hold
        preprocess_corpus(docs, folder.name, N=case["N"])
        scales = np.logspace(0, np.log10(2048.0), case["N"])
        data = WikiTextMMapDataset(folder.name, block, torch.from_numpy(np.exp(-np.log(2.0) / scales)).float())
    pick = rng.choice(len(data), size=case["B"], replace=len(data) < case["B"])
    pick[0] = next(i for i, c in enumerate(data.chunks) if c[1] == len(docs[0]))
    data.get_batch(pick[:1])  # the corpus goes to the GPU once, with the first batch
    return dict(folder=folder, data=data, pick=pick)


def _model_inputs(case, seed):
    d = _to_dev(synthetic.make_doc_batch(case["B"], case["T"], case["V"], case["N"], seed=seed))
    torch.manual_seed(seed)
    with torch.device(DEV):
        d["model"] = SlotTransformerLM(case["V"], case["D"], case["layers"], case["H"], N=case["N"], dropout=0.0,
                                       max_hl=4096.0)
    d["mask"] = d["unique"] >= 0
    return d


_INPUTS = {"attention": _attention_inputs, "eval": _attention_inputs, "dense": _dense_inputs,
           "scan": _token_batch, "gating": _gating_inputs, "rows": _rows_inputs, "factored": _factored_inputs,
           "corpus": _corpus_inputs, "batch": _batch_inputs, "model": _model_inputs}


def _inputs(case, seed):
    return _INPUTS[case["kind"]](case, seed)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    for k in _LEAVES.get(case["kind"], ()):
        s[k].requires_grad_(True)
    return s


#: What the backward gives gradients of.
_LEAVES = {"attention": ("Q", "E_k", "E_v", "W"), "dense": ("Q", "E_k", "E_v"), "gating": ("x", "W", "w", "b"),
           "rows": ("x", "w", "e", "lw", "lb", "a", "b"), "factored": ("Q", "E_k", "E_v", "W")}


# ---- one pass ----------------------------------------------------------------------------

def run(s):
    return _RUN[s["case"]["kind"]](s, s["case"])


def _run_attention(s, case):
    C = precompute_boundaries(s["x"], s["unique"], s["rhos"], 64, s["c_base"])
    O = FlashEMAFunction.apply(s["Q"], s["x"], s["E_k"], s["E_v"], s["W"], s["rhos"], case["V"], s["unique"],
                               s["unique"].shape[1], C, True, 64, True, case["precision"])
    return [O, *torch.autograd.grad(O, [s[k] for k in _LEAVES["attention"]], s["dO"])]


def _run_dense(s, case):
    O = dense_flash_ema_forward(s["Q"], s["x"], s["E_k"], s["E_v"], s["rhos"], s["pe"], case["H"])
    return [O, *torch.autograd.grad(O, [s["Q"], s["E_k"], s["E_v"], s["pe"].weight], s["dO"])]


def _run_eval(s, case):
    with torch.no_grad():
        C_seq = compute_query_ema_history(s["x"], s["rhos"], case["V"], s["c_base"], s["unique"])
        C = precompute_boundaries(s["x"], s["unique"], s["rhos"], 64, s["c_base"])
        O = flash_ema_forward(s["Q"], s["x"], s["E_k"], s["E_v"], s["W"], s["rhos"], case["V"], s["unique"],
                              s["unique"].shape[1], C, precision=case["precision"])[0]
    return [C_seq, O]


def _run_scan(s, case):
    return list(compute_query_ema_history(s["x"], s["rhos"], case["V"], s["c_base"], s["unique"], return_state=True))


def _run_gating(s, case):
    y = GatedQueryFunction.apply(s["x"], s["C"], s["W"].t(), s["w"], s["b"], True)
    return [y, *torch.autograd.grad(y, [s[k] for k in _LEAVES["gating"]], s["dy"])]


def _run_rows(s, case):
    y = rms_norm(s["x"], s["w"], 1e-6)
    z = layer_norm(s["e"], s["lw"], s["lb"], 1e-5)
    m = swiglu_product(s["a"], s["b"])
    return [y, z, m, *torch.autograd.grad([y, z, m], [s[k] for k in _LEAVES["rows"]], [s["dy"], s["de"], s["dm"]])]


def _run_factored(s, case):
    O = factored_ema_forward(s["Q"], s["x"], s["E_k"], s["E_v"], s["rhos"], s["W"], case["H"], c_base=s["c_base"],
                             unique_slots=s["unique"], pad_mask=s["unique"] >= 0)
    return [O, *torch.autograd.grad(O, [s[k] for k in _LEAVES["factored"]], s["dO"])]


def _run_corpus(s, case):
    return corpus_states(s["tokens"], s["docs"], s["rhos"])


def _run_batch(s, case):
    return list(s["data"].get_batch(s["pick"]))


def _run_model(s, case):
    model = s["model"]
    logits = model(s["x"], unique_slots=s["unique"], c_base=s["c_base"], pad_mask=s["mask"])
    loss = F.cross_entropy(logits.view(-1, case["V"]), s["targets"].view(-1), ignore_index=-1)
    names, weights = zip(*model.named_parameters())
    return {"logits": logits, **dict(zip(names, torch.autograd.grad(loss, weights)))}


_RUN = {"attention": _run_attention, "dense": _run_dense, "eval": _run_eval, "scan": _run_scan,
        "gating": _run_gating, "rows": _run_rows, "factored": _run_factored, "corpus": _run_corpus,
        "batch": _run_batch, "model": _run_model}


# ---- what a pass needs and how close it is ---------------------------------------------

def work(case):
    """Each input read once and each output written once; the gate's matrix products and the
    per-element products of the attention over its (step, slot) pairs."""
    k = case["kind"]
    if k in ("attention", "dense", "eval"):
        B, T, H, hd, N, V = (case[q] for q in ("B", "T", "H", "hd", "N", "V"))
        D, K = H * hd, _slots(T + case.get("history", 0), V)
        pairs, rows = B * T * K, B * T * D
        state = B * K * N if case.get("history") else 0
        if k == "eval":
            return {"bytes": 4 * (2 * rows + 2 * B * K * D + state + B * T * N) + 8 * B * (T + K),
                    "flops": pairs * (2 * N * D + 4 * D)}
        return {"bytes": 4 * (4 * rows + 4 * B * K * D + state + 2 * N * D) + 8 * B * (T + K),
                "flops": pairs * (6 * N * D + 14 * D)}
    if k == "scan":
        B, T, N, V = (case[q] for q in ("B", "T", "N", "V"))
        K = _slots(T + case["history"], V)  # the whole state comes back
        return {"bytes": 4 * B * N * (T + 2 * K) + 8 * B * (T + K) + 4 * B * K, "flops": 2 * B * T * N}
    if k == "gating":
        rows, D, N = case["B"] * case["T"], case["D"], case["N"]
        # forward: x, C, y; backward: dy, x, C, dx (the gate's input can be recomputed)
        return {"bytes": 4 * (rows * (5 * D + 2 * N) + 2 * N * D), "flops": rows * (4 * N * D + 30 * D)}
    if k == "rows":
        r, e, D, h = case["rows"], case["slots"], case["D"], case["hidden"]
        return {"bytes": 4 * 5 * (r + e) * D + 2 * 8 * r * h, "flops": 20 * ((r + e) * D + r * h)}
    if k == "factored":
        B, T, H, hd, N, V = (case[q] for q in ("B", "T", "H", "hd", "N", "V"))
        D, K = H * hd, _slots(T + case["history"], V)
        return {"bytes": 4 * (4 * B * T * D + 4 * V * D + B * K * N + 2 * N * D) + 8 * B * (T + K),
                "flops": 6.0 * B * (K + T) * N * hd * D + 23 * B * D * T * (T - 1) / 2}
    if k == "corpus":
        return {"bytes": case["T"] * (8 + 4 * case["N"]), "flops": 2 * case["T"] * case["N"]}
    if k == "batch":
        K = _slots(case["block"] + case["median"], case["V"])
        span = case["median"] + case["block"]
        return {"bytes": case["B"] * (4 * span + 8 * K * case["N"] + 9 * K + 24 * case["block"]), "flops": 0}
    B, T, D, N, V, layers = (case[q] for q in ("B", "T", "D", "N", "V", "layers"))
    K = _slots(T + 1000, V)
    ff = 256 * ((int(8 * D / 3) + 255) // 256)
    dense = 6 * (B * T * (2 * D * D + 3 * D * ff) + 2 * B * K * D * D) + B * T * K * (6 * N * D + 14 * D)
    return {"bytes": 4 * (2 * V * D + B * T * V), "flops": layers * dense + 6 * B * T * D * V}


def tolerance(case):
    """Four times what two correct evaluations were seen to differ by, or what each was seen to
    be from 64 bits, whichever is larger."""
    k = case["kind"]
    if k == "attention" and case["precision"] == "fp32":
        return {"rel": 3e-5, "max": 1e-2}
    if k in ("attention", "dense"):
        return {"rel": 1e-2, "max": 0.5}  # bf16 operands of the dW_pe product: 2e-3 to 3e-3 of its values
    if k == "eval":
        return {"rel": 5e-5, "max": 1e-2}  # split fp16 operands of the gate, no bf16 product
    if k == "model":
        return {"rel": 2e-2, "max": 0.9}  # the attention's roundings through the layers and the softmax
    if k == "rows":
        return {"rel": 1e-3, "max": 2e-2}  # bf16 results, rounded once
    if k == "batch":
        return {"rel": 1e-5, "max": 1e-4}  # ids, masks and counts are whole numbers: the same
    if k == "factored":
        return {"rel": 3e-5, "max": 5e-3}  # split bf16 operands of the state products
    return {"rel": 1e-5, "max": 1e-3}  # 32-bit sums


# ---- the same in 64 bits ---------------------------------------------------------------

def exact(case, seed):
    """run()'s results for these inputs from plain torch in 64 bits, None where there are none
    or where they would take long."""
    k = case["kind"]
    if k in ("attention", "eval", "dense"):
        elements = case["B"] * case["T"] * _slots(case["T"] + case.get("history", 0), case["V"]) * case["H"] * case["hd"]
        if elements > 1e11 or (k == "eval" and case["B"] * case["T"] > 20000):
            return None
    if k == "factored" and _cost(case) > 4e10:
        return None
    s = _inputs(case, seed)
    with torch.enable_grad():
        return _EXACT[k](s, case)


def _f64(t):
    return t.detach().to(torch.float64)


def _counters(x, slots, rhos, c0, start, stop, state):
    """Decayed counters [B, t, K, N] of steps [start, stop) and the state after them."""
    rows = []
    for t in range(start, stop):
        c = state * rhos
        rows.append(c)
        state = c + (slots == x[:, t:t + 1]).to(c.dtype).unsqueeze(-1)
    return torch.stack(rows, 1), state


def _attend(Q, C, E_k, E_v, W, valid, absent):
    """One block of steps: Q [B, t, H, hd], C [B, t, K, N], E [B, K, H, hd], W [N, H, hd]."""
    B, t, H, hd = Q.shape
    gate = F.silu((C.reshape(-1, C.shape[-1]) @ W.reshape(W.shape[0], -1)).view(B, t, -1, H, hd))
    s = (gate * (Q.unsqueeze(2) * E_k.unsqueeze(1))).sum(-1) / math.sqrt(hd)
    s = s.masked_fill(~valid[:, None, :, None], float("-inf"))
    m = s.amax(2, keepdim=True).clamp(min=0).detach()
    w = torch.exp(s - m)
    w = w / (w.sum(2, keepdim=True) + absent[:, None, None, None] * torch.exp(-m))
    return (gate * (w.unsqueeze(-1) * E_v.unsqueeze(1))).sum(2)


def _attention64(Q, x, E_k, E_v, W, rhos, slots, c0, V, dO=None):
    """O [B, T, H, hd], and with dO the gradients of Q, E_k [B, K, H, hd], E_v and W [N, H, hd]."""
    B, T, H, hd = Q.shape
    valid = slots >= 0
    absent = (V - valid.sum(1)).to(torch.float64)
    state = torch.zeros(B, slots.shape[1], rhos.shape[0], dtype=torch.float64, device=DEV) if c0 is None else c0
    step = max(1, min(T, int(2.5e8 / max(1, B * slots.shape[1] * max(H * hd, rhos.shape[0])))))
    E_k, E_v, W = (t.detach().requires_grad_(dO is not None) for t in (E_k, E_v, W))
    O, dQ, sums = torch.empty_like(Q), torch.empty_like(Q), None
    for t in range(0, T, step):
        C, state = _counters(x, slots, rhos, c0, t, min(T, t + step), state)
        q = Q[:, t:t + step].detach().requires_grad_(dO is not None)
        with torch.set_grad_enabled(dO is not None):
            o = _attend(q, C, E_k, E_v, W, valid, absent)
        O[:, t:t + step] = o.detach()
        if dO is not None:
            g = torch.autograd.grad(o, (q, E_k, E_v, W), dO[:, t:t + step])
            dQ[:, t:t + step] = g[0]
            sums = list(g[1:]) if sums is None else [a + b for a, b in zip(sums, g[1:])]
    return (O, dQ, *sums) if dO is not None else O


def _heads(t, H):
    return t.unflatten(-1, (H, -1))


def _exact_attention(s, case):
    H = case["H"]
    O, dQ, dk, dv, dW = _attention64(
        _f64(s["Q"]).transpose(1, 2).contiguous(), s["x"], _heads(_f64(s["E_k"]), H), _heads(_f64(s["E_v"]), H),
        _heads(_f64(s["W"]), H), _f64(s["rhos"]), s["unique"], _f64(s["c_base"]), case["V"],
        _f64(s["dO"]).transpose(1, 2))
    return [O.transpose(1, 2), dQ.transpose(1, 2), dk.flatten(2), dv.flatten(2), dW.flatten(1)]


def _distinct_rows(x):
    """Each row's distinct ids, padded with -1."""
    rows = [torch.unique(r) for r in x]
    K = max(len(r) for r in rows)
    return torch.stack([F.pad(r, (0, K - len(r)), value=-1) for r in rows])


def _exact_dense(s, case):
    H = case["H"]
    slots = _distinct_rows(s["x"])
    at = slots.clamp(min=0)
    real = (slots >= 0)[..., None, None].to(torch.float64)
    E_k, E_v = _f64(s["E_k"]), _f64(s["E_v"])
    O, dQ, dk, dv, dW = _attention64(
        _heads(_f64(s["Q"]), H), s["x"], _heads(E_k[at], H), _heads(E_v[at], H), _heads(_f64(s["pe"].weight).t(), H),
        _f64(s["rhos"]), slots, None, case["V"], _heads(_f64(s["dO"]), H))
    put = lambda e, g: torch.zeros_like(e).index_add_(0, at.reshape(-1), (g * real).flatten(2).flatten(0, 1))  # noqa: E731
    return [O.flatten(2), dQ.flatten(2), put(E_k, dk), put(E_v, dv), dW.flatten(1).t()]


def _history64(s):
    """C_seq [B, T, N], and the lazy state [B, K, N] after each slot's last occurrence."""
    x, slots, rhos, A = s["x"], s["unique"], _f64(s["rhos"]), _f64(s["c_base"])
    B, T = x.shape
    N = rhos.shape[0]
    valid = slots >= 0
    ids, order = torch.where(valid, slots, torch.full_like(slots, 1 << 40)).sort(1)
    at = order.gather(1, torch.searchsorted(ids, x))  # the slot of each token
    b = torch.arange(B, device=DEV)
    lazy, last = A.clone(), torch.zeros(B, slots.shape[1], dtype=torch.float64, device=DEV)
    out = torch.empty(B, T, N, dtype=torch.float64, device=DEV)
    for t in range(T):
        k = at[:, t]
        row = lazy[b, k] * rhos ** (t - last[b, k]).unsqueeze(-1)
        out[:, t] = row
        lazy[b, k] = row + 1
        last[b, k] = t
    return out, lazy


def _exact_eval(s, case):
    H = case["H"]
    O = _attention64(_f64(s["Q"]).transpose(1, 2).contiguous(), s["x"], _heads(_f64(s["E_k"]), H),
                     _heads(_f64(s["E_v"]), H), _heads(_f64(s["W"]), H), _f64(s["rhos"]), s["unique"],
                     _f64(s["c_base"]), case["V"])
    return [_history64(s)[0], O.transpose(1, 2)]


def _exact_scan(s, case):
    out, lazy = _history64(s)
    return [out, lazy, None]


def _gate64(x, C, W, w, b):
    return F.layer_norm(x * F.silu((C + 1) @ W.t()), (x.shape[-1],), w, b, 1e-5)


def _exact_gating(s, case):
    leaf = [_f64(s[k]).requires_grad_(True) for k in _LEAVES["gating"]]
    y = _gate64(leaf[0], _f64(s["C"]), *leaf[1:])
    return [y, *torch.autograd.grad(y, leaf, _f64(s["dy"]))]


def _rms64(x, w, eps):
    return w * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _exact_rows(s, case):
    leaf = [_f64(s[k]).requires_grad_(True) for k in _LEAVES["rows"]]
    x, w, e, lw, lb, a, b = leaf
    outs = [_rms64(x, w, 1e-6), F.layer_norm(e, (e.shape[-1],), lw, lb, 1e-5), F.silu(a) * b]
    return [*outs, *torch.autograd.grad(outs, leaf, [_f64(s["dy"]), _f64(s["de"]), _f64(s["dm"])])]


def _exact_factored(s, case):
    """The attention with a linear gate and no softmax, by a state per step:
    o_t = sum_n (q_t W_n)^T S_n with S_n <- rho_n S_n before each step and, after it,
    + e_k e_v^T of the step's token; S_n starts as the slots' sum weighted by c_base."""
    H, N = case["H"], case["N"]
    B, T = s["x"].shape
    leaf = [_f64(s[k]).requires_grad_(True) for k in _LEAVES["factored"]]
    Q, E_k, E_v, W = leaf
    rhos, u = _f64(s["rhos"]), s["unique"]
    c = _f64(s["c_base"]) * (u >= 0).unsqueeze(-1)
    powers = rhos.unsqueeze(0) ** torch.arange(T + 1, dtype=torch.float64, device=DEV).unsqueeze(1)  # [T+1, N]
    G = powers @ W  # [T+1, D]
    t = torch.arange(T, device=DEV)
    lag = t.view(-1, 1) - t.view(1, -1)

    def one(b, q, ek, ev, w, G, uk, uv):
        q, w, G, ek, ev, uk, uv = (_heads(z, H) for z in (q, w, G, ek, ev, uk, uv))
        outs = []
        for h in range(H):
            gate = G[:, h][lag.clamp(min=0)] * (lag > 0).unsqueeze(-1)  # [T, T, hd]
            A = (gate * ek[:, h].unsqueeze(0) * q[:, h].unsqueeze(1)).sum(-1)
            S = (c[b].t().unsqueeze(1) * uk[:, h].t().unsqueeze(0)) @ uv[:, h]  # [N, hd, hd]
            carried = torch.einsum("tn,tni->ti", powers[1:], ((q[:, h].unsqueeze(0) * w[:, h].unsqueeze(1)) @ S).transpose(0, 1))
            outs.append(A @ ev[:, h] + carried)
        return torch.stack(outs, 1).flatten(1)

    O = torch.empty(B, T, Q.shape[2], dtype=torch.float64, device=DEV)
    sums = [torch.zeros_like(z) for z in leaf]
    dO = _f64(s["dO"])
    for b in range(B):
        ids = u[b].clamp(min=0)
        o = one(b, Q[b], E_k[s["x"][b]], E_v[s["x"][b]], W, powers @ W, E_k[ids], E_v[ids])
        O[b] = o.detach()
        for z, g in zip(sums, torch.autograd.grad(o, leaf, dO[b])):
            z += g
    return [O, *sums]


def _exact_corpus(s, case):
    """Each position's occurrences of its (document, token) before it, by doubling the reach
    along the sorted chains."""
    T = s["tokens"].numel()
    if T * case["N"] > 3e8:
        return None
    key = (s["docs"].long() << 32) | s["tokens"].long()
    key, order = torch.sort(key, stable=True)
    pos = order.to(torch.float64)
    state = torch.ones(T, case["N"], dtype=torch.float64, device=DEV)
    rhos = _f64(s["rhos"])
    first = torch.ones(T, dtype=torch.bool, device=DEV)
    first[1:] = key[1:] != key[:-1]
    head = torch.cummax(torch.where(first, torch.arange(T, device=DEV), 0), 0).values
    reach = 1
    longest = int((torch.arange(T, device=DEV) - head).max()) + 1
    while reach < longest:
        back = torch.arange(T, device=DEV) - reach
        ok = back >= head
        i = ok.nonzero().squeeze(1)
        add = state[back[i]] * rhos ** (pos[i] - pos[back[i]]).unsqueeze(1)
        state[i] += add
        reach *= 2
    out = torch.empty_like(state)
    out[order] = state
    return out


def _exact_batch(s, case):
    """c_base from the corpus itself; the rest is whole numbers."""
    data = s["data"]
    rhos = torch.as_tensor(data.rhos, dtype=torch.float64)
    slots = data.get_batch(s["pick"])[1].cpu()
    mask = torch.zeros(slots.shape, dtype=torch.bool)
    out = torch.zeros(*slots.shape, case["N"], dtype=torch.float64)
    for i, p in enumerate(s["pick"]):
        start, end, doc = data.chunks[int(p)]
        begin = data.doc_starts[doc]
        history = torch.from_numpy(np.array(data.tokens[begin:start])).long()
        chunk = torch.from_numpy(np.array(data.tokens[start:end])).long()
        n = len(torch.unique(torch.cat([history, chunk])))
        mask[i, :n] = True
        if len(history):
            ids, inv = torch.unique(history, return_inverse=True)
            age = torch.arange(len(history), 0, -1, dtype=torch.float64).unsqueeze(1)
            sums = torch.zeros(len(ids), case["N"], dtype=torch.float64).index_add_(0, inv, rhos ** age)
            at = torch.searchsorted(ids, slots[i, :n]).clamp(max=len(ids) - 1)
            out[i, :n] = torch.where((ids[at] == slots[i, :n]).unsqueeze(1), sums[at], 0.0)
    return [None, None, None, None, out, None, None]


def _exact_model(s, case):
    H, N, V = case["H"], case["N"], case["V"]
    names = [n for n, _ in s["model"].named_parameters()]
    P = {n: _f64(p).requires_grad_(True) for n, p in s["model"].named_parameters()}
    x, slots, rhos = s["x"], s["unique"], _f64(s["model"].ema_rhos)
    B, T = x.shape
    c0 = _f64(s["c_base"])
    if slots.shape[1] < 16:
        slots = F.pad(slots, (0, 16 - slots.shape[1]), value=-1)
        c0 = F.pad(c0, (0, 0, 0, 16 - c0.shape[1]))
    valid = slots >= 0
    absent = (V - valid.sum(1)).to(torch.float64)
    E = P["embed.weight"]
    # the query side takes a token without a slot (the padding's token 0) from zero
    extra = (~(slots.unsqueeze(1) == x.unsqueeze(2)).any(2))
    q = dict(x=x, unique=slots, rhos=rhos, c_base=c0)
    if bool(extra.any()):
        q["unique"] = torch.cat([slots, torch.where(extra.any(1, keepdim=True), x.new_zeros(B, 1), x.new_full((B, 1), -1))], 1)
        q["c_base"] = F.pad(c0, (0, 0, 0, 1))
    C_seq = _history64(q)[0]
    step = max(1, min(T, int(1.5e8 / (B * slots.shape[1] * case["D"]))))
    with torch.no_grad():
        blocks, state = [], c0
        for t in range(0, T, step):
            blocks.append(state)
            state = _counters(x, slots, rhos, c0, t, min(T, t + step), state)[1]

    def block(t, state, Q, E_k, E_v, W):
        with torch.no_grad():
            C = _counters(x, slots, rhos, c0, t, min(T, t + step), state)[0]
        return _attend(Q, C, E_k, E_v, W, valid, absent)

    h = E[x]
    for i in range(case["layers"]):
        p = lambda n: P[f"layers.{i}.{n}"]  # noqa: E731
        memory = F.layer_norm(E[slots.clamp(min=0)], (case["D"],), p("attn.ln_kv.weight"), p("attn.ln_kv.bias"), 1e-5)
        E_k, E_v = (_heads(memory @ p(f"attn.{n}.weight").t(), H) for n in ("k_proj", "v_proj"))
        pe = p("attn.pe_proj.weight")
        gated = _gate64(_rms64(h, p("attn_norm.weight"), 1e-6), C_seq, pe, p("attn.ln_q.weight"), p("attn.ln_q.bias"))
        Q = _heads(gated @ p("attn.q_proj.weight").t(), H)
        W = _heads(pe.t(), H)
        O = torch.cat([checkpoint(block, t, blocks[j], Q[:, t:t + step], E_k, E_v, W, use_reentrant=False)
                       for j, t in enumerate(range(0, T, step))], 1)
        h = h + O.flatten(2) @ p("attn.o_proj.weight").t()
        n = _rms64(h, p("ffn_norm.weight"), 1e-6)
        h = h + (F.silu(n @ p("ffn.w1.weight").t()) * (n @ p("ffn.w3.weight").t())) @ p("ffn.w2.weight").t()
    logits = _rms64(h, P["final_norm.weight"], 1e-6) @ E.t()
    loss = F.cross_entropy(logits.view(-1, V), s["targets"].view(-1), ignore_index=-1)
    return {"logits": logits, **dict(zip(names, torch.autograd.grad(loss, [P[n] for n in names])))}


_EXACT = {"attention": _exact_attention, "dense": _exact_dense, "eval": _exact_eval, "scan": _exact_scan,
          "gating": _exact_gating, "rows": _exact_rows, "factored": _exact_factored, "corpus": _exact_corpus,
          "batch": _exact_batch, "model": _exact_model}
