"""The workloads whose speed this package is judged by: what a draft training program has the
package do, over the range of sizes it meets, each through a public entry point.

Kinds of cases:

  attention  DSpark block-sparse attention of one packed row (or an unpacked batch): the forward's
             integer metadata and tile plan, the forward and, unless the case is an evaluation, the
             backward to Q, K and V (`direct_cp_attention_from_kv`)
  loss       the selective head's cross-entropy and softmax-L1 from bf16 logits, forward and
             backward (`ce_l1_from_logits`; without a teacher, cross-entropy alone)
  head       the head's objective: vocabulary GEMM, loss, dlogits, dgrad GEMM
             (`selective_head_objective`)
  sampled    the L1 between temperature / top-p / top-k filtered distributions, forward and backward
             (`compiled_l1_from_logits`)
  qk         per-head Q/K RMSNorm, key join and RoPE, forward and backward (`dspark_qk_norm_rope`)
  row        what surrounds a step's tensors: packing documents into a row, sampling anchors, the
             DSpark targets, the row's mask tensors and its sparse tile lists
  step       one whole training step of the one-layer draft model: forward, objective, backward,
             AdamW (`dspark_layer_step`)

`listed()` gives the standing cases and `draw()` more of the same ranges; `prepare()` makes what a
program holds before the call, `run()` is one pass, `work()` what the pass cannot do without,
`exact()` the same result in 64 bits by plain torch.
"""

import math
import random

import torch

from aspec_amd.anchors import anchor_sampling_seed, sample_document_anchor_positions
from aspec_amd.collate import DFlashPackingCollator
from aspec_amd.direct_cp import DirectCPMetadata, direct_cp_attention_from_kv
from aspec_amd.draft_layer import DSparkDraftLayerModel, FusedBF16Optimizer, dspark_layer_step, layer_batch
from aspec_amd.dspark_qk_norm_rope import dspark_qk_norm_rope
from aspec_amd.head_loss import selective_head_objective
from aspec_amd.loss import ce_l1_from_logits
from aspec_amd.sampling import compiled_l1_from_logits
from aspec_amd.targets import dspark_targets
from aspec_amd.thd_attention import thd_fixed_aux
from aspec_amd.thd_sparse_metadata import build_thd_sparse_pair
from aspec_amd.workloads import from_layout

DEV = "cuda"
HEAD_DIM = 128
GAMMA = 4.0                       # decay of the loss weights within a block
CE_ALPHA, L1_ALPHA = 0.1, 0.9
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


# ---- the cases -----------------------------------------------------------------------------------
def _attention(name, context, docs, stride, block, heads, kv_heads, *, dtype="bf16", batch=1, window=0,
               causal=False, backward=True, layout=0):
    """`docs` documents of uneven lengths packed into `context` tokens, an anchor every `stride`
    tokens of a document, `block` draft tokens per anchor. docs = 0: an unpacked batch of `batch`
    rows of `context` tokens each."""
    return {"name": name, "kind": "attention", "context": context, "docs": docs, "stride": stride,
            "block": block, "heads": heads, "kv_heads": kv_heads, "dtype": dtype, "batch": batch,
            "window": window, "causal": causal, "backward": backward, "layout": layout}


def listed():
    return [
        # A short packed row: four documents under a thousand tokens each, some forty draft blocks.
        # Latency and launches count.
        _attention("attention_short_row", 2767, 4, 64, 16, 32, 8),
        # The ordinary row: one 4096-token document, 512 blocks of 16 draft tokens, GQA 32/8.
        _attention("attention_4k_row", 4096, 1, 8, 16, 32, 8),
        # A ragged 32K row of many short documents, an anchor every 32 tokens: tile skipping and
        # load balance.
        _attention("attention_ragged_32k", 32736, 44, 32, 16, 32, 8, layout=3),
        # The long-context row of the published attention study's shape: twelve documents in 131072
        # tokens, blocks of 7.
        _attention("attention_128k_row", 131072, 12, 21, 7, 32, 8, layout=7),
        # Evaluation of an unpacked fp16 batch with a context window: forward only, GQA 40/8.
        _attention("attention_eval_f16", 6001, 0, 16, 16, 40, 8, dtype="f16", batch=2, window=2048,
                   backward=False),
        # The head's loss of one row's blocks over the draft vocabulary, against an indexed teacher.
        {"name": "loss_32k_vocab", "kind": "loss", "rows": 8192, "vocab": 32000, "teacher_rows": 4096, "l1": True},
        # The same over the full target vocabulary, a chunk of rows at a time.
        {"name": "loss_152k_vocab", "kind": "loss", "rows": 2048, "vocab": 151936, "teacher_rows": 1024, "l1": True},
        # The head's whole objective in the ordinary row.
        {"name": "head_objective", "kind": "head", "rows": 8192, "hidden": 4096, "vocab": 32000, "teacher_rows": 4096},
        # The L1 under sampling: a filtered teacher against a filtered draft.
        {"name": "sampled_l1", "kind": "sampled", "rows": 2048, "vocab": 32000, "teacher_rows": 1024,
         "t_temp": 0.8, "t_top_p": 0.95, "t_top_k": 50, "d_temp": 1.2, "d_top_p": 0.9, "d_top_k": -1},
        # Q/K preparation of the ordinary row.
        {"name": "qk_norm_rope", "kind": "qk", "context": 4096, "draft": 8192, "heads": 32, "kv_heads": 8,
         "batch": 1, "dtype": "bf16"},
        # Row preparation of 23 documents in an 8K row with its hidden states.
        {"name": "row_prepare", "kind": "row", "row": 8192, "docs": 23, "anchors": 48, "block": 16,
         "hidden": 4096, "layout": 5},
        # The whole training step of a one-layer draft model, three documents in a 4096-token row.
        {"name": "layer_step", "kind": "step", "context": 4096, "docs": 3, "stride": 8, "block": 16,
         "hidden": 4096, "heads": 32, "kv_heads": 8, "ffn": 12288, "vocab": 32000, "layout": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sampling(rng):
    return rng.choice([1.0, 0.7, 0.8, 1.2]), rng.choice([1.0, 0.9, 0.95, 0.8]), rng.choice([-1, 20, 50, 200])


def draw(rng):
    kind = rng.choice(["attention"] * 6 + ["loss"] * 4 + ["sampled"] * 2 + ["qk"] * 2 + ["head", "row", "step"])
    if kind == "attention":
        while True:
            packed = rng.random() < 0.8
            context = _log_int(rng, 700, 90000 if packed else 12000)
            heads, kv_heads = rng.choice([(32, 8), (32, 8), (32, 8), (40, 8), (64, 8), (16, 8), (28, 4), (12, 4), (8, 8)])
            c = _attention("", context, rng.randint(1, max(1, min(48, context // 400))) if packed else 0,
                           _log_int(rng, 6, 80), rng.choice([4, 7, 8, 16, 16, 16, 31]), heads, kv_heads,
                           dtype=rng.choice(["bf16"] * 4 + ["f16"]), batch=1 if packed else rng.randint(1, 4),
                           window=rng.choice([0, 0, 0, 1024, 3000]), causal=rng.random() < 0.15,
                           backward=rng.random() < 0.85, layout=rng.randrange(1 << 16))
            queries = context // c["stride"] * c["block"] * c["batch"]
            if 64 <= queries <= 45000 and work(c)["flops"] <= 2.0e13:
                break
    elif kind in ("loss", "sampled"):
        most = 8192 * 32000 if kind == "loss" else 2048 * 32000
        vocab = _log_int(rng, 3000, 152064)
        vocab = vocab if rng.random() < 0.25 else vocab // 64 * 64
        rows = _log_int(rng, 48, max(49, min(8192, most // vocab)))
        c = {"kind": kind, "rows": rows, "vocab": vocab,
             "teacher_rows": rng.choice([0, max(1, rows // 2), max(1, rows // 3)])}
        if kind == "loss":
            c["l1"] = rng.random() < 0.8
        else:
            for side in "td":
                c[side + "_temp"], c[side + "_top_p"], c[side + "_top_k"] = _sampling(rng)
            if (c["t_temp"], c["t_top_p"], c["t_top_k"]) == (1.0, 1.0, -1):
                c["t_top_p"] = 0.9
    elif kind == "qk":
        c = {"kind": kind, "context": _log_int(rng, 200, 8192), "draft": _log_int(rng, 100, 8192),
             **dict(zip(("heads", "kv_heads"), rng.choice([(32, 8), (40, 8), (16, 8), (64, 8), (12, 4)]))),
             "batch": rng.choice([1, 1, 2]), "dtype": rng.choice(["bf16", "bf16", "f16"])}
    elif kind == "head":
        rows = _log_int(rng, 256, 8192)
        c = {"kind": kind, "rows": rows, "hidden": rng.choice([2048, 2560, 4096]),
             "vocab": rng.choice([8192, 16000, 32000, 32768]), "teacher_rows": max(1, rows // 2)}
    elif kind == "row":
        row = _log_int(rng, 1024, 16384)
        c = {"kind": kind, "row": row, "docs": rng.randint(1, max(1, row // 300)), "anchors": rng.randint(8, 64),
             "block": rng.choice([7, 8, 16]), "hidden": rng.choice([2048, 4096]), "layout": rng.randrange(1 << 16)}
    else:
        hidden, heads, kv_heads, ffn = rng.choice([(2048, 16, 8, 6144), (2560, 32, 8, 9728), (4096, 32, 8, 12288)])
        c = {"kind": kind, "context": _log_int(rng, 1024, 4096), "docs": rng.randint(1, 4),
             "stride": rng.randint(8, 40), "block": rng.choice([7, 8, 16]), "hidden": hidden, "heads": heads,
             "kv_heads": kv_heads, "ffn": ffn, "vocab": 32000, "layout": rng.randrange(1 << 16)}
    c.pop("name", None)
    return c


# ---- layouts -------------------------------------------------------------------------------------
def _lengths(total, docs, seed):
    """`docs` uneven document lengths (log-normal shares, at least 48 tokens) that sum to `total`."""
    rng = random.Random(seed)
    docs = max(1, min(docs, total // 64))
    share = [rng.lognormvariate(0.0, 0.8) for _ in range(docs)]
    free = total - 48 * docs
    lengths = [48 + int(free * s / sum(share)) for s in share]
    lengths[-1] += total - sum(lengths)
    return lengths


def _blocks(c):
    """Per block (row, document start, document end, anchor), row by row; a packed row's documents
    lie end to end, an unpacked row is one document."""
    rows = [[c["context"]]] * c["batch"] if not c["docs"] else [_lengths(c["context"], c["docs"], c["layout"])]
    out = []
    for b, lengths in enumerate(rows):
        start = 0
        for n in lengths:
            out += [(b, start, start + n, start + u) for u in range(0, n - c["block"], c["stride"])]
            start += n
    return out


def _intervals(c):
    """Visible context [begin, end) of each block and the row it lies in."""
    w = c["window"]
    return [(b, max(s, a - w) if w else s, a) for b, s, _, a in _blocks(c)]


def _pairs(c):
    block = c["block"]
    own = block * (block + 1) // 2 if c["causal"] else block * block
    return sum((hi - lo) * block + own for _, lo, hi in _intervals(c))


# ---- preparation ---------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def _logits(g, rows, vocab):
    """Logits with a few likely tokens per row over a broad tail, as a trained head gives them."""
    x = torch.randn(rows, vocab, generator=g, device=DEV) * 2.0
    hot = torch.randint(0, vocab, (rows, 8), generator=g, device=DEV)
    x.scatter_add_(1, hot, torch.rand(rows, 8, generator=g, device=DEV) * 8.0)
    return x


def _head_rows(c, g):
    """Draft logits, the frozen teacher table near them and the teacher's row indices."""
    rows, vocab = c["rows"], c["vocab"]
    table = _logits(g, c["teacher_rows"] or rows, vocab)
    index = (torch.randint(0, c["teacher_rows"], (rows,), generator=g, device=DEV) if c["teacher_rows"] else None)
    x = torch.empty(rows, vocab, dtype=torch.bfloat16, device=DEV)
    for r in range(0, rows, 1024):
        part = table[index[r:r + 1024]] if index is not None else table[r:r + 1024]
        x[r:r + 1024] = (0.8 * part + torch.randn(part.shape, generator=g, device=DEV)).to(torch.bfloat16)
    return x, table.to(torch.bfloat16), index


def _targets(g, rows, vocab):
    """Labels and decay weights of rows of blocks of 16; a tenth of the rows carries no label."""
    t = torch.randint(0, vocab, (rows,), generator=g, device=DEV)
    live = torch.rand(rows, generator=g, device=DEV) > 0.1
    w = torch.exp(-(torch.arange(rows, device=DEV) % 16).float() / GAMMA) * live
    return torch.where(live, t, -100), w / w.sum().clamp(min=1.0)


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    if kind == "attention":
        dtype, batch, hq, hkv = DTYPES[c["dtype"]], c["batch"], c["heads"], c["kv_heads"]
        blocks = _blocks(c)
        per_row = len(blocks) // batch
        nq, nk = per_row * c["block"], c["context"] + per_row * c["block"]
        leaf = lambda n, h, s: _randn(g, batch, n, h, HEAD_DIM, dtype=dtype, scale=s).transpose(1, 2).requires_grad_(c["backward"])  # noqa: E731
        long = lambda v: torch.tensor(v, dtype=torch.long, device=DEV).reshape(batch, -1)  # noqa: E731
        meta = {"anchors": long([a for *_, a in blocks]),
                "keep": torch.ones(batch, per_row, dtype=torch.bool, device=DEV),
                "positions": torch.arange(c["context"], device=DEV).repeat(batch, 1), "docs": None, "anchor_docs": None}
        if c["docs"]:
            lengths = torch.tensor(_lengths(c["context"], c["docs"], c["layout"]), device=DEV)
            meta["docs"] = torch.repeat_interleave(torch.arange(lengths.numel(), device=DEV), lengths)[None]
            meta["anchor_docs"] = meta["docs"][0][meta["anchors"][0]][None]
        s = {"q": leaf(nq, hq, 1.0), "k": leaf(nk, hkv, 1.0), "v": leaf(nk, hkv, 0.5), "meta": meta}
        if c["backward"]:
            s["dout"] = _randn(g, batch, nq, hq, HEAD_DIM, dtype=dtype).transpose(1, 2)
    elif kind == "loss":
        x, table, index = _head_rows(c, g)
        targets, w = _targets(g, c["rows"], c["vocab"])
        s = {"logits": x.requires_grad_(), "teacher": table if c["l1"] else None,
             "index": index if c["l1"] else None, "targets": targets, "w_ce": CE_ALPHA * w, "w_l1": L1_ALPHA * w}
    elif kind == "head":
        table = _randn(g, c["teacher_rows"], c["hidden"])
        weight = _randn(g, c["vocab"], c["hidden"], scale=2.0 * c["hidden"] ** -0.5)
        index = torch.randint(0, c["teacher_rows"], (c["rows"],), generator=g, device=DEV)
        hidden = (0.8 * table[index].float() + 0.6 * torch.randn(c["rows"], c["hidden"], generator=g, device=DEV)).to(torch.bfloat16)
        targets, w = _targets(g, c["rows"], c["vocab"])
        s = {"hidden": hidden.requires_grad_(), "weight": weight, "weight_t": weight.t().contiguous(),
             "teacher": table @ weight.t(), "index": index, "targets": targets, "w_ce": CE_ALPHA * w, "w_l1": L1_ALPHA * w}
    elif kind == "sampled":
        x, table, index = _head_rows(c, g)
        s = {"logits": x.requires_grad_(), "teacher": table, "index": index,
             "grad": torch.rand(c["rows"], generator=g, device=DEV) / c["rows"],
             "target": (c["t_temp"], c["t_top_p"], c["t_top_k"]), "draft": (c["d_temp"], c["d_top_p"], c["d_top_k"])}
    elif kind == "qk":
        dtype, b, lc, ld, hq, hkv = DTYPES[c["dtype"]], c["batch"], c["context"], c["draft"], c["heads"], c["kv_heads"]
        inv = 1.0 / (1e6 ** (torch.arange(0, HEAD_DIM, 2, device=DEV).float() / HEAD_DIM))
        phase = torch.outer(torch.arange(lc + 64, device=DEV).float(), inv).repeat(1, 2)
        pos = torch.randint(0, lc, (b, ld), generator=g, device=DEV)
        s = {"q": _randn(g, b, ld, hq * HEAD_DIM, dtype=dtype).requires_grad_(),
             "kc": _randn(g, b, lc, hkv * HEAD_DIM, dtype=dtype).requires_grad_(),
             "kd": _randn(g, b, ld, hkv * HEAD_DIM, dtype=dtype).requires_grad_(),
             "wq": (1 + 0.1 * _randn(g, HEAD_DIM)).to(dtype).requires_grad_(),
             "wk": (1 + 0.1 * _randn(g, HEAD_DIM)).to(dtype).requires_grad_(),
             "cos": phase.cos()[None, None].to(dtype), "sin": phase.sin()[None, None].to(dtype),
             "pos": pos, "pos_c": torch.arange(lc, device=DEV).repeat(b, 1),
             "gq": _randn(g, b, ld, hq, HEAD_DIM, dtype=dtype), "gk": _randn(g, b, lc + ld, hkv, HEAD_DIM, dtype=dtype)}
    elif kind == "row":
        features = []
        for i, n in enumerate(_lengths(c["row"] - c["row"] // 50, c["docs"], c["layout"])):
            features.append({
                "input_ids": torch.randint(0, 150000, (1, n), generator=g, device=DEV),
                "loss_mask": (torch.rand(1, n, generator=g, device=DEV) > 0.2).long(),
                "hidden_states": _randn(g, 1, n, 3 * c["hidden"]),
                "last_hidden_states": _randn(g, 1, n, c["hidden"]),
                "_aspec_work": {"execution_id": "e%d" % i}})
        s = {"features": features, "collator": DFlashPackingCollator(c["row"]), "seed": seed,
             "generator": torch.Generator(device=DEV)}
    else:
        w = _step_workload(c)
        model = DSparkDraftLayerModel(hidden=c["hidden"], heads=c["heads"], kv_heads=c["kv_heads"], ffn=c["ffn"],
                                      vocab=c["vocab"], draft_vocab=c["vocab"], device=DEV, seed=seed)
        s = {"model": model, "batch": layer_batch(model, w, seed=seed, decay_gamma=GAMMA),
             "optimizer": FusedBF16Optimizer(model, lr=1e-4, total_steps=100000, warmup_ratio=0.0)}
    return {"case": c, **s}


def _step_workload(c):
    import numpy as np

    lengths = _lengths(c["context"], c["docs"], c["layout"])
    anchors, docs, start = [], [], 0
    for d, n in enumerate(lengths):
        own = list(range(start, start + n - c["block"], c["stride"]))
        anchors += own
        docs += [d] * len(own)
        start += n
    return from_layout("step", lengths, np.asarray(anchors), np.asarray(docs), c["block"], q_heads=c["heads"],
                       kv_heads=c["kv_heads"])


# ---- one pass ------------------------------------------------------------------------------------
def _metadata(c, m):
    """A step's mask metadata: new in every step, shared by its layers."""
    return DirectCPMetadata(m["anchors"], m["keep"], m["positions"], c["block"], 0, 1, None,
                            context_doc_ids=m["docs"], anchor_doc_ids=m["anchor_docs"],
                            sequence_length=c["context"], backend="hip", context_window=c["window"] or None,
                            draft_is_causal=c["causal"])


def run(state):
    c, s = state["case"], state
    kind = c["kind"]
    if kind == "attention":
        meta = _metadata(c, s["meta"])
        if not c["backward"]:
            with torch.no_grad():
                return direct_cp_attention_from_kv(s["q"], s["k"], s["v"], meta)
        out, lse = direct_cp_attention_from_kv(s["q"], s["k"], s["v"], meta)
        return out, lse, *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"])
    if kind == "loss":
        ce, l1, argmax = ce_l1_from_logits(s["logits"], s["targets"], s["teacher"], teacher_indices=s["index"],
                                           return_argmax=True)
        if c["l1"]:
            return ce, l1, argmax, *torch.autograd.grad((ce, l1), s["logits"], (s["w_ce"], s["w_l1"]))
        return ce, argmax, *torch.autograd.grad(ce, s["logits"], s["w_ce"])
    if kind == "head":
        objective, ce, l1 = selective_head_objective(s["hidden"], s["weight"], s["targets"], s["teacher"],
                                                     ce_weights=s["w_ce"], l1_weights=s["w_l1"],
                                                     teacher_indices=s["index"], weight_t=s["weight_t"])
        return objective, ce, l1, *torch.autograd.grad(objective, s["hidden"])
    if kind == "sampled":
        l1 = compiled_l1_from_logits(s["logits"], s["teacher"], s["target"], s["draft"], teacher_indices=s["index"])
        return l1, *torch.autograd.grad(l1, s["logits"], s["grad"])
    if kind == "qk":
        q, k = dspark_qk_norm_rope(s["q"], s["kc"], s["kd"], s["wq"], s["wk"], 1e-6, s["cos"], s["sin"], s["pos"],
                                   s["pos_c"], s["pos"], c["heads"], c["kv_heads"], HEAD_DIM)
        return q, k, *torch.autograd.grad((q, k), (s["q"], s["kc"], s["kd"], s["wq"], s["wk"]), (s["gq"], s["gk"]))
    if kind == "row":
        return _run_row(c, s)
    loss, norm = dspark_layer_step(s["model"], s["optimizer"], s["batch"], ce_alpha=CE_ALPHA, l1_alpha=L1_ALPHA)
    opt = s["optimizer"]
    return loss, norm, opt.exp_avg, opt.master, opt.flat


def _run_row(c, s):
    row = s["collator"](s["features"])
    s["generator"].manual_seed(anchor_sampling_seed(s["seed"], 0, 0, 0))
    anchors, keep = sample_document_anchor_positions(row["loss_mask"], row["ctx_doc_ids"],
                                                     row["packed_document_lengths"], c["anchors"], c["block"],
                                                     s["generator"])
    t = dspark_targets(anchors, keep, row["input_ids"], row["loss_mask"], c["block"], loss_decay_gamma=GAMMA,
                       ctx_doc_ids=row["ctx_doc_ids"])
    positions = torch.arange(c["row"], device=anchors.device)[None]
    meta = DirectCPMetadata(anchors, keep, positions, c["block"], 0, 1, None, context_doc_ids=row["ctx_doc_ids"],
                            anchor_doc_ids=row["ctx_doc_ids"].gather(1, anchors), sequence_length=c["row"])
    aux = thd_fixed_aux(meta, anchors.device)
    queries = anchors.shape[1] * c["block"]
    pair = build_thd_sparse_pair(aux_tensors=aux, block_size=c["block"], query_length=queries,
                                 key_length=c["row"] + queries, query_head_dim=HEAD_DIM, value_head_dim=HEAD_DIM)
    lists = [getattr(side, n) for side in (pair.forward, pair.backward)
             for n in ("mask_block_cnt", "mask_block_idx", "full_block_cnt", "full_block_idx")]
    names = ("input_ids", "loss_mask", "ctx_doc_ids", "base_position_ids", "attention_mask", "cu_seqlens",
             "hidden_states", "last_hidden_states")
    return {"row": [row[n] for n in names], "anchors": [anchors, keep], "aux": aux, "lists": lists,
            "targets": [t.label_index, t.target_ids, t.prev_ids, t.teacher_index, t.eval_mask, t.weights]}


# ---- what a pass cannot do without ---------------------------------------------------------------
def work(case):
    c = case
    kind = c["kind"]
    if kind == "attention":
        nq = len(_blocks(c)) * c["block"]
        nk = c["context"] * c["batch"] + nq
        q, kv = nq * c["heads"] * HEAD_DIM * 2, nk * c["kv_heads"] * HEAD_DIM * 2
        flops = (14 if c["backward"] else 4) * c["heads"] * HEAD_DIM * _pairs(c)
        both = 4 * q + 4 * kv if c["backward"] else 2 * q + 2 * kv  # q, out[, dout, dq], k, v[, dk, dv]
        return {"bytes": both + nq * c["heads"] * 4, "flops": flops}
    if kind in ("loss", "sampled"):
        # the draft rows once, the teacher rows that are used once, the gradient once
        used = min(c["rows"], c["teacher_rows"] or c["rows"]) if kind == "sampled" or c["l1"] else 0
        return {"bytes": (2 * c["rows"] + used) * c["vocab"] * 2 + c["rows"] * 24, "flops": 0}
    if kind == "head":
        r, h, v = c["rows"], c["hidden"], c["vocab"]
        return {"bytes": 2 * (2 * r * h + 2 * v * h + c["teacher_rows"] * v), "flops": 4 * r * h * v}
    if kind == "qk":
        q = c["batch"] * c["draft"] * c["heads"] * HEAD_DIM * 2
        k = c["batch"] * (c["context"] + c["draft"]) * c["kv_heads"] * HEAD_DIM * 2
        return {"bytes": 4 * (q + k) + 2 * (c["context"] + 64) * HEAD_DIM * 2, "flops": 0}
    if kind == "row":
        return {"bytes": c["row"] * (2 * 4 * c["hidden"] * 2 + 2 * 16 + 24), "flops": 0}
    h, f, t = c["hidden"], c["ffn"], c["context"]
    w = _step_workload(c)
    nq = w.num_queries
    at = {"batch": 1, "window": 0, "causal": False, **c}
    d = HEAD_DIM
    weights = 3 * h * h + (2 * c["heads"] + 2 * c["kv_heads"]) * d * h + 3 * f * h
    gemm = (2 * 2 * t * 3 * h * h                                     # context projection: forward, weight
            + 3 * 2 * nq * 2 * c["heads"] * d * h                      # q and o projections
            + 3 * 2 * (t + nq) * 2 * c["kv_heads"] * d * h             # k and v projections
            + 3 * 2 * nq * 3 * f * h                                   # MLP
            - 2 * nq * (c["heads"] + 2 * c["kv_heads"]) * d * h        # the embedding is frozen
            + 2 * 2 * nq * h * c["vocab"] + 2 * t * h * c["vocab"])    # head forward, dgrad; teacher
    attn = 14 * c["heads"] * d * _pairs(at)
    return {"bytes": weights * 30 + 2 * c["vocab"] * h * 2 + 2 * t * 4 * h, "flops": gemm + attn}


def tolerance(case):
    """About four times the relative error against `exact()`, which is what rounding once to the
    result's type leaves: 1.8e-3 for bf16 gradients of 32-bit sums, 2.9e-3 (bf16) and 4e-4 (fp16)
    for attention, whose probabilities and dS are rounded too. Where the bf16 logits' own rounding
    decides the sign of p - q, the gradients through the head are 2.1e-2 off (head) and 1.1e-2 (step)."""
    kind = case["kind"]
    if kind == "row":
        return "exact"
    if kind == "attention":
        return {"rel": 1.2e-2 if case["dtype"] == "bf16" else 1.6e-3}
    return {"rel": {"head": 8e-2, "step": 4e-2}.get(kind, 7e-3)}


# ---- the same in 64 bits -------------------------------------------------------------------------
def _exact_attention(c, blocks, q, k, v, dout):
    """q [B, Hq, Nq, D], k / v [B, Hkv, T + Nq, D] (any dtype) -> out, lse and, with dout, dq, dk, dv
    in fp64. `blocks`: per block (row, context begin, context end)."""
    f64 = torch.float64
    hkv, G, B, T = k.shape[1], q.shape[1] // k.shape[1], c["block"], c["context"]
    scale = HEAD_DIM ** -0.5
    out = torch.zeros(q.shape, dtype=f64, device=DEV)
    lse = torch.full(q.shape[:3], -1.0e30, dtype=f64, device=DEV)
    grads = [torch.zeros(x.shape, dtype=f64, device=DEV) for x in (q, k, v)] if dout is not None else None
    step = max(1, 2048 // B)
    for row in range(q.shape[0]):
        mine = [(lo, hi) for b, lo, hi in blocks if b == row]
        for n0 in range(0, len(mine), step):
            part = mine[n0:n0 + step]
            lo, hi = min(x for x, _ in part), max(x for _, x in part)
            r = slice(n0 * B, (n0 + len(part)) * B)
            begin = torch.tensor([x for x, _ in part], device=DEV).repeat_interleave(B)[:, None]
            end = torch.tensor([x for _, x in part], device=DEV).repeat_interleave(B)[:, None]
            pos = torch.arange(lo, hi, device=DEV)[None]
            i = torch.arange(len(part) * B, device=DEV)
            own = i[:, None] // B == i[None] // B
            if c["causal"]:
                own &= i[None] <= i[:, None]
            seen = torch.cat(((pos >= begin) & (pos < end), own), dim=1)
            keys = torch.cat((torch.arange(lo, hi, device=DEV), T + n0 * B + i))
            for h in range(hkv):
                kk, vv = k[row, h, keys].to(f64), v[row, h, keys].to(f64)
                for head in range(h * G, (h + 1) * G):
                    qq = q[row, head, r].to(f64)
                    p = (qq @ kk.t() * scale).masked_fill_(~seen, -math.inf)
                    l = torch.logsumexp(p, dim=1)
                    p = p.sub_(l[:, None]).exp_()
                    o = p @ vv
                    out[row, head, r], lse[row, head, r] = o, l
                    if dout is None:
                        continue
                    g = dout[row, head, r].to(f64)
                    grads[2][row, h].index_add_(0, keys, p.t() @ g)
                    ds = p.mul_((g @ vv.t()).sub_((g * o).sum(1, keepdim=True))).mul_(scale)
                    grads[0][row, head, r] = ds @ kk
                    grads[1][row, h].index_add_(0, keys, ds.t() @ qq)
    return (out, lse, *grads) if dout is not None else (out, lse)


def _l1_parts(p, q, g):
    """Row L1 of two distributions and the gradient of g * L1 to the first one's logits."""
    sign = torch.sign(p - q)
    return (p - q).abs().sum(1), g[:, None] * p * (sign - (p * sign).sum(1, keepdim=True))


def _exact_loss(c, s):
    x, outs = s["logits"], ([], [], [])
    for r in range(0, c["rows"], 256):
        e = slice(r, r + 256)
        xs = x[e].detach().double()
        lse = torch.logsumexp(xs, dim=1)
        p = (xs - lse[:, None]).exp()
        live = s["targets"][e] != -100
        t = s["targets"][e].clamp(min=0)
        outs[0].append(torch.where(live, lse - xs.gather(1, t[:, None])[:, 0], 0.0))
        w = s["w_ce"][e].double() * live
        d = w[:, None] * p
        d.scatter_add_(1, t[:, None], -w[:, None])
        if s["teacher"] is not None:
            y = (s["teacher"][s["index"][e]] if s["index"] is not None else s["teacher"][e]).double()
            l1, dl = _l1_parts(p, torch.softmax(y, dim=1), s["w_l1"][e].double())
            outs[1].append(l1)
            d += dl
        outs[2].append(d)
    if "hidden" in s:
        return [torch.cat(o) for o in outs]
    ce, dx = torch.cat(outs[0]), torch.cat(outs[2])
    return (ce, torch.cat(outs[1]), None, dx) if outs[1] else (ce, None, dx)


def _filtered(x, sampling):
    """Probabilities on the joint top-k / top-p support, ties by token index."""
    temp, top_p, top_k = sampling
    x = (x - x.amax(1, keepdim=True)) / temp
    order = torch.argsort(x, dim=1, descending=True, stable=True)
    p = torch.softmax(x, dim=1).gather(1, order)
    keep = torch.ones_like(p, dtype=torch.bool)
    if top_p < 1.0:
        keep &= p.cumsum(1) - p <= float(torch.tensor(top_p, dtype=torch.float32))
    if 0 < top_k < x.shape[1]:
        keep[:, top_k:] = False
    keep = torch.zeros_like(keep).scatter_(1, order, keep)
    return torch.softmax(x.masked_fill(~keep, -math.inf), dim=1)


def _exact_sampled(c, s):
    l1, dx = [], []
    for r in range(0, c["rows"], 256):
        e = slice(r, r + 256)
        y = s["teacher"][s["index"][e]] if s["index"] is not None else s["teacher"][e]
        p, q = _filtered(s["logits"][e].detach().double(), s["draft"]), _filtered(y.double(), s["target"])
        a, b = _l1_parts(p, q, s["grad"][e].double() / s["draft"][0])
        l1.append(a)
        dx.append(b)
    return torch.cat(l1), torch.cat(dx)


def _rope(x, w, cos, sin, eps=1e-6):
    """RMSNorm of each head row times w, then rotary embedding; x [..., H, D], cos / sin [..., 1, D]."""
    n = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w
    a, b = n.chunk(2, dim=-1)
    return n * cos + torch.cat((-b, a), dim=-1) * sin


def _exact_qk(c, s):
    leaves = [s[n].detach().double().requires_grad_() for n in ("q", "kc", "kd", "wq", "wk")]
    q, kc, kd, wq, wk = leaves
    b, hq, hkv = c["batch"], c["heads"], c["kv_heads"]
    table = lambda t, pos: t[0, 0].double()[pos][:, :, None]  # noqa: E731
    joined = torch.cat((s["pos_c"], s["pos"]), dim=1)
    out_q = _rope(q.view(b, -1, hq, HEAD_DIM), wq, table(s["cos"], s["pos"]), table(s["sin"], s["pos"]))
    out_k = _rope(torch.cat((kc, kd), dim=1).view(b, -1, hkv, HEAD_DIM), wk, table(s["cos"], joined),
                  table(s["sin"], joined))
    grads = torch.autograd.grad((out_q, out_k), leaves, (s["gq"].double(), s["gk"].double()))
    return out_q.detach(), out_k.detach(), *grads


class _ExactAttention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, c, blocks):
        ctx.save_for_backward(q, k, v)
        ctx.rest = c, blocks
        return _exact_attention(c, blocks, q, k, v, None)[0]

    @staticmethod
    def backward(ctx, dout):
        return *_exact_attention(*ctx.rest, *ctx.saved_tensors, dout)[2:], None, None


def _exact_step(c, s):
    m, b = s["model"], s["batch"]
    named = [(n, p) for n, p in m.named_parameters() if p.requires_grad]
    P = {n: p.detach().double().requires_grad_() for n, p in named}
    norm = lambda x, w: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + m.eps) * w  # noqa: E731
    T, nq, d = c["context"], b["draft_input_ids"].shape[1], HEAD_DIM
    table = lambda t, pos: t[0, 0].double()[pos[0]][:, None]  # noqa: E731
    ctx = norm(b["target_hidden"][0].double() @ P["context_proj"].t(), P["context_norm"])
    draft = m.embed_tokens[b["draft_input_ids"][0]].double()
    x = norm(draft, P["input_layernorm"])
    both = torch.cat((ctx, x))
    pos, joined = b["draft_positions"], torch.cat((b["context_positions"], b["draft_positions"]), dim=1)
    q = _rope((x @ P["q_proj"].t()).view(nq, -1, d), P["q_norm"], table(m.rope_cos, pos), table(m.rope_sin, pos), m.eps)
    k = _rope((both @ P["k_proj"].t()).view(T + nq, -1, d), P["k_norm"], table(m.rope_cos, joined),
              table(m.rope_sin, joined), m.eps)
    v = (both @ P["v_proj"].t()).view(T + nq, -1, d)
    at = {"batch": 1, "window": 0, "causal": False, **c}
    o = _ExactAttention.apply(*(t.transpose(0, 1)[None] for t in (q, k, v)), at, _intervals(at))
    h = draft + o[0].transpose(0, 1).reshape(nq, -1) @ P["o_proj"].t()
    gate, up = (norm(h, P["post_attention_layernorm"]) @ P["gate_up_proj"].t()).chunk(2, dim=1)
    hidden = norm(h + (torch.nn.functional.silu(gate) * up) @ P["down_proj"].t(), P["final_norm"])
    head = m.lm_head.double()
    t = b["targets"]
    w = t.weights.reshape(-1).double()
    w = w / w.sum().clamp(min=1e-6)
    z = {"logits": (hidden @ head.t()).detach(), "teacher": b["teacher_hidden"][0].double() @ head.t(),
         "index": t.teacher_index.reshape(-1), "targets": t.target_ids.reshape(-1), "w_ce": CE_ALPHA * w,
         "w_l1": L1_ALPHA * w, "hidden": True}
    ce, l1, dz = _exact_loss({"rows": nq}, z)
    grads = torch.autograd.grad(hidden, [P[n] for n, _ in named], dz @ head)
    flat = torch.cat([g.reshape(-1) for g in grads])
    total = flat.norm()
    avg = 0.1 * torch.clamp(s["optimizer"].max_grad_norm / (total + 1e-6), max=1.0) * flat
    return (z["w_ce"] @ ce + z["w_l1"] @ l1), total, torch.cat((avg, avg.new_zeros(s["optimizer"].exp_avg.numel() - avg.numel()))), None, None


def exact(case, seed):
    c, s = case, prepare(case, seed)
    kind = c["kind"]
    if kind == "attention":
        return _exact_attention(c, _intervals(c), *(s[n].detach() for n in ("q", "k", "v")), s.get("dout"))
    if kind == "loss":
        return _exact_loss(c, s)
    if kind == "head":
        hidden, weight = s["hidden"].detach().double(), s["weight"].double()
        ce, l1, dz = _exact_loss(c, {**s, "logits": hidden @ weight.t()})
        return s["w_ce"].double() @ ce + s["w_l1"].double() @ l1, ce, l1, dz @ weight
    if kind == "sampled":
        return _exact_sampled(c, s)
    if kind == "qk":
        return _exact_qk(c, s)
    if kind == "row":
        return None
    return _exact_step(c, s)
