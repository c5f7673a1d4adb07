"""The calls by which a user of this framework spends GPU time, at the sizes they are made with.

Seven paths, each through its public entry points:

* `loop`      `calculate_divergence` per conversation on fp32 logits, `Losses.add_losses`, `Losses.backward`, `Losses.log`:
              the training loop of a program that only swapped two imports;
* `batch`     `distill_loss_batch_indexed` on the model's own [B, S, V] logits with `Losses`, training (forward and backward)
              or validation (no gradient, student alone scaled by the temperature);
* `topk`      `div_topk`: forward or reverse KL against stored top-K rows, loss and gradient in one call;
* `dense`     `div_dense`: forward KL, reverse KL or JSD against a dense teacher;
* `producer`  `teacher_topk`: what a teacher's logits become in the dataset;
* `multi`     `fkl_multi_teacher`: several stored teachers with another vocabulary, weighed and remapped;
* `marginal`  `rkl_marginalised`: a dense teacher of another tokenizer, marginalised along a byte-trie map.
"""
import math

import torch

import llm_distillery_amd as D
from llm_distillery_amd import synthetic, vocab_utils

DEV = "cuda"
CHUNK = 4096
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
BYTES = {"fp32": 4, "bf16": 2, "fp16": 2}


def listed():
    return [
        # one short exchange (a question and its answer) through the drop-in loop: launches and host work decide
        {"name": "loop_short", "path": "loop", "convos": 1, "tokens": 131, "vocab": 32000, "k": 400},
        # the default configuration: four conversations of 2048 tokens, vocabulary cropped to 32000, 400 stored entries a token
        {"name": "loop_default", "path": "loop", "convos": 4, "tokens": 2048, "vocab": 32000, "k": 400},
        # a full training batch of long conversations straight from a bf16 model of a 128k vocabulary
        {"name": "batch_train", "path": "batch", "train": True, "convos": 8, "tokens": 4096, "vocab": 128256, "pitch": 128256,
         "k": 200, "T": 1.0, "dtype": "bf16"},
        # a validation batch: ragged conversations, padded vocabulary cropped to the tokenizer's size, no gradient
        {"name": "batch_val_crop", "path": "batch", "train": False, "convos": 4, "tokens": 1021, "vocab": 151665, "pitch": 151936,
         "k": 200, "T": 2.0, "dtype": "bf16"},
        # forward KL on stored rows: a whole batch of a 128k vocabulary
        {"name": "fkl_128k", "path": "topk", "kind": "fkl", "rows": 32768, "vocab": 128256, "pitch": 128256, "k": 200, "T": 1.0,
         "dtype": "bf16", "masked": 0.0},
        # forward KL on an odd vocabulary stored without padding, odd row count, padding tokens among the rows
        {"name": "fkl_50257_odd", "path": "topk", "kind": "fkl", "rows": 4093, "vocab": 50257, "pitch": 50257, "k": 100, "T": 1.5,
         "dtype": "bf16", "masked": 0.1},
        # reverse KL on stored rows
        {"name": "rkl_128k", "path": "topk", "kind": "rkl", "rows": 8192, "vocab": 128256, "pitch": 128256, "k": 200, "T": 1.0,
         "dtype": "bf16", "masked": 0.0},
        # one conversation against a dense fp32 teacher, its tail padding
        {"name": "dense_fkl_512", "path": "dense", "kind": "fkl", "rows": 512, "vocab": 32000, "T": 1.0, "dtype": "fp32",
         "teacher": "fp32", "masked": 0.1},
        # JSD on a batch with ragged lengths
        {"name": "dense_jsd", "path": "dense", "kind": "jsd", "rows": 8192, "vocab": 32000, "T": 2.0, "dtype": "bf16",
         "teacher": "bf16", "masked": 0.25},
        # collecting a teacher's distributions: a batch of logits to stored rows
        {"name": "producer_128k", "path": "producer", "rows": 32768, "vocab": 128256, "pitch": 128256, "k": 200, "dtype": "bf16",
         "masked": 0.0},
        # three stored teachers of a 152k vocabulary onto a 128k student
        {"name": "multi_3", "path": "multi", "teachers": 3, "rows": 8192, "vocab": 128256, "teacher_vocab": 152064, "k": 200,
         "dtype": "bf16"},
        # a dense teacher of another tokenizer: 152k ids onto 32k
        {"name": "marginal_32k", "path": "marginal", "rows": 8192, "vocab": 32000, "teacher_vocab": 152064, "alphabet": 16, "T": 1.5,
         "dtype": "bf16"},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _vocab(rng, most=200064):
    """A vocabulary a tokenizer has, or any width."""
    if rng.random() < 0.5:
        return rng.choice([v for v in (32000, 32100, 50257, 50304, 100277, 128256, 151665, 151936) if v <= most])
    return _log(rng, 8000, most)


def _pitch(rng, vocab):
    """Columns of the stored rows: the vocabulary's own, or padded as model heads are."""
    return rng.choice([vocab, -(-vocab // 64) * 64, -(-vocab // 256) * 256])


def draw(rng):
    path = rng.choice(["loop", "batch", "topk", "dense", "producer", "multi", "marginal"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    most = 4 << 30                                        # logits of one pass, bytes
    if path == "loop":
        v, b = _vocab(rng), rng.randint(1, 8)
        return {"path": path, "convos": b, "tokens": min(_log(rng, 16, 4096), most // (4 * v * b)), "vocab": v, "k": _log(rng, 20, 500)}
    if path == "batch":
        v, b = _vocab(rng), rng.randint(1, 16)
        return {"path": path, "train": rng.random() < 0.7, "convos": b, "tokens": max(32, min(_log(rng, 64, 4096), most // (2 * v * b))),
                "vocab": v, "pitch": _pitch(rng, v), "k": _log(rng, 20, 500), "T": rng.choice([1.0, 1.5, 2.0]), "dtype": half}
    if path == "topk":
        v, dt = _vocab(rng), rng.choice(["fp32", half, half])
        return {"path": path, "kind": rng.choice(["fkl", "fkl", "rkl"]), "rows": min(_log(rng, 1, 32768), most // (BYTES[dt] * v)),
                "vocab": v, "pitch": _pitch(rng, v), "k": _log(rng, 10, 500), "T": rng.choice([1.0, 1.5, 2.0]), "dtype": dt,
                "masked": rng.choice([0.0, 0.1, 0.3])}
    if path == "dense":
        v = _vocab(rng)
        dt, te = rng.choice([("fp32", "fp32"), ("bf16", "bf16"), ("bf16", "bf16"), ("bf16", "fp32"), ("fp32", "bf16"), ("fp16", "fp16")])
        return {"path": path, "kind": rng.choice(["fkl", "rkl", "jsd"]), "rows": min(_log(rng, 1, 16384), most // (8 * v)), "vocab": v,
                "T": rng.choice([1.0, 1.5, 2.0]), "dtype": dt, "teacher": te, "masked": rng.choice([0.0, 0.1, 0.25])}
    if path == "producer":
        v, dt = _vocab(rng), rng.choice(["fp32", half, half])
        v = min(v, 131072) if dt == "fp32" else v
        return {"path": path, "rows": min(_log(rng, 8, 32768), most // (BYTES[dt] * v)), "vocab": v, "pitch": _pitch(rng, v),
                "k": _log(rng, 20, 400), "dtype": dt, "masked": rng.choice([0.0, 0.1, 0.3])}
    if path == "multi":
        v = _vocab(rng)
        return {"path": path, "teachers": rng.randint(2, 4), "rows": min(_log(rng, 16, 16384), most // (2 * v)), "vocab": v,
                "teacher_vocab": _vocab(rng), "k": _log(rng, 20, 400), "dtype": half}
    v, t = rng.choice([32000, _log(rng, 8000, 36000) // 8 * 8]), max(32000, _vocab(rng))      # students: whole 16-byte chunks only
    return {"path": path, "rows": _log(rng, 16, 8192), "vocab": v, "teacher_vocab": rng.choice([t, -(-t // 64) * 64]),
            "alphabet": rng.choice([4, 8, 16, 256]), "T": rng.choice([1.0, 1.5, 2.0]), "dtype": half}


# ------------------------------------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _stored_rows(n, vocab, k, g):
    """Top-K rows as the dataset holds them: distinct ids, crowded towards the low ids as a tokenizer's frequent tokens are, in
    no order of id; descending fp16 log-probs of a peaked distribution of which the K entries hold nearly everything."""
    edge = torch.linspace(0, 1, k + 1, device=DEV, dtype=torch.float64).square().mul(vocab - k).long() + torch.arange(k + 1, device=DEV)
    low, width = edge[:-1], edge[1:] - edge[:-1]
    ids = low + (torch.rand((n, k), generator=g, device=DEV) * width).long().clamp_(max=width - 1)
    ids = torch.gather(ids, 1, torch.rand((n, k), generator=g, device=DEV).argsort(1))
    score = torch.randn((n, k), generator=g, device=DEV) * 2.5
    logp = torch.log_softmax(score.sort(1, descending=True).values, 1) - 0.02
    return logp.half(), ids.to(torch.int32)


def _student_logits(n, pitch, dtype, g, vocab, t_val=None, t_idx=None, where=None, std=2.0):
    """[n, pitch] logits: noise, and in the rows `where` (all, if None) at the stored row's ids its log-probs, a row level and noise."""
    x = torch.empty((n, pitch), dtype=dtype, device=DEV)
    for a in range(0, n, CHUNK):
        b = min(n, a + CHUNK)
        x[a:b] = torch.randn((b - a, pitch), generator=g, device=DEV, dtype=dtype) * std
    if t_val is not None:
        where = torch.arange(n, device=DEV) if where is None else where
        level = math.log(vocab) + std * std / 2 + 2.0
        v = t_val.float() + level + torch.randn(t_val.shape, generator=g, device=DEV)
        x.view(-1).scatter_(0, (where.unsqueeze(1) * pitch + t_idx).flatten(), v.to(dtype).flatten())
    return x


def _row_map(rows, masked, g):
    """The teacher row of each logits row (None: its own number), the rows that have one, and how many; the masked rows lie in
    stretches as padding does."""
    if not masked:
        return None, None, rows
    valid = torch.rand((-(-rows // 16),), generator=g, device=DEV).repeat_interleave(16)[:rows] >= masked
    valid[0] = True
    where = torch.nonzero(valid).flatten()
    return synthetic.row_map_from_valid(valid), where, where.numel()


class _Logged:
    """The logger a training program hands to `Losses`."""

    def __init__(self):
        self.values = {}

    def log(self, values, step):
        self.values.update(values)


def prepare(case, seed):
    return {"case": case, **globals()["_prepare_" + case["path"]](case, _generator(seed))}


def _prepare_loop(c, g):
    convos = []
    for _ in range(c["convos"]):
        t_val, t_idx = _stored_rows(c["tokens"], c["vocab"], c["k"], g)
        x = _student_logits(c["tokens"], c["vocab"], torch.float32, g, c["vocab"], t_val, t_idx)
        avoid = torch.tensor([c["tokens"] // 2], dtype=torch.long, device=DEV)
        convos.append((x.requires_grad_(True), t_val.float(), t_idx.long(), t_idx[:-1, 0].long(), avoid))
    return {"convos": convos}


def _ranges(c):
    """Conversations of two turns, every second one shorter than the padded length: (content ranges, length) each."""
    lengths = [c["tokens"] - (b % 2) * (c["tokens"] // 5) for b in range(c["convos"])]
    return [([(n // 16, n // 3), (n // 2, n)], n) for n in lengths]


def _prepare_batch(c, g):
    ranges, lengths = zip(*_ranges(c))
    index = D.BatchIndex(ranges, lengths, c["tokens"], c["tokens"], DEV)
    t_val, t_idx = _stored_rows(index.total, c["vocab"], c["k"], g)
    where = torch.nonzero(index.row_map >= 0).flatten()
    x = _student_logits(c["convos"] * c["tokens"], c["pitch"], DTYPES[c["dtype"]], g, c["vocab"], t_val, t_idx, where)
    tokens = torch.randint(0, c["vocab"], (c["convos"], c["tokens"]), generator=g, device=DEV)
    teachers = [(t_val[a:a + n], t_idx[a:a + n]) for a, n in zip(index.offsets, index.counts)]
    for b, pos in enumerate(index.label_pos):           # most labels are among the stored ids, as a teacher's own text is
        keep = torch.rand((pos.numel(),), generator=g, device=DEV) < 0.9
        tokens[b][pos[keep]] = teachers[b][1][:pos.numel(), 0].long()[keep]
    return {"x": x.view(c["convos"], c["tokens"], c["pitch"]).requires_grad_(c["train"]), "index": index, "tokens": tokens,
            "teachers": teachers}


def _prepare_topk(c, g):
    row_map, where, n = _row_map(c["rows"], c["masked"], g)
    t_val, t_idx = _stored_rows(n, c["vocab"], c["k"], g)
    x = _student_logits(c["rows"], c["pitch"], DTYPES[c["dtype"]], g, c["vocab"], t_val, t_idx, where)
    return {"x": x[:, :c["vocab"]], "t_val": t_val, "t_idx": t_idx, "row_map": row_map, "n": n}


def _prepare_dense(c, g):
    row_map, where, n = _row_map(c["rows"], c["masked"], g)
    s, t = DTYPES[c["dtype"]], DTYPES[c["teacher"]]
    x = torch.empty((c["rows"], c["vocab"]), dtype=s, device=DEV)
    y = torch.empty((c["rows"], c["vocab"]), dtype=t, device=DEV)
    for a in range(0, c["rows"], CHUNK):
        b = min(c["rows"], a + CHUNK)
        z = torch.randn((b - a, c["vocab"]), generator=g, device=DEV) * 2.0
        x[a:b] = z
        y[a:b] = 0.8 * z + torch.randn(z.shape, generator=g, device=DEV) * 1.5
    return {"x": x, "t": y if where is None else y[where], "row_map": row_map, "n": n}


def _prepare_producer(c, g):
    _, where, n = _row_map(c["rows"], c["masked"], g)
    t_val, t_idx = _stored_rows(c["rows"], c["vocab"], c["k"], g)
    x = _student_logits(c["rows"], c["pitch"], DTYPES[c["dtype"]], g, c["vocab"], t_val, t_idx)
    return {"x": x[:, :c["vocab"]], "rows": None if where is None else where.to(torch.int32), "n": n}


def _prepare_multi(c, g):
    vals, idxs = zip(*(_stored_rows(c["rows"], c["teacher_vocab"], c["k"], g) for _ in range(c["teachers"])))
    x = _student_logits(c["rows"], c["vocab"], DTYPES[c["dtype"]], g, c["vocab"], std=3.0)
    id_map = torch.randint(0, c["vocab"], (c["teacher_vocab"],), generator=g, device=DEV, dtype=torch.int32)
    id_map[torch.rand((c["teacher_vocab"],), generator=g, device=DEV) < 0.05] = -1
    return {"x": x, "vals": list(vals), "idxs": list(idxs), "weights": (0.4, 0.3, 0.2, 0.1)[:c["teachers"]], "id_map": id_map}


def _prepare_marginal(c, g):
    student = synthetic.random_byte_vocab(c["vocab"], 501, all_single_bytes=True, alphabet=c["alphabet"])
    teacher = synthetic.random_byte_vocab(c["teacher_vocab"], 502, alphabet=c["alphabet"])
    plan = vocab_utils.MarginalPlan(vocab_utils.longest_prefix_map(student, teacher), c["vocab"], DEV)
    x = torch.randn((c["rows"], c["vocab"]), generator=g, device=DEV, dtype=DTYPES[c["dtype"]]) * 2.0
    p = torch.empty((c["rows"], c["teacher_vocab"]), device=DEV)
    for a in range(0, c["rows"], CHUNK):
        b = min(c["rows"], a + CHUNK)
        p[a:b] = torch.softmax(torch.randn((b - a, c["teacher_vocab"]), generator=g, device=DEV) * 2.0, dim=-1)
    return {"x": x, "p": p, "plan": plan}


# ------------------------------------------------------------------------------------------------ one pass

def run(state):
    return globals()["_run_" + state["case"]["path"]](state)


def _run_loop(s):
    logger = _Logged()
    losses = D.Losses(logger)
    for x, t_val, t_idx, labels, avoid in s["convos"]:
        x.grad = None
        losses.add_losses(D.calculate_divergence(x, t_val, t_idx, labels, 2.0, avoid))
    losses.backward(1)
    losses.log(1)
    return {"logged": logger.values, "grads": [convo[0].grad for convo in s["convos"]]}


def _run_batch(s):
    c, logger = s["case"], _Logged()
    x, index, crop = s["x"], s["index"], c["vocab"] if c["vocab"] < c["pitch"] else None
    losses = D.Losses(logger, validation=not c["train"])
    if c["train"]:
        x.grad = None
        losses.add_batch(D.distill_loss_batch_indexed(x, index, s["tokens"], s["teachers"], 2.0, temperature=c["T"], crop_to_size=crop))
        losses.backward(1)
    else:
        with torch.no_grad():
            losses.add_batch(D.distill_loss_batch_indexed(x, index, s["tokens"], s["teachers"], 2.0, temperature=c["T"],
                                                          crop_to_size=crop, teacher_temperature=1.0))
    losses.log(1)
    return {"logged": logger.values, "grad": x.grad}


def _run_topk(s):
    c = s["case"]
    row_loss, grad = D.div_topk(c["kind"], s["x"], s["t_val"], s["t_idx"], row_map=s["row_map"], T=c["T"], grad_scale=1.0 / s["n"])
    return D.reduce_sum(row_loss, 1.0 / s["n"]), row_loss, grad


def _run_dense(s):
    c = s["case"]
    row_loss, grad = D.div_dense(c["kind"], s["x"], s["t"], row_map=s["row_map"], T=c["T"], grad_scale=1.0 / s["n"])
    return D.reduce_sum(row_loss, 1.0 / s["n"]), row_loss, grad


def _run_producer(s):
    return D.teacher_topk(s["x"], s["case"]["k"], rows=s["rows"])


def _run_multi(s):
    n = s["case"]["rows"]
    row_loss, grad = D.fkl_multi_teacher(s["x"], s["vals"], s["idxs"], s["weights"], s["id_map"], grad_scale=1.0 / n)
    return D.reduce_sum(row_loss, 1.0 / n), row_loss, grad


def _run_marginal(s):
    n = s["case"]["rows"]
    row_loss, grad = vocab_utils.rkl_marginalised(s["x"], s["p"], s["plan"], T=s["case"]["T"], grad_scale=1.0 / n)
    return D.reduce_sum(row_loss, 1.0 / n), row_loss, grad


# ------------------------------------------------------------------------------------------------ what a pass cannot do without

def work(case):
    """Every input once, every output once; operations: an exponential and about five more on each logit that is read."""
    c, path = case, case["path"]
    if path == "loop":
        n = c["convos"] * c["tokens"]
        return {"bytes": n * (c["vocab"] * 8 + c["k"] * 12), "flops": 8 * n * c["vocab"]}
    if path == "batch":
        n, eb = sum(b - a for ranges, _ in _ranges(c) for a, b in ranges), BYTES[c["dtype"]]
        out = c["convos"] * c["tokens"] * c["pitch"] * eb if c["train"] else 0
        return {"bytes": n * (c["vocab"] * eb + c["k"] * 6) + out, "flops": (8 if c["train"] else 5) * n * c["vocab"]}
    if path == "multi":
        n, eb = c["rows"], BYTES[c["dtype"]]
        return {"bytes": n * (2 * c["vocab"] * eb + c["teachers"] * c["k"] * 6), "flops": 6 * n * c["vocab"]}
    if path == "marginal":
        n, eb = c["rows"], BYTES[c["dtype"]]
        return {"bytes": n * (c["teacher_vocab"] * 4 + 2 * c["vocab"] * eb), "flops": n * (c["teacher_vocab"] + 10 * c["vocab"])}
    live, eb = int(c["rows"] * (1 - c["masked"])), BYTES[c["dtype"]]
    if path == "producer":
        return {"bytes": live * (c["vocab"] * eb + c["k"] * 6), "flops": 5 * live * c["vocab"]}
    if path == "dense":
        return {"bytes": live * c["vocab"] * (eb + BYTES[c["teacher"]]) + c["rows"] * c["vocab"] * eb, "flops": 14 * live * c["vocab"]}
    if c["kind"] == "rkl":                                # the logits at the teacher's ids and the gradient
        return {"bytes": live * c["k"] * (6 + eb) + c["rows"] * c["vocab"] * eb, "flops": 20 * live * c["k"]}
    return {"bytes": live * (c["vocab"] * eb + c["k"] * 6) + c["rows"] * c["vocab"] * eb, "flops": 6 * live * c["vocab"]}


def tolerance(case):
    """About four times what the outputs differ by from the same formulas in float64 on reduced rows: a gradient's rounding to
    its 16-bit type (measured: 2e-3 bf16, up to 1.1e-3 fp16, where the mean's scale puts small entries among the subnormal
    numbers; largest entry 4e-3), fp32 sums elsewhere (the composite's gradients 7e-6, largest entry 3e-4 where its terms cancel;
    the other fp32 gradients 5e-7 and 2e-5, losses 8e-6), the fp16 store of log-probs (2.3e-4, largest 4.8e-4).  Ids of a
    producer's rows are the same ones: equal values are ordered by id."""
    if case["path"] == "producer":
        return {"rel": 1e-3, "max": 2e-3, "differ": 0.0}
    if case["path"] == "loop":
        return {"rel": 2.5e-5, "max": 1.2e-3}
    if case["dtype"] == "fp32" or case.get("train") is False:
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 6e-3 if case["dtype"] == "bf16" else 4e-3, "max": 1.6e-2}
