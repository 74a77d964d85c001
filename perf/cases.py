"""The sampler's work as its callers issue it, for timing: single rows, a decode
frame, served batches, long pools, text vocabularies, large and disabled
top-k, and the heads with their sample, all through the C-ABI of
include/d3s_sampler.h (the ctypes binding in drama3-mlx_amd/d3s.py).

A case is a dict of plain values:
  kind    "sample" (d3s_sample), "frame" (a decode step's ten draws) or
          "head" (d3s_linear_sample_bf16)
  rows    rows of logits (frames side by side for "frame")
  vocab   V; pad: elements between a row's end and the next row's start
  dtype   "f32" or "bf16" logits
  k       uniform columns a row; 0: top-k disabled (k = V)
  u       "given" (drawn earlier), "fill" (d3s_uniform_fill, then the sample: a
          new draw each call) or "seeded" (d3s_sample_seeded, one launch)
  per_row per-row temperature and top_p arrays instead of scalars
  banned  index 0 (eos) banned on half of the rows
  probs   ask for every rank's probability and index as well as the ids
  logits  the rows' distribution (LOGITS below)
The row lengths 4096, 4097, 8192 and 151936, the temperatures, k = 30 and
the distributions are those of drama3-mlx_amd/d3s_workloads.py and bench.py; the
other lengths are generic.

Every output is compared bit for bit ("exact"): d3s_sampler.h fixes each
operation's rounding and order (an exact fixed-point row sum, the heads' gemv
order), so a correct implementation returns the same ids, candidates,
probabilities and logits whatever its launch shape.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("drama3-mlx_amd"))
import d3s  # noqa: E402

# sigma of the normal logits, raised entries a row, their least and greatest height
LOGITS = {
    "backbone": (2.5, 5, 8.0, 8.0),   # a confident head: five likely tokens
    "batch": (2.5, 8, 4.0, 10.0),     # rows of different confidence
    "codebook": (2.0, 12, 2.0, 8.0),  # codec codes: a short head over a flat tail
    "text": (3.0, 20, 6.0, 6.0),      # a language model's vocabulary
    "flat": (0.3, 0, 0.0, 0.0),       # near-flat rows: nearly every rank kept
}

EOS, SEM_START, CODE_VOCAB = 151645, 151669, 4096
CODEBOOKS = 9


def _sample(name, rows, vocab, dtype, k, u, logits, temperature, top_p, **kw):
    c = dict(name=name, kind="sample", rows=rows, vocab=vocab, pad=0, dtype=dtype, k=k, u=u, logits=logits,
             temperature=temperature, top_p=top_p, per_row=False, banned=False, probs=False)
    c.update(kw)
    return c


def listed():
    return [
        # one step of one stream: the backbone head's row, its draw in the same launch
        _sample("row", 1, 4097, "f32", 30, "seeded", "backbone", 0.7, 0.7),
        # one decode frame of one stream: the repetition-aware main token and the
        # nine codebooks one after the other (each head waits for the code before)
        dict(name="frame", kind="frame", rows=1, vocab=4097, codes=4096, k=30, temperature=0.7, top_p=0.7),
        # a serving step: 256 streams, two kinds of request (per-row parameters)
        _sample("batch", 256, 4097, "f32", 30, "given", "batch", 0.7, 0.7, per_row=True),
        # offline scoring: 512 such batches in one call, inputs far past every cache
        _sample("pool", 131072, 4097, "f32", 30, "given", "batch", 0.7, 0.7, per_row=True),
        # a text vocabulary, bf16 logits straight from the head
        _sample("text", 64, 151936, "bf16", 30, "given", "text", 1.0, 0.9),
        # the same vocabulary with the logits raised to fp32, as most serving code
        # does before sampling, a smaller batch and a common top-k
        _sample("text_f32", 16, 151936, "f32", 50, "given", "text", 0.7, 0.9),
        # a large top-k with every rank's probability kept (log-probs of a rollout)
        _sample("large_k", 32, 151936, "bf16", 1000, "fill", "text", 1.0, 0.95, probs=True),
        # top-p only: the whole row ranked, a new draw for every rank
        _sample("nucleus", 4096, 4097, "f32", 0, "fill", "flat", 1.0, 0.95, banned=True),
        # the same with the distribution returned, a smaller batch
        _sample("nucleus_probs", 1024, 4097, "f32", 0, "fill", "backbone", 1.0, 0.95, probs=True),
        # top-p only over a text vocabulary
        _sample("nucleus_text", 64, 151936, "bf16", 0, "fill", "text", 1.0, 0.9),
        # the backbone head of one stream: gemv and sample
        dict(name="head", kind="head", rows=1, hidden=2048, vocab=4097, k=30, temperature=0.7, top_p=0.7),
        # the same head for a served batch
        dict(name="head_batch", kind="head", rows=64, hidden=2048, vocab=4097, k=30, temperature=0.7, top_p=0.7),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.choice(["rows", "rows", "frame", "text", "text", "large_k", "nucleus", "nucleus", "nucleus_text", "head",
                       "head"])
    dtype = rng.choice(["f32", "bf16"])
    pad = rng.choice([0, 0, rng.randint(1, 64)])
    temperature, top_p = rng.choice([(0.7, 0.7), (1.0, 0.9), (1.0, 0.95), (0.6, 0.95)])
    kw = dict(pad=pad, per_row=rng.random() < 0.5, banned=rng.random() < 0.25)
    if what == "rows":  # rows one wave holds
        vocab = rng.choice([_log(rng, 257, 8192), rng.randint(4000, 4200)])
        rows = _log(rng, 1, 100000 * 4097 // max(4097, vocab))
        k = rng.randint(1, min(64, vocab))
        u = "seeded" if rows <= 1024 and vocab <= 6000 and rng.random() < 0.5 else "given"
        return _unnamed(_sample("", rows, vocab, dtype, k, u, rng.choice(["backbone", "batch", "codebook"]),
                                temperature, top_p, probs=rng.random() < 0.25, **kw))
    if what == "frame":
        return dict(kind="frame", rows=_log(rng, 1, 256), vocab=rng.choice([4097, rng.randint(2049, 6000)]),
                    codes=rng.choice([4096, 2048, 1024]), k=rng.randint(20, 64), temperature=temperature, top_p=top_p)
    if what == "text":  # wide rows, small k
        vocab = _log(rng, 8193, 270000)
        rows = _log(rng, 1, 64 * 151936 // max(vocab, 32768))
        return _unnamed(_sample("", rows, vocab, dtype, rng.randint(1, 64), "given", "text", temperature, top_p,
                                probs=rng.random() < 0.25, **kw))
    if what == "large_k":
        vocab = _log(rng, 8193, 270000)
        rows = _log(rng, 1, 32 * 151936 // max(vocab, 32768))
        return _unnamed(_sample("", rows, vocab, dtype, _log(rng, 65, 4096), "fill", "text", temperature, top_p,
                                probs=rng.random() < 0.5, **kw))
    if what == "nucleus":  # rows one workgroup holds, k above 64
        vocab = _log(rng, 512, 8192)
        rows = _log(rng, 1, 4096 * 4097 // max(vocab, 4097))
        k = rng.choice([0, 0, _log(rng, 65, vocab)])
        probs = rng.random() < 0.3
        return _unnamed(_sample("", rows, vocab, dtype, k, "fill", rng.choice(["flat", "backbone", "batch"]),
                                temperature, top_p, probs=probs, **kw))
    if what == "nucleus_text":
        vocab = _log(rng, 20000, 270000)
        rows = _log(rng, 1, 64 * 151936 // max(vocab, 32768) // 2)
        return _unnamed(_sample("", rows, vocab, dtype, 0, "fill", "text", temperature, top_p, **kw))
    hidden, vocab = 128 * rng.randint(4, 32), rng.choice([4096, 4097, _log(rng, 1000, 8192)])
    rows = _log(rng, 1, max(1, min(256, 64 * 2048 * 4097 // (hidden * vocab))))
    return dict(kind="head", rows=rows, hidden=hidden, vocab=vocab, k=rng.randint(20, 64),
                temperature=temperature, top_p=top_p)


def _unnamed(case):
    del case["name"]
    return case


def _k(case):
    return min(case["k"] or case["vocab"], case["vocab"])


def _rows_of_logits(case, g, rows, vocab, stride, dtype, kind):
    sigma, n, lo, hi = LOGITS[kind]
    x = torch.randn(rows, stride, device="cuda", generator=g).mul_(sigma)
    if n:
        at = torch.randint(0, vocab, (rows, n), device="cuda", generator=g)
        up = torch.rand(rows, n, device="cuda", generator=g).mul_(hi - lo).add_(lo)
        x.scatter_add_(1, at, up)
    return x if dtype == "f32" else x.to(torch.bfloat16)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = dict(case=case, seed=seed, kind=case["kind"], rows=case["rows"], vocab=case["vocab"])
    rows, vocab = case["rows"], case["vocab"]
    new = lambda shape, dtype: torch.empty(shape, dtype=dtype, device="cuda")  # noqa: E731
    if case["kind"] == "sample":
        k = _k(case)
        s["k"], s["stride"] = k, vocab + case["pad"]
        s["dtype"] = d3s.DTYPE_F32 if case["dtype"] == "f32" else d3s.DTYPE_BF16
        s["logits"] = _rows_of_logits(case, g, rows, vocab, s["stride"], case["dtype"], case["logits"])
        if case["u"] != "seeded":
            s["u"] = new((rows, k), torch.float32)
            if case["u"] == "given":
                s["u"].uniform_(generator=g)
        T, P = case["temperature"], case["top_p"]
        if case["per_row"]:  # the first half as given, the others another request's
            first = torch.arange(rows, device="cuda") < (rows + 1) // 2
            s["T"] = torch.where(first, T, 1.0).float()
            s["P"] = torch.where(first, P, 0.9).float()
            T, P = ("ptr", s["T"].data_ptr()), ("ptr", s["P"].data_ptr())
        s["temperature"], s["top_p"] = T, P
        if case["banned"]:
            s["banned"] = torch.where(torch.rand(rows, device="cuda", generator=g) < 0.5, 0, -1).to(torch.int32)
        s["out"] = dict(ids=new((rows,), torch.int32))
        if case["probs"]:
            s["out"].update(probs=new((rows, k), torch.float32), cand=new((rows, k), torch.int32))
    elif case["kind"] == "frame":
        s["logits"] = _rows_of_logits(case, g, rows, vocab, vocab, "bf16", "backbone")
        s["codes"] = [_rows_of_logits(case, g, rows, case["codes"], case["codes"], "bf16", "codebook")
                      for _ in range(CODEBOOKS)]
        s["u"] = torch.rand(2 + CODEBOOKS, rows, case["k"], device="cuda", generator=g)
        # the last 16 main tokens, some of them likely now
        likely = s["logits"].float().topk(16, dim=1).indices
        seen = torch.rand(rows, 16, device="cuda", generator=g) < 0.25
        other = torch.randint(1, vocab, (rows, 16), device="cuda", generator=g)
        s["history"] = (SEM_START + torch.where(seen, likely, other) - 1).to(torch.int32)
        s["params"] = d3s.ras_params(temperature=case["temperature"], top_p=case["top_p"], top_k=case["k"],
                                     retry_top_k=case["k"], eos_id=EOS, semantic_start=SEM_START,
                                     semantic_end=SEM_START + CODE_VOCAB - 1, code_vocab=CODE_VOCAB)
        s["out"] = dict(frame=new((2 + CODEBOOKS, rows), torch.int32))
    else:
        K, k = case["hidden"], case["k"]
        x = torch.randn(rows, K, device="cuda", generator=g)
        w = torch.randn(vocab, K, device="cuda", generator=g).mul_(2.5 / math.sqrt(K))
        s["x"], s["w"] = x.to(torch.bfloat16), w.to(torch.bfloat16)
        s["u"] = torch.rand(rows, k, device="cuda", generator=g)
        s["out"] = dict(logits=new((rows, vocab), torch.bfloat16), ids=new((rows,), torch.int32))
    return s


def _ptr(t):
    return None if t is None else t.data_ptr()


def _ok(rc):
    if rc != d3s.OK:
        raise RuntimeError(f"the sampler returned {rc}")


def run(s):
    case, out, L = s["case"], s["out"], d3s.lib()
    stream = torch.cuda.current_stream().cuda_stream or None
    rows, vocab = s["rows"], s["vocab"]
    if s["kind"] == "sample":
        probs, cand, banned = _ptr(out.get("probs")), _ptr(out.get("cand")), _ptr(s.get("banned"))
        if case["u"] == "seeded":
            _ok(d3s.sample_seeded_raw(s["logits"].data_ptr(), s["dtype"], rows, vocab, s["stride"], s["seed"], 1,
                                      s["k"], s["temperature"], s["top_p"], banned, out["ids"].data_ptr(), probs,
                                      cand, stream=stream))
            return out
        u = s["u"].data_ptr()
        if case["u"] == "fill":
            _ok(L.d3s_uniform_fill(u, rows * s["k"], s["seed"], 1, stream))
        _ok(d3s.sample_raw(s["logits"].data_ptr(), s["dtype"], rows, vocab, s["stride"], u, s["k"],
                           s["temperature"], s["top_p"], banned, out["ids"].data_ptr(), probs, cand, stream=stream))
    elif s["kind"] == "frame":
        k, n = case["k"], rows * 4
        u, frame = s["u"].data_ptr(), out["frame"].data_ptr()
        _ok(d3s.sample_ras_raw(s["logits"].data_ptr(), d3s.DTYPE_BF16, rows, vocab, vocab, u, u + n * k,
                               s["history"].data_ptr(), 16, s["params"], frame, frame + n, stream=stream))
        for j, logits in enumerate(s["codes"]):
            _ok(d3s.sample_raw(logits.data_ptr(), d3s.DTYPE_BF16, rows, case["codes"], case["codes"],
                               u + (2 + j) * n * k, k, case["temperature"], case["top_p"], None,
                               frame + (2 + j) * n, stream=stream))
    else:
        _ok(L.d3s_linear_sample_bf16(s["x"].data_ptr(), s["w"].data_ptr(), rows, case["hidden"], vocab,
                                     out["logits"].data_ptr(), s["u"].data_ptr(), case["k"], None, None,
                                     case["temperature"], case["top_p"], out["ids"].data_ptr(), None, None, None, 0,
                                     stream))
    return out


def work(case):
    rows, vocab, k = case["rows"], case["vocab"], _k(case)
    if case["kind"] == "sample":
        read = rows * vocab * (4 if case["dtype"] == "f32" else 2)
        # uniforms: read once; a fill writes them as well
        read += rows * k * 4 * {"given": 1, "fill": 2, "seeded": 0}[case["u"]]
        read += rows * 4 * (2 * case["per_row"] + case["banned"])
        return {"bytes": read + rows * 4 + (8 * rows * k if case["probs"] else 0), "flops": 4 * rows * vocab}
    if case["kind"] == "frame":
        n = rows * (vocab + CODEBOOKS * case["codes"])
        return {"bytes": 2 * n + (2 + CODEBOOKS) * rows * (4 * k + 4) + 64 * rows, "flops": 4 * n}
    K = case["hidden"]
    return {"bytes": 2 * (rows * K + vocab * K + rows * vocab) + 4 * rows * (k + 1), "flops": 2 * rows * K * vocab}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The probabilities and the heads' logits in 64 bits.  Ids and candidates
    are choices that the 32-bit definition fixes (ties, cuts at a boundary):
    they have no 64-bit value of their own."""
    if case["kind"] == "head":
        s = prepare(case, seed)
        return {"logits": s["x"].double() @ s["w"].double().t(), "ids": None}
    if case["kind"] != "sample" or not case["probs"]:
        return None
    s = prepare(case, seed)
    k, rows, vocab = s["k"], case["rows"], case["vocab"]
    T = s["T"] if "T" in s else torch.full((rows,), case["temperature"], device="cuda")
    P = s["P"] if "P" in s else torch.full((rows,), case["top_p"], device="cuda")
    out = torch.empty(rows, k, dtype=torch.float64, device="cuda")
    step = max(1, (64 << 20) // vocab)
    for r in range(0, rows, step):
        x = s["logits"][r:r + step, :vocab].double()
        if "banned" in s:
            x[:, 0].masked_fill_(s["banned"][r:r + step] == 0, -math.inf)
        x = x / T[r:r + step, None].double().clamp_min(1e-5)
        lse = x.logsumexp(1, keepdim=True)
        v = x.topk(k, dim=1).values
        c = (v - lse).exp().cumsum(1)
        drop = c > P[r:r + step, None].double()
        drop[:, 0] = False
        keep = drop.long().cumsum(1) == 0
        e = (v - v[:, :1]).exp() * keep
        out[r:r + step] = e / e.sum(1, keepdim=True)
    return {"ids": None, "probs": out, "cand": None}
