"""Timed cases of the token-sampling path: what a program that samples with
this library calls, over the sizes, data types and options it meets.

A pass is one call of the sampler (``Sampler.sample``, or ``Sampler.sample_raw``
with arguments prepared once, as a C caller does), or one replay of a captured
graph of decode steps on the device history ring. Its outputs are the tokens,
their probabilities, the flags and, where there is one, the ring. The logits
follow the distributions of the benchmark configurations
(gemmaedge_amd/workloads.py): ``peaked`` is a confident model's row (normal,
sigma 3, with a few high peaks), ``zipf`` a heavy-tailed one, ``flat`` a row
where nearly every token counts (normal, sigma 0.1).
"""
import math

import numpy as np
import torch

from gemmaedge_amd import sampler as S

# Fields that a case need not name.
DEFAULTS = dict(call="sample", rows=1, vocab=262144, dtype="f32", values="peaked", pad=0, temperature=1.0, top_k=64,
                top_p=0.95, min_p=0.0, softcap=30.0, penalty=1.0, history=0, steps=1, mixed=False)


def listed():
    return [
        # The smallest call: one decode step of one session with the default parameters, and
        # the repetition penalty over its last 128 tokens.
        dict(name="decode_1", call="raw", penalty=1.1, history=128),
        # Deterministic decoding of a few sessions.
        dict(name="greedy_8_bf16", call="raw", rows=8, dtype="bf16", temperature=0.0, penalty=1.1, history=256),
        # A small model with an odd vocabulary: its rows are not aligned to 16 bytes.
        dict(name="small_vocab_4_bf16", call="raw", rows=4, vocab=32003, dtype="bf16", top_k=50, temperature=0.8),
        # A decode loop as one graph: the history grows on the device, stop tokens are checked there.
        dict(name="decode_graph_4x32", call="graph", rows=4, steps=32, penalty=1.1, history=512),
        # The ordinary serving batch.
        dict(name="batch_64_top40", call="raw", rows=64, temperature=0.7, top_k=40, top_p=0.9, penalty=1.15, history=2048),
        # Requests of many users in one batch, each with its own parameters: greedy, top-k, top-p alone, min-p.
        dict(name="mixed_48_bf16", rows=48, dtype="bf16", penalty=1.05, history=512, mixed=True),
        # A large batch with an odd vocabulary, min-p and top-k.
        dict(name="odd_vocab_96_top200", rows=96, vocab=100003, top_k=200, top_p=1.0, min_p=0.02),
        # The largest top-k that selection serves, heavy-tailed rows.
        dict(name="batch_256_top1024", rows=256, values="zipf", top_k=1024, top_p=0.99, penalty=1.05, history=512),
        # Top-p alone, one session in float32.
        dict(name="nucleus_1", top_k=0, penalty=1.1, history=128),
        # Top-p alone, a serving batch in float32.
        dict(name="nucleus_64", rows=64, top_k=0, temperature=0.8, top_p=0.9),
        # Top-p alone over near-uniform rows (high temperature), where most of the vocabulary
        # stays in: the largest batches, in both types.
        dict(name="nucleus_512_bf16_flat", rows=512, dtype="bf16", values="flat", top_k=0, top_p=0.9, temperature=1.3),
        dict(name="nucleus_512_flat", rows=512, values="flat", top_k=0, top_p=0.9, temperature=1.3),
    ]


def _spread(rng, lo, hi):
    """A whole number of lo..hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("top_k", "top_k", "large_k", "nucleus", "nucleus", "greedy", "mixed", "graph"))
    c = dict(kind=kind, dtype=rng.choice(("f32", "bf16")), values=rng.choice(("peaked", "peaked", "zipf", "flat")))
    most = {"graph": 16, "mixed": 128, "nucleus": 256 if c["dtype"] == "f32" else 512}  # at most the largest listed case's time
    c["rows"] = _spread(rng, 1, most.get(kind, 512))
    # Model vocabularies are round or odd numbers alike.
    c["vocab"] = 262144 if rng.random() < 0.3 else _spread(rng, 16000, 262144)
    if rng.random() < 0.4:
        c["vocab"] -= c["vocab"] % 128
    if rng.random() < 0.25:
        c["pad"] = rng.randint(1, 640)  # rows of a wider buffer (a padded head)
    c["softcap"] = rng.choice((30.0, 30.0, 0.0))
    c["temperature"] = 0.0 if kind == "greedy" else round(rng.uniform(0.5, 1.4), 3)
    c["top_k"] = {"top_k": _spread(rng, 2, 64), "large_k": _spread(rng, 65, 1024), "nucleus": 0, "greedy": 64,
                  "mixed": 64, "graph": _spread(rng, 2, 64)}[kind]
    c["top_p"] = round(rng.choice((1.0, rng.uniform(0.8, 0.99), rng.uniform(0.8, 0.99))), 3)
    c["min_p"] = rng.choice((0.0, 0.0, 0.05))
    if rng.random() < 0.6 or kind == "graph":
        c["penalty"] = round(rng.uniform(1.02, 1.3), 3)
        c["history"] = _spread(rng, 16, 4096)
    if kind == "graph":
        c.update(call="graph", steps=rng.randint(8, 32))
    else:
        c["call"] = rng.choice(("raw", "sample"))
    c["mixed"] = kind == "mixed"
    return c


def _full(case):
    return {**DEFAULTS, **case}


def _configs(c):
    """The row's SamplingConfig: one for every row, or one each (mixed batches)."""
    base = dict(temperature=c["temperature"], top_k=c["top_k"], top_p=c["top_p"], min_p=c["min_p"], softcap=c["softcap"],
                repetition_penalty=c["penalty"])
    if not c["mixed"]:
        return [S.SamplingConfig(**base)]
    styles = (dict(), dict(temperature=0.0), dict(temperature=0.7, top_k=40, top_p=0.9), dict(top_k=20, top_p=1.0, min_p=0.05),
              dict(temperature=0.8, top_k=0, top_p=0.9), dict(temperature=1.2, top_k=500))
    return [S.SamplingConfig(**{**base, **styles[r % len(styles)]}) for r in range(c["rows"])]


def _logits(c, gen):
    """[steps * rows, vocab] logits in a buffer of vocab + pad columns."""
    rows, v = c["rows"] * c["steps"], c["vocab"]
    buf = torch.empty(rows, v + c["pad"], device="cuda")
    x = buf[:, :v]
    if c["values"] == "zipf":  # log of Zipf(1.1) over a random order of the tokens, with noise
        for r in range(rows):
            order = torch.randperm(v, generator=gen, device="cuda")
            x[r] = -1.1 * torch.log(order.float() + 1.0) + 0.5 * torch.randn(v, generator=gen, device="cuda")
    else:
        buf.normal_(0.0, 3.0 if c["values"] == "peaked" else 0.1, generator=gen)
        if c["values"] == "peaked":
            at = torch.randint(v, (rows, 20), generator=gen, device="cuda")
            up = 6.0 + 4.0 * torch.rand(rows, 20, generator=gen, device="cuda")
            x.scatter_add_(1, at, up)
    return (buf.bfloat16() if c["dtype"] == "bf16" else buf)[:, :v]


def _inputs(case, seed):
    c = _full(case)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    logits = _logits(c, gen)
    uniforms = torch.rand(c["steps"], c["rows"], generator=gen, device="cuda")
    history = torch.randint(c["vocab"], (c["rows"], c["history"]), generator=gen, device="cuda", dtype=torch.int32)
    return c, logits, uniforms, history


def prepare(case, seed):
    c, logits, uniforms, history = _inputs(case, seed)
    rows, vocab, steps = c["rows"], c["vocab"], c["steps"]
    s = dict(call=c["call"], logits=logits, uniforms=uniforms)
    s["configs"] = configs = _configs(c)
    s["row_params"] = None
    if c["mixed"]:  # the parameters of the batch's requests, on the device until a request ends
        packed = (S.SampleParams * rows)(*[x.params() for x in configs])
        s["row_params"] = torch.frombuffer(bytearray(packed), dtype=torch.uint8).cuda()
    s["tokens"] = torch.empty(steps, rows, dtype=torch.int32, device="cuda")
    s["probs"] = torch.empty(steps, rows, dtype=torch.float32, device="cuda")
    s["flags"] = torch.empty(steps, rows, dtype=torch.int32, device="cuda")
    s["history"] = s["offsets"] = None
    s["sampler"] = sampler = S.Sampler(rows, vocab, c["history"] + steps)
    if c["call"] == "graph":
        _capture(s, c, history)
        return s
    if c["history"]:
        s["history"] = history.reshape(-1)
        s["offsets"] = torch.arange(rows + 1, device="cuda", dtype=torch.int32) * c["history"]
    if c["call"] == "raw":
        a = S.SampleArgs()
        a.logits = logits.data_ptr()
        a.dtype = S.GE_DTYPE_BF16 if c["dtype"] == "bf16" else S.GE_DTYPE_F32
        a.rows, a.vocab, a.row_stride = rows, vocab, logits.stride(0)
        a.params = configs[0].params()
        a.row_params = None if s["row_params"] is None else s["row_params"].data_ptr()
        if c["history"]:
            a.history, a.history_offsets = s["history"].data_ptr(), s["offsets"].data_ptr()
        a.uniforms = uniforms.data_ptr()
        a.tokens_out, a.probs_out, a.flags_out = (s[k].data_ptr() for k in ("tokens", "probs", "flags"))
        s["args"] = a
    return s


def _capture(s, c, history):
    """A graph of `steps` decode steps of `rows` sessions, each from its prompt's ring."""
    rows, steps = c["rows"], c["steps"]
    capacity = c["history"] + steps
    s["ring"] = torch.zeros(rows, capacity, dtype=torch.int32, device="cuda")
    s["ring"][:, :c["history"]] = history
    s["prompt_len"] = torch.full((rows,), c["history"], dtype=torch.int32, device="cuda")
    s["ring_len"] = s["prompt_len"].clone()
    s["stop"] = torch.tensor([1, 106], dtype=torch.int32, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(s["graph"], stream=side):
        torch.add(s["prompt_len"], 0, out=s["ring_len"])  # the sessions begin after their prompts
        for t in range(steps):
            s["sampler"].sample(s["logits"][t * rows:(t + 1) * rows], s["configs"][0], uniforms=s["uniforms"][t],
                                ring=s["ring"], ring_len=s["ring_len"], tokens=s["tokens"][t], probs=s["probs"][t],
                                flags=s["flags"][t], stop_tokens=s["stop"])
    torch.cuda.current_stream().wait_stream(side)


def run(s):
    if s["call"] == "graph":
        s["graph"].replay()
        return dict(tokens=s["tokens"], probs=s["probs"], flags=s["flags"], ring=s["ring"], ring_len=s["ring_len"])
    if s["call"] == "raw":
        rc = s["sampler"].sample_raw(s["args"], torch.cuda.current_stream())
        if rc != S.GE_OK:
            raise S.SamplerError(rc, S.last_error())
    else:
        s["sampler"].sample(s["logits"], s["configs"] if s["row_params"] is not None else s["configs"][0],
                            uniforms=s["uniforms"], history=s["history"], history_offsets=s["offsets"], tokens=s["tokens"][0],
                            probs=s["probs"][0], flags=s["flags"][0], row_params=s["row_params"])
    return dict(tokens=s["tokens"], probs=s["probs"], flags=s["flags"])


def work(case):
    """Each logit and each history id read once, the uniforms in, tokens, probabilities and
    flags out; a softcap, a scaling and an exponential count as one operation each."""
    c = _full(case)
    n = c["rows"] * c["steps"]
    size = 2 if c["dtype"] == "bf16" else 4
    ids = c["history"] * n + (c["rows"] * c["steps"] * (c["steps"] - 1) // 2 if c["call"] == "graph" else 0)
    return {"bytes": n * (c["vocab"] * size + 16) + 4 * ids, "flops": 3.0 * n * c["vocab"]}


def tolerance(case):
    """The sampler promises the CPU sampler's tokens and probabilities bit for bit, whatever
    the order in which a kernel takes the row."""
    return "exact"


def _prob64(x, u, ids, p):
    """(token, probability) of one row in float64, from the definition."""
    f32 = lambda v: float(np.float32(v))  # noqa: E731  the parameters are floats
    v = x.double()
    if p.softcap > 0:
        v = f32(p.softcap) * torch.tanh(v / f32(p.softcap))
    if ids is not None and len(ids):
        t = torch.unique(ids.long())
        w = v[t]
        v[t] = torch.where(w > 0, w / f32(p.repetition_penalty), w * f32(p.repetition_penalty))
    if p.temperature <= 0:
        return int(v.argmax()), 1.0
    k = min(p.top_k, v.numel()) if p.top_k else v.numel()
    v, at = torch.topk(v, k)
    q = torch.exp((v - v[0]) / f32(p.temperature))
    q /= q.sum()
    n = int((q >= q[0] * f32(p.min_p)).sum())
    cum = torch.cumsum(q[:n], 0)
    hit = int(torch.searchsorted(cum, f32(p.top_p)))  # the first sum at or above top_p; at least two tokens stay
    keep = max(1, min(n, max(hit + 1, 2)))
    pos = min(int(torch.searchsorted(cum[:keep], float(u) * float(cum[keep - 1]))), keep - 1)
    return int(at[pos]), float(q[pos])


def exact(case, seed):
    """The probabilities; tokens and flags have no value in 64 bits (near-equal logits are
    ordered by their values in float32, and the draw's sums are float32 by definition)."""
    c, logits, uniforms, history = _inputs(case, seed)
    configs = _configs(c)
    out = torch.empty(c["steps"], c["rows"], dtype=torch.float64)
    for r in range(c["rows"]):
        ids = history[r].clone()
        for t in range(c["steps"]):
            token, out[t, r] = _prob64(logits[t * c["rows"] + r], uniforms[t, r], ids, configs[r % len(configs)])
            if c["call"] == "graph":
                ids = torch.cat([ids, torch.tensor([token], dtype=ids.dtype, device=ids.device)])
    none = dict(tokens=None, probs=out, flags=None)
    return dict(none, ring=None, ring_len=None) if c["call"] == "graph" else none
