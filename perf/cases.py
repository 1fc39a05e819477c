"""Performance cases: the calls that a program serving Qwen3-0.6B or Qwen3-1.7B makes of this package.

Four kinds of call, each through the public operators of ``torch.ops.qwen_megakernel_C``:

* ``decode``   one token of one sequence (``decode_logits``), the batch-1 decode step;
* ``batch``    one token of each of several sequences at their own positions (``decode_batch``);
* ``prompt``   the tokens of one or more prompts, from position 0 or after a context
               (``forward_tokens``): a prefill, a new turn of a conversation, several users' prompts;
* ``sample``   one draw per logits row (``sample``): temperature, top-k, top-p.

Model calls run one to four decoder layers and the LM head, which every call of these entry points
ends with, so that a change of rounding does not travel through 28 layers; one case is the whole
28-layer model.  Weights are the repository's synthetic ones, N(0, 0.02) in bf16, with norm weights
around 1; cached keys and values are N(0, 1), as in its long-context tests.  Model calls return the
logits, the K/V caches and, for ``decode``, the final hidden state; their greedy tokens are the
logits' argmax and are left out, because a tie between two bf16 logits may fall either way.
"""

import math

import torch

V, NQ, NKV, D = 151936, 16, 8, 128
HIDDEN = {"0.6b": 1024, "1.7b": 2048}
EPS, THETA = 1e-6, 1e6
SCALE = 1.0 / math.sqrt(D)


def listed():
    return [
        # the smallest call: temperature / top-k / top-p draws for a batch of four, after a batched step
        {"name": "sample-4", "kind": "sample", "rows": 4, "temperature": 0.8, "top_k": 50, "top_p": 0.9},
        # interactive decoding of one sequence in the middle of a 2048-position cache
        {"name": "decode-1k", "kind": "decode", "model": "0.6b", "layers": 4, "context": 1023},
        # the same over a long document
        {"name": "decode-8k", "kind": "decode", "model": "0.6b", "layers": 4, "context": 8191},
        # four sequences after 512-token prompts, the repository's batch-4 benchmark
        {"name": "batch-4", "kind": "batch", "model": "1.7b", "layers": 4, "batch": 4, "low": 513, "high": 768},
        # a small server batch, sequences of very different lengths
        {"name": "batch-8-ragged", "kind": "batch", "model": "0.6b", "layers": 4, "batch": 8, "low": 5, "high": 1500},
        # three long conversations decoded together
        {"name": "batch-3-6k", "kind": "batch", "model": "0.6b", "layers": 4, "batch": 3, "low": 5000, "high": 6100},
        # a larger server batch
        {"name": "batch-48", "kind": "batch", "model": "0.6b", "layers": 2, "batch": 48, "low": 100, "high": 1000},
        # a one-line question, the whole model
        {"name": "prompt-23", "kind": "prompt", "model": "0.6b", "layers": 28, "prompts": 1, "low": 23, "high": 23, "start": 0},
        # the repository's benchmark prompt
        {"name": "prompt-128", "kind": "prompt", "model": "0.6b", "layers": 4, "prompts": 1, "low": 128, "high": 128, "start": 0},
        # a prompt that fills the default cache
        {"name": "prompt-2048", "kind": "prompt", "model": "0.6b", "layers": 4, "prompts": 1, "low": 2048, "high": 2048, "start": 0},
        # a new turn of 100 tokens after 6000 positions of conversation
        {"name": "turn-100-after-6k", "kind": "prompt", "model": "0.6b", "layers": 4, "prompts": 1, "low": 100, "high": 100, "start": 6000},
        # four users' prompts of uneven length in one forward, the larger model
        {"name": "prompts-4-ragged", "kind": "prompt", "model": "1.7b", "layers": 4, "prompts": 4, "low": 411, "high": 613, "start": 0},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["sample"] + ["decode"] * 3 + ["batch"] * 4 + ["prompt"] * 5)
    model = rng.choice(["0.6b", "0.6b", "1.7b"])
    layers = rng.randint(2, 4)
    if kind == "sample":
        filters = rng.choice([(0, 1.0), (rng.randint(2, 200), 1.0), (0, rng.uniform(0.5, 0.99)),
                              (rng.randint(2, 200), rng.uniform(0.5, 0.99))])
        return {"kind": kind, "rows": _log(rng, 1, 48), "temperature": rng.uniform(0.5, 1.5), "top_k": filters[0],
                "top_p": filters[1]}
    if kind == "decode":
        return {"kind": kind, "model": model, "layers": layers, "context": _log(rng, 1, 16000)}
    if kind == "batch":
        batch = _log(rng, 2, 48)
        high = _log(rng, 30, min(8000, 48 * 1000 // batch))
        return {"kind": kind, "model": model, "layers": 2 if batch > 16 else layers, "batch": batch,
                "low": rng.randint(1, high), "high": high}
    if rng.random() < 0.25:  # several prompts, from position 0
        prompts = rng.randint(2, 6)
        high = _log(rng, 8, 2048 // prompts)
        return {"kind": kind, "model": model, "layers": layers, "prompts": prompts, "low": rng.randint(1, high),
                "high": high, "start": 0}
    start = rng.choice([0, _log(rng, 10, 7000)])
    n = _log(rng, 1, 2048 if start == 0 else max(64, min(2048, 2_000_000 // start)))
    return {"kind": kind, "model": model, "layers": layers, "prompts": 1, "low": n, "high": n, "start": start}


def _spread(n, low, high):
    """n whole numbers from low to high, evenly spaced, in an order that is not sorted."""
    step = (high - low) / max(1, n - 1)
    vals = [low + int(round(step * i)) for i in range(n)]
    return vals[::2] + vals[1::2][::-1]


def _calls(case):
    """(sequences, per token (sequence, position), emitted rows, positions a cache must hold)."""
    if case["kind"] == "decode":
        return 1, [(0, case["context"])], [0], case["context"] + 1
    if case["kind"] == "batch":
        pos = _spread(case["batch"], case["low"], case["high"])
        return case["batch"], list(enumerate(pos)), list(range(case["batch"])), max(pos) + 1
    toks, emit = [], []
    for s, n in enumerate(_spread(case["prompts"], case["low"], case["high"])):
        toks += [(s, case["start"] + i) for i in range(n)]
        emit.append(len(toks) - 1)
    return case["prompts"], toks, emit, max(p for _, p in toks) + 1


def _rope(n):
    inv = 1.0 / (THETA ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    f = torch.outer(torch.arange(n, dtype=torch.float32), inv)
    e = torch.cat((f, f), -1)
    return e.cos().bfloat16().cuda(), e.sin().bfloat16().cuda()


def _inputs(case, seed):
    """Weights, caches and tokens of a model call, or the logits and counters of a draw, from the seed."""
    g = torch.Generator("cuda").manual_seed(seed)

    def normal(*shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=g, device="cuda") * std + mean).bfloat16()

    if case["kind"] == "sample":
        # logits as a model gives them: bf16 values in fp32, a few tokens well above the rest
        x = normal(case["rows"], V, std=2.0).float()
        top = torch.randint(0, V, (case["rows"], 64), generator=g, device="cuda")
        x.scatter_add_(1, top, torch.rand(case["rows"], 64, generator=g, device="cuda") * 8)
        counters = torch.randint(0, 1 << 40, (case["rows"],), generator=g, device="cuda")
        return {"logits": x.bfloat16().float(), "counters": counters, "seed": seed & 0x7FFFFFFF}
    h = HIDDEN[case["model"]]
    i = 3 * h
    nseq, toks, emit, need = _calls(case)
    size = -(-need // 256) * 256  # the cache: a multiple of 256 positions
    layers = []
    for _ in range(case["layers"]):
        layers += [normal(h, std=0.1, mean=1.0), normal(NQ * D, h, std=0.02), normal(NKV * D, h, std=0.02),
                   normal(NKV * D, h, std=0.02), normal(D, std=0.1, mean=1.0), normal(D, std=0.1, mean=1.0),
                   normal(h, NQ * D, std=0.02), normal(h, std=0.1, mean=1.0), normal(i, h, std=0.02),
                   normal(i, h, std=0.02), normal(h, i, std=0.02)]
    shape = (nseq, case["layers"], NKV, size, D)
    cos, sin = _rope(size)
    return {
        "embed": normal(V, h, std=0.02), "layers": layers, "final_norm": normal(h, std=0.1, mean=1.0),
        "cos": cos, "sin": sin, "k": normal(*shape), "v": normal(*shape),
        "tokens": torch.randint(0, V, (len(toks),), generator=g, device="cuda", dtype=torch.int32),
        "seqs": torch.tensor([s for s, _ in toks], dtype=torch.int32, device="cuda"),
        "positions": torch.tensor([p for _, p in toks], dtype=torch.int32, device="cuda"),
        "emit": torch.tensor(emit, dtype=torch.int32, device="cuda"), "context": need,
    }


def prepare(case, seed):
    import qwen_megakernel  # noqa: F401  (registers torch.ops.qwen_megakernel_C)

    ops = torch.ops.qwen_megakernel_C
    s = _inputs(case, seed)
    s["case"], s["ops"] = case, ops
    if case["kind"] == "sample":
        s["out"] = torch.empty(case["rows"], dtype=torch.int32, device="cuda")
        return s
    h = HIDDEN[case["model"]]
    rows = s["emit"].numel()
    s["out"] = torch.empty(rows, dtype=torch.int32, device="cuda")
    s["logits"] = torch.empty(rows, V, dtype=torch.float32, device="cuda")
    if case["kind"] == "decode":
        s["k"], s["v"] = s["k"][0], s["v"][0]
        ptrs = torch.tensor([t.data_ptr() for t in s["layers"]], dtype=torch.int64)
        s["packed"] = ptrs.view(torch.uint8).cuda()
        s["hidden"] = torch.empty(h, dtype=torch.bfloat16, device="cuda")
        s["normed"] = torch.empty(h, dtype=torch.float32, device="cuda")
        s["token"] = int(s["tokens"][0])
        return s
    if case["kind"] == "batch":
        need = ops.decode_batch_workspace_bytes(h, s["tokens"].numel(), s["context"])
    else:
        need = ops.forward_workspace_bytes(h, s["tokens"].numel(), rows, s["context"])
    s["ws"] = torch.empty(need, dtype=torch.uint8, device="cuda")
    return s


def run(s):
    case, ops = s["case"], s["ops"]
    if case["kind"] == "sample":
        ops.sample(s["logits"], case["temperature"], case["top_k"], case["top_p"], s["seed"], s["counters"], s["out"])
        return {"tokens": s["out"]}
    if case["kind"] == "decode":
        ops.decode_logits(s["out"], s["logits"][0], s["token"], s["embed"], s["packed"], s["final_norm"], s["embed"],
                          s["cos"], s["sin"], s["k"], s["v"], s["hidden"], s["normed"], case["layers"],
                          case["context"], s["k"].shape[-2], SCALE)
        return {"logits": s["logits"], "k": s["k"], "v": s["v"], "hidden": s["hidden"], "normed": s["normed"]}
    if case["kind"] == "batch":
        ops.decode_batch(s["tokens"], s["positions"], s["out"], s["logits"], s["embed"], s["layers"], s["final_norm"],
                         s["embed"], s["cos"], s["sin"], s["k"], s["v"], s["ws"], case["layers"], s["context"], SCALE)
    else:
        ops.forward_tokens(s["tokens"], s["seqs"], s["positions"], s["emit"], s["out"], s["logits"], s["embed"],
                           s["layers"], s["final_norm"], s["embed"], s["cos"], s["sin"], s["k"], s["v"], s["ws"],
                           case["layers"], s["context"], SCALE)
    return {"logits": s["logits"], "k": s["k"], "v": s["v"]}


def work(case):
    if case["kind"] == "sample":
        n = case["rows"] * V
        return {"bytes": 4 * n + 12 * case["rows"], "flops": 8 * n}  # a draw: scale, hash, two logarithms, compare
    h, n_layers = HIDDEN[case["model"]], case["layers"]
    nseq, toks, emit, _ = _calls(case)
    layer = (NQ + 2 * NKV) * D * h + NQ * D * h + 9 * h * h  # q, k, v; o; gate, up, down (MLP width 3 h)
    last = {}
    for s, p in toks:
        last[s] = max(last.get(s, 0), p + 1)
    attended = sum(p + 1 for _, p in toks)
    kv = 2 * NKV * D * 2  # K and V bytes of one position and layer
    rows, t = len(emit), len(toks)
    # K/V rows that no token of the call computes are read, the others written
    read = (sum(last.values()) - t) * kv
    return {
        "bytes": n_layers * (2 * layer + read + t * kv) + 2 * V * h + 2 * t * h + 4 * rows * V,
        "flops": 2 * t * n_layers * layer + 4 * attended * NQ * D * n_layers + 2 * rows * V * h,
    }


def tolerance(case):
    """Measured on one token's logits, two to four layers: the package's own three forms of the step (the
    decode kernel, the batched step, the forward) differ by 0.004 to 0.011 where a bf16 rounding flips
    between their orders of the same sums, so other correct orders are held to about three times that."""
    if case["kind"] == "sample":
        return "exact"
    return {"rel": 0.03}


def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def exact(case, seed):
    """The same call in float64 with no rounding in between (a draw gives whole numbers only)."""
    if case["kind"] == "sample":
        return None
    s = _inputs(case, seed)
    seqs, pos = s["seqs"].long(), s["positions"].long()
    cos, sin = s["cos"][pos].double()[:, None], s["sin"][pos].double()[:, None]

    def rot(x):
        return x * cos + torch.cat((-x[..., D // 2:], x[..., : D // 2]), -1) * sin

    k64, v64 = s["k"].double(), s["v"].double()
    x = s["embed"][s["tokens"].long()].double()
    t = x.shape[0]
    for n in range(case["layers"]):
        ln1, wq, wk, wv, qn, kn, wo, ln2, wg, wu, wd = s["layers"][11 * n: 11 * n + 11]
        y = _rms(x, ln1)
        q = rot(_rms((y @ wq.double().t()).view(t, NQ, D), qn))
        k64[seqs, n, :, pos] = rot(_rms((y @ wk.double().t()).view(t, NKV, D), kn))
        v64[seqs, n, :, pos] = (y @ wv.double().t()).view(t, NKV, D)
        att = torch.empty(t, NQ, D, dtype=torch.float64, device="cuda")
        for b in range(k64.shape[0]):
            mine = (seqs == b).nonzero()[:, 0]
            c = int(pos[mine].max()) + 1
            late = torch.arange(c, device="cuda")[None, :] > pos[mine][:, None]
            for head in range(NQ):
                sc = q[mine, head] @ k64[b, n, head // 2, :c].t() * SCALE
                att[mine, head] = torch.softmax(sc.masked_fill_(late, -math.inf), -1) @ v64[b, n, head // 2, :c]
        x = x + att.view(t, NQ * D) @ wo.double().t()
        y = _rms(x, ln2)
        x = x + (torch.nn.functional.silu(y @ wg.double().t()) * (y @ wu.double().t())) @ wd.double().t()
    last = x[s["emit"].long()]
    normed = _rms(last, s["final_norm"])
    logits = normed @ s["embed"].double().t()
    if case["kind"] == "decode":
        return {"logits": logits, "k": k64[0], "v": v64[0], "hidden": last[0], "normed": normed[0]}
    return {"logits": logits, "k": k64, "v": v64}
