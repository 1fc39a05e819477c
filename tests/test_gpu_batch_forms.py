"""GPU parity of the batched step and the batched forward at the edges of their kernels' tiles: contexts
that end on and beside a 128-position attention chunk, and token counts beside the row tiles of the
projections and of the LM head.  Every sequence is checked against the exact oracle on its own cache, and
every cache row past a sequence's context holds NaN, which must reach no output.
"""

import pytest
import torch

from parity import LITERAL, Tally, check_kv_rows, check_rows, exact_oracle, oracle_steps, with_rope

pytestmark = pytest.mark.gpu


def _decode_steps(shape, exact06, weights_gpu, c0s, layers, max_seq, steps=2):
    from qwen_megakernel.model import BatchDecoder

    B = len(c0s)
    bd = BatchDecoder(weights=with_rope(weights_gpu, max_seq, "cuda"), batch_size=B, max_seq_len=max_seq,
                      num_layers=layers, verbose=False)
    g = torch.Generator("cuda").manual_seed(B)
    bd._k_cache.fill_(float("nan"))
    bd._v_cache.fill_(float("nan"))
    for b, c0 in enumerate(c0s):
        k = torch.randn(layers, 8, max(c0, 1), 128, generator=g, device="cuda").bfloat16()
        v = torch.randn(layers, 8, max(c0, 1), 128, generator=g, device="cuda").bfloat16()
        bd.load_kv(b, k, v, c0)
    feed, lgs = [[11 + 7 * b] for b in range(B)], [[] for _ in range(B)]
    for _ in range(steps):
        nxt, logits = bd.step_logits([f[-1] for f in feed])
        assert torch.isfinite(logits).all()
        for b in range(B):
            feed[b].append(nxt[b])
            lgs[b].append(logits[b].cpu())
    t = Tally(f"batched step, contexts {c0s}")
    for b in range(B):
        orc = exact_oracle(exact06, shape, max_seq, num_layers=layers)
        n = c0s[b] + steps
        kc, vc = (torch.zeros_like(x[b]) for x in (bd._k_cache, bd._v_cache))
        kc[:, :, :n], vc[:, :, :n] = bd._k_cache[b, :, :, :n], bd._v_cache[b, :, :, :n]
        ref = oracle_steps(orc, kc, vc, c0s[b], feed[b][:-1])
        check_rows(t, ref, feed[b][1:], torch.stack(lgs[b]), bar=LITERAL)
        check_kv_rows(f"sequence {b}", orc, kc, vc, c0s[b], steps)
    print(t)


@pytest.mark.parametrize("c0s", [(0, 1, 126, 127, 128), (255, 256, 300, 0, 129, 64),
                                 tuple(range(110, 146, 2)), (383, 8200), tuple(range(112, 144)),
                                 tuple(range(112, 144)) + (256,), tuple(range(0, 126, 3))[:34]],
                         ids=["5seq-first-chunk-edge", "6seq-second-chunk-edge", "18seq-two-row-tiles", "2seq-65-chunks",
                              "32seq-raw", "33seq-finished-q", "34seq-rows"])
def test_decode_batch_attention_chunk_edges(shape, exact06, weights_gpu, c0s):
    """attn_chunk_*: contexts ending at, before and after a chunk's edge, a token in a chunk of its own,
    more than 64 chunks (two rounds of pairs), from raw projections (up to 32 sequences, the most of gemm_rows)
    and finished q (33, the first of the general projections), and contexts of at most 128 positions above
    32 sequences (attention_rows)."""
    _decode_steps(shape, exact06, weights_gpu, c0s, layers=2, max_seq=(max(c0s) + 2 + 63) // 64 * 64)


@pytest.mark.parametrize("batch", [32, 36])
def test_decode_batch_invalid_entries(weights_gpu, batch):
    """A token id outside the vocabulary and a position outside max_context among valid sequences, on both
    sides of gemm_rows' limit: they emit -1 and write no cache row, and the other sequences' logits and rows are
    the bits of the same step without them (every row of a batch is computed alike)."""
    from qwen_megakernel.model import _Forward, _ops

    V, layers, S = 151936, 2, 256
    fwd = _Forward(_ops(), weights_gpu, layers)
    g = torch.Generator("cuda").manual_seed(batch)
    k0 = torch.randn(batch, layers, 8, S, 128, generator=g, device="cuda").bfloat16()
    v0 = torch.randn(batch, layers, 8, S, 128, generator=g, device="cuda").bfloat16()
    ids, pos = [31 * b for b in range(batch)], [(29 * b) % 200 for b in range(batch)]
    got = []
    for bad in (False, True):
        i, p = list(ids), list(pos)
        if bad:
            i[3], p[batch - 2] = V, 200
        k, v = k0.clone(), v0.clone()
        out = torch.empty(batch, dtype=torch.int32, device="cuda")
        logits = torch.empty(batch, V, dtype=torch.float32, device="cuda")
        fwd.decode(_t(i), _t(p), out, logits, k, v, 200)
        got.append((out, logits, k, v))
    rest = [b for b in range(batch) if b not in (3, batch - 2)]
    for a, b in zip(*got):
        assert torch.equal(a[rest], b[rest])
    out, _, k, v = got[1]
    for b in (3, batch - 2):
        assert int(out[b]) == -1 and torch.equal(k[b], k0[b]) and torch.equal(v[b], v0[b])


def test_decode_batch_several_chunks(shape, exact06, weights_gpu):
    """More chunks than workgroups (40 sequences, a context bound of 12 chunks: 9 workgroups per head, some of
    which take two), contexts at the edges of the chunks taken second, against the oracle."""
    c0s = tuple(range(3, 31)) + (1151, 1152, 1153, 1278, 1279, 1280, 1400, 1498, 127, 128, 1023, 700)
    _decode_steps(shape, exact06, weights_gpu, c0s, layers=2, max_seq=1536, steps=1)


@pytest.mark.parametrize("batch", [5, 40])
def test_decode_batch_does_not_depend_on_the_bound(weights_gpu, batch):
    """The same step with max_context at its longest sequence and far above it (each workgroup several
    chunks, nearly all of which no token reaches): the same bits."""
    from qwen_megakernel.model import _Forward, _ops

    V, layers, S = 151936, 2, 16384 if batch == 5 else 4096
    w = with_rope(weights_gpu, S, "cuda")
    fwd = _Forward(_ops(), w, layers)
    g = torch.Generator("cuda").manual_seed(batch)
    k0 = torch.randn(batch, layers, 8, S, 128, generator=g, device="cuda").bfloat16()
    v0 = torch.randn(batch, layers, 8, S, 128, generator=g, device="cuda").bfloat16()
    pos = [(37 * b) % 300 for b in range(batch)]
    got = []
    for bound in (max(pos) + 1, S):
        k, v = k0.clone(), v0.clone()
        out = torch.empty(batch, dtype=torch.int32, device="cuda")
        logits = torch.empty(batch, V, dtype=torch.float32, device="cuda")
        fwd.decode(_t(range(batch)), _t(pos), out, logits, k, v, bound)
        got.append((out, logits, k, v))
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rows", [17, 32, 33, 64, 65, 200])
def test_lm_head_row_groups(weights_gpu, rows):
    """lm_head_tiled (more than 16 emitted rows, groups of 32 or 64): logits within one bf16 ulp of the
    same rows emitted four at a time (lm_head_rows, another order of the same fp32 sums of bf16 products:
    both round to a neighbour of the exact sum), and each token the first index of its own maximum.  One
    emitted row is outside the batch: it emits -1."""
    from qwen_megakernel.model import _Forward, _ops

    V, T = 151936, 200
    fwd = _Forward(_ops(), weights_gpu, 1)
    k = torch.zeros(1, 1, 8, 256, 128, dtype=torch.bfloat16, device="cuda")
    v = torch.zeros_like(k)

    def i32(x):
        return torch.tensor(x, dtype=torch.int32, device="cuda")

    g = torch.Generator().manual_seed(rows)
    ids = i32(torch.randint(0, V, (T,), generator=g).tolist())
    seqs, pos = i32([0] * T), torch.arange(T, dtype=torch.int32, device="cuda")

    def emit(which):
        out = torch.empty(len(which), dtype=torch.int32, device="cuda")
        logits = torch.empty(len(which), V, dtype=torch.float32, device="cuda")
        fwd(ids, seqs, pos, i32(which), out, logits, k, v, T)
        return out.cpu(), logits

    which = torch.randperm(T, generator=g)[:rows].tolist()
    which[rows // 2] = T + 5
    out, logits = emit(which)
    assert int(out[rows // 2]) == -1
    for r0 in range(0, rows, 4):
        o4, l4 = emit(which[r0:r0 + 4])
        for r in range(len(o4)):
            if which[r0 + r] >= T:
                assert int(o4[r]) == -1
                continue
            x, y = logits[r0 + r], l4[r]
            ulp = torch.exp2(torch.floor(torch.log2(y.abs().clamp_min(1e-3))) - 7)
            assert ((x - y).abs() <= 1.01 * ulp).all()
            assert int(out[r0 + r]) == int(torch.argmax(x.cpu()))


@pytest.fixture(scope="module")
def qwen3_1p7b():
    from oracle.qwen3_exact import ExactWeights
    from qwen_megakernel.shapes import QWEN3_1_7B
    from qwen_megakernel.weights import make_weights, to_device

    w = make_weights(QWEN3_1_7B, seed=0, num_layers=2, max_seq_len=256)
    return QWEN3_1_7B, ExactWeights(w, QWEN3_1_7B, num_layers=2), to_device(w, "cuda")


@pytest.mark.parametrize("model,n", [("0.6b", n) for n in (15, 16, 17, 32, 33)] + [("1.7b", n) for n in (9, 17, 32)])
def test_prompt_row_tiles(request, model, n):
    """gemm_rows' row tiles (one up to 16 tokens, two up to 32; for the larger model the residual products'
    16-column tiles at two) and the first count past them: every row of a prompt after 5 positions, 2
    layers, and its K/V rows."""
    from qwen_megakernel.weights import make_prompt

    from parity import decoder

    if model == "0.6b":
        shape, exact, weights = (request.getfixturevalue(f) for f in ("shape", "exact06", "weights_gpu"))
    else:
        shape, exact, weights = request.getfixturevalue("qwen3_1p7b")
    V, start, S = 151936, 5, 256
    dec = decoder(weights, num_layers=2, max_seq_len=S)
    dec.prefill(make_prompt(start, shape.vocab, seed=8))
    ids = make_prompt(n, shape.vocab, seed=n)

    def i32(x):
        return torch.tensor(x, dtype=torch.int32, device="cuda")

    out = torch.empty(n, dtype=torch.int32, device="cuda")
    logits = torch.empty(n, V, dtype=torch.float32, device="cuda")
    dec._forward(i32(ids), i32([0] * n), i32(list(range(start, start + n))), i32(list(range(n))), out, logits,
                 dec._k_cache, dec._v_cache, start + n)
    orc = exact_oracle(exact, shape, S, num_layers=2)
    ref = oracle_steps(orc, dec._k_cache, dec._v_cache, start, ids)
    print(check_rows(Tally(f"{model} {n} rows"), ref, out.cpu().tolist(), logits.cpu(), bar=LITERAL))
    check_kv_rows(f"{model} {n} rows", orc, dec._k_cache, dec._v_cache, start, n)


@pytest.mark.parametrize("n,start", [(33, 1400), (100, 1300), (600, 700)])
def test_prompt_does_not_depend_on_the_cache_slots(weights_gpu, n, start):
    """One prompt after a context, in a cache of one sequence and in the last of 16 (the others empty): the
    same calls, so the same logits and K/V rows bit for bit (the key chunks are cut for the call's own tiles)."""
    from qwen_megakernel.model import BatchDecoder
    from qwen_megakernel.weights import make_prompt

    V, layers, S = 151936, 2, 1536
    got = []
    for slots in (1, 16):
        bd = BatchDecoder(weights=weights_gpu, batch_size=slots, max_seq_len=S, num_layers=layers, verbose=False)
        bd.prefill(slots - 1, make_prompt(start, V, seed=3))
        _, logits = bd.prefill(slots - 1, make_prompt(n, V, seed=4), return_logits=True)
        got.append((logits.cpu(), bd._k_cache[slots - 1].cpu(), bd._v_cache[slots - 1].cpu()))
    assert torch.isfinite(got[0][0]).all()
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("order", ["interleaved", "ragged", "after-context", "one-chunk-tiles", "many-short-runs"])
def test_attention_tiles_of_several_sequences(shape, exact06, weights_gpu, order):
    """The MFMA attention's tiles over a call of several sequences, 2 layers, every sequence's last rows
    against the oracle: prompts whose tiles end inside the call, tokens in no tile (two sequences token by
    token: one run each; 130 runs of 3), an invalid token inside a prompt, and the
    same over key chunks after a context, and after one with more tiles than tile chunks (20 runs of 10)."""
    from qwen_megakernel.model import BatchDecoder
    from qwen_megakernel.weights import make_prompt

    V, layers, S = 151936, 2, 1408
    start = {"after-context": 900, "one-chunk-tiles": 300}.get(order, 0)
    lens = {"interleaved": (170, 170), "ragged": (65, 1, 190, 130), "after-context": (70, 33),
            "one-chunk-tiles": (10,) * 20, "many-short-runs": (3,) * 130}[order]
    bd = BatchDecoder(weights=weights_gpu, batch_size=len(lens), max_seq_len=S, num_layers=layers, verbose=False)
    bd._k_cache.fill_(float("nan"))
    bd._v_cache.fill_(float("nan"))
    if start:
        for b in range(len(lens)):
            bd._forward(*_one(make_prompt(start, V, seed=50 + b), b), bd._k_cache, bd._v_cache, start)
    prompts = [make_prompt(n, V, seed=90 + b) for b, n in enumerate(lens)]
    toks = [(b, i) for b, n in enumerate(lens) for i in range(n)]
    if order == "interleaved":
        toks.sort(key=lambda x: (x[1], x[0]))
    ids, seqs, pos = [prompts[b][i] for b, i in toks], [b for b, _ in toks], [start + i for _, i in toks]
    bad = len(toks) // 2 if order == "ragged" else None
    if bad is not None:  # an invalid token splits its prompt's run
        ids.insert(bad, V + 7), seqs.insert(bad, seqs[bad]), pos.insert(bad, 0)
        toks.insert(bad, (-1, -1))
    want = sorted(set(toks.index((b, i)) for b, n in enumerate(lens) if b % 19 == 0 or len(lens) < 10
                      for i in (0, n // 2, n - 1)))
    out = torch.empty(len(want), dtype=torch.int32, device="cuda")
    logits = torch.empty(len(want), V, dtype=torch.float32, device="cuda")
    bd._forward(_t(ids), _t(seqs), _t(pos), _t(want), out, logits, bd._k_cache, bd._v_cache, start + max(lens))
    assert torch.isfinite(logits).all()
    t = Tally(f"{order} tiles")
    for b in sorted(set(toks[w][0] for w in want)):
        mine = [k for k, w in enumerate(want) if toks[w][0] == b]
        n = start + lens[b]
        kc, vc = (torch.zeros_like(x[b]) for x in (bd._k_cache, bd._v_cache))
        kc[:, :, :n], vc[:, :, :n] = bd._k_cache[b, :, :, :n], bd._v_cache[b, :, :, :n]
        orc = exact_oracle(exact06, shape, S, num_layers=layers)
        ref = oracle_steps(orc, kc, vc, start, prompts[b], emit=[toks[want[k]][1] for k in mine])
        check_rows(t, ref, [int(out[k]) for k in mine], logits[mine].cpu(), bar=LITERAL)
    print(t)


@pytest.mark.parametrize("n,runs", [
    (330, [(0, 1), (63, 2), (511, 1), (512, 2), (598, 1)]),
    (70, [(3326, 1), (3327, 1), (3328, 4), (40, 3), (-1, 1)]),
    (1990, [(8190, 1), (8191, 1), (8192, 2), (511, 1), (-1, 1)]),
    (2100, [(100, 3), (700, 1), (5, 20), (-1, 1)]),
    (330, [(p, 1) for p in list(range(0, 500, 4)) + [508, 509, 510, 511, 512, 570]]),
], ids=["short", "split", "whole", "long-call", "many"])
def test_tokens_beside_a_prompt(shape, exact06, weights_gpu, n, runs):
    """Tokens in no attention tile beside a prompt of n tokens, in each of the three kernels that take them, 2
    layers: runs of fewer tokens than a tile's smallest count, at the edges of what is taken by a wave
    (position 511), of the scores that LDS holds at once (3328 positions beside tile chunks, 8192 beside
    whole tiles), a call of more tokens than the plan holds in LDS, more of them than workgroups take ("many"), and an invalid one (position -1)."""
    from qwen_megakernel.model import BatchDecoder
    from qwen_megakernel.weights import make_prompt

    V, layers = 151936, 2
    S = (max([n] + [p + k for p, k in runs]) + 63) // 64 * 64
    bd = BatchDecoder(weights=with_rope(weights_gpu, S, "cuda"), batch_size=1 + len(runs), max_seq_len=S,
                      num_layers=layers, verbose=False)
    bd._k_cache.fill_(float("nan"))
    bd._v_cache.fill_(float("nan"))
    g = torch.Generator("cuda").manual_seed(n + len(runs))
    for b, (p, _) in enumerate(runs, 1):
        if p > 0:
            bd.load_kv(b, torch.randn(layers, 8, p, 128, generator=g, device="cuda").bfloat16(),
                       torch.randn(layers, 8, p, 128, generator=g, device="cuda").bfloat16(), p)
    # half of the runs before the prompt, half after it
    order = list(range(1, 1 + len(runs) // 2)) + [0] + list(range(1 + len(runs) // 2, 1 + len(runs)))
    own = [make_prompt(n, V, seed=1)] + [make_prompt(k, V, seed=70 + b) for b, (_, k) in enumerate(runs)]
    start = [0] + [p for p, _ in runs]
    toks = [(b, i) for b in order for i in range(len(own[b]))]
    ids, seqs, pos = [own[b][i] for b, i in toks], [b for b, _ in toks], [start[b] + i for b, i in toks]
    check = [b for b in order if b and (len(runs) < 20 or b % 21 == 0 or start[b] > 500)]
    want = [k for k, (b, _) in enumerate(toks) if b in check]
    out = torch.empty(len(want), dtype=torch.int32, device="cuda")
    logits = torch.empty(len(want), V, dtype=torch.float32, device="cuda")
    bd._forward(_t(ids), _t(seqs), _t(pos), _t(want), out, logits, bd._k_cache, bd._v_cache, max(pos) + 1)
    t = Tally(f"{len(runs)} runs beside {n} tokens")
    for b in check:
        mine = [k for k, w in enumerate(want) if toks[w][0] == b]
        if start[b] < 0:
            assert [int(out[k]) for k in mine] == [-1]
            continue
        m = start[b] + len(own[b])
        kc, vc = (torch.zeros_like(x[b]) for x in (bd._k_cache, bd._v_cache))
        kc[:, :, :m], vc[:, :, :m] = bd._k_cache[b, :, :, :m], bd._v_cache[b, :, :, :m]
        orc = exact_oracle(exact06, shape, S, num_layers=layers)
        ref = oracle_steps(orc, kc, vc, start[b], own[b])
        check_rows(t, ref, [int(out[k]) for k in mine], logits[mine].cpu(), bar=LITERAL)
        check_kv_rows(f"sequence {b}", orc, kc, vc, start[b], len(own[b]))
    print(t)


def _t(values):
    return torch.tensor([int(v) for v in values], dtype=torch.int32, device="cuda")


def _one(ids, seq):
    """Arguments of a forward of one whole prompt from position 0 that emits its last row."""
    n = len(ids)
    return (_t(ids), _t([seq] * n), _t(range(n)), _t([n - 1]), torch.empty(1, dtype=torch.int32, device="cuda"),
            torch.empty(1, 151936, dtype=torch.float32, device="cuda"))
