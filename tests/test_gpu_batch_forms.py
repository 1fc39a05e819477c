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
                                 tuple(range(110, 146, 2)), (383, 8200)],
                         ids=["5seq-first-chunk-edge", "6seq-second-chunk-edge", "18seq-general", "2seq-65-chunks"])
def test_decode_batch_attention_chunk_edges(shape, exact06, weights_gpu, c0s):
    """attn_chunk_*: contexts ending at, before and after a chunk's edge, a token in a chunk of its own,
    more than 64 chunks (two rounds of pairs), from raw projections (up to 16 sequences) and finished q."""
    _decode_steps(shape, exact06, weights_gpu, c0s, layers=2, max_seq=(max(c0s) + 2 + 63) // 64 * 64)
