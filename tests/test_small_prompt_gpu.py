"""Prompt steps of small models (widths the tile GEMM's epilogues do not take): one launch per product with the RMSNorm in
front and RoPE, residual and SwiGLU behind. Logits and ids of a prompt and of a continuation against the oracle, at the
16-token tile's edges, the step's longest and one past it, a width over three K steps per wave, vocabularies on either
side of the tile GEMM's line and an odd one.
"""
import numpy as np
import pytest

from helpers import assert_prefill_ids

pytestmark = pytest.mark.gpu

# (dim, heads, ffn, vocab, ctx, prompt tokens, continuation tokens)
CASES = [
    (288, 6, 768, 1000, 64, 16, 17),
    (288, 6, 768, 1000, 64, 2, 1),
    (288, 6, 768, 32000, 64, 15, 3),   # 2000 tiles of logits, on the small kernel
    (288, 6, 768, 32000, 64, 33, 3),   # 6000: the tile GEMM
    (288, 6, 768, 1001, 48, 33, 15),   # kv == head size at the end
    (96, 4, 1024, 500, 320, 256, 2),
    (96, 4, 1024, 500, 320, 257, 2),   # past the longest small step
    (800, 10, 992, 640, 40, 31, 9),    # head size 80
    (32, 2, 64, 64, 32, 5, 5),         # one K step
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_small_prompt_steps(ctx, vk, oracle, case):
    dim, heads, ffn, vocab, n_ctx, first, second = case
    print(f"[small] {case}", flush=True)
    cfg = oracle.make_cfg(n_layer=2, dim=dim, n_head=heads, ffn=ffn, vocab=vocab, ctx=n_ctx)
    ref = oracle.Model(cfg=cfg, seed=31)
    model = vk.Model(ctx, config=vk.llama_config(2, dim, heads, ffn, vocab, n_ctx), seed=31)
    try:
        pos = 0
        for n in (first, second):
            toks = oracle.prompt_tokens(32 + n, n, vocab)
            want_ids, want, _ = ref.step(toks, pos, want_logits=True)
            ids = model.step(toks, pos)
            got = model.last_logits(n).astype(np.float32)
            err = float(np.max(np.abs(got - want.astype(np.float32))))
            assert err <= 2e-2, f"{n} tokens at {pos}: max|dlogit| {err}"
            if float(np.sort(want[-1].astype(np.float32))[-1] - np.sort(want[-1].astype(np.float32))[-2]) > 2e-2:
                assert_prefill_ids(ids, want_ids, want, what=str(case)) if n > 1 else None
            pos += n
    finally:
        ref.close()
        model.close()
