"""Prompt attention with two groups of waves sharing the rows' key blocks, at the edges of its blocks: the last key block of
the later group absent, of one key, or full; a first row block with one key block for two groups; head sizes 64 and 128;
and the grid on which one group takes over. Logits against the oracle (one layer, so a step's attention shows in them).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (dim, heads, cached tokens, step tokens)
CASES = [
    (256, 2, 0, 129),    # first row block sees one key block: the later group has none
    (256, 2, 128, 1 + 1),  # third block of two keys
    (256, 2, 64, 128),   # three blocks
    (256, 4, 191, 65),   # four full blocks, head size 64
    (256, 4, 320, 3),    # six blocks, the last of three keys, head size 64
    (128, 2, 0, 300),    # head size 64
    (512, 4, 0, 700),    # 44 workgroups, eleven key blocks
]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_prompt_attention_groups(ctx, vk, oracle, case):
    dim, heads, before, tokens = case
    print(f"[attention] {case}", flush=True)
    n_ctx = before + tokens
    cfg = oracle.make_cfg(n_layer=1, dim=dim, n_head=heads, ffn=256, vocab=500, ctx=n_ctx)
    ref = oracle.Model(cfg=cfg, seed=51)
    model = vk.Model(ctx, config=vk.llama_config(1, dim, heads, 256, 500, n_ctx), seed=51)
    try:
        pos = 0
        for n in (before, tokens):
            if n == 0:
                continue
            toks = oracle.prompt_tokens(52 + n, n, 500)
            _, want, _ = ref.step(toks, pos, want_logits=True)
            model.step(toks, pos)
            err = float(np.max(np.abs(model.last_logits(n).astype(np.float32) - want.astype(np.float32))))
            assert err <= 2e-2, f"{n} tokens at {pos}: max|dlogit| {err}"
            pos += n
    finally:
        ref.close()
        model.close()
