"""Prompt attention with two groups of waves sharing the rows' key blocks, at the edges of its blocks: the last key block of
the later group absent, of one key, or full; a first row block with one key block for two groups; head sizes 64 and 128;
and either side of the grid on which one group takes over. Logits against the oracle (one layer, so a step's attention shows in them),
and the rows whose max lies past them.
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
    (1024, 16, 0, 1000), # 256 workgroups, the most for two groups on 256 CUs
    (1024, 16, 0, 1030), # 272: one group, head size 64
    (512, 4, 3900, 65),  # long chain
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


# (dim, heads, step tokens): one pass (kv <= 128), two groups, one group (512 workgroups), a head size off the matrix cores
MAX_CASES = [(256, 2, 128), (256, 2, 300), (256, 4, 700), (1024, 16, 2048), (288, 6, 200)]


@pytest.mark.parametrize("case", MAX_CASES, ids=str)
def test_the_max_runs_over_the_whole_row(ctx, vk, oracle, case):
    """The softmax shader subtracts the max of the whole row, later positions included
    (src/shaders/vkllm_softmax.comp:42-96), so a row one of whose later scores exceeds its own by more than the
    exponent's range (104 with subnormals) is 0 / 0, in every form of the prompt attention and wherever in the row that
    score lies. The weights spread the scores with a deviation of 70; which rows it takes comes from the scores in
    float64, rows with a head between 86 (exp normal; 1 for fp16's rounding of scores up to 1024) and 106 left out."""
    dim, heads, tokens = case
    print(f"[attention max] {case}", flush=True)
    hd, std, seed = dim // heads, (70 / dim) ** 0.5, 53
    cfg = oracle.make_cfg(n_layer=1, dim=dim, n_head=heads, ffn=64, vocab=500, ctx=tokens, weight_std=std)
    ref = oracle.Model(cfg=cfg, seed=seed)
    try:
        embd, wq, wk = (ref.weight(t).view(np.float16).astype(np.float64).reshape(-1, dim) for t in (0, 2, 3))
    finally:
        ref.close()
    toks = oracle.prompt_tokens(54, tokens, 500)
    x = embd[toks]
    x /= np.sqrt(np.mean(x * x, -1, keepdims=True) + 1e-5)
    angle = np.arange(tokens)[:, None] / 10000.0 ** (np.arange(0, hd, 2) / hd)
    c, s = np.cos(angle)[None], np.sin(angle)[None]

    def rotated(w):
        v = (x @ w.T).reshape(tokens, heads, hd).transpose(1, 0, 2)
        a, b = v[..., 0::2], v[..., 1::2]
        return np.stack((c * a - s * b, s * a + c * b), -1).reshape(heads, tokens, hd)

    scores = rotated(wq) @ rotated(wk).transpose(0, 2, 1) / np.sqrt(hd)
    assert np.max(np.abs(scores)) < 1024
    own = np.where(np.tri(tokens, dtype=bool), scores, -np.inf).max(-1)
    excess = scores.max(-1) - own  # [head, row]
    undefined, defined = (excess > 106).any(0), (excess < 86).all(0)
    assert undefined.sum() >= 10 and defined.sum() >= 10
    model = vk.Model(ctx, config=vk.llama_config(1, dim, heads, 64, 500, tokens, std=std), seed=seed)
    try:
        model.step(toks, 0)
        got = np.isnan(model.last_logits(tokens)).any(-1)
    finally:
        model.close()
    assert not got[defined].any(), f"rows {np.flatnonzero(got & defined)[:8]} have no later score that large"
    assert got[undefined].all(), f"rows {np.flatnonzero(~got & undefined)[:8]} of {undefined.sum()} are 0 / 0"
