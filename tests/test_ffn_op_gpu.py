"""FFN_UP_AND_GATE on the matrix cores and the streaming GEMV, against a float64 product of the same fp16 operands.

Packed fp16 rows take the tile GEMM (K in whole 64-wide steps) or, one row, the streaming GEMV; the sizes below sit at
the edges of those rules and of the kernels' tiles, with an operand or two that must stay on the generic kernel. The
op rounds once: the bar is one fp16 ulp of the exact result plus what the fp32 sums may be off (dot_atol), carried
through up * silu(gate).
"""
import numpy as np
import pytest

from helpers import assert_fp16_close, dot_atol

pytestmark = pytest.mark.gpu

# (rows as (B, C, M), K, F)
CASES = [
    ((1, 1, 1), 64, 8),         # one row: one vector
    ((1, 1, 1), 4096, 11008),   # 7B
    ((1, 1, 1), 5120, 13825),   # 13B widths, odd F
    ((1, 1, 1), 11272, 40),     # longer than a wave holds: generic
    ((1, 1, 2), 64, 8),         # smallest tile product
    ((1, 1, 37), 4096, 11008),  # 7B, one row of tiles
    ((1, 1, 129), 512, 1000),   # F % 32 != 0, whole K
    ((1, 1, 129), 4096, 1000),  # F % 32 != 0, K split: the reduce leaves out the columns past F
    ((1, 1, 200), 4096, 11008), # 7B, K split
    ((1, 1, 300), 320, 5000),   # F % 32 != 0 through the tile epilogue
    ((1, 1, 300), 192, 5000),   # the same, rows shorter than the ring
    ((2, 3, 50), 256, 96),      # batched rows as one matrix
    ((1, 1, 1024), 256, 22016), # 256 x 256 tiles
    ((1, 1, 16), 288, 768),     # K % 64 != 0
    ((1, 1, 17), 64, 100),      # F % 8 != 0: generic
]
SPLIT = {((1, 1, 129), 4096, 1000): (64, 128, 5), ((1, 1, 200), 4096, 11008): (256, 192, 2)}  # tile and K ranges


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{'x'.join(map(str, c[0]))}-{c[1]}-{c[2]}")
def test_ffn_up_and_gate_paths(ctx, vk, case):
    rows, K, F = case
    print(f"[ffn] rows={rows} K={K} F={F}", flush=True)
    if case in SPLIT:
        assert vk.gemm_plan(rows[2], (2 * F + 63) // 64 * 64, K) == SPLIT[case]
    rng = np.random.default_rng(K + F + rows[2])
    x = rng.standard_normal((*rows, K), dtype=np.float32).astype(np.float16)
    wu, wg = ((rng.standard_normal((1, 1, F, K), dtype=np.float32) / np.sqrt(K)).astype(np.float16) for _ in range(2))
    tx, tu, tg = ctx.tensor_from(x), ctx.tensor_from(wu), ctx.tensor_from(wg)
    out = ctx.tensor([*rows, F], vk.F16, op=vk.OP_FFN_UP_AND_GATE, srcs=[tx, tu, tg])
    try:
        vk.check("ffn_up_and_gate", ctx.run_op("ffn_up_and_gate", out))
        got = ctx.download(out).reshape(-1, F)
    finally:
        for t in (out, tx, tu, tg):
            ctx.free(t)
    x2 = x.reshape(-1, K)
    up, gate = (x2.astype(np.float64) @ w[0, 0].astype(np.float64).T for w in (wu, wg))
    act = gate / (1.0 + np.exp(-gate))
    atol = dot_atol(x2, wu[0, 0]) * np.abs(act) + 1.1 * dot_atol(x2, wg[0, 0]) * np.abs(up) + 2.0 ** -22 * np.abs(up * act)
    assert_fp16_close(got, (up * act).astype(np.float16), what="ffn", atol=atol + 2.0 ** -24)
