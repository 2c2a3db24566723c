"""MATMUL on the batched matrix-core kernel against the same product in float64: both orders of B, broadcast batches,
strided, permuted and unaligned rows, ragged M, N and K, a scale and SiLU. The reference rounds once, to fp16, so the
bar is one ulp plus what the fp32 sums may be off (dot_atol).
"""
import ctypes

import numpy as np
import pytest

from helpers import assert_fp16_close, dot_atol

pytestmark = pytest.mark.gpu

# (batch of A, batch of B, M, N, K, B as [N, K], scale, act)
CASES = [
    ((1, 3), (1, 3), 512, 512, 128, True, 0.088, 0),   # scores of a 512-token prompt
    ((1, 32), (1, 32), 300, 300, 128, True, 0.088, 0), # ragged M and N on 128 x 128 tiles
    ((1, 32), (1, 32), 260, 128, 301, False, 1.0, 0),  # P.V over an odd number of positions: unaligned rows of A
    ((1, 2), (1, 2), 64, 64, 64, False, 1.0, 0),       # N == K, B in its own order by shape: [N, K]
    ((1, 6), (1, 6), 16, 16, 48, True, 0.144, 0),      # the tiny model's scores: less than one K step
    ((1, 6), (1, 6), 17, 48, 33, False, 1.0, 0),
    ((1, 1), (1, 1), 2, 1, 1, False, 1.0, 0),          # smallest
    ((2, 3), (1, 1), 65, 63, 65, True, 1.0, 1),        # broadcast B, one past and one short of a tile
    ((1, 1), (2, 3), 65, 63, 129, False, 0.5, 1),      # broadcast A, ragged [K, N] columns
    ((1, 1), (4, 1), 1, 200, 70, False, 1.0, 0),       # one row against [K, N]
    ((1, 1), (1, 1), 130, 129, 7, True, 2.0, 0),       # rows shorter than a vector
    ((1, 4), (1, 4), 1024, 1024, 256, False, 1.0, 0),
]


def view_of(ctx, vk, x, pad, made):
    """x on the device, its rows in rows `pad` elements longer (a view of a wider tensor)"""
    wide = np.full((*x.shape[:-1], x.shape[-1] + pad), np.inf, x.dtype)  # what lies past a row must not be read into it
    wide[..., :x.shape[-1]] = x
    base = ctx.tensor_from(wide)
    made.append(base)
    if pad == 0:
        return base
    ref = vk.TensorP()
    vk.check("copy_ref", vk.lib().vkllm_tensor_copy_ref(ctx.vp, base, ctypes.byref(ref)))
    ref.contents.shapes[3] = x.shape[-1]
    made.append(ref)
    return ref


@pytest.mark.parametrize("pad", [0, 3], ids=["packed", "padded"])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_matmul_batched(ctx, vk, case, pad):
    ab, bb, M, N, K, tb, scale, act = case
    print(f"[matmul] {case} pad={pad}", flush=True)
    rng = np.random.default_rng(M + N + K)
    a = rng.standard_normal((*ab, M, K), dtype=np.float32).astype(np.float16)
    b = rng.standard_normal((*bb, *((N, K) if tb else (K, N))), dtype=np.float32).astype(np.float16)
    ob = tuple(max(x, y) for x, y in zip(ab, bb))
    made = []
    ta, tb_ = view_of(ctx, vk, a, pad, made), view_of(ctx, vk, b, pad, made)
    out = ctx.tensor([*ob, M, N], vk.F16, op=vk.OP_MATMUL, srcs=[ta, tb_], params=vk.MatmulParams(scale, act))
    try:
        vk.check("matmul", ctx.run_op("matmul", out))
        got = ctx.download(out).reshape(*ob, M, N)
    finally:
        for t in [out, *reversed(made)]:
            ctx.free(t)
    transposed = tb or N == K  # by shape: a square B is read as [N, K]
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = (a64 @ (np.swapaxes(b64, -1, -2) if transposed else b64)) * scale
    atol = dot_atol(a, b, transposed=transposed) * scale
    if act:
        atol = 1.1 * atol + 2.0 ** -21 * np.abs(want)
        want = want / (1.0 + np.exp(-want))
    assert_fp16_close(got, want.astype(np.float16), what=str(case), atol=atol + 2.0 ** -24)


def test_matmul_rows_past_the_ring_kernels_offsets(ctx, vk):
    """Rows of more than 2^22 elements (the LDS-ring tile kernel's byte offsets are 32-bit): +-1 at a few places, the
    last ones included, so the sums are whole numbers and exact."""
    M, N, K = 2, 8, (1 << 22) + 64
    print(f"[matmul] {M}x{N}x{K}", flush=True)
    rng = np.random.default_rng(3)
    at = np.unique(np.concatenate([rng.integers(0, K, 500), [0, (1 << 22) - 1, 1 << 22, K - 1]]))
    a, b = np.zeros((1, 1, M, K), np.float16), np.zeros((1, 1, N, K), np.float16)
    a[..., at], b[..., at] = (rng.choice([-1.0, 1.0], (1, 1, n, at.size)) for n in (M, N))
    ta, tb = ctx.tensor_from(a), ctx.tensor_from(b)
    out = ctx.tensor([1, 1, M, N], vk.F16, op=vk.OP_MATMUL, srcs=[ta, tb], params=vk.MatmulParams(1.0, 0))
    try:
        vk.check("matmul", ctx.run_op("matmul", out))
        got = ctx.download(out).reshape(M, N)
    finally:
        for t in (out, ta, tb):
            ctx.free(t)
    want = a[0, 0][:, at].astype(np.float64) @ b[0, 0][:, at].astype(np.float64).T
    assert np.array_equal(got.astype(np.float64), want)
