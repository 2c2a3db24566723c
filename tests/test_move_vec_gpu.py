"""COPY, UPDATE_ROWS and BIN moving 16-byte vectors: bit-exact over element types, permuted views and row widths at and off
the vector size (those stay element by element), rows at the end of a cache, and every BIN operation.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def permuted(ctx, vk, base, axes, made):
    ref = vk.TensorP()
    vk.check("copy_ref", vk.lib().vkllm_tensor_copy_ref(ctx.vp, base, ctypes.byref(ref)))
    vk.check("permute", vk.lib().vkllm_tensor_permute(ctx.vp, ref, (ctypes.c_uint32 * 4)(*axes)))
    made.append(ref)
    return ref


@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["f16", "f32"])
@pytest.mark.parametrize("W", [1, 4, 8, 12, 40, 128])
def test_copy_and_update_rows(ctx, vk, dtype, W):
    print(f"[move] W={W} {dtype.__name__}", flush=True)
    rng = np.random.default_rng(W)
    x = rng.standard_normal((2, 5, 3, W)).astype(dtype)  # seen as [2, 3, 5, W]
    cache = rng.standard_normal((2, 3, 9, W)).astype(dtype)
    made = [ctx.tensor_from(x)]
    src = permuted(ctx, vk, made[0], (0, 2, 1, 3), made)
    out = ctx.tensor([2, 3, 5, W], vk.DTYPE_OF[np.dtype(dtype)], op=vk.OP_COPY, srcs=[src])
    kc = ctx.tensor([2, 3, 9, W], vk.DTYPE_OF[np.dtype(dtype)], op=vk.OP_UPDATE_ROWS, srcs=[src],
                    params=vk.UpdateRowsParams(4))
    made += [out, kc]
    want = x.transpose(0, 2, 1, 3)
    try:
        ctx.upload(kc, cache)
        vk.check("copy", ctx.run_op("copy", out))
        vk.check("update_rows", ctx.run_op("update_rows", kc))
        got, got_kc = ctx.download(out).reshape(want.shape), ctx.download(kc).reshape(cache.shape)
    finally:
        for t in reversed(made):
            ctx.free(t)
    assert np.array_equal(got, want)
    cache[:, :, 4:] = want
    assert np.array_equal(got_kc, cache)


@pytest.mark.parametrize("op", [0, 1, 2, 3])
@pytest.mark.parametrize("shape", [(1, 1, 1, 8), (1, 1, 3, 5), (2, 3, 7, 40), (1, 1, 33, 256)], ids=str)
def test_bin_vectors(ctx, vk, shape, op):
    rng = np.random.default_rng(op)
    a, b = (rng.standard_normal(shape).astype(np.float16) for _ in range(2))
    a.flat[0], b.flat[0] = np.float16(np.inf), np.float16(0.0)
    ta, tb = ctx.tensor_from(a), ctx.tensor_from(b)
    out = ctx.tensor(list(shape), vk.F16, op=vk.OP_BIN, srcs=[ta, tb], params=ctypes.c_int32(op))
    try:
        vk.check("bin", ctx.run_op("bin", out))
        got = ctx.download(out).reshape(shape)
    finally:
        for t in (out, ta, tb):
            ctx.free(t)
    a32, b32 = a.astype(np.float32), b.astype(np.float32)
    with np.errstate(all="ignore"):
        want = [a32 + b32, a32 - b32, a32 * b32, a32 / b32][op].astype(np.float16)
    assert np.array_equal(got, want, equal_nan=True)
