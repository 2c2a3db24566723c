"""SOFTMAX on fp16 rows held in a wave's registers, against the float64 softmax of the same fp16 scores: row widths at the
edges of a vector, a lane's share and the kernel's instances, packed and in rows of a wider tensor (unaligned starts),
with and without the causal mask. The op rounds once: one fp16 ulp plus the fp32 exponential's and quotient's error.
"""
import ctypes

import numpy as np
import pytest

from helpers import assert_fp16_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pad", [0, 3], ids=["packed", "padded"])
@pytest.mark.parametrize("mask", [None, 0, 5], ids=["all", "causal", "offset5"])
@pytest.mark.parametrize("W", [1, 7, 8, 9, 17, 48, 511, 512, 513, 1024, 1031, 2048, 2050, 4096, 4097])
def test_softmax_row_widths(ctx, vk, W, mask, pad):
    print(f"[softmax] W={W} mask={mask} pad={pad}", flush=True)
    rng = np.random.default_rng(W + pad)
    x = (3.0 * rng.standard_normal((2, 3, 9, W), dtype=np.float32)).astype(np.float16)
    x[0, 0, 0] = np.float16(-65504.0)  # a row of the type's lowest value is uniform
    x[1, 2, 8, 0] = np.float16(60.0)   # and a dominant first element
    wide = np.full((2, 3, 9, W + pad), np.inf, np.float16)
    wide[..., :W] = x
    base = ctx.tensor_from(wide)
    src = vk.TensorP()
    vk.check("copy_ref", vk.lib().vkllm_tensor_copy_ref(ctx.vp, base, ctypes.byref(src)))
    src.contents.shapes[3] = W
    out = ctx.tensor([2, 3, 9, W], vk.F16, op=vk.OP_SOFTMAX, srcs=[src],
                     params=vk.SoftmaxParams(0 if mask is None else 1, mask or 0))
    try:
        vk.check("softmax", ctx.run_op("softmax", out))
        got = ctx.download(out).reshape(x.shape)
    finally:
        for t in (out, src, base):
            ctx.free(t)
    s = x.astype(np.float64)
    e = np.exp(s - s.max(-1, keepdims=True))  # the maximum is over the whole row
    if mask is not None:
        e = np.where(np.arange(W)[None, :] > np.arange(9)[:, None] + mask, 0.0, e)
    with np.errstate(divide="ignore", invalid="ignore"):
        want = e / e.sum(-1, keepdims=True)
    ok = e.sum(-1) > 1e-30  # a causal row whose every entry underflows in fp32 has no defined quotient
    assert_fp16_close(got[ok], want[ok].astype(np.float16), what="softmax", atol=2.0 ** -20 * want[ok] + 2.0 ** -25)
    if mask is not None:
        later = np.broadcast_to(np.arange(W)[None, :] > np.arange(9)[:, None] + mask, x.shape)
        assert not got[later].any()
