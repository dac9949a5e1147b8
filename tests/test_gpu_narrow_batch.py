"""Batches of small maps on the narrow kernel (images per workgroup by the number of
workgroups) and the size above which a fast-sampler call takes the tile kernel."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def case(dcn, batch, h, w):
    s = dcn.DeformConvShape(batch, 128, h, w, 64, h, w, 3, 3, 1, 1, 1, 1, 1, 1, 1, 16)
    rng = np.random.default_rng(batch * 1000 + h)
    c = s.counts()
    x = rng.standard_normal(c["input"]).astype(np.float16)
    off = (rng.standard_normal(c["offset"]) * 4).astype(np.float16)
    msk = rng.random(c["mask"]).astype(np.float16)
    wt = (rng.standard_normal(c["weight"]) * 0.03).astype(np.float16)
    b = (rng.standard_normal(64) * 0.1).astype(np.float16)
    return s, x, off, msk, wt, b


# Images per workgroup: 1 (the flat kernel), 3 + 2 (5 maps of 100 tiles), 4, 9 + 8 (17 maps).
@pytest.mark.parametrize("sampler", [1, 0], ids=["fast", "exact"])
@pytest.mark.parametrize("batch,h,w", [(16, 16, 16), (5, 40, 40), (12, 48, 48), (17, 33, 61), (4, 3, 5)])
def test_batch_equals_single_images(gpu_ctx, dcn, batch, h, w, sampler):
    s, x, off, msk, wt, b = case(dcn, batch, h, w)
    one = dataclasses.replace(s, batch=1)
    c1 = one.counts()
    print("case: narrow batch", batch, h, w, sampler, flush=True)
    gpu_ctx.set_fused_config(0, 0, sampler, dcn.VARIANT_NARROW)
    try:
        packed = gpu_ctx.prepack(s, wt, b)
        out = np.asarray(gpu_ctx.run_float16_prepacked(s, x, off, msk, packed))
        part = lambda v, i, n: v[i * n:(i + 1) * n]
        for i in range(batch):
            o1 = gpu_ctx.run_float16_prepacked(one, part(x, i, c1["input"]), part(off, i, c1["offset"]),
                                               part(msk, i, c1["mask"]), packed)
            assert np.array_equal(part(out, i, c1["output"]).view(np.uint16), np.asarray(o1).view(np.uint16)), i
    finally:
        gpu_ctx.set_fused_config(0, 0, -1, 0)


@pytest.mark.parametrize("batch,h,w,variant", [(1, 116, 256, 5), (1, 116, 264, 7), (8, 64, 64, 7), (8, 64, 61, 5)])
def test_tile_kernel_above_928_tiles(gpu_ctx, dcn, batch, h, w, variant):
    """The fast sampler's choice on both sides of 928 tiles of 32 pixels (a width off 8 stays
    narrow), the exact sampler's at 1024. Narrow and tile kernel sum the same 1152 FP16
    products in FP32 in other orders and round once: they differ by at most one FP16 step
    plus that order's error, 1152 * 2^-24 * sum |terms| (each side)."""
    s, x, off, msk, wt, b = case(dcn, batch, h, w)
    print("case: tile above 928", batch, h, w, flush=True)
    assert gpu_ctx.get_fused_config(s)["variant"] == variant
    packed = gpu_ctx.prepack(s, wt, b)
    got = np.asarray(gpu_ctx.run_float16_prepacked(s, x, off, msk, packed)).astype(np.float32)
    gpu_ctx.set_fused_config(0, 0, dcn.SAMPLER_EXACT)
    try:
        assert gpu_ctx.get_fused_config(s)["variant"] == dcn.VARIANT_NARROW
        gpu_ctx.set_fused_config(0, 0, -1, dcn.VARIANT_NARROW)
        want = np.asarray(gpu_ctx.run_float16_prepacked(s, x, off, msk, packed)).astype(np.float32)
    finally:
        gpu_ctx.set_fused_config(0, 0, -1, 0)
    # |samples| <= max |x|: a bound of every output's terms.
    scale = np.abs(x).max() * np.abs(wt.astype(np.float32)).reshape(64, -1).sum(1).max() + np.abs(b).max()
    bound = np.abs(want) * 2.0 ** -10 + 2.0 ** -24 + 2 * 1152 * 2.0 ** -24 * float(scale)
    assert np.all(np.abs(got - want) <= bound), float(np.max(np.abs(got - want) / bound))
