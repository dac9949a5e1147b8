"""Batches of small maps on the narrow kernel (images per workgroup by the number of
workgroups)."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dcn():
    import jasnamacos_amd.deform_conv as module
    return module


@pytest.fixture(scope="module")
def gpu_ctx(dcn):
    return dcn.HipDeformConv(0)


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
