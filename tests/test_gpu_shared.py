"""GPU tests of the shared-sample kernel behind the plain-weight forwards (FP32 and FP16):
bit for bit the CPU oracle's result at the sizes where its tiling can go wrong."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (batch, Cin, H, W, Cout, Ho, Wo, Kh, Kw, ph, pw, sh, sw, dh, dw, groups, offset_groups), offset range
SHAPES = [
    ((3, 16, 5, 7, 64, 5, 7, 3, 3, 1, 1, 1, 1, 1, 1, 1, 2), 2.0),      # a pixel tile across images
    ((1, 24, 6, 2, 20, 6, 2, 3, 3, 1, 1, 1, 1, 1, 1, 1, 3), 2.0),      # two columns: every pair moved or not
    ((1, 24, 6, 1, 20, 6, 1, 3, 3, 1, 1, 1, 1, 1, 1, 1, 3), 2.0),      # one column: the one-thread kernel
    ((1, 40, 9, 11, 33, 9, 11, 3, 3, 1, 1, 1, 1, 1, 1, 1, 5), 9.0),    # a half stage, 33 channels
    ((2, 36, 8, 9, 30, 4, 5, 3, 3, 1, 1, 2, 2, 1, 1, 3, 3), 3.0),      # 12 channels per group, stride 2
    ((2, 30, 8, 9, 34, 8, 9, 3, 3, 1, 1, 1, 1, 1, 1, 2, 2), 3.0),      # odd channel counts, 17 outputs a group
    ((1, 17, 8, 8, 5, 8, 8, 3, 3, 1, 1, 1, 1, 1, 1, 1, 17), 3.0),      # one channel in the last stage
    ((1, 19, 8, 8, 17, 7, 7, 2, 2, 0, 0, 1, 1, 1, 1, 1, 1), 3.0),      # 4 taps, 12 samples in the last stage
    ((1, 48, 7, 7, 16, 7, 7, 1, 3, 0, 1, 1, 1, 1, 1, 4, 2), 3.0),      # an offset group over two conv groups
    ((1, 8, 7, 9, 12, 7, 9, 5, 5, 2, 2, 1, 1, 1, 1, 1, 2), 3.0),       # 25 taps: the one-thread kernel
    ((1, 16, 65, 66, 70, 65, 66, 3, 3, 1, 1, 1, 1, 1, 1, 1, 2), 12.0),  # over 256 pixel tiles, 64 + 6 channels
    ((1, 16, 50, 60, 24, 50, 60, 3, 3, 1, 1, 1, 1, 2, 2, 1, 4), 12.0),  # 188 pixel tiles, 24 channels, dilation
    ((1, 32, 70, 64, 24, 70, 64, 3, 3, 1, 1, 1, 1, 1, 1, 2, 2), 12.0),  # over 256 workgroups of 12 channels
    ((1, 4, 9, 10, 1, 9, 10, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1), 3.0),       # 36 weights in all: less than a stage
    ((1, 16, 9, 10, 1, 9, 10, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1), 3.0),      # one output channel, one whole stage
    ((1, 33, 9, 10, 2, 9, 10, 2, 2, 1, 1, 1, 1, 1, 1, 1, 1), 3.0),      # two whole stages and one channel
    ((2, 24, 33, 40, 24, 33, 40, 3, 3, 1, 1, 1, 1, 1, 1, 24, 24), 3.0),  # depthwise: the one-thread kernel
]


@pytest.mark.parametrize("dims,scale", SHAPES, ids=lambda t: "x".join(map(str, t)) if isinstance(t, tuple) else str(t))
@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
def test_shared_kernel_bit_exact(gpu_ctx, dcn, oracle, dims, scale, half):
    s = dcn.DeformConvShape(*dims)
    rng = np.random.default_rng(sum(dims) + half)
    c = s.counts()
    d = [rng.standard_normal(c["input"]), rng.uniform(-scale, scale, c["offset"]), rng.uniform(0, 1, c["mask"]),
         rng.uniform(-0.2, 0.2, c["weight"]), rng.uniform(-0.1, 0.1, c["bias"])]
    d[1][::7] = np.round(d[1][::7])  # whole offsets: samples exactly on rows, columns and edges
    d[1][::101] = 1e4
    d[3][::5] = 0.0
    d = [a.astype(np.float16 if half else np.float32) for a in d]
    print("case:", dims, scale, "f16" if half else "f32", flush=True)
    if half:
        out, ref = gpu_ctx.run_float16(s, *d), oracle.forward_f16_direct(s, *d)
        assert np.array_equal(out.view(np.uint16), ref.view(np.uint16))
    else:
        out, ref = gpu_ctx.run_float32(s, *d), oracle.forward_f32(s, *d)
        assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))


def test_shared_kernel_nonfinite(gpu_ctx, dcn, oracle):
    """Infinities and NaN in every operand, the last and first columns among them: the
    same non-finite pattern and the same bits elsewhere as the oracle."""
    s = dcn.DeformConvShape(1, 24, 9, 10, 40, 9, 10, 3, 3, 1, 1, 1, 1, 1, 1, 1, 3)
    rng = np.random.default_rng(5)
    c = s.counts()
    x = rng.standard_normal((24, 9, 10)).astype(np.float32)
    x[3, 4, 9], x[5, 2, 0], x[7, 8, 8] = np.inf, -np.inf, np.nan
    off = rng.uniform(-2, 2, c["offset"]).astype(np.float32)
    off[11], off[400], off[900] = np.nan, np.inf, -np.inf
    mask = rng.uniform(0, 1, c["mask"]).astype(np.float32)
    mask[17] = np.inf
    w = rng.uniform(-0.2, 0.2, c["weight"]).astype(np.float32)
    w[100] = np.inf
    b = np.full(c["bias"], -0.0, np.float32)
    print("case: non-finite operands", flush=True)
    out, ref = gpu_ctx.run_float32(s, x, off, mask, w, b), oracle.forward_f32(s, x, off, mask, w, b)
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(out[~np.isnan(ref)].view(np.uint32), ref[~np.isnan(ref)].view(np.uint32))
