"""GPU tests of SPyNet's convolutions on large tiles (many images, or large ones). A layer runs
them above 8192 pixels over the batch: a pair of at most 4096 runs 16-pixel tiles throughout, and
a batch has to give its bits; a larger pair is compared with the oracle chain."""
from __future__ import annotations

import numpy as np
import pytest

import spynet_reference as sr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,frames", [(64, 64, 18), (32, 96, 24), (96, 32, 24), (160, 160, 5)])
def test_clip_flows_equal_pairs(gpu_ctx, h, w, frames):
    """Bit for bit. At 160x160 the pairs run large tiles in the two finest levels too, in one of them
    of fewer rows."""
    import torch

    dev = lambda a: torch.from_numpy(np.asarray(a, np.float16).view(np.int16)).cuda()  # noqa: E731
    weights = sr.spynet_weights(np.random.default_rng(h + w))
    wd = {k: dev(v) for k, v in weights.items()}
    clip = [sr.smooth_frame(np.random.default_rng(t // 3), h, w, shift=(0.7 * t, -0.9 * t)) for t in range(frames)]
    x = dev(np.concatenate(clip))
    spy = gpu_ctx.spynet(h, w, wd, max_frames=frames)
    plane = h * w
    flows = torch.zeros(2, frames - 1, 2 * plane, dtype=torch.int16, device="cuda")
    pair = torch.zeros(2, 2 * plane, dtype=torch.int16, device="cuda")
    print("case: clip flows", h, w, frames, flush=True)
    spy.clip_flows_dev(x, frames, flows)
    fr = x.view(frames, 3 * plane)
    for t in (0, 1, frames // 2, frames - 2):
        spy.flow_dev(fr[t], fr[t + 1], pair)
        torch.cuda.synchronize()
        assert torch.equal(flows[0, t], pair[0]) and torch.equal(flows[1, t], pair[1]), t
    spy.free()
    assert np.isfinite(flows.cpu().numpy().view(np.float16).astype(np.float32)).all()


def test_large_pair_matches_oracle_chain(gpu_ctx):
    """The finest level of one 96x96 pair runs large tiles: within the bars of the small pairs,
    2e-2 max and 1e-3 mean of the flow's scale."""
    import torch

    dev = lambda a: torch.from_numpy(np.array(a, np.float16).view(np.int16)).cuda()  # noqa: E731
    h = w = 96
    rng = np.random.default_rng(96)
    weights = sr.spynet_weights(rng)
    ref, sup = sr.smooth_frame(rng, h, w), sr.smooth_frame(rng, h, w, shift=(1.5, -2.0))
    spy = gpu_ctx.spynet(h, w, {k: dev(v) for k, v in weights.items()})
    flow = torch.zeros(2 * 2 * h * w, dtype=torch.int16, device="cuda")
    print("case: large pair", h, w, flush=True)
    spy.flow_dev(dev(ref), dev(sup), flow, both_directions=True)
    torch.cuda.synchronize()
    got = flow.cpu().numpy().view(np.float16).astype(np.float64).reshape(2, -1)
    spy.free()
    for i, (a, b) in enumerate(((ref, sup), (sup, ref))):
        want = sr.spynet_flow(weights, a, b, h, w).astype(np.float64)
        scale = max(1.0, np.abs(want).max())
        err = np.abs(got[i] - want)
        print(f"direction {i}: err max {err.max():.3e} mean {err.mean():.3e}, scale {scale:.3f}", flush=True)
        assert err.max() <= 2e-2 * scale and err.mean() <= 1e-3 * scale
