"""GPU tests of SPyNet's convolutions on large tiles (batches of many images): the same bits
as one pair at a time, which runs them on 16-pixel tiles."""
from __future__ import annotations

import numpy as np
import pytest

import spynet_reference as sr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,frames", [(64, 64, 18), (32, 96, 24), (96, 32, 24), (160, 160, 5)])
def test_clip_flows_equal_pairs(gpu_ctx, h, w, frames):
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
