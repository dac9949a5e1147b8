"""The automatic choice of the tile kernel is one of the shape alone: offsets and masks of any
alignment give the same bits."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE = 7  # dcn_set_fused_config's variant


@pytest.fixture(scope="module")
def torch():
    import torch as t

    return t


class Call:
    """One layer's inputs on the GPU; run(off, msk) puts the offsets and masks that many halves past
    an aligned address, and returns the output's bits."""

    def __init__(self, torch, ctx, dcn, batch, h, w, cin=128, cout=64, amplitude=6.0):
        self.torch, self.ctx = torch, ctx
        og = cin // 8
        self.shape = dcn.DeformConvShape(batch, cin, h, w, cout, h, w, 3, 3, 1, 1, 1, 1, 1, 1, 1, og)
        rng = np.random.default_rng(batch * 1000 + h + cin)
        c = self.shape.counts()
        dev = lambda a: torch.from_numpy(np.asarray(a, np.float32).astype(np.float16)).cuda()  # noqa: E731
        self.x = dev(rng.standard_normal(c["input"]))
        # Smooth motion with a residue, wide enough for split stages in some tiles.
        flow = np.repeat(rng.uniform(-amplitude, amplitude, (batch, 2, h)), w, 2).reshape(batch, 1, 2, h * w)
        self.off = dev((flow + rng.uniform(-8, 8, (batch, og * 9, 2, h * w))).ravel())
        self.msk = dev(rng.random(c["mask"]))
        self.packed = ctx.prepack_dev(self.shape, dev(rng.standard_normal(c["weight"]) * 0.03),
                                      dev(rng.standard_normal(cout) * 0.1))
        self.out = torch.empty(c["output"], dtype=torch.float16, device="cuda")

    def _at(self, t, shift):
        held = self.torch.zeros(t.numel() + 8, dtype=t.dtype, device="cuda")[shift:shift + t.numel()]
        held.copy_(t)
        return held

    def run(self, off=0, msk=0):
        self.out.zero_()
        o, m = self._at(self.off, off), self._at(self.msk, msk)
        self.ctx.forward_f16_prepacked_dev(self.shape, self.x, o, m, self.packed, self.out)
        self.torch.cuda.synchronize()
        return self.out.cpu().numpy().view(np.uint16).copy()


# 8 x 64x64: 64 tiles per XCD; 116x264: 957 tiles of 32 pixels, partial tiles below and beside;
# 96 channels of a wide layer's 32 outputs; above 1024 tiles; the exact sampler there.
@pytest.mark.parametrize("dims,sampler", [((8, 64, 64), 1), ((1, 116, 264), 1), ((1, 118, 264, 96, 32), 1),
                                          ((1, 181, 192), 1), ((1, 181, 192), 0), ((17, 64, 64, 64, 64, 30.0), 1)])
def test_alignment_does_not_change_the_bits(gpu_ctx, dcn, torch, dims, sampler):
    gpu_ctx.set_fused_config(0, 0, sampler)
    try:
        call = Call(torch, gpu_ctx, dcn, *dims)
        assert gpu_ctx.get_fused_config(call.shape)["variant"] == TILE
        want = call.run()
        for off, msk in ((1, 0), (0, 1), (3, 5), (4, 0), (2, 2)):
            print("case: tile alignment", dims, sampler, off, msk, flush=True)
            assert np.array_equal(call.run(off, msk), want), (off, msk)
        assert np.isfinite(want.view(np.float16)).all() and want.any()
    finally:
        gpu_ctx.set_fused_config(0, 0, -1, 0)


@pytest.mark.parametrize("mt", [16, 32])
def test_pinned_tile_widths_take_any_alignment(gpu_ctx, dcn, torch, mt):
    gpu_ctx.set_fused_config(mt, 0, -1, TILE)
    try:
        call = Call(torch, gpu_ctx, dcn, 2, 19, 24)
        want = call.run()
        for off, msk in ((1, 0), (0, 3), (7, 2)):
            print("case: pinned tile alignment", mt, off, msk, flush=True)
            assert np.array_equal(call.run(off, msk), want), (off, msk)
    finally:
        gpu_ctx.set_fused_config(0, 0, -1, 0)


@pytest.mark.parametrize("mt,ks", [(1, 0), (0, 12), (1, 12), (0, 8)])
def test_pinned_narrow_settings_keep_the_narrow_kernel(gpu_ctx, dcn, torch, mt, ks):
    """The automatic variant with the narrow kernel's mt or ks pinned, at 929 to 1024 tiles: the
    narrow kernel with those settings, as at every smaller size."""
    print("case: pinned narrow settings", mt, ks, flush=True)
    call = Call(torch, gpu_ctx, dcn, 8, 64, 64)
    outs = []
    try:
        for variant in (0, dcn.VARIANT_NARROW):
            gpu_ctx.set_fused_config(mt, ks, -1, variant)
            cfg = gpu_ctx.get_fused_config(call.shape)
            assert (cfg["variant"], cfg["mt"], cfg["ks"]) == (dcn.VARIANT_NARROW, 1, ks or 12)
            outs.append(call.run())
        assert np.array_equal(outs[0], outs[1])
    finally:
        gpu_ctx.set_fused_config(0, 0, -1, 0)


def test_clock_does_not_change_the_bits(gpu_ctx, dcn, torch):
    """A clock buffer leaves choice and output as they are from 929 tiles on. Where the library
    chose the tile kernel by itself, the call goes on without stamps if the buffer is too small for
    them, up to 1024 tiles."""
    print("case: tile clock", flush=True)
    call = Call(torch, gpu_ctx, dcn, 8, 64, 64)
    want, cfg = call.run(), gpu_ctx.get_fused_config(call.shape)
    assert cfg["variant"] == TILE
    need = 4 * 8 * 64 * 64 // 128  # four per 128-pixel tile
    stamps = torch.zeros(need, dtype=torch.int64, device="cuda")
    try:
        for count in (need, need - 1, 1):
            stamps.zero_()
            gpu_ctx.set_tile_clock_dev(stamps, count)
            assert gpu_ctx.get_fused_config(call.shape) == cfg
            assert np.array_equal(call.run(), want)
            started = stamps[0::4] != 0
            assert bool(started.all()) if count == need else not bool(stamps.any())
    finally:
        gpu_ctx.set_tile_clock_dev(None)
