"""GPU tests of the propagation body over many pixels: maps and batches above one workgroup
per CU, where a step runs other kernels than one 64 x 64 tile does."""
from __future__ import annotations

import numpy as np
import pytest

import body_reference as br

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t

    return t


def _dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, np.float16)).view(np.int16)).cuda()


def _host(t):
    return t.cpu().numpy().view(np.float16)


@pytest.mark.parametrize("h,w", [(5, 1), (7, 2), (1, 3), (9, 33)])
def test_temporal_prepare_narrow_maps(gpu_ctx, oracle, h, w):
    """The warps' two-column loads at the ends of rows: maps of one, two and three columns,
    flows that leave the map on every side, bit for bit the oracle's."""
    rng = np.random.default_rng(h * 10 + w)
    print("case: temporal prepare", h, w, flush=True)
    x = br.body_inputs(rng, h, w, flow_px=float(max(h, w)) + 2)
    x["flow1"][::5] = np.round(x["flow1"][::5])
    ref = oracle.temporal_prepare_f16(w, h, True, x["feat_prop"], x["feat_current"], x["feat_n2"], x["flow1"],
                                      x["prev_flow"])
    got = gpu_ctx.temporal_prepare_f16(w, h, x["feat_prop"], x["feat_current"], x["feat_n2"], x["flow1"],
                                       x["prev_flow"], True)
    for a, b in zip((got["flow2"], got["conditions"], got["deform_input"]), ref):
        assert np.array_equal(a.view(np.uint16), b.view(np.uint16))


def _step(torch, ctx, wd, x, h, w, branch, blocks, tiles=1, cb8=False):
    plane = h * w
    body = ctx.body(h, w, wd, branch=branch, blocks=blocks, tiles=tiles)
    d = {k: _dev(torch, v) for k, v in x.items() if k != "prefix"}
    prefix = [_dev(torch, p) for p in x["prefix"]] or None
    flow2 = torch.zeros(tiles * 2 * plane, dtype=torch.int16, device="cuda")
    out = torch.zeros(tiles * 64 * plane, dtype=torch.int16, device="cuda")
    if cb8:
        mirror = torch.zeros(8 * (h + 4) * (w + 4) * 8, dtype=torch.int16, device="cuda")
        prop, n2 = (_dev(torch, br.to_cb8(x[k], 64, h, w)) for k in ("feat_prop", "feat_n2"))
        body.step_cb8_dev(d["feat_current"], d["flow1"], d["prev_flow"], prop, n2, flow2, out, mirror, True, prefix)
        torch.cuda.synchronize()
        assert np.array_equal(mirror.cpu().numpy().ravel(), br.to_cb8(_host(out), 64, h, w).view(np.int16).ravel())
    else:
        body.step_dev(d["feat_current"], d["flow1"], d["prev_flow"], d["feat_prop"], d["feat_n2"], flow2, out, True,
                      prefix)
        torch.cuda.synchronize()
    body.free()
    return _host(flow2).copy(), _host(out).copy()


@pytest.mark.parametrize("h,w,branch", [(41, 110, 0), (70, 131, 2), (91, 150, 1)])
def test_large_map_step(gpu_ctx, torch, h, w, branch):
    """One map above 256 tiles of 2 x 8 pixels, two to four 16-pixel tiles per workgroup of the
    alignment: the oracle chain's tolerance, and the CB8 step's bits."""
    rng = np.random.default_rng(h + w)
    weights = br.body_weights(rng, branch, 1)
    x = br.body_inputs(rng, h, w, branch)
    wd = {k: _dev(torch, v) for k, v in weights.items()}
    print("case: large map step", h, w, branch, flush=True)
    flow2, out = _step(torch, gpu_ctx, wd, x, h, w, branch, 1)
    flow2_cb8, out_cb8 = _step(torch, gpu_ctx, wd, x, h, w, branch, 1, cb8=True)
    assert np.array_equal(out.view(np.uint16), out_cb8.view(np.uint16))
    assert np.array_equal(flow2.view(np.uint16), flow2_cb8.view(np.uint16))
    ref2, ref, _ = br.body_step(weights, x, h, w, 1)
    assert np.array_equal(flow2.view(np.uint16), ref2.view(np.uint16))
    err = np.abs(out.astype(np.float64) - ref.astype(np.float64))
    assert err.max() <= 2e-2 and err.mean() <= 1e-3


@pytest.mark.parametrize("h,w,tiles", [(21, 35, 3), (48, 50, 5), (40, 50, 7)])
def test_batched_step_equals_single_steps(gpu_ctx, torch, h, w, tiles):
    """One to four tiles per workgroup, workgroups of several images on each XCD: the same
    bits as every image alone."""
    rng = np.random.default_rng(tiles)
    weights = br.body_weights(rng, 0, 1)
    wd = {k: _dev(torch, v) for k, v in weights.items()}
    images = [br.body_inputs(rng, h, w, 0) for _ in range(tiles)]
    print("case: batched step", h, w, tiles, flush=True)
    batch = {k: np.concatenate([i[k] for i in images]) for k in images[0] if k != "prefix"}
    batch["prefix"] = []
    flow2, out = _step(torch, gpu_ctx, wd, batch, h, w, 0, 1, tiles=tiles)
    for t, x in enumerate(images):
        f, o = _step(torch, gpu_ctx, wd, x, h, w, 0, 1)
        assert np.array_equal(flow2.reshape(tiles, -1)[t].view(np.uint16), f.view(np.uint16)), t
        assert np.array_equal(out.reshape(tiles, -1)[t].view(np.uint16), o.view(np.uint16)), t
