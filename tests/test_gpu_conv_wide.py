"""GPU tests of the large-tile body convolutions (many pixels): the same bits as the
16-pixel-tile kernels, which take every call whose CB8 tensors are not 8-byte aligned."""
from __future__ import annotations

import numpy as np
import pytest

import body_reference as br

pytestmark = pytest.mark.gpu

NCHW, CB8 = 0, 1


@pytest.fixture(scope="module")
def torch():
    import torch as t

    return t


def _dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, np.float16)).view(np.int16)).cuda()


def _placed(torch, elems, shift):
    """A zeroed device tensor of `elems` halves, `shift` halves past an aligned address."""
    return torch.zeros(elems + 8, dtype=torch.int16, device="cuda")[shift:shift + elems]


def _operand(torch, a, shift):
    t = _placed(torch, a.size, shift)
    t.copy_(_dev(torch, a.ravel()))
    return t


# Height, width: one to sixteen rows per tile by the number of tiles, with partial tiles on
# both sides and maps narrower than a tile.
SIZES = [(33, 129), (90, 91), (47, 331), (131, 133), (181, 317), (1033, 3), (5, 1500)]


@pytest.mark.parametrize("h,w", SIZES, ids=lambda v: str(v))
@pytest.mark.parametrize("acts,layouts,residuals", [((2, 0), (CB8, CB8, CB8), 1), ((1, 1), (CB8, CB8, CB8), 0),
                                                    ((2, 0), (CB8, CB8, NCHW), 2), ((0, 2), (NCHW, NCHW, NCHW), 2),
                                                    ((1, 0), (NCHW, CB8, CB8), 2)])
def test_wide_pair_same_bits(gpu_ctx, torch, h, w, acts, layouts, residuals):
    rng = np.random.default_rng(h * 1000 + w + 7 * acts[0])
    plane = h * w
    print("case: wide pair", h, w, acts, layouts, residuals, flush=True)
    f16 = lambda *s, std=1.0: br.f16(rng.normal(0, std, s))  # noqa: E731
    x = f16(64, h, w)
    x[3, h // 2, w // 2], x[9, 0, 0], x[20, h - 1, w - 1] = np.inf, np.nan, -np.inf
    convs = [gpu_ctx.conv3x3(64, 64, h, w, _dev(torch, f16(64, 64, 3, 3, std=0.04)), _dev(torch, f16(64, std=0.1)))
             for _ in range(2)]
    xd = _dev(torch, br.to_cb8(x, 64, h, w))
    res = [f16(64, h, w) for _ in range(2)]

    def run(shift):
        r = [_operand(torch, br.to_cb8(a, 64, h, w) if l == CB8 else a, shift if l == CB8 else 0) if i < residuals
             else None for i, (a, l) in enumerate(zip(res, layouts[:2]))]
        out = _placed(torch, 8 * (h + 4) * (w + 4) * 8 if layouts[2] == CB8 else 64 * plane,
                      shift if layouts[2] == CB8 else 0)
        convs[0].run_pair_dev(convs[1], xd, out, layouts[2], activation1=acts[0], activation2=acts[1], res1=r[0],
                              res1_layout=layouts[0], res2=r[1], res2_layout=layouts[1])
        torch.cuda.synchronize()
        return out.cpu().numpy().view(np.uint16).copy()

    got = run(0)
    if CB8 in layouts[:residuals] + layouts[2:]:
        want = run(1)
    else:  # no CB8 tensor to misalign: two single-conv calls with misaligned CB8 outputs
        mid, out = (_placed(torch, 8 * (h + 4) * (w + 4) * 8, 1) for _ in range(2))
        r = [_dev(torch, a) for a in res]
        convs[0].run_dev(xd, mid, CB8, activation=acts[0])
        mid2 = mid.clone()
        convs[1].run_dev(mid2, out, CB8, activation=acts[1], res1=r[0], res1_layout=NCHW, res2=r[1], res2_layout=NCHW)
        torch.cuda.synchronize()
        blocks = out.cpu().numpy().view(np.uint16).reshape(8, h + 4, w + 4, 8)[:, 2:-2, 2:-2]
        want = np.ascontiguousarray(blocks.transpose(0, 3, 1, 2)).ravel()
    for c in convs:
        c.free()
    a, b = got.view(np.float16), want.view(np.float16)
    assert np.array_equal(np.isnan(a), np.isnan(b))
    assert np.array_equal(got[~np.isnan(b)], want[~np.isnan(b)])
    assert np.isfinite(a).mean() > 0.9


# (cin, cout): each channel-block count of the kernel, whole and partial last output chunk
CHANNELS = [(64, 64), (128, 64), (192, 20), (196, 64), (256, 64), (320, 64), (61, 432)]


@pytest.mark.parametrize("cin,cout", CHANNELS, ids=lambda v: str(v))
@pytest.mark.parametrize("h,w,act,residuals,layout", [(67, 131, 1, 0, CB8), (90, 401, 2, 2, CB8), (5, 1500, 0, 1, NCHW),
                                                      (1100, 8, 1, 2, CB8)])
def test_wide_conv_same_bits(gpu_ctx, torch, cin, cout, h, w, act, residuals, layout):
    """One conv on tiles of 4 and 8 rows against the 16-pixel-tile kernel."""
    rng = np.random.default_rng(cin * 7 + cout + h)
    print("case: wide conv", cin, cout, h, w, act, residuals, layout, flush=True)
    f16 = lambda *s, std=1.0: br.f16(rng.normal(0, std, s))  # noqa: E731
    x = f16(cin, h, w)
    x[cin - 1, 0, 0], x[0, h - 1, w // 2] = np.inf, np.nan
    conv = gpu_ctx.conv3x3(cin, cout, h, w, _dev(torch, f16(cout, cin, 3, 3, std=0.04)), _dev(torch, f16(cout, std=0.1)))
    xd = _dev(torch, br.to_cb8(x, cin, h, w))
    res = [f16(cout, h, w) for _ in range(2)]
    res_l = [CB8, NCHW]
    cb = (cout + 7) // 8

    def run(shift):
        r = [_operand(torch, br.to_cb8(a, cout, h, w) if l == CB8 else a, shift if l == CB8 else 0) if i < residuals
             else None for i, (a, l) in enumerate(zip(res, res_l))]
        out = _placed(torch, cb * 8 * (h + 4) * (w + 4) if layout == CB8 else cout * h * w, shift if layout == CB8 else 0)
        conv.run_dev(xd, out, layout, activation=act, res1=r[0], res1_layout=CB8, res2=r[1], res2_layout=NCHW)
        torch.cuda.synchronize()
        return out.cpu().numpy().view(np.uint16).copy()

    got, want = run(0), run(1)
    conv.free()
    a, b = got.view(np.float16), want.view(np.float16)
    assert np.array_equal(np.isnan(a), np.isnan(b))
    assert np.array_equal(got[~np.isnan(b)], want[~np.isnan(b)])
    assert np.isfinite(a).mean() > 0.9


@pytest.mark.parametrize("cin", [64, 196])
def test_wide_conv_input_alignment(gpu_ctx, torch, cin):
    """An input 8 bytes past a 16-byte boundary (the 16-pixel kernel): the same bits."""
    h, w = 67, 131
    rng = np.random.default_rng(cin)
    print("case: conv input alignment", cin, flush=True)
    f16 = lambda *s, std=1.0: br.f16(rng.normal(0, std, s))  # noqa: E731
    x = br.to_cb8(f16(cin, h, w), cin, h, w)
    conv = gpu_ctx.conv3x3(cin, 64, h, w, _dev(torch, f16(64, cin, 3, 3, std=0.04)), _dev(torch, f16(64, std=0.1)))
    outs = []
    for shift in (0, 4):
        xd = _operand(torch, x, shift)
        out = _placed(torch, 8 * (h + 4) * (w + 4) * 8, 0)
        conv.run_dev(xd, out, CB8, activation=1)
        torch.cuda.synchronize()
        outs.append(out.cpu().numpy())
    conv.free()
    assert np.array_equal(outs[0], outs[1]) and outs[0].any()
