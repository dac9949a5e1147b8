"""Workloads that this library's speed is measured on, each through the public Python entry
points (jasnamacos_amd.deform_conv).

The framework's work is BasicVSR++ second-order propagation: the modulated deformable
convolution of its alignment (128 -> 64 channels, 3 x 3, 16 offset groups), the propagation
body around it, the four-branch clip that runs the body over a video tile, and the SPyNet
flows that feed it. The operator is called on its own too, in FP16, BF16 and FP32 and with
plain (unpacked) weights. Sizes are those of the benchmark configurations (64 x 64 tiles, 16
tiles, a 180 x 320 map, 30-frame clips) and ragged ones around them.

Every case is a dict: "kind" says which entry point, the rest its sizes.
  dcn     forward_f16_prepacked_dev / forward_bf16_prepacked_dev, weights packed once
  direct  forward_f32_dev / forward_f16_dev: plain OIHW weights, any shape
  pair    Conv3x3.run_pair_dev: a residual block of the backbone
  body    one captured propagation step (the aligned feature and the backbone)
  clip    one captured four-branch clip
  spynet  every first-order flow of a clip
"""
import math

import torch

from jasnamacos_amd import deform_conv as dc

_KEEP = {}


def _context():
    """The one context a program keeps on its device."""
    if "ctx" not in _KEEP:
        _KEEP["ctx"] = dc.HipDeformConv(0)
    return _KEEP["ctx"]


# ---- the cases -------------------------------------------------------------------------

def _dcn(name, dtype, batch, height, width, flow, cin=128, cout=64, groups=16):
    case = {"kind": "dcn", "dtype": dtype, "batch": batch, "height": height, "width": width, "flow": flow,
            "cin": cin, "cout": cout, "offset_groups": groups}
    return dict(case, name=name) if name else case


def _direct(name, dtype, batch, height, width, cin=128, cout=64, groups=1, offset_groups=16, stride=1, flow=6.0):
    case = {"kind": "direct", "dtype": dtype, "batch": batch, "height": height, "width": width, "cin": cin,
            "cout": cout, "groups": groups, "offset_groups": offset_groups, "stride": stride, "flow": flow}
    return dict(case, name=name) if name else case


def _body(name, tiles, height, width, branch):
    case = {"kind": "body", "tiles": tiles, "height": height, "width": width, "branch": branch, "blocks": 5}
    return dict(case, name=name) if name else case


def listed():
    return [
        # The alignment layer on a small odd crop: launches and latency.
        _dcn("dcn_crop_f16", "f16", 1, 23, 37, 6.0),
        # The reference's own benchmark of the operator: one 64 x 64 tile.
        _dcn("dcn_tile_f16", "f16", 1, 64, 64, 6.0),
        # A frame's tiles in one call.
        _dcn("dcn_tiles16_f16", "f16", 16, 64, 64, 12.0),
        # A whole quarter-scale 720p map with large motion.
        _dcn("dcn_map_f16", "f16", 1, 180, 320, 32.0),
        # The same layer in a BF16 model.
        _dcn("dcn_tiles16_bf16", "bf16", 16, 64, 64, 12.0),
        # runFloat32: the operator in FP32, bit-identical to the CPU definition.
        _direct("dcn_tile_f32", "f32", 1, 64, 64),
        # FP16 with plain weights, an odd size: a caller that does not prepack.
        _direct("dcn_plain_f16", "f16", 2, 45, 61),
        # One residual block of the backbone on a whole map.
        {"kind": "pair", "height": 180, "width": 320, "name": "block_map"},
        # One propagation step of one tile: latency-bound, replayed per frame.
        _body("body_tile", 1, 64, 64, 0),
        # One propagation step of a frame's tiles at once.
        _body("body_tiles16", 16, 64, 64, 3),
        # A short window of one tile through all four branches.
        {"kind": "clip", "frames": 10, "tiles": 1, "height": 64, "width": 64, "blocks": 5, "name": "clip_tile"},
        # All first-order flows of a 30-frame clip.
        {"kind": "spynet", "frames": 30, "height": 64, "width": 64, "name": "flows_clip30"},
    ]


def _log(rng, low, high):
    """A whole number spread over low..high by its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["dcn", "dcn", "dcn", "dcn", "direct", "direct", "pair", "body", "body", "clip", "spynet"])
    if kind == "dcn":
        pixels = _log(rng, 600, 65536)
        height = rng.randint(16, 181)
        batch = max(1, min(16, round(pixels / (height * height * rng.uniform(0.8, 2.0)))))
        width = max(16, min(321, pixels // (batch * height)))
        cin, cout, groups = rng.choice([(128, 64, 16), (128, 64, 16), (128, 64, 16), (64, 64, 8)])
        return _dcn(None, rng.choice(["f16", "f16", "bf16"]), batch, height, width,
                    round(rng.uniform(2.0, 32.0), 1), cin, cout, groups)
    if kind == "direct":
        dtype = rng.choice(["f32", "f16"])
        pixels = _log(rng, 500, 8192)
        height = rng.randint(12, 91)
        width = max(12, min(160, pixels // height))
        if rng.random() < 0.7:  # the alignment layer
            return _direct(None, dtype, 1, height, width, flow=round(rng.uniform(1.0, 16.0), 1))
        groups = rng.choice([1, 2, 4])  # some other deformable layer
        cin = groups * 4 * rng.randint(2, 12)
        return _direct(None, dtype, rng.randint(1, 3), height, width, cin, groups * rng.randint(3, 24), groups,
                       rng.choice([1, 2, 4]), rng.choice([1, 2]), round(rng.uniform(1.0, 8.0), 1))
    if kind == "pair":
        pixels = _log(rng, 1000, 57600)
        height = rng.randint(24, 180)
        return {"kind": "pair", "height": height, "width": max(16, min(320, pixels // height))}
    if kind == "body":
        tiles = _log(rng, 1, 16)
        side = rng.randint(32, 64) if tiles > 1 else rng.randint(32, 160)
        return _body(None, tiles, side, rng.randint(32, 64) if tiles > 1 else rng.randint(32, 160), rng.randint(0, 3))
    if kind == "clip":
        return {"kind": "clip", "frames": rng.randint(3, 9), "tiles": rng.choice([1, 1, 2, 3]),
                "height": rng.randint(32, 64), "width": rng.randint(32, 64), "blocks": 5}
    return {"kind": "spynet", "frames": rng.randint(2, 30), "height": 32 * rng.randint(1, 2),
            "width": 32 * rng.randint(1, 2)}


# ---- inputs ----------------------------------------------------------------------------

_DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


class _Random:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def normal(self, *size, std=1.0):
        return torch.randn(size, generator=self.gen, device="cuda") * std

    def uniform(self, *size, bound=1.0):
        return (torch.rand(size, generator=self.gen, device="cuda") * 2 - 1) * bound

    def smooth(self, images, height, width, bound):
        """[images][2][height][width]: an 8 x 8 grid of U(-bound, bound), bilinearly upsampled."""
        grid = self.uniform(images, 2, 8, 8, bound=bound)
        return torch.nn.functional.interpolate(grid, size=(height, width), mode="bilinear", align_corners=True)


def _out_size(case):
    stride = case.get("stride", 1)
    return (case["height"] - 1) // stride + 1, (case["width"] - 1) // stride + 1


def _shape(case):
    stride = case.get("stride", 1)
    ho, wo = _out_size(case)
    return dc.DeformConvShape(case["batch"], case["cin"], case["height"], case["width"], case["cout"], ho, wo, 3, 3,
                              1, 1, stride, stride, 1, 1, case.get("groups", 1), case["offset_groups"])


def _dcn_inputs(case, seed):
    """x ~ N(0, 1); He-uniform weights; offsets 10 tanh(N(0, 1)) around a smooth flow (dy, dx);
    masks sigmoid(N(0, 1)), as conv_offset and its transform give them."""
    r = _Random(seed)
    dtype = _DTYPE[case["dtype"]]
    b, cin, cout, og = case["batch"], case["cin"], case["cout"], case["offset_groups"]
    ho, wo = _out_size(case)
    fan_in = cin // case.get("groups", 1) * 9
    x = r.normal(b, cin, case["height"], case["width"])
    residue = 10 * torch.tanh(r.normal(b, og * 9, 2, ho, wo))
    offset = residue + r.smooth(b, ho, wo, case["flow"])[:, None]
    mask = torch.sigmoid(r.normal(b, og * 9, ho, wo))
    weight = r.uniform(cout, cin // case.get("groups", 1), 3, 3, bound=math.sqrt(6 / fan_in))
    bias = r.uniform(cout, bound=0.1)
    return [t.to(dtype).contiguous() for t in (x, offset, mask, weight, bias)]


_OFFSET_LAYERS = [(196, 64), (64, 64), (64, 64), (64, 432)]


def _body_weights(r, branch, blocks):
    w = {}

    def conv(name, cin, cout):
        w[name.replace("#", "w")] = r.normal(cout, cin, 3, 3, std=0.02).half()
        w[name.replace("#", "b")] = r.normal(cout, std=0.02).half()

    for i, (cin, cout) in enumerate(_OFFSET_LAYERS):
        conv("offset_#%d" % i, cin, cout)
    conv("dcn_#", 128, 64)
    for i in range(1 + 2 * blocks):
        conv("backbone_#%d" % i, 64 * (branch + 2) if i == 0 else 64, 64)
    return w


def _body_inputs(case, seed):
    """A step's features ~ N(0, 1) and smooth flows of up to 4 px, weights ~ N(0, 0.02)."""
    r = _Random(seed)
    t, h, w = case["tiles"], case["height"], case["width"]
    d = {"weights": _body_weights(r, case["branch"], case["blocks"])}
    for name in ("feat_current", "feat_prop", "feat_n2"):
        d[name] = r.normal(t, 64, h, w).half()
    for name in ("flow1", "prev_flow"):
        d[name] = r.smooth(t, h, w, 4.0).half().contiguous()
    d["prefix"] = [r.normal(t, 64, h, w).half() for _ in range(case["branch"])]
    return d


def _clip_inputs(case, seed):
    r = _Random(seed)
    n, t, h, w = case["frames"], case["tiles"], case["height"], case["width"]
    return {
        "weights": [_body_weights(r, b, case["blocks"]) for b in range(4)],
        "spatial": r.normal(n, t, 64, h, w).half(),
        "backward": r.smooth((n - 1) * t, h, w, 4.0).half().reshape(n - 1, t, 2, h, w).contiguous(),
        "forward": r.smooth((n - 1) * t, h, w, 4.0).half().reshape(n - 1, t, 2, h, w).contiguous(),
    }


_PAIR_STD = 0.04


def _pair_inputs(case, seed):
    r = _Random(seed)
    h, w = case["height"], case["width"]
    return {"x": r.normal(64, h, w).half(),
            "weight": [r.normal(64, 64, 3, 3, std=_PAIR_STD).half() for _ in range(2)],
            "bias": [r.normal(64, std=0.02).half() for _ in range(2)]}


_SPYNET_LAYERS = [(8, 32), (32, 64), (64, 32), (32, 16), (16, 2)]


def _spynet_inputs(case, seed):
    """Frames in [0, 1] of drifting sinusoids; He-normal 7 x 7 weights, a small flow layer."""
    r = _Random(seed)
    n, h, w = case["frames"], case["height"], case["width"]
    y = torch.arange(h, device="cuda", dtype=torch.float32)[:, None]
    x = torch.arange(w, device="cuda", dtype=torch.float32)[None, :]
    step = torch.arange(n, device="cuda", dtype=torch.float32)[:, None, None, None, None]
    waves = 6
    freq = r.uniform(2, 3, waves, 1, 1, bound=0.3)
    amp = r.uniform(3, waves, 1, 1).abs()
    phase = r.uniform(3, waves, 1, 1, bound=math.pi)
    drift = r.uniform(2, 1, 1, 1, 1, bound=1.5)
    value = torch.sin(freq[0] * (y + drift[0] * step) + freq[1] * (x + drift[1] * step) + phase) * amp
    frames = (0.5 + 0.1 * value.sum(2)).clamp(0, 1).half().contiguous()
    weights = {}
    for level in range(6):
        for i, (cin, cout) in enumerate(_SPYNET_LAYERS):
            std = 0.04 if i == 4 else math.sqrt(2 / (cin * 49))
            weights["w%d_%d" % (level, i)] = r.normal(cout, cin, 7, 7, std=std).half()
            weights["b%d_%d" % (level, i)] = r.normal(cout, std=0.01).half()
    return {"frames": frames, "weights": weights}


# ---- what a program has in hand, and one pass -------------------------------------------

def prepare(case, seed):
    ctx = _context()
    kind = case["kind"]
    stream = torch.cuda.current_stream()
    if kind in ("dcn", "direct"):
        x, offset, mask, weight, bias = _dcn_inputs(case, seed)
        shape = _shape(case)
        out = torch.empty(case["batch"], case["cout"], *_out_size(case), dtype=x.dtype, device="cuda")
        state = {"kind": kind, "dtype": case["dtype"], "ctx": ctx, "shape": shape, "x": x, "offset": offset,
                 "mask": mask, "weight": weight, "bias": bias, "out": out, "stream": stream}
        if kind == "dcn":
            pack = ctx.prepack_bf16_dev if case["dtype"] == "bf16" else ctx.prepack_dev
            state["packed"] = pack(shape, weight, bias, stream=stream)
            ctx.reserve(shape)
        return state
    if kind == "pair":
        d = _pair_inputs(case, seed)
        h, w = case["height"], case["width"]
        cb8 = torch.zeros(8, h + 4, w + 4, 8, dtype=torch.float16, device="cuda")
        cb8[:, 2:2 + h, 2:2 + w] = d["x"].reshape(8, 8, h, w).permute(0, 2, 3, 1)
        convs = [ctx.conv3x3(64, 64, h, w, d["weight"][i], d["bias"][i], stream=stream) for i in range(2)]
        return {"kind": kind, "x": cb8, "convs": convs, "keep": d, "out": torch.zeros_like(cb8), "stream": stream}
    if kind == "body":
        d = _body_inputs(case, seed)
        t, h, w = case["tiles"], case["height"], case["width"]
        body = ctx.body(h, w, d["weights"], branch=case["branch"], blocks=case["blocks"], stream=stream, tiles=t)
        flow2 = torch.empty(t, 2, h, w, dtype=torch.float16, device="cuda")
        out = torch.empty(t, 64, h, w, dtype=torch.float16, device="cuda")
        graph = body.capture(d["feat_current"], d["flow1"], d["prev_flow"], d["feat_prop"], d["feat_n2"], flow2, out,
                             True, d["prefix"] or None)
        return {"kind": kind, "graph": graph, "body": body, "keep": d, "flow2": flow2, "out": out, "stream": stream}
    if kind == "clip":
        d = _clip_inputs(case, seed)
        n, t, h, w = case["frames"], case["tiles"], case["height"], case["width"]
        clip = ctx.clip(h, w, n, d["weights"], blocks=case["blocks"], stream=stream, tiles=t)
        out = torch.empty(4, n, t, 64, h, w, dtype=torch.float16, device="cuda")
        graph = clip.capture(d["spatial"], d["backward"], d["forward"], out)
        return {"kind": kind, "graph": graph, "clip": clip, "keep": d, "out": out, "stream": stream}
    d = _spynet_inputs(case, seed)
    n, h, w = case["frames"], case["height"], case["width"]
    net = ctx.spynet(h, w, d["weights"], max_frames=n, stream=stream)
    return {"kind": kind, "net": net, "frames": d["frames"], "count": n, "stream": stream,
            "out": torch.empty(2, n - 1, 2, h, w, dtype=torch.float16, device="cuda")}


def run(state):
    s = state
    kind, out, stream = s["kind"], s["out"], s["stream"]
    if kind == "dcn":
        call = s["ctx"].forward_bf16_prepacked_dev if s["dtype"] == "bf16" else s["ctx"].forward_f16_prepacked_dev
        call(s["shape"], s["x"], s["offset"], s["mask"], s["packed"], out, stream=stream)
        return out
    if kind == "direct":
        call = s["ctx"].forward_f32_dev if s["dtype"] == "f32" else s["ctx"].forward_f16_dev
        call(s["shape"], s["x"], s["offset"], s["mask"], s["weight"], s["bias"], out, stream=stream)
        return out
    if kind == "pair":
        s["convs"][0].run_pair_dev(s["convs"][1], s["x"], out, dc.TENSOR_CB8, activation1=2, activation2=0,
                                   res1=s["x"], res1_layout=dc.TENSOR_CB8, stream=stream)
        return out
    if kind == "body":
        s["graph"].launch(stream)
        return {"feat_prop": out, "flow2": s["flow2"]}
    if kind == "clip":
        s["graph"].launch(stream)
        return out
    s["net"].clip_flows_dev(s["frames"], s["count"], out, stream=stream)
    return out


# ---- what a pass cannot do without --------------------------------------------------------

def _conv_flops(pixels, cin, cout, taps):
    return 2.0 * pixels * cin * cout * taps


def _body_work(tiles, plane, branch, blocks, step=True):
    """Bytes and flops of one step (or, without `step`, of a branch's first step)."""
    px = tiles * plane
    layers = [(64 * (branch + 2), 64)] + [(64, 64)] * (2 * blocks)
    features = 1 + branch + 1  # feat_current, prefix; the output
    flows = 0
    if step:
        layers = layers + _OFFSET_LAYERS + [(128, 64)]
        features += 2  # feat_prop, feat_n2
        flows = 6  # flow1, prev_flow, flow2
    flops = sum(_conv_flops(px, cin, cout, 9) for cin, cout in layers)
    weights = sum((cin * 9 + 1) * cout * 2 for cin, cout in layers)
    return (features * 64 + flows) * px * 2.0 + weights, flops


def work(case):
    kind = case["kind"]
    if kind in ("dcn", "direct"):
        b, cin, cout, og = case["batch"], case["cin"], case["cout"], case["offset_groups"]
        ho, wo = _out_size(case)
        per_group = cin // case.get("groups", 1)
        values = (b * cin * case["height"] * case["width"] + b * og * 27 * ho * wo + b * cout * ho * wo
                  + cout * per_group * 9 + cout)
        return {"bytes": float(values * (4 if case["dtype"] == "f32" else 2)),
                "flops": _conv_flops(b * ho * wo, per_group, cout, 9)}
    plane = case["height"] * case["width"]
    if kind == "pair":
        return {"bytes": 2.0 * (2 * 64 * plane + 2 * 64 * (64 * 9 + 1)), "flops": 2 * _conv_flops(plane, 64, 64, 9)}
    if kind == "body":
        nbytes, flops = _body_work(case["tiles"], plane, case["branch"], case["blocks"])
        return {"bytes": nbytes, "flops": flops}
    if kind == "clip":
        n, t = case["frames"], case["tiles"]
        steps = [_body_work(t, plane, b, case["blocks"], i > 0) for b in range(4) for i in range(n)]
        # Inputs once (features, both directions' flows, weights) and every propagated feature once.
        weights = sum(_body_work(0, plane, b, case["blocks"])[0] for b in range(4))
        return {"bytes": 2.0 * t * plane * (64 * n + 4 * (n - 1) + 4 * 64 * n) + weights,
                "flops": sum(f for _, f in steps)}
    pairs = 2 * (case["frames"] - 1)
    flops = sum(_conv_flops(pairs * (case["height"] >> i) * (case["width"] >> i), cin, cout, 49)
                for i in range(6) for cin, cout in _SPYNET_LAYERS)
    weights = 6 * sum((cin * 49 + 1) * cout * 2 for cin, cout in _SPYNET_LAYERS)
    return {"bytes": 2.0 * plane * (3 * case["frames"] + 2 * pairs) + weights, "flops": flops}


# ---- how far another correct implementation may be off ------------------------------------

# About four times what each path was measured to be off its FP64 result (FP16 DCN 4.4e-4,
# BF16 2.3e-3, FP32 2.2e-6, plain FP16 2.1e-4, a block 2.4e-4, a step 9.2e-4, a clip 6.6e-4,
# flows 6.8e-4).
_TOLERANCE = {
    "dcn f16": {"rel": 2e-3},
    "dcn bf16": {"rel": 1e-2},
    "direct f32": {"rel": 1e-5},
    "direct f16": {"rel": 1e-3},
    "pair": {"rel": 1e-3},
    "body": {"rel": 4e-3},
    "clip": {"rel": 4e-3},
    "spynet": {"rel": 4e-3},
}


def tolerance(case):
    key = case["kind"] + (" " + case["dtype"] if "dtype" in case else "")
    return dict(_TOLERANCE[key])


# ---- the same results in 64 bits ---------------------------------------------------------

def _sample_zero(x, y, xx):
    """Bilinear samples with zeros outside: x [N][C][H][W] at y, xx [N][P] -> [N][C][P]."""
    n, c, h, w = x.shape
    flat = x.reshape(n, c, h * w)
    y0, x0 = torch.floor(y), torch.floor(xx)
    ly, lx = y - y0, xx - x0
    total = 0
    for dy, wy in ((0, 1 - ly), (1, ly)):
        for dx, wx in ((0, 1 - lx), (1, lx)):
            yi, xi = y0 + dy, x0 + dx
            inside = (yi >= 0) & (yi < h) & (xi >= 0) & (xi < w)
            index = (yi.clamp(0, h - 1) * w + xi.clamp(0, w - 1)).long()
            value = torch.gather(flat, 2, index[:, None].expand(n, c, index.shape[1]))
            total = total + value * (wy * wx * inside)[:, None]
    return total


def _deform(x, offset, mask, weight, bias, offset_groups, groups=1, stride=1):
    """The operator over FP64 tensors, 3 x 3 taps, padding 1."""
    b, cin, h, w = x.shape
    ho, wo = mask.shape[-2:]
    cout = weight.shape[0]
    dev = x.device
    offset = offset.reshape(b, offset_groups, 9, 2, ho * wo)
    mask = mask.reshape(b, offset_groups, 9, ho * wo)
    oy = (torch.arange(ho, device=dev, dtype=x.dtype) * stride - 1).repeat_interleave(wo)
    ox = (torch.arange(wo, device=dev, dtype=x.dtype) * stride - 1).repeat(ho)
    planes = x.reshape(b * offset_groups, cin // offset_groups, h, w)
    out = torch.zeros(b, groups, cout // groups, ho * wo, device=dev, dtype=x.dtype)
    for k in range(9):
        y = (oy + k // 3 + offset[:, :, k, 0]).reshape(b * offset_groups, -1)
        xx = (ox + k % 3 + offset[:, :, k, 1]).reshape(b * offset_groups, -1)
        s = _sample_zero(planes, y, xx) * mask[:, :, k].reshape(b * offset_groups, 1, -1)
        s = s.reshape(b, groups, cin // groups, ho * wo)
        wk = weight[:, :, k // 3, k % 3].reshape(groups, cout // groups, cin // groups)
        for g in range(groups):
            out[:, g] += torch.matmul(wk[g], s[:, g])
    return out.reshape(b, cout, ho, wo) + bias[None, :, None, None]


def _conv(x, weight, bias):
    """k x k convolution with zero padding k / 2 over FP64 tensors [N][C][H][W]."""
    n, c, h, w = x.shape
    k = weight.shape[-1]
    padded = torch.nn.functional.pad(x, (k // 2,) * 4)
    out = torch.zeros(n, weight.shape[0], h * w, device=x.device, dtype=x.dtype)
    for ky in range(k):
        for kx in range(k):
            out += torch.matmul(weight[:, :, ky, kx], padded[:, :, ky:ky + h, kx:kx + w].reshape(n, c, h * w))
    return out.reshape(n, -1, h, w) + bias[None, :, None, None]


def _grid(h, w, dev):
    y, x = torch.meshgrid(torch.arange(h, device=dev, dtype=torch.float64),
                          torch.arange(w, device=dev, dtype=torch.float64), indexing="ij")
    return y.reshape(1, -1), x.reshape(1, -1)


def _warp_zero(x, flow):
    n, c, h, w = x.shape
    y, xx = _grid(h, w, x.device)
    return _sample_zero(x, y + flow[:, 1].reshape(n, -1), xx + flow[:, 0].reshape(n, -1)).reshape(n, c, h, w)


def _leaky(x):
    return torch.where(x < 0, 0.1 * x, x)


def _backbone(w, x, blocks):
    f = _leaky(_conv(x, w["backbone_w0"], w["backbone_b0"]))
    for i in range(blocks):
        t = torch.relu(_conv(f, w["backbone_w%d" % (1 + 2 * i)], w["backbone_b%d" % (1 + 2 * i)]))
        f = f + _conv(t, w["backbone_w%d" % (2 + 2 * i)], w["backbone_b%d" % (2 + 2 * i)])
    return f


def _step(w, feat_current, flow1, prev_flow, feat_prop, feat_n2, prefix, blocks, second_order):
    flow2 = flow1 + _warp_zero(prev_flow, flow1) if second_order else torch.zeros_like(flow1)
    h = torch.cat([_warp_zero(feat_prop, flow1), feat_current, _warp_zero(feat_n2, flow2), flow1, flow2], 1)
    for i in range(3):
        h = _leaky(_conv(h, w["offset_w%d" % i], w["offset_b%d" % i]))
    raw = _conv(h, w["offset_w3"], w["offset_b3"])
    yx1, yx2 = flow1.flip(1).repeat(1, 72, 1, 1), flow2.flip(1).repeat(1, 72, 1, 1)
    offset = 10 * torch.tanh(raw[:, :288]) + torch.cat([yx1, yx2], 1)
    mask = torch.sigmoid(raw[:, 288:])
    aligned = _deform(torch.cat([feat_prop, feat_n2], 1), offset, mask, w["dcn_w"], w["dcn_b"], 16)
    out = aligned + _backbone(w, torch.cat([feat_current, *prefix, aligned], 1), blocks)
    return flow2, out


def _doubles(v):
    if isinstance(v, dict):
        return {k: _doubles(x) for k, x in v.items()}
    if isinstance(v, list):
        return [_doubles(x) for x in v]
    return v.double()


def _exact_clip(case, seed):
    d = _doubles(_clip_inputs(case, seed))
    n, t, h, w, blocks = case["frames"], case["tiles"], case["height"], case["width"], case["blocks"]
    out = torch.zeros(4, n, t, 64, h, w, device="cuda", dtype=torch.float64)
    zero = torch.zeros(t, 64, h, w, device="cuda", dtype=torch.float64)
    for b in range(4):
        backward = b % 2 == 0
        flows = d["backward" if backward else "forward"]
        order = list(range(n))[::-1] if backward else list(range(n))
        for i, f in enumerate(order):
            prefix = [out[k, f] for k in range(b)]
            if i == 0:
                out[b, f] = _backbone(d["weights"][b], torch.cat([d["spatial"][f], *prefix, zero], 1), blocks)
                continue
            flow1 = flows[f if backward else f - 1]
            prev_frame = order[i - 1]
            prev_flow = flows[prev_frame if backward else prev_frame - 1] if i > 1 else flow1
            n2 = out[b, order[i - 2]] if i > 1 else zero
            out[b, f] = _step(d["weights"][b], d["spatial"][f], flow1, prev_flow, out[b, prev_frame], n2, prefix,
                              blocks, i > 1)[1]
    return out


def _sample_border(x, y, xx):
    h, w = x.shape[-2:]
    return _sample_zero(x, y.clamp(0, h - 1), xx.clamp(0, w - 1))


def _exact_spynet(case, seed):
    d = _doubles(_spynet_inputs(case, seed))
    w, n = d["weights"], case["frames"]
    dev = d["frames"].device
    mean = torch.tensor([0.485, 0.456, 0.406], device=dev, dtype=torch.float64)[None, :, None, None]
    std = torch.tensor([0.229, 0.224, 0.225], device=dev, dtype=torch.float64)[None, :, None, None]
    levels = [(d["frames"] - mean) / std]
    for _ in range(5):
        f = levels[0]
        levels.insert(0, f.reshape(n, 3, f.shape[2] // 2, 2, f.shape[3] // 2, 2).mean((3, 5)))
    images = 2 * (n - 1)
    flow = torch.zeros(images, 2, 1, 1, device=dev, dtype=torch.float64)
    for level in range(6):
        f = levels[level]
        h, wd = f.shape[-2:]
        reference, support = torch.cat([f[:-1], f[1:]]), torch.cat([f[1:], f[:-1]])
        y, x = _grid(h, wd, dev)
        if level == 0:
            flow = torch.zeros(images, 2, h, wd, device=dev, dtype=torch.float64)
        else:
            sh, sw = flow.shape[-2:]
            flow = 2 * _sample_border(flow, (y * (sh - 1) / max(h - 1, 1)).expand(images, -1),
                                      (x * (sw - 1) / max(wd - 1, 1)).expand(images, -1)).reshape(images, 2, h, wd)
        warped = _sample_border(support, y + flow[:, 1].reshape(images, -1), x + flow[:, 0].reshape(images, -1))
        z = torch.cat([reference, warped.reshape(images, 3, h, wd), flow], 1)
        for i in range(5):
            z = _conv(z, w["w%d_%d" % (level, i)], w["b%d_%d" % (level, i)])
            if i < 4:
                z = torch.relu(z)
        flow = flow + z
    return flow.reshape(2, n - 1, 2, case["height"], case["width"])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("dcn", "direct"):
        x, offset, mask, weight, bias = _doubles(_dcn_inputs(case, seed))
        return _deform(x, offset, mask, weight, bias, case["offset_groups"], case.get("groups", 1),
                       case.get("stride", 1))
    if kind == "pair":
        d = _doubles(_pair_inputs(case, seed))
        x, h, w = d["x"][None], case["height"], case["width"]
        t = torch.relu(_conv(x, d["weight"][0], d["bias"][0]))
        y = x + _conv(t, d["weight"][1], d["bias"][1])
        out = torch.zeros(8, h + 4, w + 4, 8, device="cuda", dtype=torch.float64)
        out[:, 2:2 + h, 2:2 + w] = y.reshape(8, 8, h, w).permute(0, 2, 3, 1)
        return out
    if kind == "body":
        d = _doubles(_body_inputs(case, seed))
        flow2, out = _step(d["weights"], d["feat_current"], d["flow1"], d["prev_flow"], d["feat_prop"], d["feat_n2"],
                           d["prefix"], case["blocks"], True)
        return {"feat_prop": out, "flow2": flow2}
    if kind == "clip":
        return _exact_clip(case, seed)
    return _exact_spynet(case, seed)
