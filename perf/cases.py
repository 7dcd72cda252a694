"""The work that a user of dcnv2_amd has it do, as timed cases.

Each case is one deformable convolution call (``dcn_v2_conv`` on separate
offset and mask tensors, ``dcn_v2_conv_om`` on the predictor's raw output, as
``DCN.forward`` calls it), forward alone under ``no_grad`` or forward and
backward through autograd.  ``listed`` holds the layers this repository's own
workloads, training harness, benchmark and tests use; ``draw`` gives layers of
the same kinds over the whole range of sizes.
"""
from __future__ import annotations

import math

import torch

from dcnv2_amd.dcn_v2_mm import dcn_v2_conv, dcn_v2_conv_om

_DTYPE = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _case(name, B, C, H, W, Cout, k, dtype, train, stride=1, pad=None, dil=1, dg=1, wg=1,
          om=False, nhwc=False, offsets="normal:1.0"):
    return {"name": name, "B": B, "C": C, "H": H, "W": W, "Cout": Cout, "k": k, "stride": stride,
            "pad": (k // 2) * dil if pad is None else pad, "dil": dil, "dg": dg, "wg": wg,
            "dtype": dtype, "train": train, "om": om, "nhwc": nhwc, "offsets": offsets}


def listed():
    return [
        # the smallest layer of workloads.py: latency and launches count
        _case("small_fp32_fwd", 1, 16, 32, 32, 32, 3, "fp32", False),
        # the README layer of workloads.py: inference, and a training step
        _case("readme_fp16_fwd", 8, 64, 128, 128, 256, 3, "fp16", False, offsets="normal:2.0"),
        _case("readme_fp16_train", 8, 64, 128, 128, 256, 3, "fp16", True, offsets="normal:2.0"),
        # the detection neck of workloads.py: four deformable groups, bf16 training
        _case("neck_bf16_dg4_train", 16, 256, 64, 64, 256, 3, "bf16", True, dg=4,
              offsets="normal:1.5"),
        # the strided, dilated layer of workloads.py with far-reaching offsets
        _case("stress_fp16_s2_d2_train", 2, 128, 256, 256, 128, 3, "fp16", True, stride=2, dil=2,
              offsets="uniform:16.0"),
        # train.py's network (fp32, 224 x 224 images, batch 32): a first-stage 1x1 layer, the
        # 1x1 layers of its longest stage (14 x 14 maps) in both directions, and its widest
        # (7 x 7 maps)
        _case("resnet_56_fp32_1x1_train", 32, 64, 56, 56, 256, 1, "fp32", True, om=True),
        _case("resnet_14_fp32_1x1_train", 32, 1024, 14, 14, 256, 1, "fp32", True, om=True),
        _case("resnet_7_fp32_1x1_train", 32, 512, 7, 7, 2048, 1, "fp32", True, om=True),
        # a 3x3 layer in the reference's own data type
        _case("conv3x3_fp32_train", 4, 128, 56, 56, 128, 3, "fp32", True),
        # one level of a feature pyramid of 800 x 1333 images: an odd map size
        _case("pyramid_ragged_bf16_train", 2, 256, 25, 42, 256, 3, "bf16", True),
        # bench.py's weight-group layer, inference
        _case("wgroups_fp16_fwd", 8, 128, 128, 128, 256, 3, "fp16", False, wg=2),
        # serving one image with channels_last activations
        _case("serve_fp16_nhwc_fwd", 1, 256, 50, 84, 256, 3, "fp16", False, nhwc=True),
    ]


def _out_size(case):
    ext = case["dil"] * (case["k"] - 1) + 1
    return ((case["H"] + 2 * case["pad"] - ext) // case["stride"] + 1,
            (case["W"] + 2 * case["pad"] - ext) // case["stride"] + 1)


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fwd16", "train16", "train16", "resnet", "resnet", "fwd32", "train32"])
    limit = 2.4e11  # the listed detection neck's operations
    while True:
        if kind == "resnet":  # train.py's 1x1 layers: map size and widths of a stage
            hw = rng.choice([7, 14, 28, 56, _log(rng, 7, 56)])
            c = _case("", _log(rng, 1, 64), 64 * _log(rng, 1, 16), hw, hw, 64 * _log(rng, 1, 32), 1,
                      "fp32", True, om=True)
        else:
            half = kind.endswith("16")
            k = rng.choice([3, 3, 3, 1, 5] if half else [3, 3, 1])
            stride = rng.choice([1, 1, 1, 2])
            dil = rng.choice([1, 1, 2]) if k > 1 else 1
            dg = rng.choice([1, 1, 2, 4])
            wide = rng.random() < 0.7  # widths of whole 64s, as networks have them; odd ones too
            c = _case("", _log(rng, 1, 16), (64 if wide else 4) * dg * _log(rng, 1, 4 if wide else 24),
                      _log(rng, 8, 200), _log(rng, 8, 200),
                      64 * _log(rng, 1, 6) if wide else _log(rng, 16, 320), k,
                      rng.choice(["fp16", "bf16"]) if half else "fp32", kind.startswith("train"),
                      stride=stride, dil=dil, dg=dg, om=rng.random() < 0.3,
                      nhwc=half and rng.random() < 0.25,
                      offsets=rng.choice(["normal:0.5", "normal:1.0", "normal:2.0", "uniform:8.0"]))
        w = work(c)
        # fp32 operations are counted at the cost of the fp32 matrix rate
        if w["flops"] * (8 if c["dtype"] == "fp32" else 1) <= limit and w["bytes"] <= 1.2e9:
            del c["name"]
            return c


def _inputs(case, seed):
    """Values of the call, from the seed alone: activations and output gradients
    N(0, 1), weights of variance 2 / fan-in, mask logits N(0, 1), offsets in
    pixels as the case states."""
    dt = _DTYPE[case["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, C, H, W, Cout, k = (case[n] for n in ("B", "C", "H", "W", "Cout", "k"))
    kk, (Ho, Wo) = k * k, _out_size(case)

    def normal(*shape, std=1.0):
        return torch.randn(shape, generator=g, device="cuda") * std

    t = {"input": normal(B, C, H, W)}
    dist, _, arg = case["offsets"].partition(":")
    noff = 2 * case["dg"] * kk
    if dist == "normal":
        off = normal(B, noff, Ho, Wo, std=float(arg))
    else:
        off = (torch.rand((B, noff, Ho, Wo), generator=g, device="cuda") * 2 - 1) * float(arg)
    logit = normal(B, case["dg"] * kk, Ho, Wo)
    cw = C // case["wg"]
    t["weight"] = normal(Cout, cw, k, k, std=math.sqrt(2.0 / (cw * kk)))
    t["bias"] = normal(Cout, std=0.1)
    if case["om"]:
        t["om"] = torch.cat((off, logit), dim=1)
    else:
        t["offset"], t["mask"] = off, torch.sigmoid(logit)
    if case["train"]:
        t["grad_output"] = normal(B, Cout, Ho, Wo)
    t = {n: v.to(dt) for n, v in t.items()}
    if case["nhwc"]:
        for n in ("input", "grad_output"):
            if n in t:
                t[n] = t[n].contiguous(memory_format=torch.channels_last)
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    if case["train"]:
        for n, v in t.items():
            if n != "grad_output":
                v.requires_grad_(True)
    return {"case": case, "t": t}


def _forward(case, t):
    geo = (case["stride"], case["pad"], case["dil"], case["dg"])
    if case["om"]:
        return dcn_v2_conv_om(t["input"], t["weight"], t["om"], t["bias"], *geo)
    return dcn_v2_conv(t["input"], t["weight"], t["mask"], t["offset"], t["bias"], *geo)


def _leaves(case):
    return ("input", "weight", "om", "bias") if case["om"] else \
        ("input", "weight", "mask", "offset", "bias")


def run(state):
    case, t = state["case"], state["t"]
    if not case["train"]:
        with torch.no_grad():
            return {"output": _forward(case, t)}
    out = _forward(case, t)
    names = _leaves(case)
    grads = torch.autograd.grad(out, [t[n] for n in names], t["grad_output"])
    res = {"output": out.detach()}
    res.update({"grad_" + n: g for n, g in zip(names, grads)})
    return res


def work(case):
    """Every input read once and every output written once; the convolution's
    multiplications and additions, and those of its two gradient products."""
    B, C, H, W, Cout, k = (case[n] for n in ("B", "C", "H", "W", "Cout", "k"))
    Ho, Wo = _out_size(case)
    kk, esz = k * k, 4 if case["dtype"] == "fp32" else 2
    x, w, n = B * C * H * W, Cout * (C // case["wg"]) * kk, B * Cout * Ho * Wo
    om = 3 * B * case["dg"] * kk * Ho * Wo
    elems = x + w + om + Cout + n
    flops = 2.0 * n * (C // case["wg"]) * kk
    if case["train"]:  # grad_output read; the gradients of input, weight, offset, mask, bias written
        elems += n + x + w + om + Cout
        flops *= 3
    return {"bytes": float(elems * esz), "flops": flops}


def tolerance(case):
    # About four times the error seen against `exact` (fp32 7.5e-7: sums of up to a few hundred
    # thousand products in another order; fp16 2.9e-4 and bf16 2.3e-3: results and sampled
    # columns rounded once to the type).
    return {"rel": {"fp32": 5e-6, "fp16": 1.2e-3, "bf16": 1e-2}[case["dtype"]]}


def exact(case, seed):
    """The same call in 64 bits, image by image: bilinear samples with zeros
    outside the image, columns times weight, and the analytic gradients.  The
    sample positions are the operator's own (whole grid position plus offset,
    in fp32), since the offset's gradient jumps where a position crosses a
    whole number."""
    t = _inputs(case, seed)
    B, C, H, W, Cout, k = (case[n] for n in ("B", "C", "H", "W", "Cout", "k"))
    G, wg, kk, (Ho, Wo) = case["dg"], case["wg"], k * k, _out_size(case)
    N, HW, Cg = Ho * Wo, H * W, C // G
    dev, f64 = "cuda", torch.float64
    x = t["input"].to(f64).reshape(B, G, Cg, HW)
    w = t["weight"].to(f64).reshape(wg, Cout // wg, (C // wg) * kk)
    bias = t["bias"].to(f64)
    if case["om"]:
        off, logit = t["om"][:, :2 * G * kk], t["om"][:, 2 * G * kk:]
        mask = torch.sigmoid(logit.to(f64))
    else:
        off, mask = t["offset"], t["mask"].to(f64)
    off = off.float().reshape(B, G, kk, 2, N)
    mask = mask.reshape(B, G, kk * N)
    go = t["grad_output"].to(f64).reshape(B, wg, Cout // wg, N) if case["train"] else None

    tap = torch.arange(kk, device=dev)
    pix = torch.arange(N, device=dev)
    by = (pix // Wo * case["stride"] - case["pad"])[None] + (tap // k * case["dil"])[:, None]
    bx = (pix % Wo * case["stride"] - case["pad"])[None] + (tap % k * case["dil"])[:, None]

    out = torch.empty(B, Cout, N, dtype=f64, device=dev)
    gx = torch.zeros_like(x) if case["train"] else None
    gw = torch.zeros_like(w)
    goff = torch.empty(B, G, kk, 2, N, dtype=f64, device=dev) if case["train"] else None
    gmask = torch.empty(B, G, kk * N, dtype=f64, device=dev) if case["train"] else None
    for b in range(B):
        y = (by.float() + off[b, :, :, 0]).reshape(G, kk * N).to(f64)
        xx = (bx.float() + off[b, :, :, 1]).reshape(G, kk * N).to(f64)
        y0, x0 = torch.floor(y), torch.floor(xx)
        ly, lx = y - y0, xx - x0
        corners = []
        for dy, dx in ((0, 0), (0, 1), (1, 0), (1, 1)):
            cy, cx = y0 + dy, x0 + dx
            ok = (cy >= 0) & (cy < H) & (cx >= 0) & (cx < W)
            idx = torch.where(ok, cy * W + cx, torch.zeros_like(cy)).long()
            idx = idx[:, None].expand(G, Cg, kk * N)
            corners.append((idx, ok.to(f64)[:, None], torch.gather(x[b], 2, idx) * ok[:, None]))
        ly, lx = ly[:, None], lx[:, None]
        hy, hx = 1 - ly, 1 - lx
        bw = (hy * hx, hy * lx, ly * hx, ly * lx)
        val = sum(wq * v for wq, (_, _, v) in zip(bw, corners))
        m = mask[b][:, None]
        # rows of the weight are (channel, tap)
        cols = (val * m).reshape(wg, (C // wg) * kk, N)
        out[b] = torch.matmul(w, cols).reshape(Cout, N) + bias[:, None]
        if not case["train"]:
            continue
        gw += torch.matmul(go[b], cols.transpose(1, 2).contiguous())
        gcol = torch.matmul(w.transpose(1, 2).contiguous(), go[b]).reshape(G, Cg, kk * N)
        gmask[b] = (gcol * val).sum(1)
        gval = gcol * m
        v00, v01, v10, v11 = (v for _, _, v in corners)
        goff[b, :, :, 0] = (gval * (hx * (v10 - v00) + lx * (v11 - v01))).sum(1).reshape(G, kk, N)
        goff[b, :, :, 1] = (gval * (hy * (v01 - v00) + ly * (v11 - v10))).sum(1).reshape(G, kk, N)
        for wq, (idx, ok, _) in zip(bw, corners):
            gx[b].scatter_add_(2, idx, gval * wq * ok)
    res = {"output": out.reshape(B, Cout, Ho, Wo)}
    if case["train"]:
        goff = goff.reshape(B, 2 * G * kk, Ho, Wo)
        gmask = gmask.reshape(B, G * kk, Ho, Wo)
        res["grad_input"] = gx.reshape(B, C, H, W)
        res["grad_weight"] = gw.reshape(Cout, C // wg, k, k)
        if case["om"]:
            s = mask.reshape(gmask.shape)
            res["grad_om"] = torch.cat((goff, gmask * s * (1 - s)), dim=1)
        else:
            res["grad_mask"], res["grad_offset"] = gmask, goff
        res["grad_bias"] = go.sum((0, 3)).reshape(Cout)
    return res
