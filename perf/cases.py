"""What a user of this engine has it do, over the real range of sizes: the five benchmark configurations (a quantized
convolution block, the per-channel FakeQuantize operator, ResNet-50, MobileNetV2 and the BERT-base encoder) as compiled
plans behind infer requests, from one image that somebody waits for to full batches in flight, and the operator on its
own.  Networks have seeded random weights and calibrated ranges (the repository's builders); inputs come from the seed.

A case runs in one of three ways, as an application does:
  "infer"    Infer: device buffers, the call returns when the outputs are there (latency, small batches)
  "enqueue"  one inference queued on the request's own stream (throughput, requests in flight one behind the other)
  "host"     StartAsync and Wait from the request's page-locked host blobs, u8 images in (the plug-in's ordinary path)
"""
import math

import numpy as np
import torch

from dldt_amd import FakeQuantize, builders

VOCAB = 30522
HIDDEN, HEADS, FFN = 768, 12, 3072


def listed():
    return [
        # one image through FakeQuantize -> 3x3 convolution -> bias -> ReLU: the smallest plan, launches and host work
        dict(name="block_b1", kind="block", batch=1, c=64, hw=56, oc=64, how="infer"),
        # the same block in a batch, channels and map that are no multiples of a tile
        dict(name="block_b12_ragged", kind="block", batch=12, c=72, hw=45, oc=100, how="enqueue"),
        # requantization of a large activation to u8 levels, and the operator with an f32 result on odd sizes
        dict(name="fq_u8_b32", kind="fq", batch=32, c=256, h=56, w=56, form="u8"),
        dict(name="fq_f32_ragged", kind="fq", batch=3, c=67, h=61, w=47, form="f32"),
        # an image classifier that answers one request at a time
        dict(name="resnet50_b1", kind="resnet50", batch=1, res=224, how="infer"),
        # the headline: full batches in flight, input in device memory
        dict(name="resnet50_b64", kind="resnet50", batch=64, res=224, how="enqueue"),
        # a small odd batch of u8 images from host memory and back, as the asynchronous API is used
        dict(name="resnet50_b7_host", kind="resnet50", batch=7, res=256, how="host"),
        # the depthwise network: alone and in full batches
        dict(name="mobilenet_v2_b1", kind="mobilenet_v2", batch=1, res=224, how="infer"),
        dict(name="mobilenet_v2_b64", kind="mobilenet_v2", batch=64, res=224, how="enqueue"),
        # one padded text of token ids behind an attention mask that somebody waits for
        dict(name="bert_b1_s128", kind="bert", layers=12, batch=1, seq=128, tokens=True, how="infer"),
        # a few texts of the greatest length, through a smaller encoder
        dict(name="bert_b3_s512", kind="bert", layers=6, batch=3, seq=512, tokens=True, how="infer"),
        # the encoder on full batches of long sequences
        dict(name="bert_b16_s384", kind="bert", layers=12, batch=16, seq=384, tokens=False, how="enqueue"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["block", "fq", "resnet50", "mobilenet_v2", "bert"])
    if kind == "block":
        while True:
            c = dict(kind=kind, batch=_log_int(rng, 1, 32), c=_log_int(rng, 3, 256), hw=_log_int(rng, 7, 112), oc=_log_int(rng, 8, 512))
            if c["batch"] * c["hw"] ** 2 * (c["c"] + c["oc"]) <= 3e7 and c["batch"] * c["hw"] ** 2 * c["c"] * c["oc"] * 9 <= 5e10:
                return dict(c, how="infer" if c["batch"] <= 4 else "enqueue")
    if kind == "fq":
        while True:
            c = dict(kind=kind, batch=_log_int(rng, 1, 32), c=_log_int(rng, 3, 512), h=_log_int(rng, 7, 112), w=_log_int(rng, 7, 112),
                     form=rng.choice(["u8", "f32", "nhwc"]))
            if 20000 <= c["batch"] * c["c"] * c["h"] * c["w"] <= 32 * 256 * 56 * 56:
                return c
    if kind == "bert":
        c = dict(kind=kind, layers=rng.choice([2, 3, 4, 6]), batch=_log_int(rng, 1, 16), seq=rng.choice([*range(32, 385, 32), 448, 512]), tokens=rng.random() < 0.7)
        return dict(c, how="infer" if c["batch"] <= 4 else "enqueue")
    while True:
        c = dict(kind=kind, batch=_log_int(rng, 1, 64), res=32 * rng.randint(3, 8))
        if c["batch"] * c["res"] ** 2 <= 64 * 224 ** 2:
            host = rng.random() < 0.2 and kind == "resnet50"
            return dict(c, how="host" if host else "infer" if c["batch"] <= 4 else "enqueue")


# ---- a program loads a network once and keeps the plan while inputs change -----------------------------------------------
_kept = {}
MOST_PLANS = 16


def _plan(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _kept:
        while len(_kept) >= MOST_PLANS:
            del _kept[next(iter(_kept))]
        kind, batch = case["kind"], case["batch"]
        if kind == "block":
            g = builders.conv_block(n=batch, c=case["c"], hw=case["hw"], oc=case["oc"])[0]
        elif kind == "resnet50":
            g = builders.resnet50(batch=batch, res=case["res"], u8_input=case["how"] == "host")[0]
        elif kind == "mobilenet_v2":
            g = builders.mobilenet_v2(batch=batch, res=case["res"])[0]
        else:
            tokens = case["tokens"]
            g = builders.bert_encoder(layers=case["layers"], batch=batch, seq=case["seq"], vocab=VOCAB if tokens else 0, mask=tokens)[0]
        # a request that is waited for has the device to itself: the plan is tuned for one stream, else for the default
        alone = case["how"] != "enqueue"
        _kept[key] = g.compile(0, config={"HIP_THROUGHPUT_STREAMS": "1"} if alone else None)
    return _kept[key]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "fq":
        # activations around a per-channel mean; the quantization range is the channel's own +- 3 deviations
        mean = np.random.default_rng(seed).uniform(-0.5, 0.5, case["c"]).astype(np.float32)
        x = torch.randn((case["batch"], case["c"], case["h"], case["w"]), generator=gen, device="cuda")
        x += torch.from_numpy(mean).cuda().view(1, -1, 1, 1)
        low, high = (0.0, 255.0) if case["form"] != "f32" else (mean - 3, mean + 3)
        return dict(case=case, fq=FakeQuantize(case["c"], 256, mean - 3, mean + 3, low, high), x=x)
    plan = _plan(case)
    req = plan.create_request()
    if case["how"] == "host":
        ins, outs = req.host_buffers()
        ins[0].array[...] = np.random.default_rng(seed).integers(0, 256, ins[0].array.shape, dtype=np.uint8)
        return dict(case=case, req=req, ins=ins, outs=outs)
    ins, outs = req.device_buffers()
    if case["kind"] == "bert":
        if case["tokens"]:
            ins[0].copy_(torch.randint(0, VOCAB, ins[0].shape, generator=gen, device="cuda", dtype=torch.int32))
            seq = case["seq"]
            length = torch.randint(seq // 2, seq + 1, (case["batch"], 1, 1, 1), generator=gen, device="cuda")
            ins[1].copy_(torch.where(torch.arange(seq, device="cuda").view(1, 1, 1, seq) < length, 0.0, -10000.0))
        else:
            ins[0].copy_(torch.randn(ins[0].shape, generator=gen, device="cuda"))
    else:
        high = 2.55 if case["kind"] == "block" else 1.0
        ins[0].copy_(torch.rand(ins[0].shape, generator=gen, device="cuda") * high)
    return dict(case=case, req=req, ins=ins, outs=outs)


def run(state):
    case = state["case"]
    if case["kind"] == "fq":
        if case["form"] == "f32":
            return state["fq"].run_f32(state["x"])
        if case["form"] == "u8":
            return state["fq"].run_q8(state["x"], "u8", "nchw")
        return state["fq"].run_q8(state["x"], "u8b", "nhwc")
    req, ins, outs = state["req"], state["ins"], state["outs"]
    if case["how"] == "infer":
        req.infer_device(ins, outs)
    elif case["how"] == "enqueue":
        req.enqueue(ins, outs)
    else:
        req.start(ins, outs)
        req.wait()
        return [np.array(o.array) for o in outs]     # the blobs' memory goes with the request
    return outs


def _mobilenet(res):
    """(multiply-accumulates per image, weight bytes)"""
    macs = weights = 0
    hw, ic = res // 2, 32
    macs, weights = hw * hw * 32 * 27, 32 * 27
    for t, oc, n, s in builders.MOBILENETV2_BLOCKS:
        for i in range(n):
            mid = ic * t
            out = hw // (s if i == 0 else 1)
            layer = [(hw, mid * ic if t != 1 else 0), (out, mid * 9), (out, mid * oc)]
            macs += sum(p * p * w for p, w in layer)
            weights += sum(w for _, w in layer)
            hw, ic = out, oc
    macs += hw * hw * ic * 1280 + 1280 * 1000
    return macs, weights + ic * 1280 + 1280 * 1000


def work(case):
    kind, n = case["kind"], case["batch"]
    if kind == "fq":
        e = n * case["c"] * case["h"] * case["w"]
        padded = e if case["form"] != "nhwc" else n * case["h"] * case["w"] * (-(-case["c"] // 16) * 16)
        return {"bytes": 8.0 * e if case["form"] == "f32" else 4.0 * e + padded, "flops": 0.0}
    if kind == "block":
        p = n * case["hw"] ** 2
        return {"bytes": 4.0 * p * (case["c"] + case["oc"]) + 9 * case["c"] * case["oc"], "flops": 18.0 * p * case["c"] * case["oc"]}
    if kind == "bert":
        t = n * case["seq"]
        linear = case["layers"] * (4 * HIDDEN * HIDDEN + 2 * HIDDEN * FFN)
        return {"bytes": 8.0 * t * HIDDEN + linear, "flops": 2.0 * t * (linear + case["layers"] * 2 * case["seq"] * HIDDEN)}
    image = 3 * case["res"] ** 2 * (1 if case["how"] == "host" else 4)
    if kind == "resnet50":
        macs, weights = builders.resnet50_macs(case["res"]), 25.5e6
    else:
        macs, weights = _mobilenet(case["res"])
    return {"bytes": n * (image + 4000.0) + weights, "flops": 2.0 * n * macs}


def tolerance(case):
    # integer sums and a fixed order of f32 operations behind them: the same bits, whatever computes them.  The encoder's
    # Softmax, LayerNorm and GELU are f32 sums and elementary functions to rounding, so a level of a later FakeQuantize may
    # move by one where a value lies on the boundary between two (1/127 of the range, in a small share of the values)
    return {"rel": 5e-3, "max": 0.3} if case["kind"] == "bert" else "exact"
