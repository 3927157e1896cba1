"""A convolution and the depthwise 3 x 3 layer that alone reads it in one launch (csrc/expand_dw.hip), in every form it
has, against the two layers' own kernels bit for bit: bands and columns with remainders, strides, padding, one K step and three,
channels that fill a workgroup's and that do not, fewer units than compute units and more, the three epilogues."""
import numpy as np
import pytest
import torch

from dldt_amd import HipieError
from dldt_amd.builders import QuantizedNet
from dldt_amd.graph import Plan

pytestmark = pytest.mark.gpu

#        n, c, h, w, channels (images of 3: a 3 x 3 convolution of stride 2), stride and padding of the depthwise layer, top of the range (above 6: the Clamp stays), ReLU6 or not
CASES = {
    "columns_17": (1, 16, 13, 17, 48, 1, 1, 3.0, True),
    "stride_2_odd": (3, 24, 15, 9, 80, 2, 1, 3.0, True),
    "stride_2_unpadded": (2, 16, 12, 20, 32, 2, 0, 8.0, True),
    "unpadded": (1, 64, 7, 5, 16, 1, 0, 3.0, True),
    "padded_by_2": (1, 65, 6, 6, 16, 1, 2, 8.0, True),
    "three_k_steps": (2, 160, 9, 7, 104, 1, 1, 3.0, True),
    "one_pixel": (5, 32, 1, 1, 16, 1, 1, 3.0, True),
    "wide_rows": (2, 16, 30, 111, 96, 2, 1, 3.0, True),
    "many_units": (9, 24, 40, 24, 144, 1, 1, 3.0, True),
    "small_images": (65, 16, 7, 7, 368, 1, 1, 3.0, True),
    "small_images_stride_2": (70, 24, 7, 9, 368, 2, 1, 3.0, True),
    "image": (2, 3, 33, 31, 32, 1, 1, 3.0, True),
    "image_stride_2": (3, 3, 57, 40, 40, 2, 1, 8.0, True),
    "no_scale": (3, 48, 21, 19, 70, 1, 1, 3.0, False),
    "no_scale_stride_2": (3, 48, 21, 19, 70, 2, 1, 3.0, False),
}


def _graph(n, c, h, w, oc, stride, pads, high, relu6):
    rng = np.random.default_rng(oc * h)
    net = QuantizedNet()
    a = net.input("data", (n, c, h, w), 2.0)
    conv = net.conv_relu6 if relu6 else net.conv
    k = 3 if c == 3 else 1
    mid = conv(a, rng.normal(0, 1 / np.sqrt(c), (oc, c, k, k)).astype(np.float32), rng.normal(0, 0.2, oc).astype(np.float32), high, strides=(1 + k // 2,) * 2, pads=(k // 2,) * 2)
    b = conv(mid, rng.normal(0, 0.4, (oc, 1, 3, 3)).astype(np.float32), rng.normal(0, 0.2, oc).astype(np.float32), high, strides=(stride, stride), pads=(pads, pads), grouped=True)
    net.g.result(net.conv_f32(b, rng.normal(0, 0.2, (24, oc, 1, 1)).astype(np.float32), None), "out")
    return net.g, mid["node"]


@pytest.mark.parametrize("name,form", [(n, f) for n in sorted(CASES) for f in range(4) if f < 3 or n.startswith("small")])
def test_one_launch_equals_two(name, form, tmp_path):
    g, mid = _graph(*CASES[name])
    base = {"HIP_THROUGHPUT_STREAMS": "1", "HIP_SINGLE_LAUNCH": "NO"}
    apart = g.compile(0, config=dict(base, HIP_TUNE="NO", HIP_FUSE_CONVOLUTIONS="NO"))
    default = g.compile(0, config=dict(base, HIP_TUNE="NO", HIP_FUSE_CONVOLUTIONS="YES"))
    pair = [i for i, s in enumerate(default.steps) if s["type"] == "GroupConvolution"]
    assert len(pair) == 1 and len(default.steps) == len(apart.steps) - 1
    choices = tmp_path / "choices"
    choices.write_text("".join(f"{i} {s['variant'] % 8192 + 8192 * form if i in pair else s['variant']}\n" for i, s in enumerate(default.steps)))
    fused = g.compile(0, config=dict(base, HIP_TUNE="YES", HIP_TUNE_FILE=str(choices), HIP_FUSE_CONVOLUTIONS="YES"))
    assert fused.steps[pair[0]]["variant"] >> 13 == form
    results = []
    x = torch.rand(CASES[name][:4], generator=torch.Generator(device="cuda").manual_seed(form), device="cuda") * 2
    reqs = [p.create_request() for p in (apart, fused)]
    for r in reqs:
        ins, outs = r.device_buffers()
        ins[0].copy_(x)
        outs[0].fill_(float("nan"))
        torch.cuda.synchronize()
        r.infer_device(ins, outs)
        results.append(outs[0].cpu().numpy())
    assert not np.isnan(results[0]).any() and np.abs(results[0]).max() > 0
    assert np.array_equal(results[0].view(np.uint32), results[1].view(np.uint32))
    assert reqs[0].tensor(mid) is not None
    with pytest.raises(HipieError, match="LDS only"):
        reqs[1].tensor(mid)


def _two_blocks():
    rng = np.random.default_rng(8)
    net = QuantizedNet()
    a, mids = net.input("data", (2, 16, 12, 12), 2.0), []
    for c, oc in ((16, 48), (24, 64)):
        mid = net.conv_relu6(a, rng.normal(0, 1 / np.sqrt(c), (oc, c, 1, 1)).astype(np.float32), rng.normal(0, 0.2, oc).astype(np.float32), 3.0)
        b = net.conv_relu6(mid, rng.normal(0, 0.4, (oc, 1, 3, 3)).astype(np.float32), rng.normal(0, 0.2, oc).astype(np.float32), 3.0, pads=(1, 1), grouped=True)
        mids.append(mid["node"])
        a = net.conv(b, rng.normal(0, 0.2, (24, oc, 1, 1)).astype(np.float32), None, 3.0)
    net.g.result(net.dequantize(a), "out")
    return net.g, mids


@pytest.mark.parametrize("single", ["NO", "256"])
@pytest.mark.parametrize("apart", [(), (0,), (1,), (0, 1)])
def test_layers_that_run_apart_are_two_steps(apart, single, tmp_path):
    """each has its line in the counters and its node of the executed graph; the choices survive a file and an export"""
    g, mids = _two_blocks()
    config = {"HIP_THROUGHPUT_STREAMS": "1", "HIP_SINGLE_LAUNCH": single}
    both = g.compile(0, config=dict(config, HIP_TUNE="NO", HIP_FUSE_CONVOLUTIONS="YES"))
    two = g.compile(0, config=dict(config, HIP_TUNE="NO", HIP_FUSE_CONVOLUTIONS="NO"))
    pairs = [i for i, s in enumerate(both.steps) if s["type"] == "GroupConvolution"]
    assert len(pairs) == 2 and len(both.steps) == len(two.steps) - 2
    text = "".join("%d %d\n" % (i, s["variant"] & ~4096 if i in [pairs[k] for k in apart] else s["variant"]) for i, s in enumerate(both.steps))
    (tmp_path / "choices").write_text(text)
    plan = g.compile(0, config=dict(config, HIP_TUNE="YES", HIP_TUNE_FILE=str(tmp_path / "choices")))
    assert (tmp_path / "choices").read_text() == text                     # it was taken as it is
    assert len(plan.steps) == len(both.steps) + len(apart)
    at = pairs[0]                                                         # the first block's step, or the first of its two
    for k in range(2):
        types = [s["type"] for s in plan.steps[at:at + 2]]
        if k in apart:
            assert types == ["Convolution", "GroupConvolution"] and plan.step_sources(at + 1) == [at] and plan.step_sources(at + 2) == [at + 1]
        else:
            assert types[0] == "GroupConvolution" and plan.step_sources(at + 1) == [at]
        at += 3 if k in apart else 2                                      # (behind them the projection)
    again = Plan.load(plan.export())
    assert [(s["type"], s["name"], s["variant"]) for s in again.steps] == [(s["type"], s["name"], s["variant"]) for s in plan.steps]
    x = torch.rand((2, 16, 12, 12), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda") * 2
    results = []
    for p in (two, plan, again):
        r = p.create_request(perf_count=p is plan and single == "NO")
        ins, outs = r.device_buffers()
        ins[0].copy_(x)
        torch.cuda.synchronize()
        r.infer_device(ins, outs)
        results.append(outs[0].cpu().numpy())
        if p is plan and single == "NO":
            counters = {s["name"]: s["ms"] for s in r.perf()}
            assert len(counters) == len(plan.steps) and all(ms > 0 for n, ms in counters.items() if n != "out")
            for k in range(2):
                if k in apart:
                    assert r.tensor(mids[k]).max() > 0
                else:
                    with pytest.raises(HipieError, match="LDS only"):
                        r.tensor(mids[k])
    assert np.abs(results[0]).max() > 0
    assert all(np.array_equal(results[0].view(np.uint8), v.view(np.uint8)) for v in results[1:])


def test_a_file_of_choices_apart_is_taken_as_it_is(tmp_path):
    """a tuning file from before the two layers were ever one step, as those of HIP_FUSE_CONVOLUTIONS=NO are: not measured anew"""
    g, mids = _two_blocks()
    path = tmp_path / "choices"
    config = {"HIP_THROUGHPUT_STREAMS": "1", "HIP_SINGLE_LAUNCH": "NO", "HIP_TUNE": "YES", "HIP_TUNE_FILE": str(path)}
    apart = g.compile(0, config=dict(config, HIP_FUSE_CONVOLUTIONS="NO"))
    text = path.read_text()
    assert len(text.splitlines()) == len(apart.steps)
    plan = g.compile(0, config=config)
    assert path.read_text() == text and [s["variant"] for s in plan.steps] == [s["variant"] for s in apart.steps]
    # a file with the choices of other steps is not
    path.write_text(text + "%d 0\n" % len(apart.steps))
    g.compile(0, config=config)
    assert path.read_text() != text + "%d 0\n" % len(apart.steps)
