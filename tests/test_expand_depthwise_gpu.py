"""A dense layer and the depthwise 3 x 3 layer that alone reads it, as one step of the single launch (expand_depthwise,
csrc/program.hip), against the plan's steps bit for bit: bands and columns with remainders, strides, K in one step and more and
from a table of offsets, padding at a zero point, channels that fill a tile and that do not, more units than workgroups."""
import numpy as np
import pytest
import torch

from dldt_amd import HipieError
from dldt_amd.builders import QuantizedNet

pytestmark = pytest.mark.gpu

#        n, c, h, w, channels, (kernel, stride) of the dense layer, stride and padding of the depthwise one, zero point
CASES = {
    "columns_17": (1, 16, 13, 17, 48, (1, 1), 1, 1, False),
    "stride_2_odd": (3, 24, 15, 9, 80, (1, 1), 2, 1, False),
    "stride_2_unpadded": (2, 16, 12, 20, 32, (1, 1), 2, 0, False),
    "unpadded": (1, 64, 7, 5, 16, (1, 1), 1, 0, False),
    "padded_by_2": (1, 64, 6, 6, 16, (1, 1), 1, 2, False),
    "four_k_steps": (1, 256, 9, 7, 40, (1, 1), 1, 1, False),
    "first_layer": (2, 3, 33, 31, 32, (3, 2), 1, 1, False),
    "zero_point": (2, 32, 11, 10, 56, (1, 1), 1, 1, True),
    "one_pixel": (5, 32, 1, 1, 16, (1, 1), 1, 1, False),
    "more_units_than_workgroups": (9, 16, 40, 24, 144, (1, 1), 2, 1, False),
}


def _graph(n, c, h, w, oc, dense, stride, pads, zero_point):
    rng = np.random.default_rng(oc * h)
    net = QuantizedNet()
    a = net.input("data", (n, c, h, w), 2.0)
    k, s = dense
    wd, bd = rng.normal(0, 1 / np.sqrt(c * k * k), (oc, c, k, k)).astype(np.float32), rng.normal(0, 0.2, oc).astype(np.float32)
    at = dict(strides=(s, s), pads=(k // 2, k // 2))
    mid = net.asymmetric(net.conv_f32(a, wd, bd, **at), -1.0, 3.0) if zero_point else net.conv_relu6(a, wd, bd, 3.0, **at)
    wg, bg = rng.normal(0, 0.4, (oc, 1, 3, 3)).astype(np.float32), rng.normal(0, 0.2, oc).astype(np.float32)
    b = net.conv_relu6(mid, wg, bg, 3.0, strides=(stride, stride), pads=(pads, pads), grouped=True)
    net.g.result(net.conv_f32(b, rng.normal(0, 0.2, (8, oc, 1, 1)).astype(np.float32), None), "out")
    return net.g, mid["node"]


@pytest.mark.parametrize("workgroups", [64, 256])
@pytest.mark.parametrize("name", sorted(CASES))
def test_one_step_equals_two(name, workgroups):
    g, mid = _graph(*CASES[name])
    config = {"HIP_TUNE": "NO", "HIP_THROUGHPUT_STREAMS": "1"}
    reqs = [g.compile(0, config=dict(config, HIP_SINGLE_LAUNCH=m)).create_request() for m in ("NO", str(workgroups))]
    gen = torch.Generator(device="cuda").manual_seed(workgroups)
    for _ in range(2):
        results = []
        x = torch.rand(CASES[name][:4], generator=gen, device="cuda") * 2
        for r in reqs:
            ins, outs = r.device_buffers()
            ins[0].copy_(x)
            outs[0].fill_(float("nan"))
            torch.cuda.synchronize()
            r.infer_device(ins, outs)
            results.append(outs[0].cpu().numpy())
        assert not np.isnan(results[0]).any()
        assert np.array_equal(results[0].view(np.uint8), results[1].view(np.uint8))
    assert reqs[0].tensor(mid) is not None
    with pytest.raises(HipieError, match="LDS only"):           # the form was the one compared
        reqs[1].tensor(mid)


@pytest.mark.parametrize("switch", [{"HIP_KEEP_F32": "YES"}, {"HIP_FUSE_CONVOLUTIONS": "NO"}])
def test_values_that_are_kept_are_two_steps(switch):
    g, mid = _graph(*CASES["stride_2_odd"])
    plan = g.compile(0, config=dict(switch, HIP_TUNE="NO", HIP_THROUGHPUT_STREAMS="1", HIP_SINGLE_LAUNCH="256"))
    r = plan.create_request()
    ins, outs = r.device_buffers()
    ins[0].fill_(1.0)
    torch.cuda.synchronize()
    r.infer_device(ins, outs)
    assert plan.metric("SINGLE_LAUNCH_COUNTS") == "1 0"
    assert r.tensor(mid).max() > 0
