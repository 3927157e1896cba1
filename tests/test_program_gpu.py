"""The single-launch form of a plan (csrc/program.hip) against its steps, bit for bit: tile remainders in pixels and channels,
K of one step and of many, strides, residuals, shortcuts, depthwise, pools, encoder steps; the ordering of launches on
several streams; and the way back to the steps when a launch is cancelled."""
import threading
from unittest import mock

import numpy as np
import pytest
import torch

from dldt_amd import HipieError, builders
from dldt_amd._lib import check, lib
from dldt_amd.graph import Plan

pytestmark = pytest.mark.gpu



def _beside_an_encoder(build, **kw):
    """an encoder and a network over feature maps as one graph of two branches"""
    g = builders.bert_encoder(layers=1, batch=1, seq=96, vocab=100, mask=True)[0]

    class Beside(builders.QuantizedNet):
        def __init__(self):
            super().__init__()
            self.g = g

    with mock.patch.object(builders, "QuantizedNet", Beside):
        assert build(**kw)[0] is g
    return g


GRAPHS = {
    "block_1x3x7": lambda: builders.conv_block(n=1, c=3, hw=7, oc=8)[0],
    "block_2x17x9": lambda: builders.conv_block(n=2, c=17, hw=9, oc=65)[0],
    "block_1x64x56": lambda: builders.conv_block(n=1, c=64, hw=56, oc=64)[0],
    "block_3x256x16": lambda: builders.conv_block(n=3, c=256, hw=16, oc=130)[0],
    "block_3x64x14": lambda: builders.conv_block(n=3, c=64, hw=14, oc=512)[0],
    "block_7x64x32": lambda: builders.conv_block(n=7, c=64, hw=32, oc=130)[0],
    "block_2x256x14": lambda: builders.conv_block(n=2, c=256, hw=14, oc=144)[0],
    "block_7x128x14": lambda: builders.conv_block(n=7, c=128, hw=14, oc=72)[0],
    "resnet_1": lambda: builders.resnet50(batch=1, res=64, width=16, classes=10, seed=7)[0],
    "resnet_3_u8": lambda: builders.resnet50(batch=3, res=96, u8_input=True)[0],
    "resnet_7_u8": lambda: builders.resnet50(batch=7, res=96, u8_input=True)[0],
    "mobilenet_2": lambda: builders.mobilenet_v2(batch=2, res=96)[0],
    "mobilenet_1x160": lambda: builders.mobilenet_v2(batch=1, res=160)[0],                  # maps of 80, 40, 20, 10 and 5
    "mobilenet_3x64": lambda: builders.mobilenet_v2(batch=3, res=64)[0],                    # ... of 32, 16, 8, 4 and 2
    "encoder_1x32": lambda: builders.bert_encoder(layers=1, batch=1, seq=32, vocab=100, mask=True)[0],
    "encoder_3x96": lambda: builders.bert_encoder(layers=1, batch=3, seq=96, vocab=0, mask=False)[0],
    "encoder_1x512": lambda: builders.bert_encoder(layers=1, batch=1, seq=512, vocab=100, mask=True)[0],
    "encoder_1x160": lambda: builders.bert_encoder(layers=1, batch=1, seq=160, vocab=100, mask=True)[0],       # five tiles of keys for eight waves
    "encoder_4x128": lambda: builders.bert_encoder(layers=1, batch=4, seq=128, vocab=100, mask=True)[0],       # two waves for 32 queries (64 workgroups)
    "encoder_1x448": lambda: builders.bert_encoder(layers=1, batch=1, seq=448, vocab=100, mask=True)[0],
    "encoder_and_resnet": lambda: _beside_an_encoder(builders.resnet50, batch=1, res=64, width=16, classes=10, seed=7),
    "encoder_and_mobilenet": lambda: _beside_an_encoder(builders.mobilenet_v2, batch=2, res=96),
    "encoder_2x384": lambda: builders.bert_encoder(layers=1, batch=2, seq=384, vocab=100, mask=True)[0],
}


def _fill(ins, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    for t in ins:
        if t.dtype == torch.int32:
            t.copy_(torch.randint(0, 100, t.shape, generator=gen, device="cuda", dtype=torch.int32))
        elif t.dtype == torch.uint8:
            t.copy_(torch.randint(0, 256, t.shape, generator=gen, device="cuda", dtype=torch.uint8))
        elif t.dim() == 4 and t.shape[1] == t.shape[2] == 1:          # the attention mask
            keep = torch.arange(t.shape[3], device="cuda") < t.shape[3] * 2 // 3
            t.copy_(torch.where(keep, 0.0, -10000.0).expand(t.shape))
        else:
            t.copy_(torch.rand(t.shape, generator=gen, device="cuda") * 2)


def _compile(g, mode):
    return g.compile(0, config={"HIP_SINGLE_LAUNCH": mode, "HIP_TUNE": "NO", "HIP_THROUGHPUT_STREAMS": "1"})


def _infer(req, seed):
    ins, outs = req.device_buffers()
    _fill(ins, seed)
    for o in outs:
        o.fill_(0 if o.dtype == torch.uint8 else float("nan"))
    torch.cuda.synchronize()
    req.infer_device(ins, outs)
    return [o.cpu().numpy() for o in outs]


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_single_launch_equals_steps(name):
    g = GRAPHS[name]()
    steps, single = _compile(g, "NO"), _compile(g, "YES")
    assert single.config("HIP_SINGLE_LAUNCH") == "YES"
    a, b = steps.create_request(), single.create_request()
    for seed in range(3):
        for x, y in zip(_infer(a, seed), _infer(b, seed)):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


@pytest.mark.parametrize("workgroups", ["64", "256"])
@pytest.mark.parametrize("n,hw,c,signed", [(1, 5, 8, False), (1, 28, 72, True), (3, 14, 130, False), (4, 56, 64, False)])
def test_a_residual_of_the_step_in_front_equals_steps(n, hw, c, signed, workgroups):
    """a convolution asks for its residual before it waits for the step in front: here that one writes it, as bytes and as f32"""
    rng = np.random.default_rng(hw)
    net = builders.QuantizedNet()
    g = net.g

    def weights(k):
        return (rng.standard_normal((c, c, k, k), dtype=np.float32) * np.float32(0.05)).astype(np.float32), \
            (rng.standard_normal(c, dtype=np.float32) * np.float32(0.1)).astype(np.float32)

    a = net.conv(net.input("data", (n, c, hw, hw), 2.0), *weights(3), out_high=2.0, pads=(1, 1), signed=signed)
    y = g.add(net.conv_f32(a, *weights(1)), net.dequantize(a))
    b = net.requantize(y, 2.0, signed=True)
    z = g.add(net.conv_f32(b, *weights(1)), y)
    g.result(z, "out")
    steps, single = _compile(g, "NO"), _compile(g, workgroups)
    assert single.config("HIP_SINGLE_LAUNCH") == workgroups
    one, other = steps.create_request(), single.create_request()
    for seed in range(3):
        for x, v in zip(_infer(one, seed), _infer(other, seed)):
            assert np.array_equal(x.view(np.uint8), v.view(np.uint8))


@pytest.mark.parametrize("workgroups", ["64", "128", "256"])
@pytest.mark.parametrize("batch,seq,masked", [(1, 448, False), (2, 448, True), (3, 512, True), (5, 448, True)])
def test_long_rows_whose_workgroups_cross_heads_and_elements_equal_steps(batch, seq, masked, workgroups):
    """keys, values and mask stay with a workgroup until its next unit is of another head or element: each has a mask of its own"""
    g = builders.bert_encoder(layers=1, batch=batch, seq=seq, vocab=100, mask=masked)[0]
    steps, single = _compile(g, "NO"), _compile(g, workgroups)
    assert single.config("HIP_SINGLE_LAUNCH") == workgroups
    results = []
    for plan in (steps, single):
        req = plan.create_request()
        ins, outs = req.device_buffers()
        _fill(ins, 7)
        if masked:
            keep = torch.arange(seq, device="cuda").view(1, 1, 1, seq) < torch.tensor([seq, 1, seq // 3, 33, seq - 1][:batch], device="cuda").view(batch, 1, 1, 1)
            ins[1].copy_(torch.where(keep, 0.0, -10000.0))
        torch.cuda.synchronize()
        for _ in range(2):
            for o in outs:
                o.fill_(float("nan"))
            torch.cuda.synchronize()
            req.infer_device(ins, outs)
            results.append([o.cpu().numpy() for o in outs])
    for got in results[1:]:
        for x, y in zip(results[0], got):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


@pytest.mark.parametrize("name", ["block_1x3x7", "block_3x64x14", "resnet_3_u8", "mobilenet_1x160", "encoder_3x96", "encoder_and_resnet"])
def test_results_are_there_when_the_call_returns(name):
    """The call returns by the launch's own word, before its stream has drained: results are read on another stream at once, by a
    kernel and by a copy to the host, and the request is destroyed or its next inference follows."""
    g = GRAPHS[name]()
    steps, single = _compile(g, "NO"), _compile(g, "64")
    want = [_infer(steps.create_request(), seed) for seed in range(4)]
    # (a request's stream: the first torch.cuda.Stream() makes 32 that stay, and with them every later request's hardware queue is
    # another one; test_requests_of_several_threads meets queues that two of its requests share)
    aside = steps.create_request()
    other = torch.cuda.ExternalStream(aside.stream)
    b = single.create_request()
    buffers = []
    for seed in range(4):
        ins, outs = b.device_buffers()
        _fill(ins, seed)
        buffers.append((ins, outs))
    torch.cuda.synchronize()
    for turn in range(60):
        ins, outs = buffers[turn % 4]
        for o in outs:
            o.fill_(0 if o.dtype == torch.uint8 else float("nan"))
        torch.cuda.synchronize()
        b.infer_device(ins, outs)
        with torch.cuda.stream(other):
            seen = [o.clone() if turn % 2 else o.cpu() for o in outs]
        if turn % 5 == 4:
            del b
            b = single.create_request()
        other.synchronize()
        for x, y in zip(want[turn % 4], seen):
            assert np.array_equal(x.view(np.uint8), y.cpu().numpy().view(np.uint8)), turn
    assert single.metric("SINGLE_LAUNCH_COUNTS") == "60 0"


# Together these choose every tile instance of the kernels (fragments of 16 channels x fragments of 16 pixels) and every way a
# tile's waves share its chain
@pytest.mark.parametrize("workgroups", [64, 128, 256])
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_every_size_runs_and_equals_steps(name, workgroups):
    g = GRAPHS[name]()
    steps, single = _compile(g, "NO"), _compile(g, str(workgroups))
    assert single.config("HIP_SINGLE_LAUNCH") == single.metric("SINGLE_LAUNCH_WORKGROUPS") == str(workgroups)
    assert steps.metric("SINGLE_LAUNCH_WORKGROUPS") == "0" and single.metric("SINGLE_LAUNCH_REFUSED") == ""
    a, b = steps.create_request(), single.create_request()
    for seed in range(3):
        for x, y in zip(_infer(a, seed), _infer(b, seed)):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
    assert single.metric("SINGLE_LAUNCH_COUNTS") == "3 0"       # the launches were the results compared


def test_a_step_without_a_single_launch_form_is_named():
    g = builders.bert_encoder(layers=1, batch=1, seq=64, vocab=100, mask=True)[0]
    unfused = {"HIP_FUSE_ATTENTION": "NO", "HIP_TUNE": "NO", "HIP_THROUGHPUT_STREAMS": "1"}      # products and a Softmax of their own
    plan = g.compile(0, config=dict(unfused, HIP_SINGLE_LAUNCH="YES"))
    assert plan.metric("SINGLE_LAUNCH_WORKGROUPS") == "0" and plan.metric("SINGLE_LAUNCH_REFUSED") != ""
    req = plan.create_request()
    steps = g.compile(0, config=dict(unfused, HIP_SINGLE_LAUNCH="NO")).create_request()
    for x, y in zip(_infer(steps, 0), _infer(req, 0)):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
    assert plan.metric("SINGLE_LAUNCH_COUNTS") == "0 0"


def test_single_launch_requests_on_two_streams():
    g = GRAPHS["resnet_1"]()
    steps, single = _compile(g, "NO"), _compile(g, "YES")
    want = [_infer(steps.create_request(), s) for s in range(2)]
    reqs = [single.create_request() for _ in range(2)]
    bufs = [r.host_buffers() for r in reqs]
    for s, (ins, _) in enumerate(bufs):
        dev = steps.create_request().device_buffers()[0]
        _fill(dev, s)
        ins[0].array[...] = dev[0].cpu().numpy()
    for _ in range(20):
        for r, (ins, outs) in zip(reqs, bufs):
            r.start(ins, outs)
        for r in reqs:
            r.wait()
        for (_, outs), w in zip(bufs, want):
            assert np.array_equal(outs[0].array.view(np.uint8), w[0].view(np.uint8))


def _start_device(req, ins, outs):
    check(lib().hipie_request_start(req._h, *req._ptrs(ins, outs), 1))


@pytest.mark.parametrize("memory", ["device", "host"])
def test_outputs_are_complete_in_the_order_of_a_stream_the_caller_holds(monkeypatch, memory):
    """a copy that the caller queues behind the start sees the outputs, whatever becomes of a single launch"""
    g = GRAPHS["resnet_1"]()
    want = _infer(_compile(g, "NO").create_request(), 0)[0]
    monkeypatch.setenv("HIPIE_ROLL_CALL_TICKS", "0")             # every launch is given up
    req = _compile(g, "64").create_request()
    ins, outs = req.device_buffers()
    _fill(ins, 0)
    stream = torch.cuda.ExternalStream(req.stream)
    outs[0].fill_(float("nan"))
    torch.cuda.synchronize()
    if memory == "device":
        _start_device(req, ins, outs)
        with torch.cuda.stream(stream):
            seen = outs[0].clone()
            ins[0].zero_()                                       # the inference has read its input by then
        stream.synchronize()
    else:
        hin, hout = req.host_buffers()
        hin[0].array[...] = ins[0].cpu().numpy()
        hout[0].array[...] = np.nan
        req.start(hin, hout)
        stream.synchronize()
        seen = torch.from_numpy(hout[0].array.copy())
    req.wait()
    assert np.array_equal(seen.cpu().numpy().view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("timeout", [-1, 0, 5, 10000])
def test_cancelled_launch_of_host_buffers_is_made_up_for_in_the_wait(monkeypatch, timeout):
    g = GRAPHS["resnet_1"]()
    steps = _compile(g, "NO").create_request()
    monkeypatch.setenv("HIPIE_ROLL_CALL_TICKS", "0")
    plan = _compile(g, "128")
    req = plan.create_request()
    hin, hout = req.host_buffers()
    for seed in range(2):
        want = _infer(steps, seed)[0]
        dev = steps.device_buffers()[0]
        _fill(dev, seed)
        hin[0].array[...] = dev[0].cpu().numpy()
        hout[0].array[...] = np.nan
        req.start(hin, hout)
        for _ in range(100000):
            try:
                req.wait_for(timeout)
                break
            except HipieError as e:
                assert e.status == -9 and timeout != -1          # still running, busy
        assert np.array_equal(hout[0].array.view(np.uint8), want.view(np.uint8))
        with pytest.raises(HipieError):                          # idle again
            req.wait()
    # a caller that revoked the inference gets no outputs of it, and the next one is whole
    req.start(hin, hout)
    req.cancel()
    with pytest.raises(HipieError) as e:
        req.wait()
    assert e.value.status == -13
    req.start(hin, hout)
    req.wait()
    assert np.array_equal(hout[0].array.view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("mode", ["AUTO", "YES"])
def test_a_choice_made_on_a_busy_device_is_not_kept(monkeypatch, tmp_path, mode):
    """launches that are given up while the sizes are measured: AUTO runs by steps, and neither file nor stream says why"""
    g = GRAPHS["block_2x17x9"]()
    path = tmp_path / "choices"
    monkeypatch.setenv("HIPIE_ROLL_CALL_TICKS", "0")
    plan = g.compile(0, config={"HIP_THROUGHPUT_STREAMS": "1", "HIP_SINGLE_LAUNCH": mode, "HIP_TUNE_FILE": str(path)})
    assert (plan.metric("SINGLE_LAUNCH_WORKGROUPS") == "0") == (mode == "AUTO")
    assert plan.metric("SINGLE_LAUNCH_SHARED_WORKGROUPS") == "0"
    assert "\n-" not in path.read_text() and not plan.export()[10] & 0x80


def _host_request(plan, feed):
    """(request, its host blobs) with the values of the device tensors `feed` in the inputs"""
    req = plan.create_request()
    ins, outs = req.host_buffers()
    for a, t in zip(ins, feed):
        a.array[...] = t.cpu().numpy()
    return req, ins, outs


def _feed_and_result(g, seed):
    req = _compile(g, "NO").create_request()
    out = _infer(req, seed)
    ins, _ = req.device_buffers()
    _fill(ins, seed)
    return ins, out


def _same(outs, want):
    return all(np.array_equal(o.array.view(np.uint8), w.view(np.uint8)) for o, w in zip(outs, want))


@pytest.mark.parametrize("workgroups,together", [(64, 4), (128, 2), (256, 1)])
def test_programs_in_flight_fit_the_device(workgroups, together):
    """five requests of one plan started one behind the other: as many run as programs as there are compute units for"""
    g = GRAPHS["resnet_1"]()
    plan = _compile(g, str(workgroups))
    work = [_feed_and_result(g, s) for s in range(5)]
    reqs = [_host_request(plan, feed) for feed, _ in work]
    for turn in range(1, 4):
        for r, ins, outs in reqs:
            outs[0].array[...] = np.nan
            r.start(ins, outs)
        for r, _, _ in reqs:
            r.wait()
        assert all(_same(outs, want) for (_, _, outs), (_, want) in zip(reqs, work))
        assert plan.metric("SINGLE_LAUNCH_COUNTS") == "%d 0" % (turn * together)


def test_programs_of_two_plans_and_steps_of_a_third_side_by_side():
    graphs = [GRAPHS[n]() for n in ("encoder_3x96", "mobilenet_2", "resnet_3_u8")]
    plans = [_compile(g, m) for g, m in zip(graphs, ("64", "128", "NO"))]
    work = [_feed_and_result(g, 1) for g in graphs]
    reqs = [_host_request(p, feed) for p, (feed, _) in zip(plans, work)]
    for _ in range(20):
        for r, ins, outs in reqs:
            outs[0].array[...] = np.nan
            r.start(ins, outs)
        for r, _, _ in reversed(reqs):
            r.wait()
        assert all(_same(outs, want) for (_, _, outs), (_, want) in zip(reqs, work))
    assert [p.metric("SINGLE_LAUNCH_COUNTS") for p in plans] == ["20 0", "20 0", "0 0"]


@pytest.mark.parametrize("mode", ["64", "256", "YES"])
def test_requests_of_several_threads(mode):
    """three threads that infer one request each, of two plans; every result, whichever form it took"""
    graphs = [GRAPHS["resnet_1"](), GRAPHS["encoder_1x32"]()]
    plans = [_compile(g, mode) for g in graphs]
    failed = []

    def loop(which, seed):
        try:
            torch.cuda.set_device(0)
            feed, want = work[seed]
            req = plans[which].create_request()
            _, outs = req.device_buffers()
            for _ in range(50):
                req.infer_device(feed, outs)
                if not np.array_equal(outs[0].cpu().numpy().view(np.uint8), want[0].view(np.uint8)):
                    failed.append(seed)
        except Exception as e:                                   # noqa: BLE001 (reported below)
            failed.append(e)

    work = [_feed_and_result(graphs[which], seed) for seed, which in enumerate((0, 1, 0))]
    threads = [threading.Thread(target=loop, args=(which, seed)) for seed, which in enumerate((0, 1, 0))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    assert all(p.metric("SINGLE_LAUNCH_COUNTS") != "0 0" for p in plans)


def _forms(plan):
    return plan.metric("SINGLE_LAUNCH_WORKGROUPS"), plan.metric("SINGLE_LAUNCH_SHARED_WORKGROUPS")


@pytest.mark.parametrize("config", [{"HIP_SINGLE_LAUNCH": "AUTO"}, {"HIP_SINGLE_LAUNCH": "YES", "HIP_TUNE": "NO"},
                                    {"HIP_SINGLE_LAUNCH": "128", "HIP_TUNE": "NO"}, {"HIP_TUNE": "NO"}])
def test_an_exported_plan_keeps_its_form(config):
    g = GRAPHS["resnet_1"]()
    plan = g.compile(0, config=dict(config, HIP_THROUGHPUT_STREAMS="1"))
    back = Plan.load(plan.export())
    assert _forms(back) == _forms(plan) and back.config("HIP_THROUGHPUT_STREAMS") == "1"
    assert back.export() == plan.export()
    for x, y in zip(_infer(plan.create_request(), 0), _infer(back.create_request(), 0)):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8))


def test_the_tuning_file_keeps_the_form(tmp_path):
    g = GRAPHS["resnet_1"]()
    path = tmp_path / "choices"
    config = {"HIP_THROUGHPUT_STREAMS": "1", "HIP_TUNE_FILE": str(path)}
    first = _forms(g.compile(0, config=config))
    text = path.read_text()
    assert text.endswith("-1 %s\n-2 %s\n" % first)
    steps = text[:text.index("-1 ")]
    for lone, shared in ((64, 64), (256, 128), (128, 0), (0, 0)):
        path.write_text(steps + "-1 %d\n-2 %d\n" % (lone, shared))
        assert _forms(g.compile(0, config=config)) == (str(lone), str(shared))       # taken as it is, not measured
    for damaged in ("", "-1 64\n", "-1 32\n-2 0\n", "-1 0\n-2 64\n"):
        path.write_text(steps + damaged)
        g.compile(0, config=config)                                                  # measured, and written again
        assert path.read_text().startswith(steps + "-1 ") and path.read_text().count("\n") == text.count("\n")


def test_the_memory_of_the_form_is_reported():
    """ResNet-50: 25.5 million weights, and four words per output pixel of a layer; one copy when both forms are the same"""
    g = builders.resnet50(batch=1, res=64)[0]
    assert _compile(g, "NO").metric("SINGLE_LAUNCH_BYTES") == "0"
    one = int(_compile(g, "64").metric("SINGLE_LAUNCH_BYTES"))
    assert 25.4e6 < one < 29e6
    free = torch.cuda.mem_get_info()[0]
    plan = _compile(g, "64")
    assert free - torch.cuda.mem_get_info()[0] > one
    del plan


def test_a_request_with_counters_runs_by_steps():
    g = GRAPHS["resnet_1"]()
    plan = _compile(g, "64")
    timed = plan.create_request(perf_count=True)
    want = _infer(plan.create_request(), 0)[0]
    assert np.array_equal(_infer(timed, 0)[0].view(np.uint8), want.view(np.uint8))
    assert plan.metric("SINGLE_LAUNCH_COUNTS") == "1 0"
    assert all(st["ms"] > 0 for st in timed.perf())


def test_more_requests_than_a_plan_has_slots():
    g = GRAPHS["block_1x3x7"]()
    plan = _compile(g, "64")
    want = _infer(_compile(g, "NO").create_request(), 0)[0]
    reqs = [plan.create_request() for _ in range(66)]            # 64 slots; the others run by steps
    for r in reqs:
        assert np.array_equal(_infer(r, 0)[0].view(np.uint8), want.view(np.uint8))
    assert plan.metric("SINGLE_LAUNCH_COUNTS") == "64 0"
    del reqs[10]                                                 # (r is the last one)
    again = plan.create_request()
    assert np.array_equal(_infer(again, 0)[0].view(np.uint8), want.view(np.uint8))
    assert plan.metric("SINGLE_LAUNCH_COUNTS") == "65 0"


def test_launches_that_fail_are_tried_less_and_less(monkeypatch):
    g = GRAPHS["block_2x17x9"]()
    want = _infer(_compile(g, "NO").create_request(), 0)[0]
    monkeypatch.setenv("HIPIE_ROLL_CALL_TICKS", "0")
    plan = _compile(g, "64")
    req = plan.create_request()
    given_up = []
    for i in range(1 + 4 + 1 + 20 + 1 + 84 + 1):
        before = plan.metric("SINGLE_LAUNCH_COUNTS")
        assert np.array_equal(_infer(req, 0)[0].view(np.uint8), want.view(np.uint8))
        if plan.metric("SINGLE_LAUNCH_COUNTS") != before:
            given_up.append(i)
    assert given_up == [0, 5, 26, 111] and plan.metric("SINGLE_LAUNCH_COUNTS") == "0 4"


@pytest.mark.parametrize("ticks,counts", [("", "1 0"), ("soon", "1 0"), ("-1", "1 0"), ("99999999999999999999", "1 0"), ("0", "0 1")])
def test_roll_call_deadline_is_a_number_within_its_range(monkeypatch, ticks, counts):
    monkeypatch.setenv("HIPIE_ROLL_CALL_TICKS", ticks)
    plan = _compile(GRAPHS["block_2x17x9"](), "64")
    _infer(plan.create_request(), 0)
    assert plan.metric("SINGLE_LAUNCH_COUNTS") == counts


def _at(t, offset):
    """the tensor's values `offset` elements behind a 256-byte boundary"""
    room = torch.zeros(t.numel() + 64, dtype=t.dtype, device="cuda")
    view = room[offset:offset + t.numel()].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("offset", [0, 1, 2, 4])
@pytest.mark.parametrize("name", ["block_1x64x56", "encoder_3x96"])
def test_buffers_off_the_boundary_are_left_to_the_steps(name, offset):
    """what the steps refuse (an f32 residual that is a graph input) stays refused, what they take stays right"""
    g = GRAPHS[name]()
    steps, single = _compile(g, "NO"), _compile(g, "64")
    a, b = steps.create_request(), single.create_request()
    ins, _ = a.device_buffers()
    _fill(ins, 0)
    want = _infer(a, 0)
    shifted = [_at(t, offset) for t in ins]
    outs = [_at(torch.zeros_like(o), offset) for o in a.device_buffers()[1]]
    status = []
    for r in (a, b):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        try:
            r.infer_device(shifted, outs)
            status.append(0)
            assert np.array_equal(outs[0].cpu().numpy().view(np.uint8), want[0].view(np.uint8))
        except HipieError as e:
            status.append(e.status)
    assert status[0] == status[1]
    assert status[0] == (-4 if name.startswith("encoder") and offset % 4 else 0)
    assert single.metric("SINGLE_LAUNCH_COUNTS") == ("0 0" if offset % 4 else "1 0")


def test_an_output_on_its_input_is_left_to_the_steps():
    g = builders.conv_block(n=1, c=64, hw=14, oc=64)[0]
    plan = _compile(g, "64")
    req = plan.create_request()
    want = _infer(req, 0)[0]
    ins, outs = req.device_buffers()
    _fill(ins, 0)
    req.infer_device(ins, ins)
    assert np.array_equal(ins[0].cpu().numpy().view(np.uint8), want.view(np.uint8))
    assert plan.metric("SINGLE_LAUNCH_COUNTS") == "1 0"


def test_a_request_outlives_its_plan():
    """the order in which a garbage collector finalizes a cycle that holds both"""
    g = GRAPHS["resnet_1"]()
    plan = _compile(g, "64")
    reqs = [plan.create_request() for _ in range(3)]
    for r in reqs:
        _infer(r, 0)
    lib().hipie_plan_destroy(plan._h)
    plan._h = None
    junk = [_compile(GRAPHS["block_1x3x7"](), "NO") for _ in range(3)]      # takes the freed memory
    for r in reqs:
        lib().hipie_request_destroy(r._h)
        r._h = None
    del junk


def test_cancelled_launch_runs_by_steps(monkeypatch):
    g = GRAPHS["resnet_1"]()
    steps = _compile(g, "NO")
    monkeypatch.setenv("HIPIE_ROLL_CALL_TICKS", "0")
    single = _compile(g, "YES")
    a, b = steps.create_request(), single.create_request()
    for seed in range(3):
        for x, y in zip(_infer(a, seed), _infer(b, seed)):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
