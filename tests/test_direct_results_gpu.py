"""A convolution whose f32 values are the graph's result stores them into the caller's [N, C, H, W] buffer itself, and into its own
tensor where somebody looks at that: every kernel variant the layer has and the single launch, against the copy kernel behind
the same convolution (HIP_KEEP_F32), bit for bit."""
import numpy as np
import pytest
import torch

from dldt_amd import HipieError, builders

pytestmark = pytest.mark.gpu
VARIANTS = [*range(24), 24 + 32]
ANY, LINES = [*range(6), 10, 11], [12, 14, 15, 22]        # those every layer has, those of 64 input channels and more


def _graph(relu, results):
    """a convolution whose f32 value is `results` results"""
    rng = np.random.default_rng(3)
    q = builders.QuantizedNet()
    x = q.input("data", (2, 20, 11, 11), 2.55)
    y = q.conv_f32(x, rng.standard_normal((37, 20, 3, 3), dtype=np.float32) * np.float32(0.05), rng.standard_normal(37, dtype=np.float32), pads=(1, 1), relu=relu)
    for k in range(results):
        q.g.result(y, "out%d" % k)
    return q.g


def _run(plan, x, offset=0, value=None):
    """the outputs' bits; `value`: a node whose tensor holds the first one's values as well"""
    req = plan.create_request()
    ins, outs = req.device_buffers()
    ins[0].copy_(x)
    place = [torch.full((o.numel() + 8,), float("nan"), device="cuda")[offset:offset + o.numel()].view(o.shape) for o in outs]
    torch.cuda.synchronize()
    req.enqueue(ins, place)
    torch.cuda.synchronize()
    if value is not None:
        assert np.array_equal(req.tensor(value).reshape(-1) + np.float32(0), place[0].cpu().numpy().reshape(-1))
    return [p.cpu().numpy().view(np.uint32) for p in place]


@pytest.mark.parametrize("n,c,hw,oc,more", [(1, 3, 7, 8, []), (2, 17, 9, 65, [14]), (3, 64, 14, 70, LINES), (1, 64, 33, 129, LINES),
                                            (5, 128, 8, 3, [6, 7, 16, 18, 19, 20, 21] + LINES), (2, 32, 1, 1, [14])])
def test_every_variant_stores_the_planes_that_the_copy_stores(tmp_path, n, c, hw, oc, more):
    g = builders.conv_block(n=n, c=c, hw=hw, oc=oc)[0]
    x = torch.rand((n, c, hw, hw), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda") * 2.55
    kept = g.compile(0, config={"HIP_KEEP_F32": "YES", "HIP_TUNE": "NO"})
    want = _run(kept, x)
    plan = g.compile(0, config={"HIP_TUNE": "NO"})
    types = [s["type"] for s in plan.steps]
    assert int(plan.step_rt_info(len(types) - 1, "kernels")) == (0 if hw > 1 else 1)
    ran = []
    for v in VARIANTS:
        path = tmp_path / str(v)
        text = "".join("%d %d\n" % (i, v if t.startswith("Convolution") else -1) for i, t in enumerate(types))
        path.write_text(text)
        try:
            plan = g.compile(0, config={"HIP_TUNE_FILE": str(path), "HIP_SINGLE_LAUNCH": "NO"})
        except HipieError:
            continue                                          # a variant this layer does not have
        assert path.read_text() == text and [s["variant"] for s in plan.steps if s["type"].startswith("Convolution")] == [v]
        for offset in (0, 1):                                 # (a buffer on a 4-byte boundary only)
            got = _run(plan, x, offset, g.nodes[-1]["inputs"][0])
            assert np.array_equal(got[0], want[0]), (v, offset)
        ran.append(v)
    assert ran == sorted(ANY + more)
    single = g.compile(0, config={"HIP_TUNE": "NO", "HIP_THROUGHPUT_STREAMS": "1", "HIP_SINGLE_LAUNCH": "256"})
    req = single.create_request()
    ins, outs = req.device_buffers()
    ins[0].copy_(x)
    torch.cuda.synchronize()
    req.infer_device(ins, outs)
    assert np.array_equal(outs[0].cpu().numpy().view(np.uint32), want[0])
    assert single.metric("SINGLE_LAUNCH_COUNTS") == "1 0"


@pytest.mark.parametrize("n,c,hw,oc,k,more", [(1, 3, 7, 8, 3, []), (2, 17, 9, 65, 3, [14]), (3, 64, 14, 70, 3, LINES), (1, 64, 33, 129, 3, LINES),
                                              (5, 128, 8, 3, 3, [6, 7, 16, 18, 19, 20, 21] + LINES), (2, 64, 5, 37, 1, [23]), (1, 3, 17, 9, 7, [13])])
def test_every_variant_stores_the_tensor_beside_the_planes(tmp_path, n, c, hw, oc, k, more):
    """... in the one launch, of a request whose tensor was asked for before its first inference"""
    rng = np.random.default_rng(oc)
    q = builders.QuantizedNet()
    a = q.input("data", (n, c, hw, hw), 2.55)
    node = q.conv_f32(a, rng.standard_normal((oc, c, k, k), dtype=np.float32) * np.float32(0.05), rng.standard_normal(oc, dtype=np.float32), pads=(k // 2, k // 2),
                      strides=(2, 2) if k == 7 else (1, 1))
    q.g.result(node, "out")
    x = torch.rand((n, c, hw, hw), generator=torch.Generator(device="cuda").manual_seed(4), device="cuda") * 2.55
    ref = q.g.compile(0, config={"HIP_KEEP_F32": "YES", "HIP_TUNE": "NO"}).create_request()
    ins, outs = ref.device_buffers()
    ins[0].copy_(x)
    torch.cuda.synchronize()
    ref.enqueue(ins, outs)
    torch.cuda.synchronize()
    want, planes, ran = ref.tensor(node).view(np.uint32), outs[0].cpu().numpy().view(np.uint32), []
    for v in VARIANTS:
        path = tmp_path / str(v)
        path.write_text("0 -1\n1 %d\n2 -1\n" % v)
        try:
            plan = q.g.compile(0, config={"HIP_TUNE_FILE": str(path), "HIP_SINGLE_LAUNCH": "NO"})
        except HipieError:
            continue                                          # a variant this layer does not have
        assert plan.steps[1]["variant"] == v and [int(plan.step_rt_info(i, "kernels")) for i in range(3)] == [1, 1, 0]
        req = plan.create_request()
        assert not req.tensor(node).any()
        outs[0].fill_(float("nan"))
        torch.cuda.synchronize()
        req.enqueue(ins, outs)
        torch.cuda.synchronize()
        assert np.array_equal(outs[0].cpu().numpy().view(np.uint32), planes), v
        assert np.array_equal(req.tensor(node).view(np.uint32), want), v
        ran.append(v)
    assert set(ran) >= set(ANY + more)


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("results", [1, 2])
def test_values_without_an_activation_and_with_two_results(relu, results):
    x = torch.rand((2, 20, 11, 11), generator=torch.Generator(device="cuda").manual_seed(2), device="cuda") * 2.55
    g = _graph(relu, results)
    want = _run(g.compile(0, config={"HIP_KEEP_F32": "YES", "HIP_TUNE": "NO"}), x)
    plan = g.compile(0, config={"HIP_TUNE": "NO"})
    got = _run(plan, x)
    assert len(got) == results and all(np.array_equal(a, b) for a, b in zip(got, want))
    # two readers: the value stays in a tensor and is copied twice
    assert [int(plan.step_rt_info(i, "kernels")) for i, s in enumerate(plan.steps) if s["type"] == "Result"] == ([0] if results == 1 else [1, 1])


@pytest.mark.parametrize("hw", [1, 5])
@pytest.mark.parametrize("keep", ["NO", "YES"])
def test_a_result_is_in_its_tensor_as_well(hw, keep):
    """hipie_request_tensor gives a result's values of the last inference, queued or by the single launch, never older ones"""
    rng = np.random.default_rng(hw)
    q = builders.QuantizedNet()
    x = q.input("data", (2, 32, hw, hw), 2.55)
    node = q.conv_f32(x, rng.standard_normal((37, 32, 1, 1), dtype=np.float32) * np.float32(0.2), rng.standard_normal(37, dtype=np.float32))
    q.g.result(node, "out")
    plan = q.g.compile(0, config={"HIP_TUNE": "NO", "HIP_THROUGHPUT_STREAMS": "1", "HIP_SINGLE_LAUNCH": "256", "HIP_KEEP_F32": keep})
    req = plan.create_request()
    ins, outs = req.device_buffers()
    seen = []
    for turn, run in enumerate((req.enqueue, req.infer_device, req.enqueue, req.infer_device)):
        ins[0].uniform_(0, 2.55, generator=torch.Generator(device="cuda").manual_seed(turn))
        torch.cuda.synchronize()
        run(ins, outs)
        torch.cuda.synchronize()
        seen.append(outs[0].cpu().numpy().reshape(-1))
        assert np.array_equal(req.tensor(node).reshape(-1).view(np.uint32), seen[-1].view(np.uint32))
    assert plan.metric("SINGLE_LAUNCH_COUNTS") == "2 0"
    assert all(not np.array_equal(a, b) for a, b in zip(seen, seen[1:]))


@pytest.mark.parametrize("single", ["NO", "256"])
def test_a_tensor_that_is_held_shows_the_last_inference(single):
    """the descriptor of a result's tensor, asked for once (before the first inference, or between two): the values of every
    inference behind it, queued, waited for, or replayed from a captured graph"""
    import ctypes
    from dldt_amd._lib import check, lib
    from dldt_amd.tensor import hipie_tensor
    g = _graph(True, 1)
    node = g.nodes[-1]["inputs"][0]
    plan = g.compile(0, config={"HIP_TUNE": "NO", "HIP_THROUGHPUT_STREAMS": "1", "HIP_SINGLE_LAUNCH": single})
    ins, outs = plan.create_request().device_buffers()

    def held(req):
        t = hipie_tensor()
        check(lib().hipie_request_tensor(req._h, node, ctypes.byref(t)))
        values = torch.empty(t.n * t.stride_n, dtype=torch.float32)

        def shows():
            torch.cuda.synchronize()
            check(lib().hipie_memcpy(ctypes.c_void_p(values.data_ptr()), ctypes.c_void_p(t.data), ctypes.c_size_t(4 * values.numel()), 0))
            v = torch.as_strided(values, (t.n, t.c, t.h, t.w), (t.stride_n, 1, t.stride_h, t.stride_w))
            return torch.equal(v + 0.0, outs[0].cpu())
        return shows

    def feed(seed):
        ins[0].uniform_(0, 2.55, generator=torch.Generator(device="cuda").manual_seed(seed))
        torch.cuda.synchronize()

    for asked in (0, 2):
        req = plan.create_request()
        shows = held(req) if asked == 0 else None
        for turn, run in enumerate((req.infer_device, req.enqueue, req.infer_device, req.enqueue)):
            if turn == asked and turn:
                shows = held(req)
                assert shows()
            feed(turn)
            run(ins, outs)
            if turn >= asked:
                assert shows(), (asked, turn)
    req = plan.create_request()
    stream = torch.cuda.ExternalStream(req.stream)
    feed(7)
    req.enqueue(ins, outs)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        req.enqueue(ins, outs)
    shows = held(req)
    for turn in range(3):
        feed(10 + turn)
        graph.replay()
        assert shows(), turn


def _tensor(req, node):
    import ctypes
    from dldt_amd._lib import check, lib
    from dldt_amd.tensor import hipie_tensor
    t = hipie_tensor()
    check(lib().hipie_request_tensor(req._h, node, ctypes.byref(t)))
    return t


def _image(t, n):
    """image n of a dense f32 tensor's descriptor as [C, H, W], read at once: no other stream is waited for"""
    import ctypes
    from dldt_amd._lib import check, lib
    values = torch.empty(t.stride_n, dtype=torch.float32)
    check(lib().hipie_memcpy(ctypes.c_void_p(values.data_ptr()), ctypes.c_void_p(t.data + 4 * n * t.stride_n), ctypes.c_size_t(4 * t.stride_n), 0))
    return torch.as_strided(values, (t.c, t.h, t.w), (1, t.stride_h, t.stride_w)) + 0.0


def _block(n, c, hw, oc):
    g = builders.conv_block(n=n, c=c, hw=hw, oc=oc)[0]
    return g, g.nodes[-1]["inputs"][0]


def test_the_call_that_asks_first_waits_for_an_inference_in_flight():
    from dldt_amd._lib import check, lib
    g, node = _block(32, 256, 56, 512)                              # (0.3 ms and more behind the call)
    plan = g.compile(0, config={"HIP_TUNE": "NO", "HIP_SINGLE_LAUNCH": "NO"})
    for seed in range(3):
        req = plan.create_request()
        ins, outs = req.device_buffers()
        ins[0].uniform_(0, 2.55, generator=torch.Generator(device="cuda").manual_seed(seed))
        torch.cuda.synchronize()
        check(lib().hipie_request_start(req._h, *req._ptrs(ins, outs), 1))
        seen = _image(_tensor(req, node), 31)
        req.wait()
        assert torch.equal(seen, outs[0][31].cpu())


@pytest.mark.parametrize("single", ["NO", "64"])
def test_a_tensor_asked_for_by_another_thread_shows_the_inference_beside_it(single):
    """the call comes before, while or after the inference is queued and waited for; when both have returned the values are there"""
    import threading
    import time
    g, node = _block(1, 64, 56, 64)
    plan = g.compile(0, config={"HIP_TUNE": "NO", "HIP_THROUGHPUT_STREAMS": "1", "HIP_SINGLE_LAUNCH": single})
    feed = [torch.rand((1, 64, 56, 56), generator=torch.Generator(device="cuda").manual_seed(k), device="cuda") * 2.55 for k in range(2)]
    for turn in range(60):
        req = plan.create_request()
        _, outs = req.device_buffers()
        torch.cuda.synchronize()
        seen = []

        def ask():
            until = time.perf_counter() + turn * 1e-6
            while time.perf_counter() < until:
                pass
            seen.append(_tensor(req, node))

        other = threading.Thread(target=ask)
        other.start()
        for k in range(2):
            req.infer_device([feed[k]], outs)
        other.join()
        assert torch.equal(_image(seen[0], 0), outs[0][0].cpu()), turn


def test_a_tensor_asked_for_in_a_capture_shows_the_last_inference_behind_it():
    g, node = _block(1, 64, 14, 70)
    plan = g.compile(0, config={"HIP_TUNE": "NO", "HIP_SINGLE_LAUNCH": "NO"})
    req = plan.create_request()
    ins, outs = req.device_buffers()
    later = [torch.empty_like(outs[0])]
    ins[0].uniform_(0, 2.55)
    torch.cuda.synchronize()
    req.enqueue(ins, outs)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.ExternalStream(req.stream), capture_error_mode="thread_local"):
        _tensor(req, node)
        req.enqueue(ins, later)
        _tensor(req, node)
    assert torch.equal(_image(_tensor(req, node), 0), outs[0][0].cpu())      # (nothing of the graph has run)
    for turn in range(3):
        ins[0].uniform_(0, 2.55)
        torch.cuda.synchronize()
        (graph.replay if turn != 1 else lambda: req.enqueue(ins, later))()
        torch.cuda.synchronize()
        assert torch.equal(_image(_tensor(req, node), 0), later[0][0].cpu()), turn
