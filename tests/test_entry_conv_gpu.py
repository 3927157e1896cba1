"""A graph input's FakeQuantize and the convolution behind it as one launch (csrc/entry_conv.hip) against the two, bit for bit: the
values in the caller's buffer and the levels in the tensor between them."""
import numpy as np
import pytest
import torch

from dldt_amd import builders
from dldt_amd.graph import Plan
from dldt_amd.tensor import F32

pytestmark = pytest.mark.gpu


def _graph(n, c, h, w, oc, k=3, kind="u8", act="relu"):
    """kind: the input's levels - u8, i8, u8 with a zero point, or u8 values as they are"""
    rng = np.random.default_rng(n * c + h)
    q = builders.QuantizedNet()
    if kind == "bytes":
        a = q.input("data", (n, c, h, w), 255.0, u8=True)
    elif kind == "u8":
        a = q.input("data", (n, c, h, w), 2.55)
    else:
        p = q.g.parameter("data", (n, c, h, w))
        a = q.requantize(p, 1.9, signed=True) if kind == "i8" else q.asymmetric(p, -0.7, 1.9)
    y = q.conv_f32(a, rng.standard_normal((oc, c, k, k), dtype=np.float32) * np.float32(0.1), rng.standard_normal(oc, dtype=np.float32), pads=(k // 2, k // 2), relu=act == "relu")
    if act == "clamp":
        y = q.g.clamp(y, -0.25, 0.5)
    q.g.result(y, "out")
    return q.g, a["node"]


def _compile(g, fuse, **kw):
    return g.compile(0, config=dict({"HIP_FUSE_CONVOLUTIONS": fuse, "HIP_TUNE": "NO", "HIP_SINGLE_LAUNCH": "NO"}, **kw))


def _one(plan):
    return int(plan.step_rt_info(0, "kernels")) == 0


def _run(plan, node, x, offset=0):
    req = plan.create_request()
    ins, outs = req.device_buffers()
    size = x.element_size()
    feed = torch.zeros(x.numel() + 16, dtype=x.dtype, device="cuda")[offset:offset + x.numel()].view(x.shape)
    feed.copy_(x)
    place = torch.full((outs[0].numel() + 16,), float("nan"), device="cuda")
    out = place[offset:offset + outs[0].numel()].view(outs[0].shape)
    torch.cuda.synchronize()
    assert feed.data_ptr() % (16 * size) == offset * size
    req.enqueue([feed], [out])
    torch.cuda.synchronize()
    assert torch.isnan(place[:offset]).all() and torch.isnan(place[offset + out.numel():]).all()
    return out.cpu().numpy().view(np.uint32), req.tensor(node)


def _input(g, seed):
    node = g.nodes[0]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if node["dtype"] != F32:
        return torch.randint(0, 256, node["shape"], generator=gen, device="cuda", dtype=torch.uint8)
    x = torch.randn(node["shape"], generator=gen, device="cuda") * 2
    flat = x.view(-1)
    for i, v in enumerate((float("nan"), float("inf"), -float("inf"), 0.0, -0.0, 1e-40, 3e38, -3e38)):
        flat[i * 7 % flat.numel()::41] = v
    return x


# tiles of one row and of many, a last tile of fewer rows, pixels that end inside a fragment and a wave's chunk, channels that end
# inside a quad, a pixel of four bytes, an odd and an even number of 16-byte pieces, output channels inside a tile of 32, several groups
@pytest.mark.parametrize("n,c,h,w,oc", [(1, 1, 1, 2, 1), (1, 3, 7, 7, 8), (2, 4, 9, 31, 33), (1, 5, 33, 2, 31), (3, 17, 9, 65, 65), (2, 16, 5, 64, 32), (12, 72, 45, 45, 100),
                                        (1, 64, 56, 56, 64), (2, 8, 107, 107, 301), (32, 256, 7, 7, 512), (1, 256, 112, 112, 9), (7, 30, 14, 512, 40), (5, 33, 1, 100, 130)])
def test_one_launch_equals_two(n, c, h, w, oc):
    g, node = _graph(n, c, h, w, oc)
    one, two = _compile(g, "YES"), _compile(g, "NO")
    assert _one(one) and not _one(two)
    for seed, offset in ((1, 0), (2, 1)):                    # (buffers on a 4-byte boundary only)
        x = _input(g, seed)
        got, want = _run(one, node, x, offset), _run(two, node, x, offset)
        assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0])


@pytest.mark.parametrize("kind", ["u8", "i8", "zero point", "bytes"])
@pytest.mark.parametrize("c,k,act", [(3, 3, "clamp"), (3, 7, "relu"), (20, 1, "none"), (20, 5, "clamp"), (40, 3, "none")])
def test_kinds_of_levels_filters_and_activations(kind, c, k, act):
    g, node = _graph(3, c, 13, 19, 37, k, kind, act)
    one, two = _compile(g, "YES"), _compile(g, "NO")
    assert _one(one) and not _one(two)
    x = _input(g, 3)
    got, want = _run(one, node, x), _run(two, node, x)
    assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0])


def test_what_the_kernel_does_not_take_runs_as_two():
    g, node = _graph(1, 20, 4, 600, 8)                         # a row of more pixels than a workgroup's waves hold
    assert not _one(_compile(g, "YES"))
    assert not _one(_compile(_graph(2, 20, 9, 9, 8)[0], "YES", HIP_KEEP_F32="YES"))
    assert not _one(_compile(_graph(2, 20, 9, 9, 8)[0], "AUTO"))   # (not measured)


def test_the_choice_is_kept_in_files_and_exports(tmp_path):
    g, node = _graph(2, 17, 9, 9, 65)
    x = _input(g, 5)
    want = _run(_compile(g, "NO"), node, x)
    path = tmp_path / "choices"
    tuned = _compile(g, "YES", HIP_TUNE="YES", HIP_TUNE_FILE=str(path))
    again = _compile(g, "AUTO", HIP_TUNE="YES", HIP_TUNE_FILE=str(path))
    loaded = Plan.load(tuned.export())
    for plan in (tuned, again, loaded):
        assert _one(plan) and plan.steps[1]["variant"] == tuned.steps[1]["variant"]
        got = _run(plan, node, x)
        assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0])
    assert not _one(_compile(g, "NO", HIP_TUNE="YES", HIP_TUNE_FILE=str(path)))


# images of their own, rows that two workgroups share, several groups of channels over one patch, more workgroups than find a place
@pytest.mark.parametrize("tuned", [False, True])
@pytest.mark.parametrize("n,c,h,w,oc,kind", [(1, 64, 14, 14, 64, "u8"), (12, 72, 45, 45, 72, "u8"), (3, 17, 9, 65, 130, "zero point"), (32, 64, 28, 28, 512, "u8"),
                                             (16, 96, 40, 40, 24, "bytes"), (32, 8, 112, 112, 48, "u8")])
def test_an_output_on_its_input_is_the_result_of_two_launches(n, c, h, w, oc, kind, tuned):
    """the FakeQuantize reads all of its input before the convolution stores anything where the two buffers share a byte"""
    g, node = _graph(n, c, h, w, oc, kind=kind)
    plan = _compile(g, "YES", HIP_TUNE="YES" if tuned else "NO")
    assert _one(plan)
    x = _input(g, 7)
    want = _run(_compile(g, "NO"), node, x)
    results = n * oc * h * w * 4
    size = x.numel() * x.element_size()
    # (whole, the output behind the input's start and in front of it, the last and the first of its bytes, side by side)
    for at in (0, 4 * w, -4 * w, size - 4, 4 - results, size, -results):
        start = max(0, -at)
        place = torch.zeros(start + max(size, at + results) + 64, dtype=torch.uint8, device="cuda")
        feed = place[start:start + size].view(x.dtype).view(x.shape)
        out = place[start + at:start + at + results].view(torch.float32).view(n, oc, h, w)
        req = plan.create_request()
        for run in (req.enqueue, req.infer_device):
            feed.copy_(x)
            torch.cuda.synchronize()
            run([feed], [out])
            torch.cuda.synchronize()
            got = out.cpu().numpy().view(np.uint32)
            assert np.array_equal(got, want[0]) and np.array_equal(req.tensor(node), want[1]), (at, run.__name__)


def _kernels(graph):
    """how many nodes a captured graph has"""
    import ctypes
    (path,) = {line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line}
    n = ctypes.c_size_t()
    assert ctypes.CDLL(path).hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


# as one launch, as two with and without K split over workgroups (whose workspace an inference in front of the capture makes, where
# it runs that layer); in place it is two either way
@pytest.mark.parametrize("variant,in_place", [(64 + 4, False), (64 + 14, False), (64 + 15, True), (4, True), (14, False), (15, True), (22, False)])
def test_a_captured_inference_stores_both_in_its_own_launches(tmp_path, variant, in_place):
    g, node = _graph(3, 128, 9, 31, 128)
    out_node = g.nodes[-1]["inputs"][0]
    path = tmp_path / "choices"
    path.write_text("0 -1\n1 %d\n2 -1\n" % variant)
    plan = _compile(g, "AUTO", HIP_TUNE="YES", HIP_TUNE_FILE=str(path))
    assert plan.steps[1]["variant"] == variant
    want = [_run(_compile(g, "NO"), node, _input(g, seed)) for seed in range(4)]
    req = plan.create_request()
    ins, outs = req.device_buffers()
    feed, out = ins[0], outs[0]
    apart = torch.empty_like(out)
    ins[0].copy_(_input(g, 0))
    torch.cuda.synchronize()
    req.enqueue([feed], [apart])                                   # (once before capturing, into another buffer)
    torch.cuda.synchronize()
    if in_place:
        out = feed
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=torch.cuda.ExternalStream(req.stream), capture_error_mode="thread_local"):
        req.enqueue([feed], [out])
    assert _kernels(graph) == (1 if variant & 64 and not in_place else 2)
    for seed in range(4):
        feed.copy_(_input(g, seed))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want[seed][0])
        assert np.array_equal((req.tensor(out_node) + np.float32(0)).view(np.uint32), want[seed][0]), seed
        assert np.array_equal(req.tensor(node), want[seed][1])


@pytest.mark.parametrize("n,c,h,w,oc", [(1, 3, 7, 7, 8), (2, 4, 9, 31, 33), (12, 72, 45, 45, 100), (5, 33, 1, 100, 130), (3, 20, 13, 21, 5)])
@pytest.mark.parametrize("fuse", ["YES", "NO"])
def test_an_inference_whose_tensor_is_looked_at_stores_both(n, c, h, w, oc, fuse):
    g, node = _graph(n, c, h, w, oc, act="none")
    out_node = g.nodes[-1]["inputs"][0]
    plan = _compile(g, fuse)
    keeps = _compile(g, "NO", HIP_KEEP_F32="YES")                  # (every value in its tensor, the result copied from there)
    req, ref = plan.create_request(), keeps.create_request()
    ins, outs = req.device_buffers()
    for seed in range(3):
        ins[0].copy_(_input(g, seed))
        torch.cuda.synchronize()
        ref.enqueue(ins, outs)
        torch.cuda.synchronize()
        want = outs[0].cpu().numpy().view(np.uint32)
        outs[0].fill_(float("nan"))
        torch.cuda.synchronize()
        req.enqueue(ins, outs)
        torch.cuda.synchronize()
        assert np.array_equal(outs[0].cpu().numpy().view(np.uint32), want)
        assert np.array_equal(req.tensor(out_node).view(np.uint32), ref.tensor(out_node).view(np.uint32))      # (also in the sign of zeros)
