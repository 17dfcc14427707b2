"""Which calls of the product entry points reach a kernel of the engine, which the library and which are
refused: on the CPU, with tensors that have a device and a shape but no data."""
import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx

from pylon_amd.kernels import ops


def empty(*shape, dtype=torch.bfloat16):
    return torch.empty(*shape, dtype=dtype, device="cuda:0")


@pytest.mark.parametrize("act", ["relu2", "capped", "none", "tanh"])
@pytest.mark.parametrize("rows", [8, 100, 300])
def test_what_is_no_gate_is_refused(rows, act):
    with FakeTensorMode(), pytest.raises(KeyError):
        ops.linear_glu(empty(rows, 256), empty(512, 256), out_dtype=torch.bfloat16, act=act)


# rows and sizes that reach the tiled kernel, and the rows kernel in the library's stead
@pytest.mark.parametrize("rows, n, k", [(300, 512, 256), (100, 2560, 4096), (32, 5120, 2560)])
def test_a_traced_product_is_the_librarys(rows, n, k):
    with FakeTensorMode():
        assert ops.linear(empty(rows, k), empty(n, k)).shape == (rows, n)


def test_a_compiled_product_is_the_librarys():
    """All of it one graph: a check that the compiler cannot see through would refuse or break it."""
    graphs = []
    with FakeTensorMode():
        x, w = empty(300, 256), empty(512, 256)
    compiled = torch.compile(lambda a, b: ops.linear(a, b), fullgraph=True, dynamic=False,
                             backend=lambda graph, example: graphs.append(graph) or graph.forward)
    assert compiled(x, w).shape == (300, 512)
    assert [node.target for node in graphs[0].graph.nodes if node.op == "call_function"] == [torch.nn.functional.linear]


def test_a_product_that_is_followed_is_told_from_one_that_is_not():
    x, w = torch.ones(3, 4), torch.nn.Parameter(torch.ones(2, 4), requires_grad=False)
    seen = []

    def ask(a):
        seen.append(ops._watched(a, w))
        return a * 2

    ask(x)
    ask(x.requires_grad_())
    with torch.no_grad():
        ask(x)
    x = x.detach()
    torch.vmap(ask)(x)
    torch.func.jvp(ask, (x,), (x,))
    with forward_ad.dual_level():
        ask(forward_ad.make_dual(x, x))
    make_fx(ask)(x)
    torch.jit.trace(ask, (x,), check_trace=False)
    ask(x)
    assert seen == [False, True, False, True, True, True, True, True, False]


def test_a_vector_is_the_librarys():
    x, w = torch.empty(300, 256, dtype=torch.bfloat16, device="meta"), torch.empty(256, dtype=torch.bfloat16, device="meta")

    class OnTheDevice(torch.Tensor):  # what the checks ask for, and no more
        is_cuda = True

    assert ops._wide_ok(x.as_subclass(OnTheDevice), w) is False
    with FakeTensorMode():
        assert ops.linear(empty(300, 256), empty(256)).shape == (300,)


@pytest.mark.parametrize("x_on, weight_on, current", [(1, 1, 0), (0, 1, 0), (1, 0, 0), (0, 0, 1)])
def test_operands_of_other_devices_reach_no_kernel(monkeypatch, x_on, weight_on, current):
    """The library goes to its operands' device, or refuses two; a launch would go to the current one."""
    if torch.cuda.device_count() == 1:
        pytest.skip("tensors without data can be put on any device of a machine that has none, or has two")
    monkeypatch.setattr(ops, "_raw_device", lambda: current)
    monkeypatch.setattr(ops, "_watched", lambda x, weight: False)
    launched = []
    monkeypatch.setattr(ops._lib, "call", lambda name, *args: launched.append(name))
    with FakeTensorMode():
        for rows, n, k in ((300, 512, 256), (32, 5120, 2560)):
            x = torch.empty(rows, k, dtype=torch.bfloat16, device=f"cuda:{x_on}")
            w = torch.empty(n, k, dtype=torch.bfloat16, device=f"cuda:{weight_on}")
            if x_on == weight_on:
                assert ops.linear(x, w).device == x.device
            else:
                with pytest.raises(RuntimeError):
                    ops.linear(x, w)
            with pytest.raises(ops.KernelError):
                ops.gemm_wide(x, w)
    assert not launched


@pytest.fixture
def routes(monkeypatch):
    """What the entry points launch or hand to the library, in order; nothing is computed."""
    seen = []
    monkeypatch.setattr(ops, "_raw_device", lambda: 0)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_watched", lambda x, weight: False)
    monkeypatch.setattr(ops, "_dev", lambda t, name, dtype=None: 0)
    monkeypatch.setattr(ops._lib, "compute_units", lambda: 256)
    monkeypatch.setattr(ops._lib, "call", lambda name, *args: seen.append(name.removeprefix("pylon_")))
    real = torch.nn.functional.linear
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w: (seen.append("library"), real(x, w))[1])
    with FakeTensorMode(), warnings.catch_warnings():
        warnings.simplefilter("ignore")  # data pointers of tensors without data
        yield seen


# the widest gate/up matrices, where the library's tiles hold what begins a third one of the tiled kernel: a gate goes
# there, a capped one and a squared relu stay on their float32 sums
@pytest.mark.parametrize("rows, half, own", [(320, 25600, True), (321, 25600, False), (384, 25600, False), (385, 25600, True),
                                             (350, 17408, True), (576, 19200, True), (1344, 9216, True)])
def test_activations_of_very_wide_matrices(routes, rows, half, own):
    x, w = empty(rows, 256), empty(2 * half, 256)
    ops.linear_capped(x, w, alpha=1.702, offset=1.0, limit=7.0, out_dtype=torch.bfloat16)
    ops.linear_relu2(x, w, out_dtype=torch.bfloat16)
    assert routes == ["gemm_wide"] * 2
    routes.clear()
    ops.linear_glu(x, w, out_dtype=torch.bfloat16)
    assert routes == (["gemm_wide"] if own else ["library", "silu_gate"])


# out and down of 4B, 8B and 32B sizes: few tiles, whole rounds, full portions; a q/k/v matrix; more than one rule
@pytest.mark.parametrize("rows, n, k, own", [
    (160, 2560, 9728, True), (512, 2560, 9728, False), (1300, 2560, 9728, True), (2048, 2560, 9728, False),
    (2048, 4096, 12288, True), (700, 4096, 4096, False), (1024, 5120, 25600, True), (2048, 5120, 25600, False),
    (1300, 6144, 4096, True), (2048, 6144, 4096, False)])
def test_products_of_prompt_portions(routes, rows, n, k, own):
    ops.linear(empty(rows, k), empty(n, k))
    ops.linear_for_residual(empty(rows, k), empty(n, k), out_dtype=torch.bfloat16)
    assert routes == ["gemm_wide" if own else "library"] * 2


@pytest.mark.parametrize("rows", [33, 64])
def test_a_head_with_its_rows_apart_is_the_librarys_when_followed(routes, monkeypatch, rows):
    """As one without, which is the library's at so many rows: followed for a gradient, or on another device."""
    x, apart, close = empty(rows, 4096), empty(32768, 4160)[:, :4096], empty(32768, 4096)
    ops.linear(x, apart)
    ops.linear(x, close)
    assert routes == ["gemm_rows", "library"]
    routes.clear()
    monkeypatch.setattr(ops, "_watched", lambda x, weight: True)
    ops.linear(x, apart)
    monkeypatch.setattr(ops, "_watched", lambda x, weight: False)
    monkeypatch.setattr(ops, "_raw_device", lambda: 1)
    ops.linear(x, apart)
    assert routes == ["library"] * 2
