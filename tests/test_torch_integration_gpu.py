"""The ops behave as well-formed torch custom ops: opcheck (schema, fake kernels, autograd
registration), torch.compile, autocast, save/load (cf. the reference's tests/export_test.py:89-225)."""

import io

import numpy as np
import pytest
import torch

import openequivariance_amd as oeq
from openequivariance_amd.core import problems as P
from oracle import e3nn_ref as R
from gpu_util import err, to_gpu, tp_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tp_and_inputs():
    problem = P.config2_nequip_uvu()
    tp = oeq.TensorProduct(problem)
    x, y, w, g = tp_inputs(problem, 48, seed=11)
    z_ref = R.tp_forward(R.Problem.from_spec(problem), x, y, w)
    return problem, tp, (x, y, w, g), z_ref


def test_opcheck_tp(tp_and_inputs):
    problem, tp, (x, y, w, g), _ = tp_and_inputs
    tx, ty, tw = to_gpu(x, y, w, requires_grad=True)
    (tg,) = to_gpu(g)
    torch.library.opcheck(torch.ops.oeq_amd.tp_forward.default, (tx, ty, tw, tp.kid),
                          test_utils=("test_schema", "test_faketensor", "test_autograd_registration"))
    torch.library.opcheck(torch.ops.oeq_amd.tp_backward.default, (tx, ty, tw, tg, tp.kid),
                          test_utils=("test_schema", "test_faketensor", "test_autograd_registration"))


def test_opcheck_conv():
    problem = P.config1_single_uvu()
    conv = oeq.TensorProductConv(problem, deterministic=True)
    rows = torch.tensor([0, 1, 1, 2], device="cuda")
    cols = torch.tensor([1, 0, 2, 1], device="cuda")
    perm = torch.argsort(cols, stable=True)
    X = torch.rand(3, 5, device="cuda", requires_grad=True)
    Y = torch.rand(4, 7, device="cuda", requires_grad=True)
    W = torch.rand(4, 1, device="cuda", requires_grad=True)
    torch.library.opcheck(torch.ops.oeq_amd.conv_forward.default, (X, Y, W, rows, cols, perm, conv.kid),
                          test_utils=("test_schema", "test_faketensor", "test_autograd_registration"))


def test_torch_compile(tp_and_inputs):
    problem, tp, (x, y, w, g), z_ref = tp_and_inputs
    tx, ty, tw = to_gpu(x, y, w, requires_grad=True)
    compiled = torch.compile(lambda a, b, c: tp(a, b, c) * 2.0, fullgraph=True)
    z = compiled(tx, ty, tw)
    assert err(z, 2.0 * z_ref) <= 1e-5
    z.sum().backward()
    dx_ref, _, _ = R.tp_backward(R.Problem.from_spec(problem), x, y, w, 2.0 * np.ones_like(z_ref))
    assert err(tx.grad, dx_ref) <= 1e-5


def test_autocast_runs_in_module_dtype(tp_and_inputs):
    problem, tp, (x, y, w, g), z_ref = tp_and_inputs
    tx, ty, tw = to_gpu(x, y, w)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        z = tp(tx, ty, tw)
    assert z.dtype == torch.float32 and err(z, z_ref) <= 1e-5


def test_save_load_module(tp_and_inputs):
    problem, tp, (x, y, w, g), z_ref = tp_and_inputs
    buf = io.BytesIO()
    torch.save(tp, buf)
    buf.seek(0)
    tp2 = torch.load(buf, weights_only=True)
    assert err(tp2(*to_gpu(x, y, w)), z_ref) <= 1e-5


def test_module_inside_a_model_moves_with_to():
    class Net(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.tp = oeq.TensorProduct(P.config1_single_uvu())
            self.lin = torch.nn.Linear(5, 5)

        def forward(self, x, y, w):
            return self.lin(self.tp(x, y, w))

    net = Net().to("cuda").to(torch.float64)
    x, y, w = (torch.rand(10, n, device="cuda", dtype=torch.float64) for n in (5, 7, 1))
    out = net(x, y, w)
    assert out.dtype == torch.float64 and out.shape == (10, 5)
    assert net.tp.config.irrep_dtype == np.float64


def _module_and_inputs(kind):
    """The reference's export fixtures (tests/export_test.py:18-86): 32x5e (x) 1x3e -> 32x5e, batch of
    1000 rows or the 3-node / 4-edge toy graph."""
    problem = oeq.TPProblem("32x5e", "1x3e", "32x5e", [(0, 0, 0, "uvu", True)], shared_weights=False,
                            internal_weights=False)
    gen = torch.Generator(device="cuda").manual_seed(0)
    if kind == "batch":
        n = 1000
        shapes = [(n, 352), (n, 7), (n, problem.weight_numel)]
        return oeq.TensorProduct(problem), tuple(torch.rand(*s, device="cuda", generator=gen) for s in shapes)
    rows = torch.tensor([0, 1, 1, 2], device="cuda")
    cols = torch.tensor([1, 0, 2, 1], device="cuda")
    X = torch.rand(3, 352, device="cuda", generator=gen)
    Y = torch.rand(4, 7, device="cuda", generator=gen)
    W = torch.rand(4, problem.weight_numel, device="cuda", generator=gen)
    if kind == "conv_atomic":
        return oeq.TensorProductConv(problem, deterministic=False), (X, Y, W, rows, cols)
    return oeq.TensorProductConv(problem, deterministic=True), (X, Y, W, rows, cols, torch.argsort(cols, stable=True))


KINDS = ["batch", "conv_det", "conv_atomic"]


@pytest.mark.parametrize("kind", KINDS)
def test_save_load_compile_export(kind):
    module, inputs = _module_and_inputs(kind)
    expected = module(*inputs)
    buf = io.BytesIO()
    torch.save(module, buf)
    buf.seek(0)
    loaded = torch.load(buf, weights_only=True)
    assert torch.allclose(loaded(*inputs), expected, atol=1e-5)
    assert torch.allclose(torch.compile(module)(*inputs), expected, atol=1e-5)
    exported = torch.export.export(module, args=inputs, strict=False)
    assert torch.allclose(exported.module()(*inputs), expected, atol=1e-5)


@pytest.mark.parametrize("kind", KINDS)
def test_side_stream_matches_default_stream(kind):
    """Kernels, scratch allocations and the per-call CSR build all follow torch's current stream."""
    module, inputs = _module_and_inputs(kind)
    ts = tuple(t.clone().requires_grad_(t.is_floating_point()) for t in inputs)
    expected = module(*ts)
    expected.sum().backward()
    grads = [t.grad.clone() for t in ts[:3]]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    ts2 = tuple(t.detach().clone().requires_grad_(t.is_floating_point()) for t in inputs)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(3):  # back-to-back calls reuse freed scratch blocks on this stream
            z = module(*ts2)
        z.sum().backward()
    side.synchronize()
    assert torch.allclose(z, expected, atol=1e-5)
    for a, b in zip(grads, (t.grad for t in ts2[:3])):
        assert torch.allclose(a, b / 1.0, atol=1e-4)


def test_benchmark_helpers():
    """benchmark_forward / benchmark_backward / benchmark_double_backward keep the reference's call
    signatures and return one positive sample per iteration; kernel-only time does not exceed the time
    of the whole call."""
    from openequivariance_amd.core.graph import CoordGraph, periodic_radius_graph
    problem = P.config2_nequip_uvu()
    tp = oeq.TensorProduct(problem)
    x, y, w, g = tp_inputs(problem, 20000, seed=1)
    whole = tp.benchmark_forward(2, 4, x, y, g, w)
    kernel = tp.benchmark_forward(2, 4, x, y, g, w, with_torch_overhead=False)
    # (two clocks: events inside the C ABI vs. events around the torch call; at 45 us they agree to a few %)
    assert whole.shape == (4,) and np.all(whole > 0) and np.all(kernel > 0) and kernel.min() <= 1.5 * whole.max()
    back = tp.benchmark_backward(2, 3, x, y, g, w, with_torch_overhead=False)
    assert back.shape == (3,) and np.all(back > 0)
    dd_whole = tp.benchmark_double_backward(1, 3, x, y, w, w)
    dd_kernel = tp.benchmark_double_backward(1, 3, x, y, w, w, with_torch_overhead=False)
    assert dd_whole.shape == (3,) and np.all(dd_kernel > 0) and dd_kernel.min() <= 1.5 * dd_whole.max()
    # the second-order map as numpy arrays, against the first-order kernels by linearity in dZ:
    # with zero cotangents for dY and dW, d/d(dZ) = F(A, Y, W)
    a = np.random.default_rng(3).uniform(size=x.shape).astype(np.float32)
    second = tp.double_backward_cpu(x, y, g, w, np.zeros_like(w), a, np.zeros_like(y))
    f_a = tp(*to_gpu(a, y, w)).cpu().numpy()
    assert err(second[3], f_a) <= 1e-5
    coords, rows, cols, _ = periodic_radius_graph(300, 12, 5.0, 0)
    graph = CoordGraph(coords, rows, cols)
    for det in (True, False):
        conv = oeq.TensorProductConv(problem, deterministic=det)
        for stats in (conv.benchmark_forward(1, 3, graph), conv.benchmark_backward(1, 3, graph)):
            assert len(stats["time_millis"]) == 3 and min(stats["time_millis"]) > 0
            assert stats["graph_adj_nnz"] == graph.nnz and min(stats["throughputs_gflops"]) > 0
        stats = conv.benchmark_double_backward(1, 2, graph)
        assert stats["direction"] == "double_backward" and min(stats["time_millis"]) > 0


def test_numpy_interface():
    """forward_cpu / backward_cpu / double_backward_cpu: numpy arrays in, results written into (or
    returned as) numpy arrays, as the reference's correctness harness calls them."""
    from openequivariance_amd.core.graph import CoordGraph, periodic_radius_graph
    problem = P.config2_nequip_uvu()
    ref = R.Problem.from_spec(problem)
    x, y, w, g = tp_inputs(problem, 300, seed=2)
    tp = oeq.TensorProduct(problem)
    z, dx, dy, dw = np.zeros_like(g), np.zeros_like(x), np.zeros_like(y), np.zeros_like(w)
    tp.forward_cpu(x, y, z, w)
    tp.backward_cpu(x, dx, y, dy, g, w, dw)
    for got, want in zip((z, dx, dy, dw), (R.tp_forward(ref, x, y, w),) + tuple(R.tp_backward(ref, x, y, w, g))):
        assert err(got, want) <= 1e-5
    coords, rows, cols, _ = periodic_radius_graph(50, 8.0, 4.0, 1)
    graph = CoordGraph(coords, rows, cols)
    rng = np.random.default_rng(4)
    X = rng.uniform(size=(50, problem.irreps_in1.dim)).astype(np.float32)
    Y = rng.uniform(size=(graph.nnz, problem.irreps_in2.dim)).astype(np.float32)
    W = rng.uniform(size=(graph.nnz, problem.weight_numel)).astype(np.float32)
    G = rng.uniform(size=(50, problem.irreps_out.dim)).astype(np.float32)
    for det in (True, False):
        conv = oeq.TensorProductConv(problem, deterministic=det)
        Z, dX, dY, dW = np.zeros_like(G), np.zeros_like(X), np.zeros_like(Y), np.zeros_like(W)
        conv.forward_cpu(X, Y, W, Z, graph)
        conv.backward_cpu(X, dX, Y, dY, W, dW, G, graph)
        want = (R.conv_forward(ref, X, Y, W, graph.rows, graph.cols),) + tuple(
            R.conv_backward(ref, X, Y, W, G, graph.rows, graph.cols))
        for got, w_ in zip((Z, dX, dY, dW), want):
            assert err(got, w_) <= 1e-5
        # second order with only the X cotangent: d/d(dZ) is the forward pass applied to it
        A = rng.uniform(size=X.shape).astype(np.float32)
        second = conv.double_backward_cpu(X, Y, G, W, np.zeros_like(W), A, np.zeros_like(Y), graph)
        assert err(second[3], R.conv_forward(ref, A, Y, W, graph.rows, graph.cols)) <= 1e-5


def test_conv_under_inference_mode():
    """Edge tensors made under torch.inference_mode() carry no version counter: the ops build the index of
    such an edge list at every call instead of caching it, and the results are the usual ones."""
    from openequivariance_amd._torch import ops
    from openequivariance_amd.core.graph import CoordGraph, periodic_radius_graph
    problem = P.config2_nequip_uvu()
    coords, rows, cols, _ = periodic_radius_graph(50, 8.0, 5.0, seed=3)
    g = CoordGraph(coords, rows, cols)
    rng = np.random.default_rng(3)
    X = rng.normal(size=(50, problem.irreps_in1.dim)).astype(np.float32)
    Y = rng.normal(size=(g.nnz, problem.irreps_in2.dim)).astype(np.float32)
    W = rng.normal(size=(g.nnz, problem.weight_numel)).astype(np.float32)
    z_ref = R.conv_forward(R.Problem.from_spec(problem), X, Y, W, g.rows, g.cols)
    for det in (True, False):
        conv = oeq.TensorProductConv(problem, deterministic=det)
        ops.clear_index_cache()
        with torch.inference_mode():
            tX, tY, tW = to_gpu(X, Y, W)
            tr, tc, tp = (torch.tensor(a, device="cuda") for a in (g.rows, g.cols, g.transpose_perm))
            assert tr.is_inference()
            z = conv(tX, tY, tW, tr, tc, tp if det else None)
            z2 = conv(tX, tY, tW, tr, tc, tp if det else None)
        assert err(z, z_ref) <= 1e-5 and torch.equal(z, z2)
        assert not ops._index_cache, "nothing is kept for tensors whose changes cannot be seen"


def test_nondeterministic_calls_warn_or_raise(monkeypatch):
    """torch.use_deterministic_algorithms: calls that use float atomics are errors, or Python warnings with warn_only,
    in both directions."""
    monkeypatch.setenv("OEQ_AMD_TUNE", "conv_sort=0")
    problem = P.config1_single_uvu()
    conv = oeq.TensorProductConv(problem, deterministic=False)
    x, y, w = (torch.randn(4, n, device="cuda", requires_grad=True)
               for n in (problem.irreps_in1.dim, problem.irreps_in2.dim, problem.weight_numel))
    edges = [torch.tensor([0, 1, 2, 3], device="cuda") for _ in range(2)]
    try:
        torch.use_deterministic_algorithms(True, warn_only=True)
        with pytest.warns(UserWarning, match="deterministic implementation"):
            z = conv(x, y, w, *edges)
        with pytest.warns(UserWarning, match="deterministic implementation"):
            z.sum().backward()
        torch.use_deterministic_algorithms(True)
        with pytest.raises(RuntimeError, match="deterministic implementation"):
            conv(x, y, w, *edges)
    finally:
        torch.use_deterministic_algorithms(False)
