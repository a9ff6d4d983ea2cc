"""Small-graph forms of the convolution kernels: a node's edges dealt out to several waves of a block (forward-shaped
kernels, summed through LDS) or to several walk positions (backward-shaped kernels), against the plain kernels of the
same problem and, on the smallest graphs, the oracle. Degrees from none over fewer than there are waves to a segment cut into
chunks; every kernel structure that has such a form."""

import numpy as np
import pytest
import torch

import openequivariance_amd as oeq
from openequivariance_amd._torch import ops
from openequivariance_amd.core import problems as P
from openequivariance_amd.core.graph import CoordGraph

from gpu_util import err, to_gpu
from oracle import e3nn_ref as R
from oracle.torch_ref import TorchConv

pytestmark = pytest.mark.gpu


def _f64(p):
    p.irrep_dtype = p.weight_dtype = np.float64
    return p


PROBLEMS = {
    "mace-medium": lambda: P.mace_problems()[1],          # two chunks, LDS staging
    "mace-large-f64": lambda: _f64(P.mace_problems()[0]),  # one wave per SIMD
    "config1": P.config1_single_uvu,                      # 64 rows to a wave
    "config2": P.config2_nequip_uvu,                      # two rows to a wave
    "config2-f64": lambda: _f64(P.config2_nequip_uvu()),  # two rows to a wave, staged: lanes hold the edges ahead
    "aspirin": lambda: P.nequip_problems()[1],            # one chunk; sender gradients by the sender walk
    "SevenNet-main": lambda: P.seven_net_problems()[1],   # folded multiplicities, waves share the output segments
    "SevenNet-last": lambda: P.seven_net_problems()[2],   # sender walk over long rows
    "benzene-f64": lambda: _f64(P.nequip_problems()[3]),  # several segments per wave, stores through LDS
    "wide-ragged": lambda: P.ChannelwiseTPP("96x0e+70x1o", "0e+1o+2e", "0e+1o+2e"),
}


def _graph(n, seed, hub):
    """Degrees 0, 1, 2, ... over the first nodes, random ones after that, and one node with ``hub`` edges."""
    rng = np.random.default_rng(seed)
    deg = np.concatenate([np.arange(min(n, 20)), rng.integers(0, 30, size=max(0, n - 20))])
    if hub:
        deg[-1] = hub
    rows = np.repeat(np.arange(n), deg)
    cols = rng.integers(0, n, size=len(rows))
    if hub:
        cols[rng.permutation(len(rows))[:hub]] = min(1, n - 1)
    return CoordGraph(np.zeros((n, 3)), rows.astype(np.int64), cols.astype(np.int64))


def _run(problem, tune, det, g, tensors, monkeypatch):
    monkeypatch.setenv("OEQ_AMD_TUNE", tune)
    conv = oeq.TensorProductConv(problem, deterministic=det)
    monkeypatch.delenv("OEQ_AMD_TUNE")
    e = [torch.tensor(a, device="cuda") for a in (g.rows, g.cols, g.transpose_perm)]
    x, y, w, gr, a, b, c = tensors
    out = [ops.conv_forward(x, y, w, *e, conv.kid), *ops.conv_backward(x, y, w, gr, *e, conv.kid),
           *ops.conv_double_backward(x, y, w, gr, a, b, c, *e, conv.kid)]
    again = ops.conv_forward(x, y, w, *e, conv.kid)
    assert torch.equal(again, out[0]), "the sum over the waves has a fixed order"
    return out


@pytest.mark.parametrize("name", list(PROBLEMS))
@pytest.mark.parametrize("tune,n,hub", [("", 1, 5), ("", 33, 300), ("conv_fsplit=2,conv_parts=3", 40, 0),
                                        ("conv_fsmax=100000,conv_parts=16", 700, 600),
                                        # two waves a node, a node that is walked in chunks, walk positions before and past a block
                                        ("conv_fsplit=2,conv_fsmax=4000", 512, 700),
                                        ("conv_fsplit=2,conv_fsmax=4000", 513, 700),
                                        ("", 3, 900)])
def test_small_forms_match_the_plain_kernels(name, tune, n, hub, monkeypatch):
    problem = PROBLEMS[name]()
    det = n != 33
    g = _graph(n, 3, hub)
    dt = torch.float64 if problem.irrep_dtype == np.float64 else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(1)
    dims = (problem.irreps_in1.dim, problem.irreps_in2.dim, problem.weight_numel, problem.irreps_out.dim)
    shapes = [(n, dims[0]), (g.nnz, dims[1]), (g.nnz, dims[2]), (n, dims[3]), (n, dims[0]), (g.nnz, dims[1]),
              (g.nnz, dims[2])]
    tensors = [torch.randn(*s, device="cuda", dtype=dt, generator=gen) for s in shapes]
    # (the same source as the default knobs': one compilation for both)
    plain = _run(problem, "conv_fsmax=0,conv_parts=0", det, g, tensors, monkeypatch)
    small = _run(problem, tune, det, g, tensors, monkeypatch)
    tol = 1e-12 if dt == torch.float64 else 1e-5
    for i, (got, want) in enumerate(zip(small, plain)):
        scale = max(float(want.abs().max()), 1e-30)
        assert float((got - want).abs().max()) / scale <= tol, (name, i)
    # results per edge do not depend on which position walks the edge
    assert torch.equal(small[2], plain[2]) and torch.equal(small[3], plain[3])
    if n <= 40 and g.nnz < 1000:
        x, y, w, gr, a, b, c = (t.double().cpu() for t in tensors)
        leaves = [t.requires_grad_() for t in (x, y, w)]
        z = TorchConv(R.Problem.from_spec(problem), torch.float64)(*leaves, torch.tensor(g.rows), torch.tensor(g.cols))
        first = torch.autograd.grad(z, leaves, gr.requires_grad_(), create_graph=True)
        second = torch.autograd.grad(first, [*leaves, gr], [a, b, c], allow_unused=True)
        for i, (got, want) in enumerate(zip(small, (z, *first, *second))):
            assert err(got, want.detach().numpy()) <= tol, (name, i)


@pytest.mark.parametrize("in1,in2,out", [("64x0e", "1x4e", "64x4e"), ("64x0e", "1x0e+1x2e+1x4e", "64x0e+64x2e+64x4e"),
                                         ("128x0e", "1x4e", "128x4e"), ("64x0e+64x1o", "1x3o", "64x4e"),
                                         ("64x4e", "1x4e", "64x0e")])
@pytest.mark.parametrize("det", [False, True])
def test_blocks_wider_than_the_staging_buffer(in1, in2, out, det, monkeypatch):
    """Outputs (last problem: rows of the sender walk) whose 9 components do not fit a wave's staging buffer."""
    problem = P.ChannelwiseTPP(in1, in2, out)
    g = _graph(40, 3, 60)
    rng = np.random.default_rng(1)
    x, y, w, gr = (rng.normal(size=s).astype(np.float32) for s in (
        (40, problem.irreps_in1.dim), (g.nnz, problem.irreps_in2.dim), (g.nnz, problem.weight_numel),
        (40, problem.irreps_out.dim)))
    monkeypatch.setenv("OEQ_AMD_TUNE", "conv_dxs=1" if in1 == "64x4e" else "")
    conv = oeq.TensorProductConv(problem, deterministic=det)
    e = [torch.tensor(a, device="cuda") for a in (g.rows, g.cols, g.transpose_perm)]
    tx, ty, tw = to_gpu(x, y, w, requires_grad=True)
    z = conv(tx, ty, tw, *e)
    z.backward(torch.tensor(gr, device="cuda"))
    ref = R.Problem.from_spec(problem)
    want = [R.conv_forward(ref, x, y, w, g.rows, g.cols), *R.conv_backward(ref, x, y, w, gr, g.rows, g.cols)]
    for got, exp in zip((z, tx.grad, ty.grad, tw.grad), want):
        assert err(got, exp) <= 1e-5
