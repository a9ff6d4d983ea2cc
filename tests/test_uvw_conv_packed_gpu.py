"""Forward of the fused 'uvw' convolution with lanes packed by output channel and input channel: widths at and beside the
edges of its vectors (1, 2, 4 channels), of a wave's input channels per step and of the 64-channel segments; weights that
stay in registers and weights that are streamed; the plain scheme beyond the packed one's limits; segments longer than the
64 edge numbers a wave holds and than one chunk; infinite weights next to channels that are not there."""

import numpy as np
import pytest
import torch

import openequivariance_amd as oeq
from openequivariance_amd.codegen.lower import lower
from openequivariance_amd.codegen.uvw import UvwEmitter
from openequivariance_amd.core.graph import CoordGraph
from oracle import e3nn_ref as R
from gpu_util import err, tol_of


def _problem(in1, in2, out, ins, dtype=np.float32):
    return oeq.TPProblem(in1, in2, out, [(*i, "uvw", True) for i in ins], shared_weights=False, internal_weights=False,
                         irrep_dtype=dtype, weight_dtype=dtype, label=f"{in1} x {in2} -> {out}")


# name -> (problem, does every segment fit the packed scheme)
CASES = {
    "10-48": (("10x1o+48x0e", "1x0e+1x1o", "10x1o+48x0e", [(0, 0, 0), (0, 1, 1), (1, 1, 0), (1, 0, 1)]), True),
    "64-80": (("64x0e+16x1o", "1x0e+1x1o", "80x0e+16x1o", [(0, 0, 0), (1, 1, 0), (0, 1, 1), (1, 0, 1)]), True),
    "one-channel": (("1x0e+3x1o", "1x0e+1x1o", "1x0e+1x1o", [(0, 0, 0), (1, 1, 0), (0, 1, 1), (1, 0, 1)]), True),
    "63-65": (("63x0e+65x1o", "1x0e+1x1o", "66x0e+33x1o", [(0, 0, 0), (1, 1, 0), (0, 1, 1), (1, 0, 1)]), True),
    "streamed": (("130x0e+64x1o", "1x0e+1x1o", "64x0e+32x1o", [(0, 0, 0), (1, 1, 0), (0, 1, 1), (1, 0, 1)]), True),
    "second-operand-channels": (("7x1o+20x0e", "3x1o+2x0e", "6x1o+5x0e", [(0, 0, 1), (0, 1, 0), (1, 0, 0)]), True),
    "high-l": (("5x5e+16x2e", "1x3e", "12x4e+6x3e", [(0, 0, 0), (1, 0, 0), (1, 0, 1)]), True),
    "many-jobs": (("16x3e", "25x2e", "16x3e", [(0, 0, 0)]), False),
}


def _make(name, dtype=np.float32):
    return _problem(*CASES[name][0], dtype)


@pytest.mark.parametrize("name", list(CASES))
def test_plan(name):
    em = UvwEmitter(lower(_make(name)))
    plans = [em._pack_plan(io, wc) for io, bo in enumerate(em.low.out) for wc in range(0, bo.mul, 64)]
    assert all(plans) == CASES[name][1]
    for plan, (io, wc) in zip(plans, [(io, wc) for io, bo in enumerate(em.low.out) for wc in range(0, bo.mul, 64)]):
        if plan is None:
            continue
        vw, lanes, groups, jobs, stride = plan
        assert vw * lanes == min(64, em.low.out[io].mul - wc) and 1 <= lanes * groups <= 64
        # every input channel of every path once, and the last step's reads stay inside a row of the tile
        for p in (q for q in em.low.paths if q.io == io):
            seen = sorted(uc + i for q, v, uc, nu, _ in jobs if q is p and v == 0 for i in range(nu))
            assert seen == list(range(em.low.in1[p.i1].mul))
        assert all(-(-nu // groups) * groups <= stride for *_, nu, _ in jobs)


def _graph(n, hub):
    rng = np.random.default_rng(5)
    deg = np.array([0, 1, 2, 63, 64, 65, hub] + [7] * (n - 7))
    rows = np.repeat(np.arange(n), deg)
    return CoordGraph(np.zeros((n, 3)), rows.astype(np.int64), rng.integers(0, n, size=len(rows)).astype(np.int64))


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("dtype,kahan", [(np.float32, False), (np.float32, True), (np.float64, False)])
def test_forward(name, dtype, kahan):
    problem = _make(name, dtype)
    g = _graph(20, 300)
    rng = np.random.default_rng(7)
    x, y, w = (rng.normal(size=s).astype(dtype) for s in ((20, problem.irreps_in1.dim), (g.nnz, problem.irreps_in2.dim),
                                                          (g.nnz, problem.weight_numel)))
    want = R.conv_forward(R.Problem.from_spec(problem), x, y, w, g.rows, g.cols)
    edges = [torch.tensor(a, device="cuda") for a in (g.rows, g.cols, g.transpose_perm)]
    for det in ([True] if kahan else [True, False]):
        conv = oeq.TensorProductConv(problem, deterministic=det, kahan=kahan)
        args = [torch.tensor(a, device="cuda") for a in (x, y, w)] + (edges if det else edges[:2])
        got = conv(*args)
        # (normal inputs: sums of up to 300 edges x 194 channels cancel to about their root of the terms' size)
        assert err(got, want) <= tol_of(problem), (name, det)
        assert torch.equal(got, conv(*args))


@pytest.mark.gpu
def test_infinite_weight_stays_in_its_channel():
    problem = _make("10-48")
    g = _graph(20, 300)
    gen = torch.Generator(device="cuda").manual_seed(2)
    x, y, w = (torch.randn(*s, device="cuda", generator=gen) for s in (
        (20, problem.irreps_in1.dim), (g.nnz, problem.irreps_in2.dim), (g.nnz, problem.weight_numel)))
    edges = [torch.tensor(a, device="cuda") for a in (g.rows, g.cols, g.transpose_perm)]
    conv = oeq.TensorProductConv(problem, deterministic=True)
    clean = conv(x, y, w, *edges)
    # last input channel of the first path (10 -> 10 channels, l=1): output channel 9 of every node with edges
    w[:, 9 * 10 + 9] = float("inf")
    got = conv(x, y, w, *edges)
    hit = torch.zeros(problem.irreps_out.dim, dtype=torch.bool, device="cuda")
    hit[27:30] = True
    assert torch.equal(got[:, ~hit], clean[:, ~hit])
    assert not torch.isfinite(got[1:, hit]).any()
