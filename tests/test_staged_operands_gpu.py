"""Convolution kernels with an edge's operands staged in LDS, against the oracle. Waves that walk two edges side by side:
rows of less than an instruction's 1 024 bytes, of whole instructions and with a rest, blocks without a channel for every
lane, several channels in the second operand; segments without an edge, with odd and even numbers, on either side of the
64 edges whose numbers a wave holds, and cut into chunks. Double precision, a node's outputs shared out between waves that
stage what theirs need: one, two and four of them, paths in and out of the order of their outputs. Blocks of different
widths: a wave per width, one to eight edges side by side."""

import re

import numpy as np
import pytest
import torch

import openequivariance_amd as oeq
from openequivariance_amd import runtime as rt
from openequivariance_amd._torch import ops
from openequivariance_amd.codegen.lower import lower
from openequivariance_amd.codegen.uvu import UvuEmitter, _staged_segments, conv_module
from openequivariance_amd.core import problems as P
from openequivariance_amd.core.graph import CoordGraph
from openequivariance_amd.core.layout import transpose_irrep_layout

from gpu_util import err, to_gpu, tol_of
from oracle import e3nn_ref as R

PROBLEMS = {
    "short": ("32x0e", "0e+1o", "0e+1o"),                            # 128 and 256 bytes
    "whole": ("32x0e+32x1o+32x0o+32x1e", "0e+1o", "0e+1o+1e"),       # X: one instruction
    "rest": ("32x0e+32x1o+32x2e", "0e+1o+2e", "0e+1o+2e"),
    "ragged": ("20x0e+32x1o+4x2e", "0e+1o", "0e+1o+2e"),
    "channels": ("32x0e+32x1o", "2x0e+3x1o", "0e+1o"),
    "lips": None,
    "middle": ("32x0e+32x1o+32x2e", "1o", "0e"),          # paths read one block of X, not the first
    "ragged-middle": ("30x0e+20x1o+24x2e+2x3o", "1o", "0e+3o"),  # two of the four, the first one off a 16-byte boundary
    "holes": ("32x0e+32x1o+32x2e+32x3o", "0e", "0e+2e"),  # the first and the third block, across an instruction boundary
    "ragged-holes": ("18x0e+32x1o+6x2e+20x1e+32x0o", "0e", "0e+2e+0o"),  # three runs, off 16-byte boundaries
    "chunks": ("128x0e+128x1o", "0e+1o+2e", "0e+1o+2e"),  # two waves to a node: dY of eight edges at a time
    "ragged-chunks": ("200x0e+100x1o", "0e+1o", "0e+1o+2e"),
}
# channels, largest l of the first operand and of the harmonics, paths and their order
SHARED = {"one": (128, 1, 2, range(9)), "two": (128, 2, 2, range(18)), "two-shuffled": (128, 2, 2, [k * 7 % 18 for k in range(18)]),
          "four-shuffled": (64, 3, 3, [k * 5 % 34 for k in range(34)])}
# double precision, more than the LDS of a block holds: staged for sixteen waves (with the buffer the rows are stored
# through), two segments of two chunks, more nodes to a block of the sender walk
WIDE = {"sixteen-waves": ("1024x0e+1024x1o+1024x2e+1024x3o", "0e", "0e+1o+2e+3o"),
        "two-segments": ("128x0e+128x1o+128x2e+128x3o", "0e+1o+2e+3o", "0e+0o+1o+1e+2e+2o+3o+3e+4e+4o")}
# blocks of different widths: a wave per width
WIDTHS = {"two": ("64x0e+64x1o+32x2e+32x3o", "0e+1o+2e+3o", "0e+1o+2e"), "three": ("64x0e+32x1o+16x2e", "0e+1o+2e", "0e+1o+2e+3o"),
          "halved": ("64x1o+32x2e+32x3o+32x1e", "0e+1o+2e+3o", "0e+1o+2e+3o"),
          "few-spilled": ("64x0e+64x1o+32x2e+32x3o", "0e+1o+2e+3o", "0e+1o+2e+3o"),
          "eighth": ("64x0e+64x1o+8x2e+8x1e", "0e+1o+2e", "0e+1o+2e+1e"), "ragged-widths": ("100x0e+40x1o+20x2e+9x1e", "0e+1o+2e", "0e+1o+2e+1e")}
DEGREES = [0, 1, 2, 3, 7, 8, 9, 16, 17, 31, 63, 64, 65, 0, 128, 129, 300, 5, 0]


def _problem(name, dtype, layout):
    p = P.nequip_problems()[0] if name == "lips" else P.nequix_problems()[1] if name == "nequix" else P.ChannelwiseTPP(*{**PROBLEMS, **WIDTHS, **WIDE}[name])
    p.irrep_dtype = p.weight_dtype = dtype
    p.layout = layout
    return p


def _shared(name, layout):
    mul, lx, ly, order = SHARED[name]
    paths = [(l1, l2, l3) for l1 in range(lx + 1) for l2 in range(ly + 1) for l3 in range(abs(l1 - l2), min(3, l1 + l2) + 1)]
    in1, in2 = [f"{mul}x{l}e" for l in range(lx + 1)], [f"1x{l}e" for l in range(ly + 1)]
    outs = [f"{mul}x{l3}e" for _, _, l3 in paths[:len(order)]]
    p = oeq.TPProblem("+".join(in1), "+".join(in2), "+".join(outs),
                      [(paths[k][0], paths[k][1], k, "uvu", True) for k in order], shared_weights=False,
                      internal_weights=False, label=f"shared-{name}", irrep_dtype=np.float64, weight_dtype=np.float64)
    p.layout = layout
    return p


@pytest.mark.parametrize("name", ["rest", "ragged", "channels", "lips"])
def test_these_problems_stage_their_rows(name):
    assert UvuEmitter(lower(_problem(name, np.float32, "mul_ir"))).rows_stage is not None


@pytest.mark.parametrize("name,dtype,runs", [
    ("rest", np.float32, [[0, 288, 0]]), ("middle", np.float32, [[32, 128, 0]]), ("middle", np.float64, [[32, 128, 0]]),
    ("ragged-middle", np.float32, [[28, 212, 0]]), ("ragged-middle", np.float64, [[30, 210, 0]]),
    ("holes", np.float32, [[0, 32, 0], [128, 288, 32]]),
    ("ragged-holes", np.float32, [[0, 20, 0], [112, 144, 20], [204, 236, 52]]),
    ("ragged-holes", np.float64, [[0, 18, 0], [114, 144, 18], [204, 236, 48]])])
def test_rows_are_staged_as_far_as_paths_read_them(name, dtype, runs):
    assert UvuEmitter(lower(_problem(name, dtype, "mul_ir"))).rows_stage["runs"] == runs


@pytest.mark.parametrize("problem", [("32x0e+32x1o+32x2e", "0e+1o+2e+3o", "0e+0o+1e+1o+2e+2o"),
                                     ("32x0e+32x0o+32x1e+32x1o", "3x0e+3x1o+2x2e", "0e+0o+1e+1o+2e+2o")])
def test_rows_are_staged_where_that_takes_little_scratch_memory(problem, monkeypatch):
    monkeypatch.delenv("OEQ_AMD_TUNE", raising=False)
    p = P.ChannelwiseTPP(*problem)
    p.irrep_dtype = p.weight_dtype = np.float64
    assert UvuEmitter(lower(p)).rows_stage is not None  # (in one pass with 116 and 352 bytes)
    assert rt.kernel_resources(rt.compile_source(conv_module(lower(p), True)[0]))["forward"][1] <= 80


@pytest.mark.parametrize("in2,dtype,det,staged", [("0e+1o", np.float32, True, False), ("0e+1o", np.float32, False, True),
                                                  ("0e+1o", np.float64, True, True), ("0e+1o+2e", np.float32, True, True)])
def test_short_rows_of_sorted_edges_are_not_staged(in2, dtype, det, staged, monkeypatch):
    monkeypatch.delenv("OEQ_AMD_TUNE", raising=False)
    p = P.ChannelwiseTPP("32x0e", in2, "0e+1o+2e")
    p.irrep_dtype = p.weight_dtype = dtype
    src = conv_module(lower(p), det)[0]
    forward = src[src.index(" void forward(i64"):]
    assert ("global_load_lds" in forward[:forward.index("__global__")]) == staged


@pytest.mark.parametrize("mul", [32, 64, 128])
def test_single_values_in_double_precision_are_not_staged(mul):
    for dtype, in2, staged in ((np.float64, "0e", False), (np.float64, "0e+1o", True), (np.float32, "0e", True)):
        p = P.ChannelwiseTPP(f"{mul}x0e", in2, "0e+1o")
        p.irrep_dtype = p.weight_dtype = dtype
        em = UvuEmitter(lower(p))
        assert ((em.rows_stage if mul == 32 else em.stage) is not None) == staged


@pytest.mark.parametrize("name,waves", [("one", 1), ("two", 2), ("two-shuffled", 2), ("four-shuffled", 4)])
def test_waves_that_share_the_outputs(name, waves):
    em = _staged_segments(lower(_shared(name, "mul_ir")), 8)
    assert len(em.segments) == len(em.stages) == waves


@pytest.mark.parametrize("name", list(WIDE))
def test_staging_leaves_a_block_its_lds(name, monkeypatch):
    monkeypatch.delenv("OEQ_AMD_TUNE", raising=False)
    src = conv_module(lower(_problem(name, np.float64, "mul_ir")), True)[0]
    assert rt.kernel_resources(rt.compile_source(src))["forward"][0] <= 160 * 1024


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(WIDE))
@pytest.mark.parametrize("layout,det", [("mul_ir", True), ("ir_mul", False)])
def test_rows_too_wide_for_staging_against_the_oracle(name, layout, det, monkeypatch):
    _check(_problem(name, np.float64, layout), _problem(name, np.float64, "mul_ir"), det, "conv_fsmax=0", monkeypatch)


def _long_harmonics(in2):
    """Sixteen waves to a node, and more components of the second operand than these have room to collect."""
    return oeq.TPProblem("1024x0e", in2, "1024x0e", [(0, 0, 0, "uvu", True)], shared_weights=False, internal_weights=False,
                         label="long-harmonics", irrep_dtype=np.float64, weight_dtype=np.float64)


@pytest.mark.parametrize("in2", ["1x0e+10x4e", "1x0e+80x3o"])
def test_gradients_of_long_harmonics_leave_a_block_its_lds(in2, monkeypatch):
    monkeypatch.delenv("OEQ_AMD_TUNE", raising=False)
    resources = rt.kernel_resources(rt.compile_source(conv_module(lower(_long_harmonics(in2)), True)[0]))
    assert max(lds for lds, _ in resources.values()) <= 160 * 1024


@pytest.mark.gpu
@pytest.mark.parametrize("det", [True, False])
def test_gradients_of_long_harmonics_against_the_oracle(det, monkeypatch):
    problem = _long_harmonics("1x0e+10x4e")
    _check(problem, problem, det, "conv_fsmax=0", monkeypatch)


@pytest.mark.parametrize("name,rows", [("two", [1, 2]), ("three", [1, 2, 4]), ("halved", [1, 2]), ("eighth", [1, 8]),
                                       ("ragged-widths", [1, 2, 4])])
def test_a_wave_for_every_width(name, rows):
    em = UvuEmitter(lower(_problem(name, np.float32, "mul_ir")))
    assert [g.R for g in em.plan_width_groups()] == rows
    # (forward: a third of the registers, so that a group with many outputs is halved)
    assert [g.R for g in em.plan_forward_groups()] == ([1, 2, 2] if name == "halved" else rows)


def _module(name, layout, det, tune, monkeypatch):
    monkeypatch.setenv("OEQ_AMD_TUNE", tune)
    src = conv_module(lower(_problem(name, np.float32, layout)), det)[0]
    return src, rt.kernel_resources(rt.compile_source(src))


@pytest.mark.parametrize("name", list(WIDTHS))
@pytest.mark.parametrize("layout,det", [("mul_ir", True), ("ir_mul", False)])
def test_the_module_has_a_wave_for_every_width(name, layout, det, monkeypatch):
    """The kernels that the oracle tests below are about: not others that the generator went back to."""
    src, resources = _module(name, layout, det, "conv_wgrp=7", monkeypatch)
    assert "namespace oeq_group0" in src and "namespace oeq_forward_group0" in src
    assert name == "halved" or resources["backward"][1] == 0


@pytest.mark.parametrize("tune", ["", "conv_wgrp=7"])
def test_a_forward_by_width_may_spill_a_few_bytes(tune, monkeypatch):
    src, resources = _module("few-spilled", "mul_ir", True, tune, monkeypatch)
    assert "namespace oeq_forward_group0" in src and resources["forward"][1] <= 16
    # then no lane group stands aside at a node's last edges (what a branch spills, it spills for its own lanes)
    assert ("if (done + r < count)" in src) == (resources["forward"][1] == 0)


@pytest.mark.parametrize("layout,det", [("mul_ir", True), ("ir_mul", False)])
def test_lanes_are_read_outside_of_branches(layout, det, monkeypatch):
    """A lane's value (numbers and senders of the edges ahead) is read by the whole wave, before lanes choose: a spilled
    register is reloaded for the lanes of a branch only. NequiX's main layer held to 168 registers has spilled ones."""
    src, resources = _module("nequix", layout, det, "conv_wgrp=7,conv_wb=3", monkeypatch)
    assert "namespace oeq_group1" in src
    assert not re.search(r"\?[^;\n]*__builtin_amdgcn_readlane", src)
    if not resources["backward"][1]:
        pytest.skip("this compiler fits the kernel into its registers: the oracle test below has no spilled ones")


@pytest.mark.parametrize("xcd", [1, 8])
def test_batches_take_turns_across_positions(xcd, monkeypatch):
    """The half of the dY buffer that is next belongs to the block, whatever number of batches a walk position has: with it
    begun anew at every position, a block that walks two could overwrite rows that a slower wave still adds up."""
    src, _ = _module("two", "mul_ir", True, f"conv_wgrp=7,conv_xcd={xcd}", monkeypatch)
    kernel = src[src.index("void backward(i64 node_count"):]
    assert kernel.index("int batch = 0;") < kernel.index("for (i64 wpos")
    walks = src[src.index("namespace oeq_group0"):src.index("void backward(i64 node_count")]
    assert walks.count("int& batch)") == 2 and "int batch" not in walks


@pytest.mark.gpu
@pytest.mark.parametrize("layout,det", [("mul_ir", True), ("ir_mul", False)])
def test_spilled_operands_against_the_oracle(layout, det, monkeypatch):
    _check(_problem("nequix", np.float32, layout), _problem("nequix", np.float32, "mul_ir"), det, "conv_wgrp=7,conv_wb=3",
           monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(WIDTHS))
@pytest.mark.parametrize("layout,det,tune", [("mul_ir", True, "conv_parts=1"), ("ir_mul", False, "conv_parts=3"),
                                             ("mul_ir", False, "conv_hub=40"), ("mul_ir", True, "conv_fsmax=0"),
                                             ("ir_mul", False, "conv_fsmax=0,conv_hub=40")])
def test_widths_against_the_oracle(name, layout, det, tune, monkeypatch):
    _check(_problem(name, np.float32, layout), _problem(name, np.float32, "mul_ir"), det, "conv_wgrp=7," + tune, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(PROBLEMS))
@pytest.mark.parametrize("dtype,layout,det,tune", [
    (np.float32, "mul_ir", True, "conv_fsmax=0"), (np.float32, "ir_mul", False, "conv_fsmax=0,conv_dxs=1"),
    (np.float64, "mul_ir", False, "conv_fsmax=0,conv_dxs=1"), (np.float32, "mul_ir", False, "conv_fsplit=4")])
def test_against_the_oracle(name, dtype, layout, det, tune, monkeypatch):
    _check(_problem(name, dtype, layout), _problem(name, dtype, "mul_ir"), det, tune, monkeypatch)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(SHARED))
@pytest.mark.parametrize("layout,det,tune", [("mul_ir", True, "conv_fsmax=0"), ("ir_mul", False, "conv_fsmax=0"),
                                             ("mul_ir", False, "conv_fsplit=2")])
def test_shared_outputs_against_the_oracle(name, layout, det, tune, monkeypatch):
    _check(_shared(name, layout), _shared(name, "mul_ir"), det, tune, monkeypatch)


@pytest.mark.gpu
def test_gradients_of_harmonics_where_blocks_take_several_nodes():
    """Shared weights: a bounded grid whose blocks walk one node after the other."""
    problem = oeq.TPProblem("128x0e+128x1o", "1x0e+1x1o", "128x0e+128x1o+128x1o",
                            [(0, 0, 0, "uvu", True), (0, 1, 1, "uvu", True), (1, 0, 2, "uvu", True)], shared_weights=True,
                            internal_weights=False, label="shared-chunks")
    n, rng = 5000, np.random.default_rng(3)
    rows = np.repeat(np.arange(n), rng.integers(0, 20, size=n))
    cols = rng.integers(0, n, size=len(rows))
    x, y, w, gz = (rng.normal(size=s).astype(np.float32) for s in (
        (n, problem.irreps_in1.dim), (len(rows), 4), (problem.weight_numel,), (n, problem.irreps_out.dim)))
    conv = oeq.TensorProductConv(problem)
    tx, ty, tw = to_gpu(x, y, w, requires_grad=True)
    r, c, tg = to_gpu(rows, cols, gz)
    conv(tx, ty, tw, r, c).backward(tg)
    dx, dy, dw = R.conv_backward(R.Problem.from_spec(problem), x, y, w, gz, rows, cols)
    for got, want in ((tx.grad, dx), (ty.grad, dy), (tw.grad, dw)):
        assert err(got, want) <= tol_of(problem)


@pytest.mark.gpu
@pytest.mark.parametrize("name,dtype", [("lips", np.float32), ("chunks", np.float32), ("chunks", np.float64),
                                        ("shared-weights", np.float32)])
def test_operands_that_begin_anywhere(name, dtype):
    """Contiguous views one element into a larger tensor, for kernels that bring operands into LDS 16 bytes at a time:
    the same kernels on the same values, so the same bits."""
    n, edges = len(DEGREES), []
    if name == "shared-weights":
        problem = P.FCTPP("128x0e+128x1o", "1x0e+1x1o", "128x0e+128x1o", shared_weights=True, internal_weights=False)
        module, e, weights = oeq.TensorProduct(problem), n, (problem.weight_numel,)
    else:
        problem = _problem(name, dtype, "mul_ir")
        rows = np.repeat(np.arange(n), DEGREES)
        graph = CoordGraph(np.zeros((n, 3)), rows, np.random.default_rng(3).integers(0, n, size=len(rows)))
        edges = to_gpu(graph.rows, graph.cols, graph.transpose_perm)
        module, e = oeq.TensorProductConv(problem, deterministic=True), len(rows)
        weights = (e, problem.weight_numel)
    rng = np.random.default_rng(5)
    values = to_gpu(*(rng.normal(size=s).astype(dtype) for s in (
        (n, problem.irreps_in1.dim), (e, problem.irreps_in2.dim), weights, (n, problem.irreps_out.dim))))

    def passes(place):
        x, y, w, g = (place(t).requires_grad_(True) for t in values)
        z = module(x, y, w, *edges)
        first = torch.autograd.grad(z, (x, y, w), g, create_graph=True)
        second = torch.autograd.grad(first, (x, y, w, g), [place(2 * t.detach()) for t in first])
        return [t.detach() for t in (z, *first, *second)]

    def inside(t):
        view = t.new_empty(t.numel() + 1)[1:].view(t.shape).copy_(t).detach()
        assert view.is_contiguous() and view.data_ptr() % 16
        return view

    assert all(torch.equal(p, q) for p, q in zip(passes(torch.clone), passes(inside)))
    assert ops.get_entry(module.kid).direct_loads


def _check(problem, plain, det, tune, monkeypatch):
    """Forward and backward of ``problem``, whose ``mul_ir`` form, what the oracle works in, is ``plain``."""
    dtype, layout = problem.irrep_dtype, problem.layout
    n = len(DEGREES)
    rng = np.random.default_rng(7)
    rows = np.repeat(np.arange(n), DEGREES)
    cols = np.where(rng.random(len(rows)) < 0.3, 4, rng.integers(0, n, size=len(rows)))
    g = CoordGraph(np.zeros((n, 3)), rows.astype(np.int64), cols.astype(np.int64))
    x, y, w, gz = (rng.normal(size=s).astype(dtype) for s in (
        (n, problem.irreps_in1.dim), (g.nnz, problem.irreps_in2.dim), (g.nnz, problem.weight_numel),
        (n, problem.irreps_out.dim)))
    ref = R.Problem.from_spec(plain)
    ref_z = R.conv_forward(ref, x, y, w, g.rows, g.cols)
    ref_dx, ref_dy, ref_dw = R.conv_backward(ref, x, y, w, gz, g.rows, g.cols)
    i1, i2, io = problem.irreps_in1, problem.irreps_in2, problem.irreps_out
    x, y, gz, ref_z, ref_dx, ref_dy = (transpose_irrep_layout(a, irreps, "mul_ir", layout) for a, irreps in (
        (x, i1), (y, i2), (gz, io), (ref_z, io), (ref_dx, i1), (ref_dy, i2)))
    monkeypatch.setenv("OEQ_AMD_TUNE", tune)
    conv = oeq.TensorProductConv(problem, deterministic=det)
    tx, ty, tw = to_gpu(x, y, w, requires_grad=True)
    r, c, perm, tg = to_gpu(g.rows, g.cols, g.transpose_perm, gz)
    z = conv(tx, ty, tw, r, c, perm) if det else conv(tx, ty, tw, r, c)
    z.backward(tg)
    for got, want in ((z, ref_z), (tx.grad, ref_dx), (ty.grad, ref_dy), (tw.grad, ref_dw)):
        assert err(got, want) <= tol_of(problem)
