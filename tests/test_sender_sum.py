"""The ordered sum of a sender's dX terms in double precision (codegen/common.py: fixup_backward_kernel) at row lengths that
leave remainders of its 16-byte pieces, against the same rows through the batch product."""

import numpy as np
import pytest
import torch

import openequivariance_amd as oeq
from openequivariance_amd.codegen.common import fixup_backward_kernel


@pytest.mark.parametrize("row,size,width", [(6, 8, 2), (8, 8, 2), (7, 8, 1), (8, 4, 4), (6, 4, 2), (7, 4, 1)])
def test_a_load_is_sixteen_bytes_at_most(row, size, width):
    assert f"#define FX_VEC {width}\n" in fixup_backward_kernel(row, elem_size=size)


@pytest.mark.gpu
@pytest.mark.parametrize("channels", [1, 2, 3, 4, 170])
def test_double_precision_rows(channels):
    irreps = f"{channels}x0e" + ("" if channels % 2 else f"+{channels}x1o")
    problem = oeq.TPProblem(irreps, "1x0e", irreps, [(i, 0, i, "uvu", True) for i in range(1 + (channels % 2 == 0))],
                            shared_weights=False, internal_weights=False, label="sender-sum",
                            irrep_dtype=np.float64, weight_dtype=np.float64)
    rng = np.random.default_rng(channels)
    nodes, edges = 37, 700
    rows, cols = np.sort(rng.integers(0, nodes, edges)), rng.integers(0, nodes - 1, edges)  # the last node sends nothing
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    perm = np.argsort(cols, kind="stable")
    rows, cols, perm = (torch.from_numpy(v).cuda() for v in (rows, cols, perm))
    gen = torch.Generator(device="cuda").manual_seed(channels)
    x, y, w, g = (torch.randn(*s, generator=gen, device="cuda", dtype=torch.float64) for s in
                  ((nodes, problem.irreps_in1.dim), (edges, 1), (edges, problem.weight_numel), (nodes, problem.irreps_out.dim)))
    x.requires_grad_(True)
    got, = torch.autograd.grad(oeq.TensorProductConv(problem, deterministic=True)(x, y, w, rows, cols, perm), x, g)
    z = oeq.TensorProduct(problem)(x[cols], y, w)
    want, = torch.autograd.grad(z, x, g[rows])
    assert not got[-1].any()
    # a sum of some twenty terms: as many roundings of 2^-53
    assert float((got - want).abs().max()) <= 64 * 2.0 ** -53 * float(want.abs().max())


def _wide(dtype, channels=64):
    out = [(0, 0, 0), (1, 1, 0), (0, 1, 1), (1, 0, 1), (1, 2, 1), (0, 2, 2), (1, 1, 2), (1, 2, 2)]  # l of the three irreps
    return oeq.TPProblem(f"{channels}x0e+{channels}x1o", "1x0e+1x1o+1x2e",
                         "+".join(f"{channels}x{l}{'oe'[(a + b) % 2 == 0]}" for a, b, l in out),
                         [(a, b, n, "uvu", True) for n, (a, b, _) in enumerate(out)],
                         shared_weights=False, internal_weights=False, label="default-mode-terms",
                         irrep_dtype=dtype, weight_dtype=dtype)


@pytest.mark.parametrize("channels", [32, 64, 128])
def test_default_mode_adds_by_atomics(channels):
    """Edges in any order, in both precisions: rows that a wave's atomics cover without holes."""
    from openequivariance_amd import runtime as rt
    from openequivariance_amd._torch.tensor_product_conv import build_conv_module
    modes = [build_conv_module(_wide(dtype, channels), False)[1]["dx_mode"] for dtype in (np.float32, np.float64)]
    assert modes == [rt.DX_ATOMIC, rt.DX_ATOMIC]


@pytest.mark.gpu
@pytest.mark.parametrize("channels,nodes,edges", [(32, 40, 700), (64, 37, 900), (64, 9000, 20000), (128, 40, 700)])
def test_double_precision_default_mode(channels, nodes, edges):
    """Unsorted edges, the first half of them from one sender (more than a chunk of its sum holds), none from the last node; the
    index in one launch, and in slices. Two passes agree in every bit of dY and dW; dX is added up by atomics."""
    problem = _wide(np.float64, channels)
    rng = np.random.default_rng(channels + nodes)
    rows, cols = rng.integers(0, nodes, edges), rng.integers(0, nodes - 1, edges)
    cols[:edges // 2] = 3
    shuffle = rng.permutation(edges)
    rows, cols = (torch.from_numpy(v[shuffle]).cuda() for v in (rows, cols))
    gen = torch.Generator(device="cuda").manual_seed(channels)
    x, y, w, g = (torch.randn(*s, generator=gen, device="cuda", dtype=torch.float64) for s in
                  ((nodes, problem.irreps_in1.dim), (edges, 9), (edges, problem.weight_numel), (nodes, problem.irreps_out.dim)))
    leaves = tuple(t.requires_grad_(True) for t in (x, y, w))
    conv = oeq.TensorProductConv(problem)
    got = torch.autograd.grad(conv(x, y, w, rows, cols), leaves, g)
    again = torch.autograd.grad(conv(x, y, w, rows.clone(), cols.clone()), leaves, g)
    assert all(torch.equal(a, b) for a, b in zip(got[1:], again[1:]))
    want = torch.autograd.grad(oeq.TensorProduct(problem)(x[cols], y, w), leaves, g[rows])
    assert not got[0][-1].any()
    # sums of up to n terms, in another order: their roundings add up to n 2^-53 of the terms' sizes at most
    n = int(torch.bincount(cols).max()) + 16
    for a, b in zip((*got, again[0]), (*want, want[0])):
        assert float((a - b).abs().max()) <= n * 2.0 ** -53 * float(b.abs().max())


@pytest.mark.parametrize("dtype,paths,walk", [(np.float32, 5, True), (np.float64, 4, True), (np.float64, 5, False)])
def test_up_to_which_ratio_the_senders_are_walked(dtype, paths, walk):
    """Words of an edge's weights and an output row against those of an X row: 3 with four paths, 4 with five."""
    from openequivariance_amd import runtime as rt
    from openequivariance_amd._torch.tensor_product_conv import build_conv_module
    ins = [(0, 0, 0, "uvu", True), (0, 1, 1, "uvu", True), (1, 0, 2, "uvu", True), (1, 1, 3, "uvu", True), (1, 1, 4, "uvu", True)]
    out = ["64x0e", "64x1o", "64x1o", "64x0e", "64x1e"]
    problem = oeq.TPProblem("64x0e+64x1o", "1x0e+1x1o", "+".join(out[:paths]), ins[:paths], shared_weights=False,
                            internal_weights=False, label="sender-ratio", irrep_dtype=dtype, weight_dtype=dtype)
    for deterministic in (False, True):
        assert build_conv_module(problem, deterministic)[1]["dx_mode"] == (rt.DX_SENDER_WALK if walk else rt.DX_TERMS)


@pytest.mark.parametrize("dtype,instruction", [(np.float32, "global_atomic_add_f32"), (np.float64, "global_atomic_add_f64")])
def test_atomics_are_one_instruction(dtype, instruction, tmp_path, monkeypatch):
    """Not a loop of compare-and-swap, whichever compiler it is."""
    import subprocess
    from pathlib import Path
    from openequivariance_amd import runtime as rt
    from openequivariance_amd._torch.tensor_product_conv import build_conv_module
    objdump = Path("/opt/rocm/llvm/bin/llvm-objdump")
    if not objdump.exists():
        pytest.skip("no disassembler")
    monkeypatch.setenv("OEQ_AMD_TUNE", "conv_dxm=1")
    code = rt.unpack_code(rt.compile_source(build_conv_module(_wide(dtype, 64), False)[0]))
    text = ""
    for n, blob in enumerate(code):
        (tmp_path / f"{n}.co").write_bytes(blob)
        text += subprocess.run([objdump, "-d", "--mcpu=gfx950", tmp_path / f"{n}.co"], capture_output=True, text=True, check=True).stdout
    assert instruction in text and "cmpswap" not in text


@pytest.mark.gpu
@pytest.mark.parametrize("deterministic", [False, True])
def test_no_room_for_the_terms(deterministic, monkeypatch):
    """Double precision at a ratio of 4, where the terms are the faster form: without room for them the senders are walked."""
    channels, edges, nodes = 64, 60000, 2000
    ins = [(0, 0, 0, "uvu", True), (0, 1, 1, "uvu", True), (1, 0, 2, "uvu", True), (1, 1, 3, "uvu", True), (1, 1, 4, "uvu", True)]
    problem = oeq.TPProblem(f"{channels}x0e+{channels}x1o", "1x0e+1x1o", "+".join(f"{channels}x{r}" for r in ("0e", "1o", "1o", "0e", "1e")),
                            ins, shared_weights=False, internal_weights=False, label="no-room", irrep_dtype=np.float64,
                            weight_dtype=np.float64)
    rng = np.random.default_rng(5)
    rows, cols = np.sort(rng.integers(0, nodes, edges)), rng.integers(0, nodes, edges)
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    where = [torch.from_numpy(v).cuda() for v in (rows, cols, np.argsort(cols, kind="stable"))][:3 if deterministic else 2]
    gen = torch.Generator(device="cuda").manual_seed(5)
    x, y, w, g = (torch.randn(*s, generator=gen, device="cuda", dtype=torch.float64) for s in
                  ((nodes, problem.irreps_in1.dim), (edges, 4), (edges, problem.weight_numel), (nodes, problem.irreps_out.dim)))
    leaves = tuple(t.requires_grad_(True) for t in (x, y, w))
    conv = oeq.TensorProductConv(problem, deterministic=deterministic)
    backward = lambda: torch.autograd.grad(conv(*leaves, *where), leaves, g)
    want = backward()
    terms = edges * problem.irreps_in1.dim * 8  # bytes; the results take nearly as many again
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    fill = []
    try:
        # (room in what torch holds already is filled first)
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            while True:
                fill.append(torch.empty(terms // 8, dtype=torch.uint8, device="cuda"))
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + sum(t.nbytes for t in want) + terms * 0.6) / total)
        got = backward()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    monkeypatch.setenv("OEQ_AMD_TUNE", "conv_dxs=1")
    conv = oeq.TensorProductConv(problem, deterministic=deterministic)
    assert all(torch.equal(a, b) for a, b in zip(got, backward()))
    n = int(torch.bincount(where[1]).max()) + 16
    for a, b in zip(got, want):
        assert float((a - b).abs().max()) <= n * 2.0 ** -53 * float(b.abs().max())
