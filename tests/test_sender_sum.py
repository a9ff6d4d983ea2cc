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
