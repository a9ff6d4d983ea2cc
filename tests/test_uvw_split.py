"""Split-operand matrix kernels of shared-weight 'uvw' products (codegen/uvw_split.py): which problems they take, that their
kernels cover every sub-path once, and their results at tile, step and grid boundaries against the float64 oracle."""

import numpy as np
import pytest
import torch

import openequivariance_amd as oeq
from openequivariance_amd._torch.tensor_product import build_tp_module
from openequivariance_amd.codegen.lower import lower
from openequivariance_amd.codegen.uvw_split import SplitEmitter
from openequivariance_amd.core import problems as P
from oracle import e3nn_ref as R


def _shared(in1, in2, out, dtype=np.float32):
    return P.FullyConnectedTPProblem(in1, in2, out, shared_weights=True, internal_weights=False, label="split",
                                     irrep_dtype=dtype, weight_dtype=dtype)


def _gaps():  # an input irrep that no path reads, an output irrep that no path writes
    return oeq.TPProblem("32x0e+48x1o+20x2e", "1x0e+1x1o", "32x0e+16x1e+64x1o",
                         [(0, 0, 0, "uvw", True), (0, 1, 2, "uvw", True), (1, 0, 2, "uvw", True, 0.6),
                          (1, 1, 0, "uvw", True)], shared_weights=True, internal_weights=False, label="split-gaps")


def _zero_weight():  # a path that contributes nothing, and whose weights get no gradient
    return oeq.TPProblem("64x0e+64x1o", "1x0e+1x1o", "64x0e+64x1o",
                         [(0, 0, 0, "uvw", True), (0, 1, 1, "uvw", True, 0.0), (1, 0, 1, "uvw", True)],
                         shared_weights=True, internal_weights=False, label="split-zero-weight")


# (name, problem, waves per SIMD of forward and backward)
CASES = [
    ("l2-64", P.config4_uvw_shared, 1, 1),
    ("l2-32", lambda: _shared("32x0e+32x1o+32x2e", "1x0e+1x1o+1x2e", "32x0e+32x1o+32x2e"), 1, 1),
    ("l1-64-16", lambda: _shared("64x0e+16x1o", "1x0e+1x1o", "64x0e+16x1o"), 2, 2),
    ("odd-channels", lambda: _shared("33x0e+17x1o", "1x0e+1x1o", "15x0e+7x1o"), 2, 2),
    ("two-channel-second-operand", lambda: _shared("64x0e+32x1o", "3x0e+2x1o", "64x0e+32x1o"), 1, 1),
    ("gaps", _gaps, 2, 1),
    ("zero-path-weight", _zero_weight, 2, 1),
    # sixteen input channels: the waves of dW side by side along the output channels
    ("narrow-input", lambda: _shared("16x0e+16x1o", "1x0e+1x1o", "64x0e+32x1o"), 2, 2),
    # two components of the output: two steps of dX's pipeline
    ("two-scalars", lambda: _shared("64x0e+64x1o", "1x0e+1x1o", "64x0e+32x0e"), 2, 2),
]


@pytest.mark.parametrize("name,make,wf,wb", CASES, ids=[c[0] for c in CASES])
def test_plan_covers_every_sub_path_once(name, make, wf, wb):
    low = lower(make())
    em = SplitEmitter(low)
    assert em.supported("forward") and em.supported("dx")
    assert (em.waves("forward"), em.waves("dx")) == (wf, wb)
    for plan in (em.plan("forward"), em.plan("dx"), em.plan_dw()):
        assert sorted(q.index for subs in plan for q in subs) == list(range(len(em.subs)))
    for subs in em.plan_dw():
        stages = em.stages_dw(subs)
        assert {q.index for _, _, q in stages} == {q.index for q in subs}
        assert all(any(k == kk for _, _, kk, _ in q.p.nnz) for _, k, q in stages)
    src, _, descs = build_tp_module(make())
    assert "oeq_split3(" in src and any(d[1] == "backward_w" for d in descs)


@pytest.mark.parametrize("name,make,wf,wb", CASES, ids=[c[0] for c in CASES])
def test_shares_of_dy_are_read_before_the_barrier(name, make, wf, wb):
    """A tile's step 0 writes the shares that the tile before reads: not one read of them past that tile's barrier."""
    loops = build_tp_module(make())[0].split("tile += gridDim.x, cur ^= 1)")[1:]
    found = 0
    for loop in loops:
        loop = loop[:loop.index("prow0 = row0;")]
        reads = [at for at in range(len(loop)) if loop.startswith("s_dy[cur][", at)]
        found += len(reads)
        assert loop.count("oeq_block_sync();") == 1 and all(at < loop.index("oeq_block_sync();") for at in reads)
    assert found


# (problem, sub-paths contracted before the product in the forward, and in each kernel of dW)
FOLDS = [("l2-64", 2, [0, 1, 1]), ("l2-32", 2, [2]), ("l1-64-16", 1, [1]), ("odd-channels", 1, [1]),
         ("two-channel-second-operand", 2, [2]), ("gaps", 1, [1]), ("two-scalars", 1, [0]), ("zero-path-weight", 0, [1]), ("narrow-input", 1, [1])]


@pytest.mark.parametrize("name,forward,dw", FOLDS, ids=[f[0] for f in FOLDS])
def test_contracted_first_are_paths_with_one_component_on_the_other_side(name, forward, dw):
    low = lower(next(c[1] for c in CASES if c[0] == name)())
    em = SplitEmitter(low)
    found = [q for subs in em.plan("forward") for q in em.folds("forward", subs)]
    assert len(found) == forward and all(low.out[q.p.io].d == 1 < low.in1[q.p.i1].d for q in found)
    assert not any(em.folds("dx", subs) for subs in em.plan("dx"))
    assert [len(em.folds_dw(subs)) for subs in em.plan_dw()] == dw
    for subs in em.plan_dw():
        folds = em.folds_dw(subs)
        assert all(low.in1[q.p.i1].d == 1 < low.out[q.p.io].d for q in folds)
        stages = em.stages_dw(subs, folds)
        assert {q.index for _, _, q in stages} == {q.index for q in subs} and len(stages) >= 3
        assert [sum(q is f for _, _, q in stages) for f in folds] == [1] * len(folds)


def test_takes_only_what_it_is_made_for():
    for problem in (_shared("64x0e+64x1o", "1x0e+1x1o", "64x0e+64x1o", np.float64),   # fp64
                    _shared("128x0e+128x1o", "1x0e+1x1o", "64x0e+64x1o"),             # blocks of more than 64 channels
                    _shared("8x0e+8x1o", "1x0e+1x1o", "8x0e+8x1o"),                   # tiles that are mostly padding
                    _shared("64x0e", "1x0e", "64x0e")):                               # a single component
        em = SplitEmitter(lower(problem))
        assert not em.supported("forward") and not em.supported("dx")
        assert "oeq_split3(" not in build_tp_module(problem)[0]


# A result is a sum of at most some thirty roundings of 2^-24 of its size, or a sum over rows that are as near: 2-norm.
TOL = 16 * 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("name,make,wf,wb", CASES, ids=[c[0] for c in CASES])
def test_boundaries_match_oracle(name, make, wf, wb):
    """1 to 33 rows: below, at and past a tile of 16 and a step of 32. Then three tiles for some blocks and two for the
    others, and a last tile of five rows; there the output gradient is zero but at rows where mistakes would hide, so that
    the oracle's weight gradient needs these rows only."""
    from openequivariance_amd._torch import ops
    problem = make()
    ref = R.Problem.from_spec(problem)
    tp = oeq.TensorProduct(problem)
    for B in (1, 15, 16, 17, 31, 32, 33, 16 * 256 * max(wf, wb) * 2 + 21):
        gen = torch.Generator(device="cuda").manual_seed(B)
        x, y, g = (torch.randn(B, d, device="cuda", generator=gen)
                   for d in (problem.irreps_in1.dim, problem.irreps_in2.dim, problem.irreps_out.dim))
        w = torch.randn(problem.weight_numel, device="cuda", generator=gen)
        at = sorted({r for r in (0, 15, 16, 31, 32, 4095, 4096, 4111, 8191, 8192, B // 2, B - 21, B - 6, B - 5, B - 1)
                     if 0 <= r < B}) if B > 33 else list(range(B))
        if B > 33:
            keep = torch.zeros(B, 1, device="cuda")
            keep[at] = 1.0
            g *= keep
        z = ops.tp_forward(x, y, w, tp.kid)
        dx, dy, dw = ops.tp_backward(x, y, w, g, tp.kid)
        xs, ys, gs = (t[at].cpu().numpy() for t in (x, y, g))
        want = (R.tp_forward(ref, xs, ys, w.cpu().numpy()), *R.tp_backward(ref, xs, ys, w.cpu().numpy(), gs))
        for got, exact in zip((z[at], dx[at], dy[at], dw), want):
            off = np.linalg.norm(got.cpu().numpy().astype(np.float64) - exact) / np.linalg.norm(exact)
            assert off <= TOL, (name, B, off)
        if B > 33:
            assert not (dx * (1 - keep)).any() and not (dy * (1 - keep)).any()
        again = ops.tp_backward(x, y, w, g, tp.kid)
        assert all(torch.equal(a, b) for a, b in zip((dx, dy, dw), again))
    # an infinity and a NaN stay in their rows
    x[3, 0], x[20, 1] = float("inf"), float("nan")
    z2 = ops.tp_forward(x, y, w, tp.kid)
    rows = torch.arange(len(z2), device="cuda")
    assert not torch.isfinite(z2[3]).all() and not torch.isfinite(z2[20]).all()
    clean = (rows != 3) & (rows != 20)
    assert torch.equal(z2[clean], z[clean])


# (problem, kernels on split operands of the forward and the backward pass, waves per SIMD of each)
SPILLS = [
    # as estimated, forward 712 bytes a lane at one wave per SIMD; 120 at two, a tile that is mostly padding
    (("8x0e+20x1o+48x2e", "1x0e+1x1o+1x2e+2x3o", "64x0o+40x0o+64x2o+32x3o"), 0, 1),
    (("40x0o+16x2o", "1x0e+1x1o+1x2e+1x3o", "64x0e+40x1o+8x1e"), 0, 0),
    # at two waves forward 472 and backward 100 bytes, none at one
    (("40x0e+40x2o", "1x0e+2x1o", "64x0o+48x1o+64x2e"), 1, 1),
    (("48x0e+48x1o", "1x0e+1x1o", "48x0e+48x1o"), 2, 1),
]


@pytest.mark.parametrize("irreps,wf,wb", SPILLS)
def test_kernels_that_spill_are_not_used(irreps, wf, wb):
    from openequivariance_amd import runtime as rt
    from openequivariance_amd.codegen.uvw_mfma import SPLIT_SCRATCH
    src, _, descs = build_tp_module(_shared(*irreps))
    scratch = rt.kernel_resources(rt.compile_source(src))
    for role, name, waves in ((rt.ROLE_TP_FORWARD, "forward", wf), (rt.ROLE_TP_BACKWARD, "backward", wb)):
        kernels = [d for d in descs if d[0] == role]
        body = src.split(f"void {name}(")[1].split('extern "C"')[0]
        assert ("oeq_split8" in body or "oeq_split_part" in body) == bool(waves)
        if waves:
            assert f"amdgpu_waves_per_eu({waves}, {waves})" in src.split(f"void {name}(")[0].split('extern "C"')[-1]
            assert all(d[4] == 256 * waves and scratch[d[1]][1] <= SPLIT_SCRATCH[waves] for d in kernels)


def test_cases_cover_the_forms_of_dw():
    """Waves along input and output channels, and numbers of stages, whose parity decides which operands a step begins with."""
    forms, stages = set(), set()
    for _, make, _, _ in CASES:
        em = SplitEmitter(lower(make()))
        for subs in em.plan_dw():
            forms.add(em.split_dw(subs)[:2])
            stages.add(len(em.stages_dw(subs, em.folds_dw(subs))) % 2)
    assert forms == {(4, 1), (2, 2), (1, 4)} and stages == {0, 1}


@pytest.mark.gpu
@pytest.mark.parametrize("name,make,wf,wb", CASES, ids=[c[0] for c in CASES])
def test_many_steps_a_block(name, make, wf, wb):
    """Four or five steps of dW for every block and nine or ten tiles: buffers in turn and the third copy of Y come around again.
    Against the kernels in double precision, all of the results."""
    from openequivariance_amd import runtime as rt
    from openequivariance_amd._torch import ops
    problem, double = make(), make()
    double.irrep_dtype = double.weight_dtype = np.float64
    kid, exact_kid = oeq.TensorProduct(problem).kid, oeq.TensorProduct(double).kid
    blocks = max(d[4] for d in build_tp_module(problem)[2] if d[0] in (rt.ROLE_TP_FORWARD, rt.ROLE_TP_BACKWARD))
    B = 32 * (4 * blocks + 21) + 5
    gen = torch.Generator(device="cuda").manual_seed(7)
    x, y, g = (torch.randn(B, d, device="cuda", generator=gen)
               for d in (problem.irreps_in1.dim, problem.irreps_in2.dim, problem.irreps_out.dim))
    w = torch.randn(problem.weight_numel, device="cuda", generator=gen)
    run = lambda kid, x, y, w, g: (ops.tp_forward(x, y, w, kid), *ops.tp_backward(x, y, w, g, kid))
    for got, exact in zip(run(kid, x, y, w, g), run(exact_kid, *(t.double() for t in (x, y, w, g)))):
        assert float((got.double() - exact).norm() / exact.norm()) <= TOL


def _fp32(problem):
    """The kernel set of the problem on fp32 matrix instructions."""
    from openequivariance_amd._torch import ops
    with ops._tune_env("uvw_split=0"):
        return ops.register_spec(ops.make_spec("tp", problem))


def _off(got, want):
    """The 2-norm of the difference. Infinities in the same places, NaN nowhere else (the fp32 kernels have some more: zeros
    that pad a tile meet infinities)."""
    known = ~torch.isnan(want)
    got, want = got[known], want[known]
    assert not torch.isnan(got).any() and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])
    a, b = got[torch.isfinite(got)].double(), want[torch.isfinite(got)].double()
    return float((a - b).norm() / b.norm()) if bool(b.any()) else float(a.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("name,make,wf,wb", CASES, ids=[c[0] for c in CASES])
def test_operands_that_three_parts_do_not_hold(name, make, wf, wb):
    """Infinities, the largest numbers, numbers near the smallest: rows that have one are what the fp32 instructions make of
    them, rows beside them keep their bits."""
    from openequivariance_amd._torch import ops
    problem = make()
    tp, plain = oeq.TensorProduct(problem), _fp32(problem)
    for B in (40, 16 * 256 * max(wf, wb) * 2 + 21) + ((16 * 512 * 33 + 5,) if name == "two-scalars" else ()):
        gen = torch.Generator(device="cuda").manual_seed(B)
        x, y, g = (torch.randn(B, d, device="cuda", generator=gen)
                   for d in (problem.irreps_in1.dim, problem.irreps_in2.dim, problem.irreps_out.dim))
        w = torch.randn(problem.weight_numel, device="cuda", generator=gen)
        z, (dx, dy, _) = ops.tp_forward(x, y, w, tp.kid), ops.tp_backward(x, y, w, g, tp.kid)
        rows = dict(zip(("inf", "-inf", "large x", "large dZ", "small", "smallest", "nan"), (3, 17, B // 2, B // 2 + 1, B - 9, B - 2, B - 1)))
        clean = torch.ones(B, dtype=torch.bool, device="cuda")
        clean[list(rows.values())] = False
        xs, gs, ys = x.clone(), g.clone(), y.clone()
        for t in (xs, gs):
            t[rows["inf"], 0], t[rows["-inf"], -1], t[rows["nan"], 1] = float("inf"), float("-inf"), float("nan")
            t[rows["small"]] *= 2.0 ** -112
            t[rows["smallest"]] *= 2.0 ** -124
        xs[rows["large x"], 0] = gs[rows["large dZ"], 0] = 3.4e38
        # (the other operands small, so that no result is near the end of the range)
        ys[rows["large x"]] *= 2.0 ** -40
        gs[rows["large x"]] *= 2.0 ** -40
        ys[rows["large dZ"]] *= 2.0 ** -40
        xs[rows["large dZ"]] *= 2.0 ** -40
        got = (ops.tp_forward(xs, ys, w, tp.kid), *ops.tp_backward(xs, ys, w, gs, tp.kid)[:2])
        want = (ops.tp_forward(xs, ys, w, plain), *ops.tp_backward(xs, ys, w, gs, plain)[:2])
        for n, (a, b, before) in enumerate(zip(got, want, (z, dx, dy))):
            assert torch.equal(a[clean], before[clean]), (B, n)
            for kind, r in rows.items():
                # (results near 2^-124 are sums of some hundred terms, each of which is rounded to multiples of 2^-149)
                assert _off(a[r], b[r]) <= (TOL if kind != "smallest" else 100 * 2.0 ** -25), (B, n, kind)
        # a weight that three parts do not hold: every row
        for value in (2.0 ** -120 * 1.37, float("inf")):
            wt = w.clone()
            wt[5] = value
            got = (ops.tp_forward(x, y, wt, tp.kid), *ops.tp_backward(x, y, wt, g, tp.kid)[:2])
            want = (ops.tp_forward(x, y, wt, plain), *ops.tp_backward(x, y, wt, g, plain)[:2])
            for a, b in zip(got, want):
                assert _off(a, b) <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("name,make,wf,wb", CASES, ids=[c[0] for c in CASES])
def test_weight_gradients_of_operands_that_three_parts_do_not_hold(name, make, wf, wb):
    from openequivariance_amd._torch import ops
    problem = make()
    tp, plain = oeq.TensorProduct(problem), _fp32(problem)
    for B in (40, 16 * 256 * max(wf, wb) * 2 + 21):
        gen = torch.Generator(device="cuda").manual_seed(B)
        x, y, g = (torch.randn(B, d, device="cuda", generator=gen)
                   for d in (problem.irreps_in1.dim, problem.irreps_in2.dim, problem.irreps_out.dim))
        w = torch.randn(problem.weight_numel, device="cuda", generator=gen)
        gradient = lambda x, y, g, kid=tp.kid: ops.tp_backward(x, y, w, g, kid)[2]
        dw = gradient(x, y, g)
        # powers of two change no bit: numbers near the smallest, and large ones
        for sx, sg in ((2.0 ** -100, 1.0), (1.0, 2.0 ** -100), (2.0 ** 40, 2.0 ** 20)):
            assert torch.equal(gradient(x * sx, y, g * sg) * (1 / sx) * (1 / sg), dw), (B, sx, sg)
        # sums that leave the range on the way, and come back; x near the smallest; the largest numbers, infinities, NaN
        for sx, sg in ((2.0 ** 60, 2.0 ** 40), (2.0 ** -124, 2.0 ** 30)):
            assert _off(gradient(x * sx, y, g * sg), gradient(x * sx, y, g * sg, plain)) <= 2 * TOL, (B, sx, sg)
        for where, value in ((x, 3.4e38), (g, -3.4e38), (x, float("inf")), (g, float("-inf")), (y, float("inf")), (x, float("nan"))):
            small = [t * 2.0 ** -40 if abs(value) < 1e39 else t for t in (x, y, g)]
            at = [t is where for t in (x, y, g)].index(True)
            small[at] = where.clone()
            small[at][B - 3, 0] = value
            assert _off(gradient(*small), gradient(*small, plain)) <= 2 * TOL, (B, at, value)


@pytest.mark.gpu
@pytest.mark.parametrize("irreps", [("64x0e+64x1o+64x2e", "1x0e+1x1o+1x2e"), ("64x0e+16x1o", "1x0e+1x1o")])
def test_errors_have_no_mean(irreps):
    """Y of l = 0 is one, as spherical harmonics are: nothing else gives an error either sign. Against the kernels in double
    precision, on an even number of blocks of as many tiles each."""
    from openequivariance_amd._torch import ops
    kids = [oeq.TensorProduct(_shared(*irreps, irreps[0], dtype)).kid for dtype in (np.float32, np.float64)]
    problem = _shared(*irreps, irreps[0])
    B = 16 * 512 * 4
    gen = torch.Generator(device="cuda").manual_seed(1)
    x, y, g = (torch.randn(B, d, device="cuda", generator=gen)
               for d in (problem.irreps_in1.dim, problem.irreps_in2.dim, problem.irreps_out.dim))
    y[:, 0] = 1.0
    w = torch.randn(problem.weight_numel, device="cuda", generator=gen)
    both = [(ops.tp_forward(*[t.to(d) for t in (x, y, w)], kid), ops.tp_backward(*[t.to(d) for t in (x, y, w, g)], kid)[0])
            for kid, d in zip(kids, (torch.float32, torch.float64))]
    for got, exact in zip(*both):
        off = got.double() - exact
        # (six standard deviations; columns of a row share the errors of its operands: a few times more)
        assert abs(float(off.mean())) <= 12 * float(off.std()) / off.numel() ** 0.5
