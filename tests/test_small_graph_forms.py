"""Where the small-graph form of the forward kernel puts its waves' accumulators: every value inside the slice of the
wave that writes it, every read inside a slice, and the whole inside the array that the kernel declares. And that such
forms keep to chunks where a node has many edges."""

import re

import numpy as np
import pytest

from openequivariance_amd import runtime as rt
from openequivariance_amd.codegen.common import Src
from openequivariance_amd.codegen.lower import adjoint, lower
from openequivariance_amd.codegen.uvu import LDS_LIMIT, UvuEmitter, conv_module, split_waves
from openequivariance_amd.core import problems as P


def _f64(p):
    p.irrep_dtype = p.weight_dtype = np.float64
    return p


PROBLEMS = {
    # staged operands: an output block of 9 components beside a staging buffer of 8 x 64 words (one and two chunks), and
    # beside one of more rows; the widest degrees of the family
    "64x4e": lambda: P.ChannelwiseTPP("64x0e", "1x4e", "64x4e"),
    "64x0e+2e+4e": lambda: P.ChannelwiseTPP("64x0e", "1x0e+1x2e+1x4e", "64x0e+64x2e+64x4e"),
    "128x4e": lambda: P.ChannelwiseTPP("128x0e", "1x4e", "128x4e"),
    "64x4e from 0e+1o": lambda: P.ChannelwiseTPP("64x0e+64x1o", "1x3o", "64x4e"),
    "64x6e": lambda: P.ChannelwiseTPP("64x0e", "1x6e", "64x6e"),
    "64x8e": lambda: P.ChannelwiseTPP("64x0e", "1x8e", "64x8e"),
    "64x4e of the sender walk": lambda: P.ChannelwiseTPP("64x4e", "1x4e", "64x0e"),
    "mace-medium": lambda: P.mace_problems()[1],
    "aspirin": lambda: P.nequip_problems()[1],
    "64x4e-f64": lambda: _f64(P.ChannelwiseTPP("64x0e", "1x4e", "64x4e")),  # no staging
    "64x10e-f64": lambda: _f64(P.ChannelwiseTPP("64x0e", "1x10e", "64x10e")),  # eight slices do not fit a CU
    "32x4e": lambda: P.ChannelwiseTPP("32x0e", "1x4e", "32x4e"),            # two rows to a wave
}


@pytest.mark.parametrize("name", list(PROBLEMS))
def test_slices_of_the_waves_do_not_overlap(name):
    low = lower(PROBLEMS[name]())
    em = UvuEmitter(adjoint(low) if "sender walk" in name else low, acc_budget_words=128)
    em.tr_stores = 3 if em.low.elem_size == 8 else 0  # (as conv_module sets it)
    n = em.split_count(split_waves({"conv_fsplit": -1}, "conv_fsplit", em, 1, 2), 2)
    assert n > 1
    s = Src()
    block = em.emit_conv_forward(s, 1, True, 2, 2, 8, name="forward_split", split=n)
    text = s.text()
    declared = {a: [int(v) for v in re.findall(r"\[(\d+)\]", dims)]
                for a, dims in re.findall(r"__shared__ [^;]*?T (s_\w+)((?:\[\d+\])+);", text)}
    assert sum(np.prod(d) for d in declared.values()) * em.low.elem_size <= LDS_LIMIT
    array = "s_stage" if "T* const s_red = &s_stage[0][0];" in text else "s_red"
    (stride,) = {int(v) for v in re.findall(r"mine = s_red \+ wave \* (\d+) \+ lane", text)}
    assert np.prod(declared[array]) >= block // 64 * stride
    if array == "s_stage":  # a wave must not write where another one's operands are still in use
        assert declared[array][-1] == stride
    writes = {int(v) for v in re.findall(r"mine\[(\d+)\] =", text)}
    reads = {int(v) for v in re.findall(r"first\[(\d+)\]", text)}
    assert writes and max(writes) + 64 <= stride
    assert reads == {p * em.NCH * stride + v for p in range(n) for v in writes}


def test_small_graph_forms_walk_long_segments_in_chunks():
    """A node may hold nearly all edges of a small graph (a virtual node, parallel edges, the padding of an edge list): the
    small-graph form leaves room for the rows of its extra chunks as the plain one does."""
    low = lower(P.nequip_problems()[1])
    src, dims, descs = conv_module(low, True)
    ks = rt.KernelSet(b"\x7fELFxxxx", dims, descs)
    roles = {d[0]: d for d in descs}
    for nodes, edges in ((200, 20000), (1000, 1500), (32, 600)):
        assert nodes <= roles[rt.ROLE_CONV_FORWARD_SPLIT][7]
        assert ks.conv_forward_scratch_bytes(nodes, edges) >= edges // dims["hub_limit"] * low.L3 * 4


def _forms(problem):
    src, _dims, descs = conv_module(lower(problem), True)
    scratch = {name: r[1] for name, r in rt.kernel_resources(rt.compile_source(src)).items()}
    return {d[1]: d for d in descs}, scratch


def test_small_graph_forms_only_where_they_pay():
    toluene, scratch = _forms(P.nequip_problems()[2])
    assert toluene["forward_split"][2] == 64 * 4 and scratch["forward_split"] == scratch["forward"] == 0
    assert toluene["double_backward_A_split"][2] == 64 * 8
    several_segments, _ = _forms(_f64(P.seven_net_problems()[1]))
    assert "forward_split" not in several_segments and "double_backward_A_split" not in several_segments
    assert several_segments["backward"][6] > 0
    many_rows, _ = _forms(P.config1_single_uvu())  # 64 edges to a wave
    assert not any("split" in name for name in many_rows)
    assert many_rows["backward"][6] == many_rows["double_backward_B"][6] == 0
    four_rows, _ = _forms(P.ChannelwiseTPP("16x0e+16x1o", "0e+1o", "16x0e+16x1o"))
    assert four_rows["forward_split"][2] == 64 * 4 and four_rows["forward_split"][7] <= 640
