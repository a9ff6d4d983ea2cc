"""The index of an edge list (segment starts, grouped edge ids, table of extra walk positions, walk order) against
numpy, at the sizes where its kernels hand over to each other: one-launch build up to 16 384 edges (sorted lists: 8 192) and 4 096 nodes,
grouping slice by slice up to 262 144 edges and 16 384 nodes, scan tiles of 1 024 segments, segments ranked by a wave / through a bitmap / by the whole grid."""

import numpy as np
import pytest
import torch

from openequivariance_amd import runtime as rt
from openequivariance_amd._torch.tensor_product_conv import build_conv_module
from openequivariance_amd.core import problems as P

pytestmark = pytest.mark.gpu


def _edges(nodes, edges, hubs, seed):
    """Random edge list; node 0 gets ``hubs[0]`` of the edges as receiver, node ``nodes - 1`` ``hubs[1]`` as sender."""
    rng = np.random.default_rng(seed)
    rows, cols = rng.integers(0, nodes, edges), rng.integers(0, nodes, edges)
    rows[rng.permutation(edges)[:hubs[0]]] = 0
    cols[rng.permutation(edges)[:hubs[1]]] = nodes - 1
    return rows.astype(np.int64), cols.astype(np.int64)


def _hub_table(deg, limit, cap):
    extra = np.where(deg > limit, -(-deg // limit) - 1, 0)
    ptr = np.concatenate([[0], np.cumsum(extra)])
    return ptr, np.repeat(np.arange(len(deg)), extra)[:cap]


SIZES = [
    # nodes, edges, hub edges (receiver side, sender side)
    (1, 1, (0, 0)), (3, 700, (400, 500)), (64, 1024, (0, 257)), (192, 6144, (0, 0)),
    (4096, 16384, (256, 16384)), (4096, 16384, (5000, 0)), (4097, 16384, (300, 1025)), (100, 16385, (0, 1024)),
    (1023, 20000, (2000, 3000)), (1024, 20000, (0, 0)), (8191, 50001, (0, 1030)), (8192, 40000, (255, 512)), (140001, 150000, (4000, 10)),
    # grouped slice by slice: up to 64 slices of 4 096 edges and 16 384 nodes, more than 256 edges of a node in a slice
    # through a bitmap
    (1, 20480, (0, 0)), (5000, 24576, (1536, 1542)), (16384, 262144, (262144, 70000)), (300, 262144, (0, 0)),
    (300, 262145, (0, 0)), (16385, 20000, (300, 0)), (255, 16385, (16385, 256)), (256, 69633, (0, 4097)),
    (300, 8192, (257, 0)), (300, 8193, (0, 257)),
    # beyond the slices, with segments that the whole grid ranks on both sides
    (16385, 40000, (2000, 3000)), (1000, 270000, (1025, 5000)),
]


@pytest.mark.parametrize("det", [True, False], ids=["sorted", "grouped"])
@pytest.mark.parametrize("nodes,edges,hubs", SIZES)
def test_index_pieces(nodes, edges, hubs, det, monkeypatch):
    monkeypatch.setenv("OEQ_AMD_TUNE", "conv_omin=1023")
    src, dims, descs = build_conv_module(P.config1_single_uvu(), det)
    ks = rt.get_kernel_set(src, dims, descs)
    rows, cols = _edges(nodes, edges, hubs, seed=nodes + edges)
    if det:
        order = np.lexsort((cols, rows))
        rows, cols = rows[order], cols[order]
    perm = np.lexsort((rows, cols)).astype(np.int64)
    tr, tc, tp = (torch.tensor(a, device="cuda") for a in (rows, cols, perm))
    limit = dims["hub_limit"]
    built = []
    for _ in range(2):
        nb = ks.conv_index_bytes(nodes, edges, True)
        index = torch.full((nb,), 0x5A, dtype=torch.uint8, device="cuda")
        ks.conv_index_build(nodes, edges, tr.data_ptr(), tc.data_ptr(), tp.data_ptr() if det else 0, True,
                            index.data_ptr(), nb, torch.cuda.current_stream().cuda_stream)

        def piece(name):
            off, n = ks.conv_index_piece(nodes, edges, True, name)
            return index[off:off + 8 * n].view(torch.int64).cpu().numpy()

        built.append(piece)
        for keys, ptr_name, perm_name, hub in ((rows, "rowptr", "rperm", "hub"), (cols, "colptr", "sperm", "shub")):
            deg = np.bincount(keys, minlength=nodes)
            assert np.array_equal(piece(ptr_name), np.concatenate([[0], np.cumsum(deg)]))
            if not det:
                assert np.array_equal(piece(perm_name), np.argsort(keys, kind="stable"))
            if edges >= limit:
                hubptr, hubnode = _hub_table(deg, limit, edges // limit)
                assert np.array_equal(piece(hub + "ptr"), hubptr)
                assert np.array_equal(piece(hub + "node")[:len(hubnode)], hubnode)
        if nodes >= 1023:
            assert np.array_equal(np.sort(piece("order")), np.arange(nodes))
    if nodes >= 1023:
        assert np.array_equal(built[0]("order"), built[1]("order"))


def test_indices_out_of_range_stay_out_of_the_grouping():
    """Keys that name no node are left out; nothing is read or written outside the buffers (one launch, slice by
    slice, and the five launches beyond)."""
    src, dims, descs = build_conv_module(P.config1_single_uvu(), False)
    ks = rt.get_kernel_set(src, dims, descs)
    for nodes, edges in ((50, 900), (5000, 20000), (16385, 20000), (1000, 270000)):
        rows, cols = _edges(nodes, edges, (0, 0), seed=1)
        rows[::7], cols[::5] = nodes, -3
        tr, tc = torch.tensor(rows, device="cuda"), torch.tensor(cols, device="cuda")
        nb = ks.conv_index_bytes(nodes, edges, True)
        index = torch.zeros(nb, dtype=torch.uint8, device="cuda")
        ks.conv_index_build(nodes, edges, tr.data_ptr(), tc.data_ptr(), 0, True, index.data_ptr(), nb,
                            torch.cuda.current_stream().cuda_stream)
        for keys, ptr_name, perm_name in ((rows, "rowptr", "rperm"), (cols, "colptr", "sperm")):
            ok = np.flatnonzero((keys >= 0) & (keys < nodes))
            off, n = ks.conv_index_piece(nodes, edges, True, ptr_name)
            ptr = index[off:off + 8 * n].view(torch.int64).cpu().numpy()
            assert np.array_equal(ptr, np.concatenate([[0], np.cumsum(np.bincount(keys[ok], minlength=nodes))]))
            off, n = ks.conv_index_piece(nodes, edges, True, perm_name)
            got = index[off:off + 8 * n].view(torch.int64).cpu().numpy()[:len(ok)]
            assert np.array_equal(got, ok[np.argsort(keys[ok], kind="stable")])
