"""The two gradients of a product side by side on two streams against one after the other: the same kernels on the same
operands, so the same bits, whatever has to be copied for a launch, eager and from a graph."""
import numpy as np
import pytest
import torch

import stk_amd as stk
from oracle import stk_oracle as O
from stk_amd.backend import autograd, hip_kernels
from tests import _util as U

pytestmark = pytest.mark.gpu
DEV = "cuda"
_LARGE = np.array([300, 0, 129, 384, 640, 128, 77, 256, 512, 1000, 40, 896, 512, 384, 640, 512])   # cuts the last round of a dsd
_SMALL = np.array([256, 384, 128, 512])                                                            # sdd walks block_order


def _strided(t):
    return torch.stack((t, torch.zeros_like(t)), 1)[:, 0]


def _misaligned(t):
    return torch.cat((t.new_zeros(t.size(0), 1), t), 1)[:, 1:]


def _case(pair, copied, tokens, hidden, ffn):
    topo = O.dmoe_topology(tokens, ffn, 128)
    rows, cols = topo.shape
    g = torch.Generator().manual_seed(rows + hidden)
    rand = lambda *shape: (torch.randn(*shape, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    m = U.matrix_from_topology(stk, topo, rand(len(topo.row_indices), 128, 128), DEV)
    meta = [m.row_indices, m.column_indices, m.offsets, m.column_indices_t, m.offsets_t, m.block_offsets_t]
    if copied == "indices":
        meta = [_strided(t) for t in meta]
    elif copied == "block offsets":
        meta[5] = _strided(meta[5])
    values = m.data.requires_grad_(True)
    m = stk.Matrix(m.size(), values, *meta)
    if pair == "dsd":                          # sdd and dsd
        dense, out, call = rand(cols, hidden), (rows, hidden), lambda d: stk.ops.dsd(m, d)
    elif pair == "dds":                        # dds and sdd
        dense, out, call = rand(hidden, rows), (hidden, cols), lambda d: stk.ops.dds(d, m)
    else:                                      # two dsd, or a dsd and a dds
        other = rand(cols, hidden).t() if pair == "sdd of a view" else rand(hidden, cols)
        dense, out = rand(rows, hidden), tuple(values.shape)
        call = lambda d: stk.ops.sdd(d, other, m).data
        values = other.requires_grad_(True)
    if copied == "operand":
        dense = _misaligned(dense)
    dense.requires_grad_(True)
    return (values, dense), rand(*out), lambda: call(dense)


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("copied", ["nothing", "indices", "block offsets", "operand"])
@pytest.mark.parametrize("pair", ["dsd", "dds", "sdd", "sdd of a view"])
@pytest.mark.parametrize("size", ["small", "large"])
def test_pairs_on_two_streams(size, pair, copied, captured, monkeypatch):
    monkeypatch.setattr(autograd, "OVERLAP_FROM", 0.0)
    monkeypatch.setattr(autograd, "JOINT_GRADIENTS", False)
    monkeypatch.setattr(autograd, "JOINT_DSD_GRADIENTS", False)
    leaves, dy, call = _case(pair, copied, *((_SMALL, 256, 512) if size == "small" else (_LARGE, 1024, 4096)))
    launches = []
    for name in ("sdd", "dsd", "dds"):
        def recorded(*args, launch=getattr(hip_kernels, name), **kwargs):
            launches.append(hip_kernels._stream())
            launch(*args, **kwargs)
        monkeypatch.setattr(hip_kernels, name, recorded)

    def gradients(overlap):
        monkeypatch.setattr(autograd, "OVERLAP_GRADIENTS", overlap)
        out = call()
        launches.clear()
        grads = torch.autograd.grad(out, leaves, dy)
        assert len(launches) == 2 and (len(set(launches)) == 2) == overlap
        return grads

    hip_kernels.release_workspaces()       # (the first launch on the side stream makes its own)
    torch.cuda.synchronize()
    got = gradients(True)
    want = gradients(False)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert all(torch.isfinite(t.float()).all() and t.float().abs().sum() > 0 for t in want)
    if not captured:
        for _ in range(3):
            assert all(torch.equal(a, b) for a, b in zip(gradients(True), want))
        return
    # (torch hands its 32 streams out in turn, the side stream among them)
    stream = next(s for s in iter(torch.cuda.Stream, None) if s.cuda_stream not in hip_kernels.CONCURRENT_STREAMS)
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        gradients(True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = gradients(True)
    for _ in range(3):
        with torch.no_grad():
            dy.mul_(-0.5)
        graph.replay()
        torch.cuda.synchronize()
        again = [t.clone() for t in got]
        want = gradients(False)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(again, want))
