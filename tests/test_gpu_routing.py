"""GPU parity of the token routing around the dMoE products: stk_route, stk_padded_gather,
stk_padded_scatter and its weight gradient, through the C ABI.

Index outputs and both copies must match the oracle bit for bit (the order of the fp32 operations in
the scatter is part of its definition); the weight gradient is a long fp32 dot product and is held to
a tolerance written at its test.
"""
import numpy as np
import pytest
import torch

import stk_amd as stk
from oracle import stk_oracle as O
from stk_amd.backend import hip_kernels
from tests import _util as U
from tests.test_oracle import ROUTE_CASES, ROUTE_KAT, route_experts

pytestmark = pytest.mark.gpu
DEV = "cuda"
FIELDS = ("indices", "bin_ids", "bins", "padded_bins", "slot_rows", "row_slots")


def _assert_route(got, want, what=""):
    for k in FIELDS:
        g = getattr(got, k)
        assert g.dtype == torch.int32 and g.is_cuda, (what, k)
        assert np.array_equal(g.cpu().numpy(), getattr(want, k)), (what, k)


def _bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy()


def _round(a, dtype):
    """fp32 numpy -> 16-bit torch (round to nearest even on the host)."""
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dtype)


def test_route_known_answer_on_device():
    top = torch.tensor(ROUTE_KAT["top_experts"], dtype=torch.int32, device=DEV)
    r = stk.ops.route(top, 3, 4)
    assert r.top_k == 2 and r.blocking == 4
    for k in FIELDS:
        assert getattr(r, k).cpu().tolist() == ROUTE_KAT[k], k


@pytest.mark.parametrize("tokens,top_k,experts,blocking,seed", ROUTE_CASES)
def test_route_cases_on_device(tokens, top_k, experts, blocking, seed):
    top = route_experts(tokens, top_k, experts, seed)
    dev_top = torch.from_numpy(top).to(DEV)
    _assert_route(stk.ops.route(dev_top, experts, blocking), O.route(top, experts, blocking), "exact")
    cap = stk.ops.route_capacity(top.size, experts, blocking)
    _assert_route(stk.ops.route(dev_top, experts, blocking, padded_rows=cap), O.route(top, experts, blocking, padded_rows=cap), "capacity")
    # int64 choices (what torch.topk returns) take the same path
    _assert_route(stk.ops.route(dev_top.long(), experts, blocking), O.route(top, experts, blocking), "int64")


def _top1(tokens, experts, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(tokens, experts, generator=g).argmax(dim=1, keepdim=True).to(torch.int32)


def _zipf_top2(tokens, experts, seed, s=1.2):
    g = torch.Generator().manual_seed(seed)
    logp = -s * torch.log(torch.arange(1, experts + 1, dtype=torch.float64))
    u = torch.rand(tokens, experts, generator=g, dtype=torch.float64).clamp_min(1e-300)
    return (logp[None, :] - torch.log(-torch.log(u))).topk(2, dim=1).indices.to(torch.int32)


def _skewed(tokens, experts, seed):
    g = torch.Generator().manual_seed(seed)
    top = torch.randint(1, experts, (tokens,), generator=g, dtype=torch.int32)
    top[torch.randperm(tokens, generator=g)[:tokens // 2]] = 0
    return top[:, None]


FULL = {
    "config3 top-1": (lambda: _top1(16384, 64, 0), 128),
    "config4 zipf top-2": (lambda: _zipf_top2(32768, 64, 0), 128),
    "config5 top-1 b64": (lambda: _top1(16384, 64, 0), 64),
    "config5 skew": (lambda: _skewed(16384, 64, 0), 64),
}


@pytest.mark.parametrize("name", list(FULL))
def test_route_full_size_feeds_the_topology(name):
    make, blocking = FULL[name]
    top = make()
    experts = 64
    want = O.route(top.numpy(), experts, blocking)
    r = stk.ops.route(top.to(DEV), experts, blocking)
    _assert_route(r, want, name)
    # the padded bins are those of the block-diagonal topology the products run on
    counts = np.bincount(top.numpy().reshape(-1), minlength=experts)
    ffn = 4 * blocking
    topo = O.dmoe_topology(counts, ffn, blocking)
    m = stk.ops.dmoe_topology(r.padded_bins, blocking, r.row_slots.numel() // blocking, ffn // blocking)
    U.assert_topology_equal(m, topo, name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("top_k,weighted", [(1, False), (1, True), (2, False), (2, True), (4, True), (3, False), (6, True)])
@pytest.mark.parametrize("cols", [8, 1024, 2056])
def test_copies_bit_exact(dtype, top_k, weighted, cols):
    tokens, experts, blocking = 700, 16, 128
    top = route_experts(tokens, top_k, experts, 40 + top_k)
    want_r = O.route(top, experts, blocking)
    r = stk.ops.route(torch.from_numpy(top).to(DEV), experts, blocking)
    g = torch.Generator().manual_seed(cols + top_k)
    x = torch.randn(tokens, cols, generator=g).to(dtype)
    w = torch.rand(tokens, top_k, generator=g) if weighted else None
    dev_w = None if w is None else w.to(DEV)
    wn = None if w is None else w.numpy().reshape(-1)

    got = hip_kernels.padded_gather(x.to(DEV), r.row_slots, top_k, dev_w)
    want = _round(O.padded_gather(U.np32(x), want_r.row_slots, top_k, wn), dtype)
    assert got.dtype == dtype and got.shape == want.shape
    assert np.array_equal(_bits(got), _bits(want)), "gather"

    y = torch.randn(want_r.row_slots.size, cols, generator=g).to(dtype)
    got = hip_kernels.padded_scatter(y.to(DEV), r.slot_rows, top_k, dev_w)
    want = _round(O.padded_scatter(U.np32(y), want_r.slot_rows, top_k, wn), dtype)
    assert got.dtype == dtype and got.shape == (tokens, cols)
    assert np.array_equal(_bits(got), _bits(want)), "scatter"


def test_copies_read_strided_rows_in_place():
    tokens, experts, blocking, cols, top_k = 260, 8, 64, 256, 2
    top = route_experts(tokens, top_k, experts, 5)
    want_r = O.route(top, experts, blocking)
    r = stk.ops.route(torch.from_numpy(top).to(DEV), experts, blocking)
    g = torch.Generator().manual_seed(1)
    wide = torch.randn(tokens, 3 * cols, generator=g).bfloat16().to(DEV)
    x = wide[:, cols:2 * cols]                    # row stride 768, rows 16-byte aligned
    got = hip_kernels.padded_gather(x, r.row_slots, top_k)
    want = _round(O.padded_gather(U.np32(x), want_r.row_slots, top_k), torch.bfloat16)
    assert np.array_equal(_bits(got), _bits(want))
    odd = wide[:, 1:1 + cols]                     # rows not aligned: copied at the boundary, same result
    got = hip_kernels.padded_gather(odd, r.row_slots, top_k)
    assert np.array_equal(_bits(got), _bits(_round(O.padded_gather(U.np32(odd), want_r.row_slots, top_k), torch.bfloat16)))


def test_round_trip_and_padding_rows():
    tokens, experts, blocking, cols = 1000, 64, 128, 512
    top = _top1(tokens, experts, 3)
    r = stk.ops.route(top.to(DEV), experts, blocking)
    x = torch.randn(tokens, cols, generator=torch.Generator().manual_seed(0)).bfloat16().to(DEV)
    padded = stk.ops.padded_gather(x, r)
    assert padded.shape[0] % blocking == 0 and padded.shape[0] == int(r.padded_bins[-1])
    assert bool((padded[r.row_slots < 0] == 0).all())
    assert torch.equal(stk.ops.padded_scatter(padded, r), x)


@pytest.mark.parametrize("top_k", [1, 2])
def test_autograd(top_k):
    tokens, experts, blocking, cols = 300, 8, 64, 128
    dtype = torch.bfloat16
    top = route_experts(tokens, top_k, experts, 9)
    want_r = O.route(top, experts, blocking)
    r = stk.ops.route(torch.from_numpy(top).to(DEV), experts, blocking)
    g = torch.Generator().manual_seed(2)
    x = torch.randn(tokens, cols, generator=g).to(dtype).to(DEV).requires_grad_()
    w = torch.rand(tokens, top_k, generator=g).to(DEV).requires_grad_()
    padded = stk.ops.padded_gather(x, r)
    out = stk.ops.padded_scatter(padded, r, w)
    grad = torch.randn(tokens, cols, generator=g).to(dtype).to(DEV)
    padded.retain_grad()
    out.backward(grad)
    wn = U.np32(w).reshape(-1)
    # d/d(padded) = gather of the incoming gradient, weighted
    want = _round(O.padded_gather(U.np32(grad), want_r.row_slots, top_k, wn), dtype)
    assert np.array_equal(_bits(padded.grad), _bits(want)), "d padded"
    # d/dx = scatter of that, unweighted
    want = _round(O.padded_scatter(U.np32(want), want_r.slot_rows, top_k), dtype)
    assert np.array_equal(_bits(x.grad), _bits(want)), "d x"
    # d/dw: fp32 dot products of 128 terms of size ~1, summed in another order than the oracle's float64:
    # |error| <= 128 * 2^-24 * sum|terms| ~ 1e-3 at worst; rtol 1e-4 / atol 1e-3
    want = O.padded_scatter_weight_gradient(U.np32(padded), U.np32(grad), want_r.slot_rows, top_k)
    assert w.grad.shape == w.shape and w.grad.dtype == w.dtype
    np.testing.assert_allclose(U.np32(w.grad).reshape(-1), want, rtol=1e-4, atol=1e-3)


def test_routed_layer_against_per_token_dense():
    """route -> gather -> sdd -> dsd -> scatter equals, token by token, x W1[e] W2[e] summed over the choices."""
    tokens, experts, blocking, hidden, ffn, top_k = 500, 8, 128, 256, 256, 2
    dtype = torch.bfloat16
    top = route_experts(tokens, top_k, experts, 13)
    g = torch.Generator().manual_seed(4)
    x = torch.randn(tokens, hidden, generator=g).mul(0.5).to(dtype)
    w1 = torch.randn(hidden, experts * ffn, generator=g).mul(0.05).to(dtype)
    w2 = torch.randn(experts * ffn, hidden, generator=g).mul(0.05).to(dtype)
    weights = torch.rand(tokens, top_k, generator=g)
    r = stk.ops.route(torch.from_numpy(top).to(DEV), experts, blocking)
    padded = stk.ops.padded_gather(x.to(DEV), r)
    topo = stk.ops.dmoe_topology(r.padded_bins, blocking, padded.shape[0] // blocking, ffn // blocking, dtype=dtype)
    h = stk.ops.sdd(padded, w1.to(DEV), topo)
    y = stk.ops.dsd(h, w2.to(DEV))
    out = stk.ops.padded_scatter(y, r, weights.to(DEV))
    want = np.zeros((tokens, hidden), dtype=np.float32)
    xn, w1n, w2n = U.np32(x), U.np32(w1), U.np32(w2)
    for k in range(top_k):
        for e in range(experts):
            sel = top[:, k] == e
            hid = _round(xn[sel] @ w1n[:, e * ffn:(e + 1) * ffn], dtype).float().numpy()
            want[sel] += weights[sel, k].numpy()[:, None] * (hid @ w2n[e * ffn:(e + 1) * ffn])
    U.assert_close(out, want, dtype, "routed layer")


def test_empty_and_errors():
    r = stk.ops.route(torch.empty(0, 2, dtype=torch.int32, device=DEV), 4, 8)
    assert r.indices.numel() == 0 and r.row_slots.numel() == 0 and r.bins.cpu().tolist() == [0, 0, 0, 0]
    assert r.padded_bins.cpu().tolist() == [0, 0, 0, 0]
    x = torch.empty(0, 64, dtype=torch.bfloat16, device=DEV)
    assert stk.ops.padded_gather(x, r).shape == (0, 64)
    assert stk.ops.padded_scatter(torch.empty(0, 64, dtype=torch.bfloat16, device=DEV), r).shape == (0, 64)
    top = torch.zeros(16, 1, dtype=torch.int32, device=DEV)
    with pytest.raises(NotImplementedError):
        stk.ops.route(top, 1025, 8)
    r = stk.ops.route(top, 2, 8)
    with pytest.raises(NotImplementedError):
        stk.ops.padded_gather(torch.zeros(16, 12, dtype=torch.bfloat16, device=DEV), r)
    with pytest.raises(NotImplementedError):
        stk.ops.padded_gather(torch.zeros(16, 16, dtype=torch.float32, device=DEV), r)
    with pytest.raises(RuntimeError):
        stk.ops.route(torch.zeros(16, 1, dtype=torch.int32), 2, 8)
    with pytest.raises(AssertionError):
        stk.ops.padded_scatter(torch.zeros(16, 16, dtype=torch.bfloat16, device=DEV), r, torch.ones(3, device=DEV))


def test_weights_in_host_memory_are_refused():
    # 4 slots: the few-row product, 9000: the scattered one (or the two steps)
    for tokens, experts, hidden, ffn in ((4, 4, 128, 128), (9000, 8, 1024, 2560)):
        r = stk.ops.route(torch.randint(0, experts, (tokens, 1), dtype=torch.int32, device=DEV), experts, 128)
        rows = r.row_slots.numel()
        m = stk.ops.dmoe_topology(r.padded_bins, 128, rows // 128, ffn // 128, dtype=torch.bfloat16)
        x = torch.zeros(tokens, hidden, dtype=torch.bfloat16, device=DEV)
        rhs = torch.zeros(m.size()[1], hidden, dtype=torch.bfloat16, device=DEV)
        weights = torch.ones(tokens, 1)
        for call in (lambda: stk.ops.dsd_scatter(m, rhs, r, weights), lambda: stk.ops.padded_scatter(stk.ops.padded_gather(x, r), r, weights),
                     lambda: hip_kernels.padded_gather(x, r.row_slots, 1, weights)):
            with pytest.raises(RuntimeError, match="ROCm GPU only"):
                call()


def test_routed_layer_gradients_against_dense_autograd():
    """Backward of route -> gather -> sdd -> dsd -> weighted scatter against torch autograd on the same layer written
    with per-expert dense fp32 products.  The HIP path rounds four intermediate tensors to bf16 (2^-9 relative each), the
    reference none: every gradient must agree within 2 % of its largest element."""
    tokens, experts, blocking, hidden, ffn, top_k = 300, 4, 128, 128, 256, 2
    dtype = torch.bfloat16
    top = route_experts(tokens, top_k, experts, 17)
    g = torch.Generator().manual_seed(6)
    x0 = torch.randn(tokens, hidden, generator=g).mul(0.5).to(dtype)
    w10 = torch.randn(hidden, experts * ffn, generator=g).mul(0.1).to(dtype)
    w20 = torch.randn(experts * ffn, hidden, generator=g).mul(0.1).to(dtype)
    wt0 = torch.rand(tokens, top_k, generator=g)
    grad = torch.randn(tokens, hidden, generator=g).to(dtype)

    x, w1, w2, wt = (t.to(DEV).requires_grad_() for t in (x0, w10, w20, wt0))
    r = stk.ops.route(torch.from_numpy(top).to(DEV), experts, blocking)
    padded = stk.ops.padded_gather(x, r)
    topo = stk.ops.dmoe_topology(r.padded_bins, blocking, padded.shape[0] // blocking, ffn // blocking, dtype=dtype)
    out = stk.ops.padded_scatter(stk.ops.dsd(stk.ops.sdd(padded, w1, topo), w2), r, wt)
    out.backward(grad.to(DEV))

    xr, w1r, w2r, wtr = (t.float().requires_grad_() for t in (x0, w10, w20, wt0))
    ref = torch.zeros(tokens, hidden)
    for k in range(top_k):
        for e in range(experts):
            sel = torch.from_numpy(top[:, k] == e)
            y = (xr[sel] @ w1r[:, e * ffn:(e + 1) * ffn]) @ w2r[e * ffn:(e + 1) * ffn]
            ref = ref.index_add(0, sel.nonzero()[:, 0], wtr[sel, k][:, None] * y)
    ref.backward(grad.float())

    def close(got, want, what):
        got, want = U.np32(got), U.np32(want)
        assert got.shape == want.shape, what
        err = np.abs(got - want).max()
        assert err <= 2e-2 * np.abs(want).max(), (what, err, np.abs(want).max())

    close(out, ref, "forward")
    close(x.grad, xr.grad, "d x")
    close(w1.grad, w1r.grad, "d w1")
    close(w2.grad, w2r.grad, "d w2")
    close(wt.grad, wtr.grad, "d weights")


def test_route_at_the_largest_expert_count_and_a_million_slots():
    """1024 experts (the limit of stk_route) with 2^20 slots: 4096 tiles of slots, a table of 4 M counts."""
    rng = np.random.default_rng(3)
    experts, blocking = 1024, 128
    top = rng.integers(0, experts, size=(1 << 19, 2), dtype=np.int32)
    top[:, 1] = (top[:, 0] + 1 + rng.integers(0, experts - 1, size=1 << 19)) % experts   # a second, different expert
    top[top == 17] = 18                                                                 # an expert without slots
    want = O.route(top, experts, blocking)
    r = stk.ops.route(torch.from_numpy(top).to(DEV), experts, blocking)
    _assert_route(r, want, "large")
    assert int(r.bins[17]) == int(r.bins[16]) and int(r.padded_bins[17]) == int(r.padded_bins[16])
    # a wide row through both copies
    x = torch.randn(1 << 19, 64, generator=torch.Generator().manual_seed(0)).bfloat16().to(DEV)
    padded = hip_kernels.padded_gather(x, r.row_slots, 2)
    assert padded.shape[0] == int(r.padded_bins[-1])
    back = hip_kernels.padded_scatter(padded, r.slot_rows, 2)
    assert torch.equal(back, (x.float() * 2).bfloat16())
