"""The routed products on block rows with few tokens each: stk_sdd_gather's small tiles bit for bit against the two calls
(same sums in the same order), stk_dsd_scatter_few against the two calls' arithmetic in fp32.

Rows in use per block row are chosen at the edges of the tiles (1, 31 .. 33, 64, 65, 128, none)."""
import pytest
import torch

import stk_amd as stk
from stk_amd.backend import _lib, hip_kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"
COUNTS = ((1, 31, 33, 0, 64, 65, 5, 128), (32, 0, 0, 2, 130, 7, 1, 1), (0, 3))
#        (experts' slots, hidden, ffn, top_k)
SIZES = [(COUNTS[0], 128, 128, 1), (COUNTS[0], 384, 1280, 3), (COUNTS[1], 64, 640, 1), (COUNTS[1], 256, 2048, 2), (COUNTS[2], 1024, 9088, 1)]


def _layer(counts, hidden, ffn, top_k, dtype, spare=0):
    g = torch.Generator().manual_seed(7)
    experts = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))
    experts = torch.cat([experts, experts.new_zeros(-len(experts) % top_k)])
    top = experts[torch.randperm(len(experts), generator=g)].view(-1, top_k).to(torch.int32).to(DEV)
    tokens = top.shape[0]
    rows = sum(-(-int((top == e).sum()) // 128) * 128 for e in range(len(counts))) + 128 * spare
    r = stk.ops.route(top, len(counts), 128, padded_rows=rows)
    topo = stk.ops.dmoe_topology(r.padded_bins, 128, rows // 128, ffn // 128, dtype=dtype)
    x = torch.randn(tokens, hidden, generator=g).to(dtype).to(DEV)
    w1 = (torch.randn(hidden, len(counts) * ffn, generator=g) * hidden ** -0.5).to(dtype).to(DEV)
    w2 = (torch.randn(len(counts) * ffn, hidden, generator=g) * ffn ** -0.5).to(dtype).to(DEV)
    return x, top, r, topo, w1, w2


def _bits(t):
    return t.view(torch.int16)


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16), ids=("bf16", "f16"))
@pytest.mark.parametrize("out_in", (False, True))
@pytest.mark.parametrize("counts,hidden,ffn,top_k", SIZES)
def test_gather_sdd_of_few_rows(counts, hidden, ffn, top_k, out_in, dtype):
    x, _, r, topo, w1, _ = _layer(counts, hidden, ffn, top_k, dtype, spare=1)
    if out_in:
        w1 = w1.t().contiguous().t()
    for activation in (None, "gelu_tanh"):
        want = stk.ops.sdd_fused(stk.ops.padded_gather(x, r), w1, topo, activation)
        with torch.no_grad():
            got = stk.ops.gather_sdd(x, r, w1, topo, activation)
        assert torch.equal(_bits(got.data), _bits(want.data))


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16), ids=("bf16", "f16"))
@pytest.mark.parametrize("out_in", (False, True))
@pytest.mark.parametrize("weighted", (False, True))
@pytest.mark.parametrize("counts,hidden,ffn,top_k", [s for s in SIZES if s[1] >= 128])
def test_dsd_scatter_of_few_rows(counts, hidden, ffn, top_k, weighted, out_in, dtype):
    x, top, r, topo, _, w2 = _layer(counts, hidden, ffn, top_k, dtype)
    tokens = top.shape[0]
    weights = torch.rand(tokens, top_k, device=DEV) + 0.5 if weighted else None
    # rows that hold no token are not looked at
    h = torch.randn(topo.data.shape, device=DEV).to(dtype)
    padding = (r.row_slots < 0).view(-1, 128)[topo.row_indices.long()]
    clean, h = h.masked_fill(padding[..., None], 0.0), h.masked_fill(padding[..., None], float("nan"))
    m = stk.Matrix(topo.size(), h, topo.row_indices, topo.column_indices, topo.offsets, topo.column_indices_t, topo.offsets_t, topo.block_offsets_t)
    rhs = w2.t().contiguous().t() if out_in else w2
    call = lambda: hip_kernels.dsd_scatter_few(m.size(), m.data, m.offsets, m.column_indices, rhs, r.row_slots, r.slot_rows, top_k, weights)
    got = call()
    assert got is not None and torch.equal(_bits(got), _bits(call())), "the library has this kernel, and it is repeatable"
    with torch.no_grad():
        assert torch.equal(_bits(got), _bits(stk.ops.dsd_scatter(m, rhs, r, weights)))
    # the same in float64 from the dense matrix: a row is rounded to the value type, and so is the token's sum over its rows
    dense = torch.zeros(topo.size(), dtype=torch.float64, device=DEV)
    blocks = dense.view(topo.size()[0] // 128, 128, topo.size()[1] // 128, 128)
    blocks[topo.row_indices.long(), :, topo.column_indices.long(), :] = clean.double()
    y = (dense @ w2.double())[r.slot_rows.long()].view(tokens, top_k, -1)
    w = weights.double().view(tokens, top_k, 1) if weighted else torch.ones(tokens, top_k, 1, dtype=torch.float64, device=DEV)
    want, unit = (w * y).sum(1), {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    # half a unit of each rounded row times its weight, half a unit of the result, and the fp32 sums' error (|h| |w2| 2^-24 per term)
    bound = unit * ((w * y).abs().sum(1) + want.abs()) * 1.01 + 2.0 ** -24 * ffn ** 0.5 * 64
    assert bool(((got.double() - want).abs() <= bound).all())


def test_dsd_scatter_few_with_columns_that_are_no_multiple_of_128():
    x, top, r, topo, _, w2 = _layer(COUNTS[0], 192, 256, 1, torch.bfloat16)
    lib, n = _lib.load(), 192
    h = torch.randn(topo.data.shape, device=DEV).to(torch.bfloat16)
    (m, k), tokens, nnz = topo.size(), top.shape[0], topo.data.shape[0]
    out = torch.full((tokens, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    need = lib.stk_dsd_scatter_few_bytes(m, n, nnz, tokens)
    assert need > 0 and lib.stk_dsd_scatter_few_bytes(m, 96, nnz, tokens) == 0 and lib.stk_dsd_scatter_few_bytes(m, n, nnz, 100 * m) == 0
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    call = lambda size: lib.stk_dsd_scatter_few(m, k, n, h.data_ptr(), topo.offsets.data_ptr(), topo.column_indices.data_ptr(), w2.data_ptr(), n, 1,
                                                r.row_slots.data_ptr(), r.slot_rows.data_ptr(), None, 1, tokens, out.data_ptr(), n, nnz, 128,
                                                _lib.STK_BF16, _lib.STK_I16, ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
    assert call(need - 1) == _lib.STK_ERR_WORKSPACE
    assert call(need) == 0
    dense = torch.zeros(m, k, device=DEV)
    dense.view(m // 128, 128, k // 128, 128)[topo.row_indices.long(), :, topo.column_indices.long(), :] = h.float()
    want = (dense.double() @ w2.double())[r.slot_rows.long()]
    # one rounding of the result, fp32 sums
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())


@pytest.mark.parametrize("counts,reads", ((COUNTS[0], False), ((100, 128, 90, 128), True)))
def test_a_plan_is_built_for_the_gathered_product_only_where_it_is_read(monkeypatch, counts, reads):
    # (under inference mode, which caches none, every product that asks for a plan builds one)
    built = []
    plan = hip_kernels.fusion_plan
    monkeypatch.setattr(hip_kernels, "fusion_plan", lambda *a, **k: built.append(1) or plan(*a, **k))
    with torch.inference_mode():
        x, _, r, topo, w1, _ = _layer(counts, 128, 1280, 1, torch.bfloat16)
        stk.ops.gather_sdd(x, r, w1, topo)
    assert bool(built) == reads
    with torch.no_grad():
        x, _, r, topo, w1, _ = _layer(counts, 128, 1280, 1, torch.bfloat16)
        del topo.offsets._stk_plan, built[:]
        stk.ops.gather_sdd(x, r, w1, topo)
    assert bool(built) == reads
