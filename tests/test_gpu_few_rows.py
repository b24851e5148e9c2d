"""The routed products on block rows with few tokens each, stk_sdd_gather's small tiles and stk_dsd_scatter_few: bit for bit against
the two calls (same sums in the same order, cut where stk_dsd cuts its last round), and against float64.

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


def test_one_plan_for_a_layer_of_64_blocks():
    # (which has no gathered product: the first of its two steps finds the plan that the second will ask for)
    top = torch.arange(8, dtype=torch.int32, device=DEV).view(-1, 1)
    r = stk.ops.route(top, 8, 64)
    m = stk.ops.dmoe_topology(r.padded_bins, 64, 8, 4, dtype=torch.bfloat16)
    m = stk.Matrix(m.size(), m.data, m.row_indices, m.column_indices, m.offsets.clone(), m.column_indices_t, m.offsets_t, m.block_offsets_t)
    x = torch.randn(8, 128, device=DEV).to(torch.bfloat16)
    w1 = torch.randn(128, m.size()[1], device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        stk.ops.gather_sdd(x, r, w1, m)
    plan = m.offsets._stk_plan[1]
    assert hip_kernels.fusion_plan(m.offsets, m.column_indices, m.offsets_t, m.column_indices_t, blocking=64) is plan


# (slots of the experts, hidden, ffn, top_k, spare block rows, whether dsd cuts a tile of its last round): tiles of 64 and of 128 columns;
# one round of tiles, all of them cut, and a second one of 28; pairs and threes of block rows in the lists; no cut
SLICED = [([8] * 16, 2048, 8192, 2, 0, True), ([16] * 64, 1024, 4096, 1, 7, True), ([290, 190] + [5] * 6, 2048, 8192, 1, 0, True),
          ([4] * 8, 1024, 9088, 1, 2, False)]


def _random_layer(counts, hidden, ffn, top_k, spare, dtype=torch.bfloat16):
    _, top, r, topo, _, _ = _layer(counts, 128, 128, top_k, dtype, spare)
    topo = stk.ops.dmoe_topology(r.padded_bins, 128, r.row_slots.numel() // 128, ffn // 128, dtype=dtype)
    topo.data.normal_()
    w2 = torch.empty(len(counts) * ffn, hidden, dtype=dtype, device=DEV).normal_()
    return r, topo, w2, torch.rand(top.shape, device=DEV) + 0.5


@pytest.mark.parametrize("counts,hidden,ffn,top_k,spare,cut", SLICED)
def test_dsd_scatter_of_few_rows_is_dsd_then_scatter(monkeypatch, counts, hidden, ffn, top_k, spare, cut):
    r, m, w2, weights = _random_layer(counts, hidden, ffn, top_k, spare)
    args = (m.size(), m.data, m.offsets, m.column_indices, w2, r.row_slots, r.slot_rows, top_k, weights, m.offsets_t, m.column_indices_t)
    wants = []
    for sliced in (True, False):
        monkeypatch.setattr(hip_kernels, "SLICE_LAST_ROUND", sliced)
        wants.append(stk.ops.padded_scatter(stk.ops.dsd(m, w2), r, weights))
        got = hip_kernels.dsd_scatter_few(*args)
        assert got is not None and torch.equal(_bits(got), _bits(wants[-1])), sliced
        assert torch.equal(_bits(stk.ops.dsd_scatter(m, w2, r, weights)), _bits(got))
    assert torch.equal(*map(_bits, wants)) != cut
    # a K-major second weight, int32 indices, less room for partial tiles
    monkeypatch.setattr(hip_kernels, "SLICE_LAST_ROUND", True)
    monkeypatch.setattr(hip_kernels, "DSD_WORKSPACE_SLOTS", 100)
    m = stk.Matrix(m.size(), m.data, m.row_indices.int(), m.column_indices.int(), m.offsets.clone(), m.column_indices_t.int(), m.offsets_t, m.block_offsets_t)
    w2 = w2.t().contiguous().t()
    assert torch.equal(_bits(stk.ops.dsd_scatter(m, w2, r, weights)), _bits(stk.ops.padded_scatter(stk.ops.dsd(m, w2), r, weights)))
    hip_kernels.release_workspaces()
    monkeypatch.setattr(hip_kernels, "FUSION", False)
    assert hip_kernels.dsd_scatter_few(*args) is None


def test_dsd_scatter_of_few_rows_without_some_slots():
    # slots without a row, and rows of the layout behind the matrix: left out, like in the scatter
    r, m, w2, weights = _random_layer(COUNTS[1], 256, 2048, 2, 1)
    slot_rows, row_slots = r.slot_rows.clone(), r.row_slots.clone()
    gone = torch.arange(0, slot_rows.numel(), 3, device=DEV)
    row_slots[slot_rows[gone].long()] = -1
    slot_rows[gone] = -1
    slot_rows[1] = m.size()[0]
    row_slots[r.slot_rows[1].long()] = -1
    r = r._replace(slot_rows=slot_rows, row_slots=row_slots)
    assert hip_kernels.dsd_scatter_few(m.size(), m.data, m.offsets, m.column_indices, w2, r.row_slots, r.slot_rows, 2, weights) is not None
    assert torch.equal(_bits(stk.ops.dsd_scatter(m, w2, r, weights)), _bits(stk.ops.padded_scatter(stk.ops.dsd(m, w2), r, weights)))


def test_a_layer_of_few_rows_on_a_stream_under_autocast_and_in_a_graph():
    tokens, experts, hidden, ffn, dtype = 96, 16, 256, 4096, torch.bfloat16
    capacity = stk.ops.route_capacity(2 * tokens, experts, 128)
    x = torch.randn(tokens, hidden, device=DEV).to(dtype)
    w1, w2 = (torch.randn(*shape, device=DEV).to(dtype) * 0.05 for shape in ((hidden, experts * ffn), (experts * ffn, hidden)))
    weights, top = torch.rand(tokens, 2, device=DEV), torch.zeros(tokens, 2, dtype=torch.int32, device=DEV)
    choose = lambda seed: top.copy_(torch.rand(tokens, experts, generator=torch.Generator().manual_seed(seed)).topk(2).indices)

    def layer(routed):
        r = stk.ops.route(top, experts, 128, capacity)
        topo = stk.ops.dmoe_topology(r.padded_bins, 128, capacity // 128, ffn // 128, dtype=dtype)
        if routed:
            return stk.ops.dsd_scatter(stk.ops.gather_sdd(x, r, w1, topo, "silu"), w2, r, weights)
        h = stk.ops.sdd_fused(stk.ops.padded_gather(x, r), w1, topo, "silu")
        return stk.ops.padded_scatter(stk.ops.dsd(h, w2), r, weights)

    with torch.no_grad():
        choose(0)
        assert torch.equal(_bits(layer(True)), _bits(layer(False)))
        for autocast in (torch.float16, dtype):               # casts the products' operands, or leaves them
            with torch.autocast("cuda", dtype=autocast):
                got, want = layer(True), layer(False)
            assert got.dtype == want.dtype == autocast and torch.equal(_bits(got), _bits(want))
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            got = layer(True)
        torch.cuda.current_stream().wait_stream(side)
        assert torch.equal(_bits(got), _bits(layer(False)))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = layer(True)
        for seed in (1, 2, 3):
            choose(seed)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(_bits(out), _bits(layer(False))), seed
