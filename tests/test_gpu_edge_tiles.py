"""Dense extents that are not a multiple of the 256-wide tiles: the last tile is moved back over the one before it and
stores only what that one does not.  Every product against the dense product in fp32 on the GPU, with the scale-free
bounds of the other product tests, and no element left unwritten."""
import numpy as np
import pytest
import torch

import stk_amd as stk
from tests import _util as U

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(rows_per_expert, width, b, dtype, hidden, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    bins = torch.from_numpy(np.cumsum(np.array(rows_per_expert) * b).astype(np.int32)).to(DEV)
    topo = stk.ops.dmoe_topology(bins, b, sum(rows_per_expert), width, dtype=dtype)
    rows, cols = topo.size()
    s = stk.Matrix(topo.size(), torch.randn(topo.data.shape, device=DEV, generator=g).to(dtype), topo.row_indices, topo.column_indices, topo.offsets,
                   topo.column_indices_t, topo.offsets_t, topo.block_offsets_t)
    operand = lambda m, n: torch.randn(m, n, device=DEV, generator=g).to(dtype)
    return s, operand(cols, hidden), operand(rows, hidden), operand(hidden, rows), operand(hidden, cols)


# runs of one, two, three and more rows (lone lines, pairs, threes, fours); `many` has the work for the eight-wave tiles, and
# `more` the lines for them where block rows are walked and the extent is no multiple of 256
_FEW, _MANY, _MORE = [1, 2, 3], [1, 2, 3, 5, 4, 0, 7, 1] * 6, [1, 2, 3, 5, 4, 0, 7, 1, 22] * 6


@pytest.mark.parametrize("b,hidden", [(128, 128), (128, 384), (128, 640), (128, 1152), (64, 64), (64, 192), (64, 320), (64, 448), (64, 704), (64, 1216)])
@pytest.mark.parametrize("rows,width", [(_FEW, 3), (_MANY, 23), (_MORE, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_products_with_ragged_dense_extents(b, hidden, rows, width, dtype):
    s, v, a, u, w = _case(rows, width, b, dtype, hidden, hidden + width)
    dense = stk.ops.to_dense(s).float()
    for name, got, want in (("dsd", stk.ops.dsd(s, v), dense @ v.float()),
                            ("dsd view", stk.ops.dsd(s, w.t()), dense @ w.float().t()),
                            ("dsd t", stk.ops.dsd(s.t(), a), dense.t() @ a.float()),
                            ("dds", stk.ops.dds(u, s), u.float() @ dense),
                            ("dds view", stk.ops.dds(a.t(), s), a.float().t() @ dense),
                            ("dds t", stk.ops.dds(w, s.t()), w.float() @ dense.t())):
        U.assert_close_scaled(got, want, dtype, f"{name} {b} {hidden}", tol=dict(rtol=1e-2, atol=1.0))


@pytest.mark.parametrize("b,hidden", [(128, 384), (128, 1152), (64, 320), (64, 704)])
@pytest.mark.parametrize("view", [False, True])
def test_gradients_with_ragged_dense_extents(b, hidden, view):
    # the joint launches of sdd's gradients and the pair of dsd's against the products one by one
    dtype = torch.bfloat16
    s, v, a, u, w = _case(_MANY, 23, b, dtype, hidden, hidden)
    x = a.detach().requires_grad_(True)
    weight = (w.t().contiguous().t() if view else w).detach().requires_grad_(True)
    h = stk.ops.sdd(x, weight, s)
    v = v.detach().requires_grad_(True)
    y = stk.ops.dsd(h, v)
    dy = a
    dx, dw, dv = torch.autograd.grad(y, (x, weight, v), dy)
    dh = stk.ops.sdd(dy, v.detach().t(), s)
    assert torch.equal(dv, stk.ops.dsd(h.t(), dy))
    assert torch.equal(dw, stk.ops.dsd(dh.t(), x.detach()).t() if view else stk.ops.dds(x.detach().t(), dh))
    want = stk.ops.to_dense(dh).float() @ weight.detach().float().t()
    U.assert_close_scaled(dx, want, dtype, "dx", tol=dict(rtol=1e-2, atol=1.0))


@pytest.mark.parametrize("hidden", [384, 1152])
def test_scattered_rows_with_ragged_columns(hidden):
    g = torch.Generator(device=DEV).manual_seed(hidden)
    top = torch.randint(0, 16, (6000, 1), device=DEV, generator=g, dtype=torch.int32)
    r = stk.ops.route(top, 16, 128)
    topo = stk.ops.dmoe_topology(r.padded_bins, 128, r.row_slots.numel() // 128, 24, dtype=torch.bfloat16)
    h = stk.Matrix(topo.size(), torch.randn(topo.data.shape, device=DEV, generator=g).bfloat16(), topo.row_indices, topo.column_indices, topo.offsets,
                   topo.column_indices_t, topo.offsets_t, topo.block_offsets_t)
    w2 = torch.randn(16 * 24 * 128, hidden, device=DEV, generator=g).bfloat16()
    weights = torch.rand(6000, 1, device=DEV, generator=g)
    with torch.no_grad():
        assert torch.equal(stk.ops.dsd_scatter(h, w2, r, weights), stk.ops.padded_scatter(stk.ops.dsd(h, w2), r, weights))
