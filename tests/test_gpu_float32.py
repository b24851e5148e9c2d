"""float32 products on the GPU: the tile sizes, layouts and fallbacks of stk_amd/csrc/fp32.hip against float64 products.

The bound is the one of a sum of K products in fp32 in any order: every element is off by at most
(K + 1) 2^-24 sum |a| |b| (each product and each of the sums rounded once)."""
import numpy as np
import pytest
import torch

import stk_amd as stk
from stk_amd.backend import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(got, a, b, keep=None):
    want, bound = a.double() @ b.double(), (a.double().abs() @ b.double().abs()) * ((a.shape[1] + 1) * 2.0 ** -24)
    if keep is not None:
        want, bound = want * keep, bound * keep
    assert got.shape == want.shape
    assert ((got.double() - want).abs() <= bound).all(), float(((got.double() - want).abs() - bound).max())


def _sparse(rows, cols, density, b, gen):
    keep = (torch.rand(rows // b, cols // b, generator=gen, device=DEV) < density).float()
    keep[0, 0] = 1.0
    keep = keep.repeat_interleave(b, 0).repeat_interleave(b, 1)
    dense = torch.randn(rows, cols, generator=gen, device=DEV) * keep
    return dense, keep, stk.ops.to_sparse(dense, b)


# rows, cols of the sparse matrix, inner size, density: one block, an extent that leaves only 32-wide tiles, one that leaves
# 64-wide ones, lines of more than 64 blocks (the walk is read 64 entries at a time), enough work for the 64-wide and for
# the 128-wide tiles
@pytest.mark.parametrize("rows,cols,inner,density,b", [
    (128, 128, 128, 1.0, 128), (64, 64, 64, 1.0, 64), (256, 384, 384, 0.5, 128), (128, 192, 192, 0.7, 64), (128, 4224, 128, 1.0, 64),
    (4224, 64, 64, 0.9, 64), (1024, 1280, 1024, 0.5, 128), (4096, 4096, 4096, 0.5, 128)])
@pytest.mark.parametrize("views", [False, True])
def test_products_of_every_tile_size_and_layout(rows, cols, inner, density, b, views):
    gen = torch.Generator(device=DEV).manual_seed(rows + cols)
    dense, keep, s = _sparse(rows, cols, density, b, gen)

    def operand(m, n):
        return torch.randn(n, m, generator=gen, device=DEV).t() if views else torch.randn(m, n, generator=gen, device=DEV)

    a, w, v, u = operand(rows, inner), operand(inner, cols), operand(cols, inner), operand(inner, rows)
    _check(stk.ops.to_dense(stk.ops.sdd(a, w, s)), a, w, keep)
    _check(stk.ops.dsd(s, v), dense, v)
    _check(stk.ops.dds(u, s), u, dense)
    _check(stk.ops.dsd(s.t(), a), dense.t(), a)
    _check(stk.ops.dds(w, s.t()), w, dense.t())


# lines of very unequal lengths, empty ones among them: the number of lines (64 are ordered by length, 66 are not), and of
# tiles of the dense operand that is a multiple of the eight dies (1024), or not, with whole and partial rounds of a
# die's units
@pytest.mark.parametrize("lines,inner", [(3, 64), (9, 448), (64, 192), (64, 1024), (66, 192)])
def test_lines_of_unequal_lengths(lines, inner):
    gen, b = torch.Generator(device=DEV).manual_seed(lines * inner), 64
    keep = (torch.rand(lines, 8, generator=gen, device=DEV) < torch.linspace(0, 1.2, lines, device=DEV)[torch.randperm(lines, generator=gen, device=DEV)][:, None])
    keep = keep.float().repeat_interleave(b, 0).repeat_interleave(b, 1)
    dense = torch.randn(lines * b, 8 * b, generator=gen, device=DEV) * keep
    s = stk.ops.to_sparse(dense, b)
    v, a = torch.randn(8 * b, inner, generator=gen, device=DEV), torch.randn(inner, 8 * b, generator=gen, device=DEV)
    _check(stk.ops.dsd(s, v), dense, v)
    _check(stk.ops.dds(a, s.t()), a, dense.t())


@pytest.mark.parametrize("inner", [32, 96, 160])
def test_an_inner_size_of_odd_multiples_of_32(inner):
    gen = torch.Generator(device=DEV).manual_seed(inner)
    _, keep, s = _sparse(256, 256, 0.7, 128, gen)
    a, w = torch.randn(256, inner, generator=gen, device=DEV), torch.randn(inner, 256, generator=gen, device=DEV)
    _check(stk.ops.to_dense(stk.ops.sdd(a, w, s)), a, w, keep)


@pytest.mark.parametrize("extent,ld", [(40, 40), (128, 131), (96, 98)])
def test_ragged_extents_and_odd_strides_take_the_generic_kernels(extent, ld):
    # through the C ABI: the Python boundary asks for whole blocks and strides that are multiples of eight
    gen = torch.Generator(device=DEV).manual_seed(extent)
    dense, _, s = _sparse(256, 384, 0.6, 128, gen)
    rhs = torch.randn(384, ld, generator=gen, device=DEV)
    out = torch.full((256, ld), float("nan"), device=DEV)
    _lib.check(_lib.load().stk_dsd(256, 384, extent, s.data.data_ptr(), s.offsets.data_ptr(), s.column_indices.data_ptr(), s.offsets_t.data_ptr(),
                                   s.column_indices_t.data_ptr(), s.block_offsets_t.data_ptr(), 0, rhs.data_ptr(), ld, 1, out.data_ptr(), ld,
                                   s.data.shape[0], 128, _lib.STK_F32, _lib.STK_I16, None, None, 0, torch.cuda.current_stream().cuda_stream))
    _check(out[:, :extent], dense, rhs[:, :extent])
    assert bool(torch.isnan(out[:, extent:]).all()) or ld == extent


@pytest.mark.parametrize("activation", ["gelu_tanh", "silu"])
def test_the_fused_store_in_every_tile_size(activation):
    f = {"gelu_tanh": lambda x: torch.nn.functional.gelu(x, approximate="tanh"), "silu": torch.nn.functional.silu}[activation]
    gen = torch.Generator(device=DEV).manual_seed(3)
    for rows, cols, inner in ((128, 256, 64), (1024, 1024, 64), (4096, 4096, 64)):       # tiles of 32, 64 and 128
        _, keep, s = _sparse(rows, cols, 1.0, 128, gen)
        a, w = torch.randn(rows, inner, generator=gen, device=DEV), torch.randn(inner, cols, generator=gen, device=DEV)
        m = stk.Matrix(s.size(), torch.randn(s.data.shape, generator=gen, device=DEV), s.row_indices, s.column_indices, s.offsets,
                       s.column_indices_t, s.offsets_t, s.block_offsets_t)
        got = stk.ops.to_dense(stk.ops.sdd_fused(a, w, s, activation, m))
        want = f(a.double() @ w.double()) * stk.ops.to_dense(m).double()
        # the sums' error through a function of slope below 1.2, and the hardware's exp2 and reciprocal (1 ulp each)
        bound = (1.2 * (inner + 1) * 2.0 ** -24 * (a.double().abs() @ w.double().abs()) + 2.0 ** -19 * (a.double() @ w.double()).abs()) \
            * stk.ops.to_dense(m).double().abs() + 1e-7
        assert ((got.double() - want).abs() <= bound).all(), (rows, float(((got.double() - want).abs() / bound).max()))
