"""Format conversion and small helpers (stk/ops/matrix_ops.py:7-98).

GPU tensors are converted by the HIP kernels (block mask + wavefront
compaction + block copy); host tensors by torch statements, as the reference
does when it builds matrices on the CPU."""
import numpy as np
import torch

from stk_amd.backend import autograd as sputnik
from stk_amd.backend import hip_kernels, host_format
from stk_amd.matrix import Matrix


@torch.no_grad()
def row_indices(shape, data, offsets, column_indices):
    return sputnik.row_indices(shape, data, offsets, column_indices)


@torch.no_grad()
def to_dense(x):
    assert isinstance(x, Matrix)
    rows, cols = int(np.prod(x.shape[:-1])), x.shape[-1]
    if x.is_cuda:
        dense = hip_kernels.to_dense(x.data, x.row_indices, x.column_indices, rows, cols, x.offsets if x.is_contiguous() else None)
    else:
        dense = host_format.to_dense(x.data, x.row_indices, x.column_indices, rows, cols)
    return dense.reshape(x.size())


@torch.no_grad()
def to_sparse(x, blocking=1):
    assert x.dim() == 2
    assert x.size()[0] % blocking == 0
    assert x.size()[1] % blocking == 0
    if x.is_cuda:
        return Matrix(x.size(), *hip_kernels.to_sparse_meta(x, blocking))
    return Matrix(x.size(), *host_format.to_sparse(x, blocking))


@torch.no_grad()
def ones_like(x):
    # the transpose metadata is rebuilt, as in stk/ops/matrix_ops.py:88-93
    return Matrix(x.size(), torch.ones_like(x.data), x.row_indices, x.column_indices, x.offsets)


def sum(x):
    assert isinstance(x, Matrix)
    return x.data.sum()
