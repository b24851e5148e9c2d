"""The fusion plan that stk_dmoe_topology_plan builds in closed form against the one stk_build_plan finds by comparing the
lines of the same topology: tiles, lists and hints, bit for bit."""
import numpy as np
import pytest
import torch

import stk_amd as stk
from stk_amd.backend import _lib, hip_kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _parts(plan, br, bc, nnz):
    """What the products read of a plan: the tiles of sdd, the counts, the used part of the lists, the hints."""
    whole = plan.cpu().numpy()
    most = (nnz + br + 1) // 2
    sdd = whole[:8 + 8 * most].view(np.int32)
    body = whole[8 + 8 * most:]
    off = (3 * (br + bc) + 3) // 4 * 4
    lists = body[off:off + 4 * 5 * (2 + br + bc)].view(np.int32)
    out = {"sdd": sdd[:2 + 2 * int(sdd[0])].tolist(), "counts": lists[:10].tolist(), "hints": body[off + 4 * 5 * (2 + br + bc):][:64].tolist()}
    for d, lines in enumerate((br, bc)):
        for kind in range(5):
            base = 10 + (5 * br if d else 0) + kind * lines
            out["list", d, kind] = lists[base:base + int(lists[5 * d + kind])].tolist()
    # (bytes 24 .. 31 of a direction's hints are not used)
    out["hints"] = [v for i, v in enumerate(out["hints"]) if i % 32 < 24]
    return out


# block rows per expert, blocks per row: one expert; runs of every length up to nine, with empty experts first, in between and
# last; one block column per expert; more lone columns than a list is sorted for; an expert with over 255 block rows and one
# with half of them all (heavy with 64-blocks); the largest number of experts; odd and even widths
_CASES = [([1], 1), ([7], 5), ([0, 1, 2, 3, 0, 4, 5, 6, 7, 8, 9, 0], 4), ([3, 0, 2, 5], 1), ([0, 0, 3, 0], 7), ([1] * 40 + [0] * 200, 33),
          ([300, 4, 1, 260, 90], 3), ([64] + [1] * 63, 64), ([i % 4 for i in range(1024)], 2), ([2, 3] * 32, 32)]


@pytest.mark.parametrize("blocking,index_dtype", [(128, torch.int16), (64, torch.int16), (128, torch.int32)])
@pytest.mark.parametrize("case", range(len(_CASES)))
def test_closed_form_plan_is_the_compared_plan(case, blocking, index_dtype):
    rows, width = _CASES[case]
    block_rows = sum(rows)
    bins = torch.from_numpy(np.cumsum(np.array(rows) * blocking).astype(np.int32)).to(DEV)
    m = stk.ops.dmoe_topology(bins, blocking, block_rows, width, data=torch.empty(block_rows * width, blocking, blocking, dtype=torch.float16, device=DEV),
                              index_dtype=index_dtype)
    assert m.offsets._stk_plan[2] == blocking
    built = hip_kernels.fusion_plan(m.offsets, m.column_indices, m.offsets_t, m.column_indices_t, blocking=blocking)
    assert built is m.offsets._stk_plan[1]           # the launch of the topology left it there
    compared = hip_kernels.fusion_plan(m.offsets.clone(), m.column_indices, m.offsets_t, m.column_indices_t, blocking=blocking)
    assert compared is not built
    args = block_rows, len(rows) * width, block_rows * width
    got, want = _parts(built, *args), _parts(compared, *args)
    for key in want:
        assert got[key] == want[key], key


def test_rows_behind_the_last_bin_belong_to_the_last_expert():
    bins = torch.tensor([256, 384], dtype=torch.int32, device=DEV)
    m = stk.ops.dmoe_topology(bins, 128, 6, 3)           # three more block rows than the bins say
    compared = hip_kernels.fusion_plan(m.offsets.clone(), m.column_indices, m.offsets_t, m.column_indices_t, blocking=128)
    assert m.offsets_t.tolist() == [0, 2, 4, 6, 10, 14, 18]
    assert _parts(m.offsets._stk_plan[1], 6, 6, 18) == _parts(compared, 6, 6, 18)


# 1024 experts whose bins go up and down: their row counts, each taken on its own, add up to 512 times the rows there are
@pytest.mark.parametrize("blocking", [128, 64])
@pytest.mark.parametrize("bins,block_rows", [([5, 2, 9, 9, 4, 12], 12), ([-3, 4, -1, 8], 8), ([0, 40] * 512, 40), ([50, 10, 60], 8)])
def test_bins_that_do_not_ascend_stay_inside_the_plan(bins, block_rows, blocking):
    E, width = len(bins), 3
    nnz, columns = block_rows * width, E * width
    given = torch.tensor(bins, dtype=torch.int32, device=DEV) * blocking
    read_as = torch.cummax(given.clamp(0, block_rows * blocking), 0).values
    lib = _lib.load()
    size, guard = lib.stk_plan_bytes(block_rows, columns, nnz), 1 << 16
    ends = {}
    for name, b in (("given", given), ("read as", read_as)):
        plan = torch.full((size + guard,), 0xa5, dtype=torch.uint8, device=DEV)
        ints = [torch.full((n,), -7, dtype=torch.int32, device=DEV) for n in (block_rows + 1, nnz, nnz, columns + 1, nnz, nnz)]
        _lib.check(lib.stk_dmoe_topology_plan(b.data_ptr(), E, blocking, block_rows, width, _lib.STK_I32, *(t.data_ptr() for t in ints),
                                              plan.data_ptr(), size, torch.cuda.current_stream().cuda_stream))
        assert (plan[size:] == 0xa5).all()
        ends[name] = [t.tolist() for t in ints], _parts(plan[:size], block_rows, columns, nnz)
    assert ends["given"] == ends["read as"]
    assert sorted(ends["given"][0][5]) == list(range(nnz))     # every block has its place in the columns' order
