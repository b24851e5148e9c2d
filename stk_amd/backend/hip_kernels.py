"""Kernel boundary: the functions the autograd layer calls, backed by libstk_amd.so.

`sdd`, `dsd`, `dds` and `row_indices` keep the positional signatures of
stk/backend/triton_kernels.py (:332-339, :222-233, :278-289, :389-391), write
into a caller-allocated `out`, return None and raise AssertionError for the
same shape violations (:15-19, :243, :299, :351).  `transpose_meta`, `to_dense`
and `to_sparse` are the device versions of stk/matrix.py:105-123 and
stk/ops/matrix_ops.py:36-85.

Device tensors launch on torch's current stream without synchronising (to_sparse
and an exact route read one int back, as the reference's torch.nonzero does); for them nothing falls
back to another implementation.  Calls of the four reference functions whose tensors
all live in host memory are handed to the host library (host_kernels), which is how
the reference's plumbing configuration - products on CPU tensors - runs here.

The checks, allocations and launches are native code (csrc/native.cc); what is left here is what depends on the
switches below and on the caches: which fusion plan and which workspace a launch gets.
"""
import threading

import torch

from stk_amd.backend import _lib, host_kernels

_INDEX_DTYPES = {torch.int16: _lib.STK_I16, torch.int32: _lib.STK_I32}


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_raw_device = getattr(torch._C, "_cuda_getDevice", None)


def _stream(device=None):
    """Handle of torch's current stream on `device` (default: the current device).  Read through torch's C entry
    points where they exist: torch.cuda.current_stream() builds a Stream object, which costs several microseconds
    on a path that every launch takes."""
    if _raw_stream is not None and _raw_device is not None:
        return _raw_stream(_raw_device() if device is None or device.index is None else device.index)
    return torch.cuda.current_stream(device).cuda_stream


def _capture_id(handle):
    """Identifier of the graph capture under way on the stream `handle`, 0 outside captures.  A buffer
    allocated or filled while a capture is under way exists only in that graph's replays: the caches below keep
    such a buffer apart from launches outside that capture."""
    return _lib.native().capture_id(handle)


def follow_stream(waiting, first):
    """What is launched on the stream with the handle `waiting` from now on starts after what has been launched on `first`."""
    _lib.native().follow(waiting, first)


def _need_gpu(*tensors):
    for t in tensors:
        if not t.is_cuda:
            raise RuntimeError("stk_amd: this operation runs on a ROCm GPU only; got a tensor on " + str(t.device))


# Tile fusion across identical neighbouring block rows / columns (stk_build_plan).  Results do not
# depend on it; switching it off makes every product take the one-line-per-tile kernels.
FUSION = True


def _version_of(t):
    """In-place modification counter of a tensor, or None for a tensor that keeps none (inference mode)."""
    return None if t.is_inference() else t._version


def _plan_cache_get(tensors, blocking):
    """The cache entry on tensors[0] (`offsets`) if it describes exactly these index tensors in their
    present state, else None.  The entry keeps the other index tensors it was built from: their storage
    stays alive, so an address cannot come back with other contents, and identity plus the version
    counters say whether they still hold what the plan describes.  A plan built with the transpose
    metadata also serves a request without it."""
    cached = getattr(tensors[0], "_stk_plan", None)
    if cached is None or cached[2] != blocking:
        return None
    others, versions = cached[0], cached[5]
    if len(others) < len(tensors) - 1:
        return None
    for i, t in enumerate(tensors):
        if (i and others[i - 1] is not t) or t.is_inference() or t._version != versions[i]:
            return None
    return cached


def _plan_cache_put(tensors, blocking, plan, stream_handle, elsewhere, capture):
    """Remembers `plan` on tensors[0]; tensors without a version counter (made under inference mode)
    cannot be watched for in-place changes and are not cached.  stream_handle: the stream that the plan was built on;
    `elsewhere`: the plans of other streams on the same topology, by their handles; `capture`: the graph capture they were
    built in (0: none)."""
    versions = tuple(_version_of(t) for t in tensors)
    if None in versions:
        return False
    try:
        tensors[0]._stk_plan = (tuple(tensors[1:]), plan, blocking, stream_handle, elsewhere, versions, capture)
    except AttributeError:
        return False
    return True


# Plans of further streams that are kept with a topology.
PLAN_STREAMS = 32
_followed = threading.local()


class following:
    """Inside, plans are those of the stream with the handle `handle`: for launches on a stream that waits for what has been
    launched on that one, and that it will wait for."""

    def __init__(self, handle):
        self.handle = handle

    def __enter__(self):
        _followed.handle = self.handle

    def __exit__(self, *exc):
        _followed.handle = None


def fusion_plan(offsets, column_indices, offsets_t=None, column_indices_t=None, blocking=128):
    """Device tensor with the fusion roles of the block rows (and, when the
    transpose metadata is given, of the block columns): which neighbouring lines
    repeat each other and are computed as one 256-wide tile.  Depends on the
    topology only, so it is cached on the `offsets` tensor and rebuilt when one of
    the index tensors has been replaced or modified in place.

    Every stream that uses the topology builds a plan of its own, once: a plan is launched with on the stream that built it,
    so that neither its contents nor its memory need anything between streams.  (Sharing one takes an event behind every
    build, which cost 4.5 us of the 252 of a routed layer of 64 tokens and 20 us of the 735 of a training step of 5003, both of
    which build one on each pass.)

    Under a graph capture: a plan built before the capture is used as it is (on another stream than the one that
    built it without waiting for the build, which a capture cannot do: the build must be complete when the capture
    starts, as it is after the synchronisation with which torch.cuda.graph() begins); a plan built inside a capture
    serves that capture only, and launches outside it build their own."""
    _need_gpu(offsets, column_indices)
    want_cols = offsets_t is not None and column_indices_t is not None
    tensors = (offsets, column_indices) + ((offsets_t, column_indices_t) if want_cols else ())
    cached = _plan_cache_get(tensors, blocking)
    if cached is not None:
        handle, built_in = _stream(offsets.device), cached[6]
        if built_in == 0 and cached[3] == handle:
            return cached[1]
    followed = getattr(_followed, "handle", None)
    elsewhere = None
    if cached is not None:
        capture = _capture_id(handle)
        if followed is not None:
            handle = followed
        if built_in == capture:
            if cached[3] == handle:
                return cached[1]
            whole = (offsets,) + cached[0]    # (the plans of all streams are for the same directions)
            if _plan_cache_get(whole, blocking) is not None:
                tensors, elsewhere = whole, cached[4]
                if handle in elsewhere:
                    return elsewhere[handle]
        elif built_in == 0:
            return cached[1]
    plan = _lib.native().build_plan(*tensors, *(None,) * (4 - len(tensors)), blocking)
    if followed is not None:
        return plan      # (built on the following stream: for this launch only)
    if elsewhere is None:
        _remember_plan(tensors, blocking, plan)
    else:
        while len(elsewhere) >= PLAN_STREAMS:
            elsewhere.pop(list(elsewhere)[0], None)
        elsewhere[handle] = plan
    return plan


def _remember_plan(tensors, blocking, plan):
    """The plan has just been built on the current stream: into the cache with it."""
    handle = _stream(tensors[0].device)
    _plan_cache_put(tensors, blocking, plan, handle, {}, _capture_id(handle))


def _plan_for(data, offsets, column_indices, offsets_t, column_indices_t):
    """The fusion plan, for both directions, that a product on this topology gets; None for a product without one."""
    b = data.shape[-1]
    if FUSION and (b == 128 or b == 64) and data.shape[0] > 0:
        return fusion_plan(offsets, column_indices, offsets_t, column_indices_t, b)
    return None


def prepare_plan(data, offsets, column_indices, offsets_t, column_indices_t):
    """Builds the fusion plan of a topology for both directions if there is none yet.  sdd itself needs the block rows
    only (its signature, the reference's, has no transpose metadata), so a plan built by its first call would be built
    again, with the columns, by the dsd or dds that follows on the same topology; callers that have the whole metadata
    at hand (the autograd functions) call this first and every product finds the one plan.  Nothing is built for index tensors
    whose plan no product would find."""
    # (tensors made under inference mode keep no version counter: their plan is not cached)
    if (data.dim() == 3 and offsets.is_cuda and column_indices.numel() > 0
            and not (offsets.is_inference() or column_indices.is_inference() or offsets_t.is_inference() or column_indices_t.is_inference())):
        _plan_for(data, offsets, column_indices, offsets_t, column_indices_t)


ACTIVATIONS = {None: 0, "none": 0, "relu": 1, "gelu_tanh": 2, "gelu": 3, "silu": 4,
               # the derivatives: with the incoming gradient as the multiplier, the gradient with respect to the sums
               "relu_grad": 5, "gelu_tanh_grad": 6, "gelu_grad": 7, "silu_grad": 8}


def sdd(lhs, rhs, shape, out, offsets, row_indices, column_indices, block_order=None):
    """out[p] = lhs[block row p] @ rhs[block column p]; out is [nnz, b, b].

    block_order (optional, not in the reference signature) is a permutation of
    the blocks that sets the visiting order of workgroups for 64x64 blocks.
    """
    sdd_fused(lhs, rhs, shape, out, offsets, row_indices, column_indices, None, None, block_order)


def sdd_fused(lhs, rhs, shape, out, offsets, row_indices, column_indices, activation=None, multiplier=None,
              block_order=None, sums=None):
    """sdd whose store applies `activation` (a key of ACTIVATIONS) to the fp32 sums and, after the
    rounding, multiplies by `multiplier` ([nnz, b, b] values of a matrix with the same topology).
    `sums` (like `out`, or None) also receives the rounded sums themselves (stk_sdd_fused_sums).
    No counterpart as one call in the reference, whose callers run the activation and
    stk.ops.mul (stk/ops/eltwise_ops.py:3-28) as passes of their own over the values."""
    if not out.is_cuda:
        if ACTIVATIONS.get(activation, 1) != 0 or multiplier is not None or sums is not None:
            raise NotImplementedError("stk_amd: the fused store of sdd runs on a GPU only")
        host_kernels.matmul_dims(lhs.shape[1], lhs.shape[0], rhs.shape[0], rhs.shape[1], out.shape[-1])
        return host_kernels.sdd(lhs, rhs, shape, out, offsets, row_indices, column_indices)
    if activation not in ACTIVATIONS:
        raise ValueError(f"unknown activation {activation!r}; one of {sorted(k for k in ACTIVATIONS if k)}")
    b = out.shape[-1]
    plan = None
    if FUSION and (b == 128 or b == 64) and offsets is not None and out.shape[0] > 0:
        plan = fusion_plan(offsets, column_indices, blocking=b)
    _lib.native().sdd(lhs, rhs, out, offsets, row_indices, column_indices, plan, ACTIVATIONS[activation], multiplier, block_order, sums)


def activation_product(sums, factor, activation):
    """round(round(act(sums)) * factor) over the values of a sparse matrix (factor None: the first rounding only);
    `activation` a key of ACTIVATIONS, derivatives included (stk_activation_product)."""
    if activation not in ACTIVATIONS:
        raise ValueError(f"unknown activation {activation!r}")
    return _lib.native().activation_product(sums, factor, ACTIVATIONS[activation])


# dsd launches that fill the GPU only a few times cut the tiles of their last round into slices
# along k, which takes a workspace.  Results then differ in the last bit from the uncut sums;
# switching it off restores those.
SLICE_LAST_ROUND = True
# Partial tiles (256 KiB each) the workspace of a device has room for: 256 of them (64 MiB) let a last round of
# 128 tiles be cut in two, or one of 64 tiles in four; a launch that would like more is cut less.  The buffer is
# allocated on the first dsd that can use it and kept; release_workspaces() frees it.
DSD_WORKSPACE_SLOTS = 256
# Streams (their handles) whose dsd launches may run beside those of other streams (the autograd layer's side stream): they get
# a workspace of their own.  Everything else shares one per device, and a launch on another stream than the
# last one first waits for that stream.
CONCURRENT_STREAMS = set()
_dsd_workspaces = {}   # (device index, concurrent lane) -> [buffer, stream of the last launch]
# Held from the choice of a workspace to its launch: a thread that takes it over for another stream waits for what has been
# launched, which has to include the launch that the entry names.
_workspace_lock = threading.RLock()


def release_workspaces():
    """Frees the dsd workspaces (they are allocated again on demand)."""
    _dsd_workspaces.clear()


def _check_launch(status, ws):
    """Raises for a launch that was refused or failed.  Whatever a failed launch has left in the counters of the workspace
    `ws` is not reused; a call that was refused has not touched them."""
    if status == _lib.STK_ERR_HIP and ws is not None:
        for key in [key for key, entry in _dsd_workspaces.items() if entry[0] is ws]:
            del _dsd_workspaces[key]
    _lib.check(status)


def _workspace_choice(capturing, entry_stream, handle):
    """Which workspace a dsd launch on the stream `handle` takes.  `capturing`: a graph capture is under way on that
    stream; `entry_stream`: handle of the stream that last used the device's shared workspace (None: there is none yet).
      "private"  a buffer of the launch's own.  Every captured launch: its buffer comes out of the graph's memory pool, so
                 replays - on whatever stream, next to whatever eager launches or other graphs - share counters and
                 partial-tile slots with nobody.
      "create"   no shared workspace yet: allocate it for this stream.
      "shared"   the shared workspace, last used on this very stream: launches on one stream cannot overlap.
      "wait"     the shared workspace after waiting for the stream that used it last."""
    if capturing:
        return "private"
    if entry_stream is None:
        return "create"
    return "shared" if entry_stream == handle else "wait"


def _new_workspace(device, nbytes, counters):
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
    ws[:counters].zero_()   # (a fill kernel, also under capture; the slots behind the counters need no initial value)
    return ws


def _dsd_workspace(data, m, n):
    """Workspace of stk_dsd for a product with these sparse values, launched on the current stream, or None:
    [counters | slots], the counters zero between launches."""
    blocking = data.shape[-1]
    if not SLICE_LAST_ROUND or blocking != 128:
        return None
    lib = _lib.load()
    # (launches with little work for every compute unit do not cut their last round either)
    if lib.stk_dsd_workspace_bytes(m, n, blocking) <= 0 or lib.stk_dsd_is_small(data.shape[0], n):
        return None
    device = data.device
    handle = _stream(device)
    key = (device.index, handle in CONCURRENT_STREAMS)
    entry = _dsd_workspaces.get(key)
    counters = lib.stk_dsd_workspace_counter_bytes()
    nbytes = counters + DSD_WORKSPACE_SLOTS * lib.stk_dsd_workspace_slot_bytes()
    if entry is not None and entry[0].numel() != nbytes:
        entry = None
    choice = _workspace_choice(_capture_id(handle) != 0, None if entry is None else entry[1].cuda_stream, handle)
    if choice == "private":
        # zeroed by a fill kernel that is part of the graph; the memory goes back to the graph's pool when the
        # caller drops it, where only later allocations of the same capture, which run behind this launch, reuse it
        return _new_workspace(device, nbytes, counters)
    if choice == "create":
        entry = _dsd_workspaces[key] = [_new_workspace(device, nbytes, counters), torch.cuda.current_stream(device)]
    elif choice == "wait":
        stream = torch.cuda.current_stream(device)
        stream.wait_stream(entry[1])   # launches that share a workspace must not overlap
        entry[0].record_stream(stream)   # (dropped, its memory is not handed out again before they have ended)
        entry[1] = stream
    return entry[0]


def dsd(shape, data, offsets, row_indices, column_indices, offsets_t, column_indices_t,
        block_offsets_t, transpose_a, rhs, out):
    """out = op(sparse) @ rhs; `shape` is the logical shape of the sparse operand."""
    if not out.is_cuda:
        host_kernels.matmul_dims(shape[1], shape[0], rhs.shape[0], rhs.shape[1], data.shape[-1])
        return host_kernels.dsd(shape, data, offsets, row_indices, column_indices, offsets_t, column_indices_t, block_offsets_t,
                                transpose_a, rhs, out)
    m, k = shape
    plan = _plan_for(data, offsets, column_indices, offsets_t, column_indices_t)
    with _workspace_lock:
        ws = _dsd_workspace(data, m, out.shape[1]) if plan is not None else None
        status = _lib.native().dsd(m, k, data, offsets, column_indices, offsets_t, column_indices_t, block_offsets_t, transpose_a, rhs, out, plan, ws)
        if status != _lib.STK_OK:
            _check_launch(status, ws)


def dds(lhs, shape, data, offsets, row_indices, column_indices, offsets_t, column_indices_t,
        block_offsets_t, transpose_b, out):
    """out = lhs @ op(sparse); `shape` is the logical shape of the sparse operand."""
    if not out.is_cuda:
        host_kernels.matmul_dims(lhs.shape[1], lhs.shape[0], shape[0], shape[1], data.shape[-1])
        return host_kernels.dds(lhs, shape, data, offsets, row_indices, column_indices, offsets_t, column_indices_t, block_offsets_t,
                                transpose_b, out)
    k, n = shape
    plan = _plan_for(data, offsets, column_indices, offsets_t, column_indices_t)
    _lib.native().dds(lhs, k, n, data, offsets, column_indices, offsets_t, column_indices_t, block_offsets_t, transpose_b, out, plan)


def dsd_dds(shape, data, offsets, row_indices, column_indices, offsets_t, column_indices_t, block_offsets_t, rhs, out_dsd, lhs, out_dds):
    """out_dsd = sparse @ rhs and out_dds = lhs @ sparse for one sparse operand [m, k] = `shape`, in one launch where
    the layouts allow it (the two gradients of sdd, stk/backend/sputnik.py:274-299); otherwise the two products one
    after the other.  The results are those of dsd (without its workspace) and dds, bit for bit."""
    plan = _plan_for(data, offsets, column_indices, offsets_t, column_indices_t)
    _lib.native().dsd_dds(*shape, data, offsets, column_indices, offsets_t, column_indices_t, block_offsets_t, rhs, out_dsd, lhs, out_dds, plan)


def dsd_dsd(shape, data, offsets, row_indices, column_indices, offsets_t, column_indices_t, block_offsets_t, rhs, out, rhs_t, out_t):
    """out = sparse @ rhs and out_t = sparse^T @ rhs_t for one sparse operand [m, k] = `shape`, in one launch where the
    layouts allow it (the two gradients of an sdd whose rhs was a .t() view, stk/backend/sputnik.py:274-299); otherwise
    the two products one after the other.  The results are those of two dsd calls without the workspace, bit for bit."""
    plan = _plan_for(data, offsets, column_indices, offsets_t, column_indices_t)
    _lib.native().dsd_dsd(*shape, data, offsets, column_indices, offsets_t, column_indices_t, block_offsets_t, rhs, out, rhs_t, out_t, plan)


def sdd_dsd(shape, lhs, rhs_sdd, out_sdd, data, offsets, row_indices, column_indices, offsets_t, column_indices_t, block_offsets_t,
            transpose_a, rhs_dsd, out_dsd):
    """out_sdd = lhs @ rhs_sdd on the topology [m, n] = `shape` and out_dsd = op(sparse) @ rhs_dsd for the values `data` on the
    same topology, in one launch where the layouts allow it (the two gradients of dsd, stk/backend/sputnik.py:131-155);
    otherwise the two products one after the other.  The results are those of sdd and dsd (without its workspace), bit
    for bit."""
    plan = _plan_for(data, offsets, column_indices, offsets_t, column_indices_t)
    _lib.native().sdd_dsd(*shape, lhs, rhs_sdd, out_sdd, data, row_indices, offsets, column_indices, offsets_t, column_indices_t, block_offsets_t,
                          transpose_a, rhs_dsd, out_dsd, plan)


def row_indices(shape, data, offsets, column_indices, out):
    """out[offsets[r]:offsets[r+1]] = r for every block row r."""
    if not out.is_cuda:
        return host_kernels.row_indices(shape, data, offsets, column_indices, out)
    _lib.native().row_indices(offsets, out)


def transpose_meta(size, data, row_indices, column_indices, offsets):
    """(column_indices_t, offsets_t, block_offsets_t), stable tie order."""
    return _lib.native().transpose_meta(size[1] // data.shape[-1], row_indices, column_indices)


DMOE_PLAN_EXPERTS = 1024   # up to this many experts stk_dmoe_topology_plan builds the plan (their shares fit in LDS)


def dmoe_topology(padded_bins, blocking, block_rows, blocks_per_row, index_dtype=torch.int16):
    """(offsets, row_indices, column_indices, offsets_t, column_indices_t, block_offsets_t) of the
    block-diagonal dropless-MoE pattern, one launch, no sort.  padded_bins: int32 device tensor,
    inclusive prefix sum of the per-expert row counts (each a multiple of `blocking`).  The launch also
    builds the fusion plan, which the products on the topology then find on `offsets` (not under inference mode, where
    they could not)."""
    with_plan = (FUSION and blocking in (64, 128) and block_rows * blocks_per_row > 0 and padded_bins.numel() <= DMOE_PLAN_EXPERTS
                 and not torch.is_inference_mode_enabled())
    *meta, plan = _lib.native().dmoe_topology(padded_bins, blocking, block_rows, blocks_per_row, _INDEX_DTYPES[index_dtype] == _lib.STK_I32, with_plan)
    if plan is not None:
        offsets, _, column_indices, offsets_t, column_indices_t, _ = meta
        _remember_plan((offsets, column_indices, offsets_t, column_indices_t), blocking, plan)
    return tuple(meta)


def to_dense(data, row_indices, column_indices, rows, cols, offsets=None):
    """offsets: where given, those of the block rows (row r's blocks are the entries offsets[r] .. offsets[r + 1] - 1)."""
    return _lib.native().to_dense(data, row_indices, column_indices, rows, cols, offsets)


def to_sparse(x, blocking, index_dtype=torch.int16):
    """(data, row_indices, column_indices, offsets) of the nonzero blocks of x."""
    return to_sparse_meta(x, blocking, index_dtype)[:4]


def to_sparse_meta(x, blocking, index_dtype=torch.int16):
    """The results of to_sparse, then column_indices_t, offsets_t and block_offsets_t, or None for each of these three: they
    come with the others where the matrix has few blocks."""
    return _lib.native().to_sparse(x, blocking, _INDEX_DTYPES[index_dtype] == _lib.STK_I32)


# ---------------------------------------------------------------- token routing (no counterpart in the reference)
def route(top_experts, num_experts, blocking, padded_rows=None):
    """(indices, bin_ids, bins, padded_bins, slot_rows, row_slots) of stk_route; all int32 on the
    device of top_experts.  padded_rows: rows of the padded layout (length of row_slots); None: as many as it needs, which
    the host waits for."""
    return _lib.native().route(top_experts, num_experts, blocking, -1 if padded_rows is None else padded_rows)


def padded_gather(x, row_slots, top_k, weights=None):
    """out[r] = (weights[s]) * x[s // top_k], s = row_slots[r]; zeros where s < 0."""
    return _lib.native().padded_gather(x, row_slots, top_k, weights)


def padded_scatter(x, slot_rows, top_k, weights=None):
    """out[t] = sum_k (weights[s]) * x[slot_rows[s]], s = t * top_k + k."""
    return _lib.native().padded_scatter(x, slot_rows, top_k, weights)


def padded_scatter_weight_gradient(x, grad, slot_rows, top_k):
    """fp32 [slots]: <x[slot_rows[s]], grad[s // top_k]>."""
    return _lib.native().padded_scatter_weight_gradient(x, grad, slot_rows, top_k)


def sdd_gather_reads_plan(x, top_k, shape, blocking=128):
    """Whether sdd_gather of these token rows, or what runs where it has no kernel, makes use of a plan: not where block rows of
    128 hold few slots each."""
    return blocking != 128 or x.dim() != 2 or bool(_lib.native().sdd_gather_reads_plan(shape[0], x.shape[1], x.shape[0] * top_k))


def sdd_gather(x, row_slots, top_k, rhs, shape, out, offsets, row_indices, column_indices, activation=None):
    """out = act(sdd(padded_gather(x, row_slots, top_k), rhs)) on the topology without the padded copy of x
    (stk_sdd_gather); bit-identical to padded_gather followed by sdd_fused.  False, with nothing launched, when
    the library has no such kernel for this case (the caller then makes the two calls); True otherwise."""
    if out.shape[-1] != 128 or activation not in ACTIVATIONS or ACTIVATIONS[activation] > ACTIVATIONS["silu"] or not FUSION:
        return False
    plan = None
    if offsets is not None and out.shape[0] > 0 and sdd_gather_reads_plan(x, top_k, shape):
        plan = fusion_plan(offsets, column_indices, blocking=128)
    return _lib.native().sdd_gather(x, row_slots, top_k, rhs, *shape, out, offsets, row_indices, column_indices, plan, ACTIVATIONS[activation])


def dsd_scatter(shape, data, offsets, column_indices, offsets_t, column_indices_t, rhs, row_slots, weights, out):
    """out = padded_scatter(sparse @ rhs, top_k = 1, weights) without the padded result (stk_dsd_scatter): row r of
    the product goes to out[row_slots[r]]; bit-identical to dsd followed by padded_scatter.  False, with nothing
    launched, when the library has no such kernel for this case (the caller then makes the two calls); True otherwise."""
    m, k = shape
    n = rhs.shape[1]
    if data.shape[-1] != 128 or n < 256 or n % 64 or not FUSION or data.shape[0] == 0 or out.shape[0] == 0:
        return False
    plan = fusion_plan(offsets, column_indices, offsets_t, column_indices_t, blocking=128)
    with _workspace_lock:
        ws = _dsd_workspace(data, m, n)
        status = _lib.native().dsd_scatter(m, k, data, offsets, column_indices, rhs, row_slots, weights, out, plan, ws)
        if status == _lib.STK_ERR_UNSUPPORTED:
            return False
        _check_launch(status, ws)
    return True


def dsd_scatter_few(shape, data, offsets, column_indices, rhs, row_slots, slot_rows, top_k, weights, offsets_t=None, column_indices_t=None):
    """padded_scatter(sparse @ rhs, top_k, weights) from the rows that hold a slot alone (stk_dsd_scatter_few_as_cut); bit-identical
    to dsd followed by padded_scatter (without the transpose metadata: to a dsd without its workspace).  None, with nothing
    launched, when the library has no such kernel for this case (the block rows hold many slots, other than 128-blocks of 16-bit
    values; the caller then makes the two calls)."""
    if data.shape[-1] != 128 or data.dtype == torch.float32 or not FUSION or rhs.dim() != 2:
        return None
    m, k = shape
    # the workspace of that dsd, if it may cut its last round: the plan then says where, and the sums here are cut alike
    partial_tiles = DSD_WORKSPACE_SLOTS if SLICE_LAST_ROUND and offsets_t is not None else 0
    dsd_workspace = _lib.native().dsd_scatter_few_case(m, rhs.shape[1], data.shape[0], slot_rows.numel(), partial_tiles)
    if dsd_workspace < 0:
        return None
    plan = fusion_plan(offsets, column_indices, offsets_t, column_indices_t, 128) if dsd_workspace else None
    return _lib.native().dsd_scatter_few(m, k, data, offsets, column_indices, rhs, row_slots, slot_rows, top_k, weights, plan, dsd_workspace)
