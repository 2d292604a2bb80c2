"""Fused linear + cross-entropy with the names of the reference's
cross_entropy_triton/cross_entropy.py, on the HIP kernels of libmi_attn.so
(no Triton, no fallback).  The backward follows the reference's scheme in blocks
of rows, with the two plain gradient GEMMs left to the BLAS library behind
torch.mm.  Its dlogits come from the forward's fp32 logits where those are kept
(KEEP_BYTES below), and from one launch that computes the logits again and
applies the element-wise step to the fp32 accumulators where they are not: in a
plain cross_entropy_fused_fwd / _bwd pair the logits are never materialised."""
import ctypes as C
import threading
import weakref

import torch

from . import _lib
from .ops import _num_cus, _ptr, _require_gpu, _stream

_TAGS = {torch.bfloat16: _lib.MI_DTYPE_BF16, torch.float16: _lib.MI_DTYPE_F16}
# Rows of logits that the backward materialises at a time (the reference uses
# 2048, cross_entropy.py:367; a 288 GB device holds far larger blocks).
BWD_ROWS = 16384
# Kept logits lie in tiles of this many tokens: a block of rows read from them
# starts on a tile (BWD_ROWS is rounded down to whole tiles there, to one at least).
_KEPT_ROWS = 256
# The forward of a call that will be differentiated keeps its fp32 logits (unless
# its caller says otherwise, keep_logits) where the rows have at least KEEP_DIM
# elements and all graphs that are alive hold at most KEEP_BYTES of them on the
# device, this call included: 8 bytes per logit go through memory
# once instead of 2 * dim operations.  Forward + backward, recomputed -> kept:
# dim 4096, 8192 tokens x 128256: 28.0 -> 22.8 ms; dim 1024, 4096 x 128256:
# 4.60 -> 4.27; dim 768, 4096 x 50257: 1.84 -> 1.75; dim 512, 8192 x 128256:
# 4.96 -> 5.25; dim 256, 8192 x 32000: 0.82 -> 0.97.
KEEP_BYTES = 8 << 30
KEEP_DIM = 1024
# The two gradient products sum over the vocabulary and over the tokens; the library
# is fastest where both operands are contiguous along the summed index.
# grad_w = dlogits^T x: a transposed x costs little, a second copy of the dlogits, written
# along with the first, 0.55 us per million.  Both from _TURN_ROWS rows and _TURN_DIM
# columns on (product before -> after, cost: 8192 x 4096 x 128256: 7.85 -> 5.55, 0.61 ms;
# 4096 x 2560 x 128256: 2.49 -> 1.90, 0.29; 1000 x 2560 x 50304: 302 -> 249, 29 us; forward
# and both gradients, 100 x 2048 x 32000: 171 -> 165, 205 x 2048 x 128256: 669 -> 623, 150 x
# 4096 x 50257: 528 -> 469, but 64 x 2048 x 32000: 148 -> 149), with
# fewer columns the copy costs what it saves (4096 x 1024 x 128256: 1.07 -> 0.82, 0.29 ms)
# and x alone is turned, from _TURN_X_ROWS rows on (1.07 -> 0.94; 1000 rows: 329 -> 332 us).
# grad_x = dlogits w: a transposed w costs the same whatever the number of rows: from
# _TURN_W_ROWS rows on, where the result has at least _TURN_W_TILES tiles of 256 x 256
# (8192 x 4096 x 128256: 6.25 -> 5.34, 0.40 ms; 8192 x 1024: 1.69 -> 1.39, 0.10;
# 4096 x 2560: 2.88 -> 2.02, 0.26, but 4096 x 1024: 1.25 -> 1.34 and 2048 x 4096:
# 1.62 -> 1.37, 0.40).
# Where the result has so few tiles of 256 x 256 that _SPLIT_ROUNDS times as many still
# fit the CUs, grad_x comes from a kernel of this library that divides the vocabulary
# (the library's product leaves the other CUs idle: 1000 x 2560 x 128256: 1083 -> 604 us,
# 300 x 1024 x 50257: 158 -> 57, 2000 x 2048 x 32000: 392 -> 242, 64 x 4096 x 128256:
# 472 -> 253; with 96 tiles, 2000 x 3072, 1381 -> 1407), and from 96 tiles on where the
# library's rounds of the chip are likely to be uneven (mi_xent_grad_x_uneven_splits).
_SPLIT_ROUNDS, _SPLIT_VOCAB = 3, 8192
_TURN_ROWS, _TURN_DIM = 96, 1536
_TURN_X_ROWS, _TURN_X_DIM = 2048, 1024
_TURN_W_ROWS, _TURN_W_TILES = 4096, 128
# From KEEP_UNASKED bytes in all on, the memory is asked first: kept logits and what the
# backward allocates for its products take at most a quarter of what is free (to the
# allocator or in its cache), so that what the program allocates next still fits.
KEEP_UNASKED = 256 << 20
# Kept logits that are alive: token -> (device, bytes).  An entry leaves when its
# tensor is freed, from whichever thread that happens in (one dict operation, no lock).
_kept_live = {}
_kept_lock = threading.Lock()
_saved_hooks = getattr(torch._C._autograd, "_top_saved_tensors_default_hooks", None)


def _tag(t):
    try:
        return _TAGS[t.dtype]
    except KeyError:
        raise TypeError("fused cross-entropy supports bfloat16 and float16 tensors, got %s" % t.dtype)


def _check_xw(x, w):
    """x [T, D] and w [N, D] of one dtype on one device: the kernels take w's type from x."""
    if x.ndim != 2 or w.ndim != 2:
        raise ValueError("x and w must be 2D tensors.")
    if x.shape[1] != w.shape[1]:
        raise ValueError("x has %d columns, w has %d" % (x.shape[1], w.shape[1]))
    if w.dtype != x.dtype:
        raise TypeError("x and w must share one dtype (got %s and %s)" % (x.dtype, w.dtype))
    if w.device != x.device:
        raise ValueError("x and w must be on one device (got %s and %s)" % (x.device, w.device))


def _pad_dim(t, mult=128):
    """Rows as the kernel wants them: unit inner stride, 16-byte aligned, row
    stride a multiple of 8 and the inner size a multiple of 128 (zero columns
    do not change x @ w^T)."""
    d = t.shape[1]
    if d % mult:
        t = torch.nn.functional.pad(t, (0, mult - d % mult))
    if t.stride(1) != 1 or t.stride(0) % 8 or t.data_ptr() % 16:
        t = t.contiguous()
    return t


def _labels(y, n):
    y = y.reshape(-1)
    if y.shape[0] != n:
        raise ValueError("Dimension mismatch: x.shape[0] (%d) != y.shape[0] (%d)" % (n, y.shape[0]))
    if y.dtype not in (torch.int32, torch.int64):
        y = y.to(torch.int64)
    return y.contiguous()


def cross_entropy_fused_fwd(x, w, y):
    """(loss, lse), both fp32 [T]: lse[t] = logsumexp_n(x[t] . w[n]),
    loss[t] = lse[t] - x[t] . w[y[t]] — forward of CrossEntropyFusedFunction
    (cross_entropy.py:276-352)."""
    return _fwd(x, w, y, False)[:2]


def _free_bytes(device):
    """Device memory that an allocation could get.  (The nested form of the
    allocator's figures: 6 us, the flat one takes 260.)"""
    stats = torch.cuda.memory_stats_as_nested_dict(device)
    reserved, used = (stats[k]["all"]["current"] if k in stats else 0 for k in ("reserved_bytes", "allocated_bytes"))
    return torch.cuda.mem_get_info(device)[0] + reserved - used


def _alloc_kept(x, w, always):
    """Room for the logits of x w^T, or None: where the automatic choice (not
    `always`) finds too many of them alive or too little memory free for them and
    what the backward allocates, and where the allocation fails."""
    T, N, device = x.shape[0], w.shape[0], x.device
    nbytes = _lib.load().mi_xent_kept_bytes(T, N)
    token = object()
    with _kept_lock:
        if not always:
            live = nbytes + sum(n for d, n in list(_kept_live.values()) if d == device)
            if live > KEEP_BYTES:
                return None
            # (a capture repeats what its program ran before it, and its pool is not in these figures)
            if live > KEEP_UNASKED and not torch.cuda.is_current_stream_capturing() \
                    and 4 * (nbytes + _bwd_bytes(x, w)) > _free_bytes(device):
                return None
        _kept_live[token] = (device, nbytes)
    try:
        kept = torch.empty(nbytes // 4, device=device, dtype=torch.float32)
    except BaseException as e:
        _kept_live.pop(token, None)
        if not isinstance(e, torch.OutOfMemoryError):
            raise
        return None
    weakref.finalize(kept, _kept_live.pop, token, None).atexit = False
    return kept


def _fwd(x, w, y, keep):
    """(loss, lse, kept): kept is the logits for _kept_dlogits, or None; `keep`:
    False never, True where there is memory for them, None within the budget."""
    _require_gpu(x, w, y)
    _check_xw(x, w)
    lib = _lib.load()
    T, N = x.shape[0], w.shape[0]
    y = _labels(y, T)
    xp, wp = _pad_dim(x), _pad_dim(w)
    lse = torch.empty((T,), device=x.device, dtype=torch.float32)
    loss = torch.empty((T,), device=x.device, dtype=torch.float32)
    a = _lib.XentArgs()
    a.struct_size = C.sizeof(a)
    a.dtype = _tag(x)
    a.tokens, a.dim, a.vocab = T, xp.shape[1], N
    a.labels_i64 = 1 if y.dtype == torch.int64 else 0
    a.x, a.w, a.y = _ptr(xp), _ptr(wp), _ptr(y)
    a.x_stride = xp.stride(0) if T > 1 else xp.shape[1]
    a.w_stride = wp.stride(0) if N > 1 else wp.shape[1]
    a.lse, a.loss = _ptr(lse), _ptr(loss)
    nbytes = lib.mi_xent_fwd_workspace_bytes(C.byref(a))
    ws = torch.empty(max(nbytes, 16), device=x.device, dtype=torch.uint8)
    a.workspace, a.workspace_bytes = _ptr(ws), nbytes
    kept = None
    if keep is not False and T and N:
        kept = _alloc_kept(x, w, bool(keep))
    if kept is None:
        _lib.check(lib.mi_xent_fwd(C.byref(a), _stream()))
    else:
        _lib.check(lib.mi_xent_fwd_keep(C.byref(a), _ptr(kept), _stream()))
    return loss, lse, kept


def cross_entropy_dlogits_(logits, lse, dloss, y):
    """In place: logits[t, n] <- dloss[t] (exp(logits[t, n] - lse[t]) - [n == y[t]])
    (cross_entropy_fused_bwd_kernel, cross_entropy.py:185-266)."""
    _require_gpu(logits, lse, dloss, y)
    lib = _lib.load()
    if logits.ndim != 2 or logits.stride(1) != 1:
        raise ValueError("logits must be 2-D with unit inner stride")
    a = _lib.XentGradArgs()
    a.struct_size = C.sizeof(a)
    a.dtype = _tag(logits)
    a.rows, a.vocab = logits.shape
    a.ld = logits.stride(0) if logits.shape[0] > 1 else logits.shape[1]
    a.labels_i64 = 1 if y.dtype == torch.int64 else 0
    a.logits, a.lse, a.dloss, a.y = _ptr(logits), _ptr(lse), _ptr(dloss), _ptr(y)
    _lib.check(lib.mi_xent_dlogits(C.byref(a), _stream()))
    return logits


def cross_entropy_dlogits(x, w, y, lse, dloss):
    """dlogits [T, N] in x's dtype: dloss[t] (exp(x[t] . w[n] - lse[t]) - [n == y[t]]),
    computed by the forward's GEMM kernel with the gradient epilogue on its fp32
    accumulators (replaces the logits GEMM + element-wise kernel of
    cross_entropy.py:374, :185-266, which round the logits to x's dtype first)."""
    _require_gpu(x, w, y, lse, dloss)
    _check_xw(x, w)
    return _dlogits(x, w, y, lse, dloss, torch.empty((x.shape[0], w.shape[0]), device=x.device, dtype=x.dtype))


def _dlogits(x, w, y, lse, dloss, dl):
    lib = _lib.load()
    T, N = x.shape[0], w.shape[0]
    xp, wp = _pad_dim(x), _pad_dim(w)
    a = _lib.XentBwdArgs()
    a.struct_size = C.sizeof(a)
    a.dtype = _tag(x)
    a.tokens, a.dim, a.vocab = T, xp.shape[1], N
    a.labels_i64 = 1 if y.dtype == torch.int64 else 0
    a.x, a.w, a.y = _ptr(xp), _ptr(wp), _ptr(y)
    a.x_stride = xp.stride(0) if T > 1 else xp.shape[1]
    a.w_stride = wp.stride(0) if N > 1 else wp.shape[1]
    a.lse, a.dloss = _ptr(lse), _ptr(dloss)
    a.dlogits, a.ld = _ptr(dl), dl.stride(0) if T > 1 else N
    _lib.check(lib.mi_xent_bwd_dlogits(C.byref(a), _stream()))
    return dl


def _dlogits_rows(rows, N, like):
    """Room for dlogits [rows, N] as the two gradient products read them best:
    rows start on 16-byte boundaries, which an odd vocabulary's own pitch does
    not give, neither to the 16-byte stores of the kernels that write them nor
    to the library's loads.  Forward + backward, 8192 tokens x 2048 x 50257:
    5.31 -> 4.81 ms with padded rows, 1000 x 1024 x 50257: 0.75 -> 0.69."""
    ld = N if N % 8 == 0 else -(-N // 64) * 64
    return torch.empty((rows, ld), device=like.device, dtype=like.dtype)[:, :N]


def _kept_dlogits(kept, first, y, lse, dloss, N, dl, dl_t=None):
    """dl [rows, N] <- dlogits of the rows from `first` on (a multiple of _KEPT_ROWS),
    from the logits that _fwd kept; the values of cross_entropy_dlogits.  dl_t [N, ld]
    receives their transpose as well, its columns behind `rows` zeros."""
    if first % _KEPT_ROWS:
        raise ValueError("rows of kept logits start at a multiple of %d, not at %d" % (_KEPT_ROWS, first))
    lib = _lib.load()
    a = _lib.XentBwdArgs()
    a.struct_size = C.sizeof(a)
    a.dtype = _tag(dl)
    a.tokens, a.vocab = dl.shape[0], N
    a.labels_i64 = 1 if y.dtype == torch.int64 else 0
    a.y, a.lse, a.dloss = _ptr(y), _ptr(lse), _ptr(dloss)
    a.dlogits, a.ld = _ptr(dl), dl.stride(0) if dl.shape[0] > 1 else N
    at = C.c_void_p(kept.data_ptr() + lib.mi_xent_kept_bytes(first, N))
    if dl_t is None:
        _lib.check(lib.mi_xent_kept_dlogits(C.byref(a), at, _stream()))
    else:
        _lib.check(lib.mi_xent_kept_dlogits_both(C.byref(a), at, _ptr(dl_t), dl_t.shape[1], _stream()))
    return dl


def _can_turn(t):
    """Whether mi_transpose16 takes t (2-D)."""
    return (t.element_size() == 2 and t.stride(1) == 1 and t.shape[1] % 8 == 0 and t.stride(0) % 8 == 0 and t.stride(0) >= t.shape[1]
            and t.data_ptr() % 16 == 0)


def _room_turned(t):
    """Room for the transpose of t [r, c]: [c rounded up to 8, r rounded up to 64]."""
    return torch.empty((-(-t.shape[1] // 8) * 8, -(-t.shape[0] // 64) * 64), device=t.device, dtype=t.dtype)


def _turn(t, out):
    """out <- the transpose of t, its columns behind t's rows zeros."""
    rows, cols = t.shape
    _lib.check(_lib.load().mi_transpose16(_ptr(t), rows, cols, t.stride(0) if rows > 1 else max(cols, t.stride(0)),
                                          _ptr(out), out.shape[1], _stream()))
    return out


def _turns_x(rows, x):
    """(x, dlogits): which operands of grad_w a block of `rows` rows takes the other way round."""
    if not _can_turn(x):
        return False, False
    both = rows >= _TURN_ROWS and x.shape[1] >= _TURN_DIM
    return both or (rows >= _TURN_X_ROWS and x.shape[1] >= _TURN_X_DIM), both


def _turns_w(rows, x, w):
    """Whether grad_x of a block of `rows` rows sums over a contiguous vocabulary."""
    return (rows >= _TURN_W_ROWS and -(-rows // 256) * -(-w.shape[1] // 256) >= _TURN_W_TILES
            and w.shape[1] >= _TURN_X_DIM and _can_turn(w) and not _splits(rows, x, w))


def _splits(rows, x, w):
    """_splits_vocab, for a grad_x with the strides that it takes from x: the kernel writes whole rows."""
    if not (x.is_contiguous() or torch.empty_like(x, device="meta").is_contiguous()):
        return 0
    return _splits_vocab(rows, w)


def _splits_vocab(rows, w):
    """The ranges of the vocabulary that grad_x of a block of `rows` rows is divided into; 0: it is not."""
    N, D = w.shape
    if N < _SPLIT_VOCAB or not _can_turn(w) or w.stride(0) > 1 << 22 or N > (1 << 22) - 64:
        return 0
    lib = _lib.load()
    cus = _num_cus(lib)
    if -(-rows // 256) * -(-D // 256) * _SPLIT_ROUNDS > cus:
        return lib.mi_xent_grad_x_uneven_splits(rows, D, N, cus)
    return lib.mi_xent_grad_x_splits(rows, D, N, cus)


def _grad_x(dl, w, out, n_split):
    """out <- dl @ w, the vocabulary in n_split ranges; False without memory for their partial sums."""
    lib = _lib.load()
    a = _lib.XentGradXArgs()
    a.struct_size = C.sizeof(a)
    a.dtype = _tag(dl)
    a.tokens, a.dim, a.vocab, a.n_split = out.shape[0], out.shape[1], w.shape[0], n_split
    a.dlogits, a.w, a.grad_x = _ptr(dl), _ptr(w), _ptr(out)
    a.ld, a.w_stride, a.grad_x_stride = dl.stride(0), w.stride(0), out.shape[1]
    a.workspace_bytes = lib.mi_xent_grad_x_workspace_bytes(a.tokens, a.dim, n_split)
    try:
        ws = torch.empty(a.workspace_bytes, device=dl.device, dtype=torch.uint8)
    except torch.OutOfMemoryError:
        return False
    a.workspace = _ptr(ws)
    _lib.check(lib.mi_xent_grad_x(C.byref(a), _stream()))
    return True


def _copy_bytes(rows, x, w):
    """What the operands that blocks of `rows` rows take the other way round occupy."""
    turn_x, turn_dl = _turns_x(rows, x)
    n = rows * (turn_x * x.shape[1] + turn_dl * w.shape[0]) + _turns_w(rows, x, w) * w.numel()
    return n * x.element_size()


def _makes_copies(rows, x, w, kept):
    """Whether blocks of `rows` rows may take operands the other way round where the rules above say so:
    from KEEP_UNASKED bytes on, the copies take at most a quarter of the free memory.  (With
    kept logits that is not asked again, 25 us on a busy device: the forward has asked for the
    copies along with them, unless its caller wanted them kept whatever is free.)"""
    if kept is not None:
        return True
    n = _copy_bytes(rows, x, w)
    if n <= KEEP_UNASKED or torch.cuda.is_current_stream_capturing():   # (as in _alloc_kept)
        return n > 0
    return 4 * n <= _free_bytes(x.device)


def _bwd_bytes(x, w):
    """What the backward allocates for its dlogits and products at a time."""
    rows = min(x.shape[0], BWD_ROWS)
    n_split = _splits(rows, x, w)
    split = _lib.load().mi_xent_grad_x_workspace_bytes(rows, w.shape[1], n_split) if n_split else 0
    return rows * w.shape[0] * x.element_size() + _copy_bytes(rows, x, w) + split


def cross_entropy_fused_bwd(grad_o, x, w, y, lse, rows_per_block=None):
    """(grad_x, grad_w) in the dtypes of x and w — backward of
    CrossEntropyFusedFunction (cross_entropy.py:355-420): per block of rows,
    dlogits from the fused GEMM kernel, then the two gradient GEMMs."""
    return _bwd(grad_o, x, w, y, lse, None, rows_per_block or BWD_ROWS)


def _bwd(grad_o, x, w, y, lse, kept, step):
    _require_gpu(grad_o, x, w, y, lse)
    _check_xw(x, w)
    T = x.shape[0]
    y = _labels(y, T)
    g = grad_o.reshape(-1).to(torch.float32).contiguous()
    lse = lse.contiguous()
    if kept is not None and step % _KEPT_ROWS:
        step = max(step - step % _KEPT_ROWS, _KEPT_ROWS)
    if _makes_copies(min(T, step), x, w, kept):
        try:
            return _gradients(x, w, y, lse, g, kept, step, True)
        except torch.OutOfMemoryError:
            pass   # (whichever allocation it was, the copies are gone with the frames that held them)
    return _gradients(x, w, y, lse, g, kept, step, False)


def _gradients(x, w, y, lse, g, kept, step, copies):
    """_bwd in blocks of `step` rows; `copies`: with operands the other way round where _turns_x and
    _turns_w say so."""
    grad_x = torch.empty_like(x)
    grad_w = w_t = None
    if copies and _turns_w(min(x.shape[0], step), x, w):
        w_t = _turn(w, _room_turned(w))[:, :w.shape[0]].t()
    for s in range(0, x.shape[0], step):
        r = slice(s, min(s + step, x.shape[0]))
        grad_w = _block_gradients(x[r], w, w_t, y[r], lse[r], g[r], kept, s, copies, grad_x[r], grad_w)
    if grad_w is None:
        grad_w = torch.zeros_like(w)
    return grad_x, grad_w


def _block_gradients(x, w, w_t, y, lse, g, kept, first, copies, grad_x, grad_w):
    """grad_x of a block of rows, the first of which is row `first`, and grad_w with the block's part
    added.  (A function of its own: its dlogits and copies are freed before the next block's are made.)"""
    rows, N = x.shape[0], w.shape[0]
    dl = _dlogits_rows(rows, N, x)
    turn_x, turn_dl = _turns_x(rows, x) if copies else (False, False)
    x_t = _room_turned(x) if turn_x else None
    dl_t = _room_turned(dl) if turn_dl else None
    if kept is None:
        _dlogits(x, w, y, lse, g, dl)
        if dl_t is not None:  # (rows of dlogits are padded to whole pieces of 8, see _dlogits_rows)
            _turn(dl.as_strided((rows, dl_t.shape[0]), dl.stride()), dl_t)
    elif dl_t is None:
        _kept_dlogits(kept, first, y, lse, g, N, dl)
    else:
        _kept_dlogits(kept, first, y, lse, g, N, dl, dl_t)
    n_split = _splits_vocab(rows, w) if grad_x.is_contiguous() else 0
    if not (n_split and _grad_x(dl, w, grad_x, n_split)):
        torch.mm(dl, w if w_t is None else w_t, out=grad_x)
    d, v = dl.t(), x
    if x_t is not None:
        v = _turn(x, x_t).t()
        if dl_t is None:
            v = v[:rows]
        else:  # (the columns behind the rows are zeros in both)
            d = dl_t[:N]
    return torch.mm(d, v) if grad_w is None else grad_w.addmm_(d, v)


def _saved_hooks_set():
    """Whether hooks on saved tensors (activation checkpointing, offloading to the host),
    which would copy or drop kept logits, are or may be in force."""
    if _saved_hooks is None:
        return True
    for args in ((False,), ()):  # torch has had the getter with and without its argument
        try:
            return _saved_hooks(*args) is not None
        except TypeError:
            pass
    return True


def _keeps_logits(x, w):
    """Whether the forward may keep its logits for the backward (see KEEP_BYTES)."""
    if not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad)):
        return False
    if x.ndim != 2 or w.ndim != 2 or x.shape[1] < KEEP_DIM:
        return False
    if _saved_hooks_set():
        return False
    return _lib.load().mi_xent_kept_bytes(x.shape[0], w.shape[0]) <= KEEP_BYTES


class CrossEntropyFusedFunction(torch.autograd.Function):
    """Drop-in for the reference's autograd Function (cross_entropy.py:270-420).
    `keep_logits`: the backward reads the forward's logits instead of computing
    them again; the results are the same.  True: wherever there is memory for them;
    None: within KEEP_BYTES."""

    @staticmethod
    def forward(ctx, x, w, y, keep_logits=False):
        if y.ndim != 1 and y.shape[-1] != 1:
            raise ValueError("y must be a 1D tensor.")
        loss, lse, kept = _fwd(x, w, y, keep_logits)
        ctx.save_for_backward(x, w, y, lse, *(() if kept is None else (kept,)))
        return loss

    @staticmethod
    def backward(ctx, grad_o):
        x, w, y, lse, *kept = ctx.saved_tensors
        grad_x, grad_w = _bwd(grad_o, x, w, y, lse, kept[0] if kept else None, BWD_ROWS)
        return grad_x, grad_w, None, None


def cross_entropy_fused_triton(x, w, y, *, keep_logits=None):
    """loss [T] fp32 of softmax cross-entropy over x @ w^T (cross_entropy.py:423-425).

    `keep_logits`: whether the fp32 logits (4 bytes each) stay in memory from the
    forward to the backward, which then does not compute them again; loss and
    gradients are the same bits either way (but for the order of the gradients' fp32
    sums where memory is so short that one of the two backwards goes without its
    copies, see below).  None: where that is the faster way and KEEP_BYTES and the
    free memory allow it.  False: never.  True: always where the allocation succeeds.

    The backward holds BWD_ROWS rows of dlogits at a time and, where its products are
    faster for it and a quarter of the free memory is enough, transposed copies of
    these and of its x and w (which keep_logits=True asks for whatever is free); if an
    allocation fails with them it goes without."""
    if keep_logits is None:
        keep_logits = None if _keeps_logits(x, w) else False
    return CrossEntropyFusedFunction.apply(x, w, y, keep_logits)
