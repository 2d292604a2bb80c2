"""The native host calls (csrc/host_calls.cpp) against the general way behind them:
the same bits over the forms they take, and only those; everything else goes the
general way, with its results and its errors."""
import pytest
import torch

from tritonops_amd import _lib, masks, ops, rms

pytestmark = pytest.mark.gpu


class _Counting:
    """Stands in for the native module: counts the calls it answered."""

    def __init__(self, module, answer=True):
        self._module, self._answer, self.taken = module, answer, 0

    def __getattr__(self, name):
        def call(*args):
            out = getattr(self._module, name)(*args) if self._answer else None
            self.taken += out is not None
            return out
        return call


def _both(monkeypatch, call, native=True):
    """call() with and without the native calls: the same bits, and taken or not as `native` says."""
    real = _lib.native()
    got = []
    for answer in (True, False):
        stub = _Counting(real, answer)
        monkeypatch.setattr(_lib, "_native", stub)
        out = call()
        got.append(out if isinstance(out, (tuple, list)) else (out,))
        assert (stub.taken > 0) == (answer and native)
    monkeypatch.setattr(_lib, "_native", real)
    for a, b in zip(*got):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype
            assert torch.equal(a, b)


def _randn(*shape, dtype=torch.bfloat16, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return torch.randn(shape, device="cuda", generator=g).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("form", ["rows", "one", "three", "strided", "transposed", "empty", "mixed", "shifted"])
def test_rmsnorm(monkeypatch, dtype, form):
    x = {"rows": lambda: _randn(33, 255, dtype=dtype), "one": lambda: _randn(128, dtype=dtype),
         "three": lambda: _randn(2, 5, 1024, dtype=dtype), "strided": lambda: _randn(9, 64, dtype=dtype)[:, :48],
         "transposed": lambda: _randn(64, 9, dtype=dtype).t(), "empty": lambda: _randn(0, 64, dtype=dtype),
         "mixed": lambda: _randn(7, 96, dtype=dtype), "shifted": lambda: _randn(8 * 64 + 1, dtype=dtype)[1:].view(8, 64)}[form]()
    w = _randn(x.shape[-1], dtype=torch.float32 if form == "mixed" else dtype, seed=1)
    dy = _randn(*x.shape, dtype=dtype, seed=2)
    native = form in ("rows", "one", "three", "mixed", "shifted")
    _both(monkeypatch, lambda: rms.rmsnorm_fwd(x, w, 1e-5), native)
    _, rs = rms.rmsnorm_fwd(x, w, 1e-5)
    _both(monkeypatch, lambda: rms.rmsnorm_bwd(dy, x, w, rs, 1e-5), native)
    if native and x.dim() > 1:
        _both(monkeypatch, lambda: rms.rmsnorm_bwd(dy.transpose(0, 1).contiguous().transpose(0, 1), x, w, rs, 1e-5), False)


@pytest.mark.parametrize("D,native", [(64, True), (96, True), (128, True), (80, True)])
@pytest.mark.parametrize("causal", [True, False])
def test_dense_forward_and_backward(monkeypatch, D, native, causal):
    import tritonops_amd as ta

    cu = torch.tensor([0, 70, 70, 333, 500], device="cuda", dtype=torch.int32)
    q, k, v = _randn(1, 512, 4, D), _randn(1, 512, 2, D, seed=1), _randn(1, 512, 2, D, seed=2)
    wide = _randn(1, 512, 8, D, seed=3)[:, :, ::2]              # heads apart from each other
    for lse in (True, False):                                   # (padded head_dims: the general way pads, then calls again)
        _both(monkeypatch, lambda: ta.flash_attention(q, k, v, cu, causal=causal, return_lse=lse), native)
        _both(monkeypatch, lambda: ta.flash_attention(wide, k, v, cu, causal=causal, return_lse=lse, max_seq_len=100), native)
        b = [t.view(4, 128, -1, D).transpose(1, 2) for t in (q, k, v)]
        _both(monkeypatch, lambda: ta.flash_attention(*b, causal=causal, return_lse=lse), native)
        _both(monkeypatch, lambda: ta.flash_attention(*(t.contiguous() for t in b), causal=causal, return_lse=lse), native)
    _both(monkeypatch, lambda: ta.flash_attention(q, k, v, cu.long(), causal=causal), False)

    def train(layout):
        ts = [t.detach().requires_grad_(True) for t in ((q, k, v) if layout == "packed" else b)]
        o = ta.flash_attention(*ts, cu if layout == "packed" else None, causal=causal)
        return (o.detach(),) + torch.autograd.grad(o, ts, torch.ones_like(o) * 0.5)
    _both(monkeypatch, lambda: train("packed"), native)
    _both(monkeypatch, lambda: train("batched"), native)


def test_sparse_prefill(monkeypatch):
    import tritonops_amd as ta

    cu = torch.tensor([0, 300, 1000], device="cuda", dtype=torch.int32)
    q, k, v = _randn(1, 1000, 4, 64), _randn(1, 1000, 2, 64, seed=1), _randn(1, 1000, 2, 64, seed=2)
    for local, sink in ((128, 64), (1, 0), (0, 64), (4096, 0)):
        _both(monkeypatch, lambda: ta.flash_attn_sparse_triton(q, k, v, cu, None, local, sink))
        _both(monkeypatch, lambda: ta.flash_attn_sparse_triton(q, k, v, cu, 0.3, local, sink, max_seq_len=650))
    b = [t.view(2, 500, -1, 64).transpose(1, 2) for t in (q, k, v)]
    mask = torch.tril(torch.rand((2, 4, 8, 8)) < 0.5) | torch.eye(8, dtype=torch.bool)
    _both(monkeypatch, lambda: ta.flash_attn_sparse_triton(*b, None, block_mask=mask))
    rp, ci, st = masks.block_mask_to_csr(mask, "cuda")
    _both(monkeypatch, lambda: ta.flash_attn_sparse_triton(*b, None, row_ptr=rp, col_idx=ci, csr_strides=st))
    _both(monkeypatch, lambda: ta.flash_attn_sparse_triton(q.transpose(1, 2).contiguous().transpose(1, 2), k, v, cu, None, 128, 64), False)


@pytest.mark.parametrize("hq,hkv,D", [(8, 2, 64), (4, 4, 96), (80, 2, 128), (8, 8, 40)])
def test_decoding(monkeypatch, hq, hkv, D):
    import tritonops_amd as ta

    lens = torch.tensor([0, 1, 64, 333, 1000], device="cuda", dtype=torch.int32)
    cu = torch.cat([lens.new_zeros(1), lens.cumsum(0).to(torch.int32)])
    q, k, v = _randn(5, hq, D), _randn(5, 1024, hkv, D, seed=1), _randn(5, 1024, hkv, D, seed=2)
    pool = [t.view(80, 64, hkv, D) for t in (k, v)]
    table = torch.randperm(80, device="cuda").to(torch.int32).view(5, 16)
    packed = [t.view(1, 5120, hkv, D) for t in (k, v)]
    idx = torch.arange(15, device="cuda", dtype=torch.int32).expand(5, hkv, 15).contiguous()
    cnt = torch.tensor([[0, 1, 1, 6, 15]], device="cuda", dtype=torch.int32).t().expand(5, hkv).contiguous()
    for lse in (True, False):
        _both(monkeypatch, lambda: ta.flash_attention_decoding(q, k, v, cu, return_lse=lse))
        _both(monkeypatch, lambda: ta.flash_attention_decoding(q, k, v, None, 0.2, seq_lens=lens, max_seq_len=1000, split_tokens=192,
                                                               return_lse=lse))
        _both(monkeypatch, lambda: ta.flash_attention_decoding(q, k.transpose(1, 2).contiguous().transpose(1, 2), v, cu, return_lse=lse))
        if D != 40:   # (a pool of padded pages is another pool)
            _both(monkeypatch, lambda: ta.flash_attention_decoding(q, *pool, cu, kv_layout="paged", page_table=table, return_lse=lse))
            _both(monkeypatch, lambda: ta.flash_attention_decoding(q, *pool, cu, kv_layout="paged", page_table=table.long()), False)
        _both(monkeypatch, lambda: ta.flash_attention_decoding(q, *packed, cu, kv_layout="packed", return_lse=lse))
        _both(monkeypatch, lambda: ta.flash_attention_sparse_decoding(q, k, v, cu, 64, 200, return_lse=lse))
        _both(monkeypatch, lambda: ta.flash_attention_sparse_decoding(q, k, v, cu, block_indices=idx, block_counts=cnt, return_lse=lse))
        _both(monkeypatch, lambda: ta.flash_attention_sparse_decoding(q, k, v, None, seq_lens=lens, block_indices=idx,
                                                                      block_counts=cnt, include_last_block=False, split_blocks=2))
    if D != 40:
        _both(monkeypatch, lambda: ta.flash_attention_decoding(q, k, v, cu.long()), False)
    # lengths of another type or with gaps between them: worked out on the device first, as they were
    for c in (cu.long(), cu.float(), cu.repeat_interleave(2)[::2]):
        want = ta.flash_attention_sparse_decoding(q, k, v, cu, block_indices=idx, block_counts=cnt)
        assert torch.equal(ta.flash_attention_sparse_decoding(q, k, v, c, block_indices=idx, block_counts=cnt), want)


def test_errors_are_those_of_the_general_way():
    import tritonops_amd as ta

    q, k = _randn(1, 64, 4, 64), _randn(1, 64, 3, 64)
    cu = torch.tensor([0, 64], device="cuda", dtype=torch.int32)
    with pytest.raises(ValueError, match="multiple of heads_kv"):
        ta.flash_attention(q, k, k, cu)
    with pytest.raises(RuntimeError, match="runs on the GPU only"):
        ta.flash_attention(q, q.cpu(), q, cu)
    with pytest.raises(TypeError, match="bfloat16 or float16"):
        ta.flash_attention(q.float(), q.float(), q.float(), cu)
    with pytest.raises(_lib.MiAttnError, match="MI_ERR_ALIGNMENT"):
        flat = _randn(64 * 4 * 64 + 1)[1:].view(1, 64, 4, 64)
        ta.flash_attention(flat, flat, flat, cu)
    with pytest.raises(_lib.MiAttnError, match="MI_ERR_SCALE"):
        ta.flash_attention(q, q, q, cu, softmax_scale=-1.0)
    with pytest.raises(ValueError, match="Expected weight dim"):
        ta.rmsnorm_fwd(q, _randn(32), 1e-6)
    d = _randn(2, 4, 64)
    with pytest.raises(ValueError, match="share one dtype"):
        ta.flash_attention_decoding(d, _randn(2, 64, 4, 64).half(), _randn(2, 64, 4, 64).half(), torch.zeros(3, device="cuda", dtype=torch.int32))
    with pytest.raises(ValueError, match="integer tensor of 3 entries"):
        ta.flash_attention_decoding(d, _randn(2, 64, 4, 64), _randn(2, 64, 4, 64), cu)


def test_wrapped_tensors_and_modes_take_the_general_way(monkeypatch):
    from torch.utils._python_dispatch import TorchDispatchMode

    x, w = _randn(8, 64), _randn(64, seed=1)

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    def inside():
        with Mode():
            return rms.rmsnorm_fwd(x, w, 1e-6)
    _both(monkeypatch, inside, False)
    stub = _Counting(_lib.native())
    monkeypatch.setattr(_lib, "_native", stub)
    rms.rmsnorm_fwd(x.as_subclass(Sub), w, 1e-6)
    assert stub.taken == 0
