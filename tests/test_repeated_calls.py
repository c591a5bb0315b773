"""Calls whose geometry the thread has had before go straight to the library: they see the tensors they are given, and whatever
the geometry does not decide is looked at again."""
import numpy as np
import pytest
import torch

from flash_colsum import _hip, flash_colsum, flash_colsum_ext, flash_colsum_f32
from oracle import colsum_exact


def test_only_plain_arguments_are_recognised():
    q = torch.zeros(1, 2, 8, 64, dtype=torch.float16)
    assert _hip.call_key(0, q, q, None, False, None) is not None and _hip.call_key(0, q, q, 0.5, True, 3) is not None
    for args in [(0, torch.nn.Parameter(q), q, None, False, None), (0, q, q, torch.tensor(0.5), False, None), (0, q, q, np.float32(0.5), False, None),
                 (0, q, q, None, 1, None), (0, q, q, None, False, torch.tensor(3)), (0, None, q, None, False, None), (0, q, q, None, False, 1.5)]:
        assert _hip.call_key(*args) is None
    # kinds, dtypes and storage orders are told apart
    t = torch.zeros(1, 8, 2, 64, dtype=torch.float16).transpose(1, 2)
    keys = [_hip.call_key(kind, a, b, None, False, None) for kind in (0, 1, 2) for a, b in ((q, q), (t, q), (q.bfloat16(), q), (q, t))]
    assert len(set(keys)) == len(keys)
    assert _hip.repeated_call(keys[0], q, q) is None  # nothing known, and not on a GPU
    with pytest.raises(ValueError, match="only supports CUDA tensors"):
        flash_colsum(q, q)


@pytest.mark.filterwarnings("ignore")  # nested and compressed tensors warn that they are prototypes
def test_tensors_without_sizes_or_strides_are_refused_as_others_are():
    nested = torch.nested.nested_tensor([torch.zeros(2, 3, 8), torch.zeros(2, 5, 8)])
    compressed = torch.zeros(2, 3, 8, 8).to_sparse_csr()
    for t in (nested, compressed):
        assert t.ndim == 4 and _hip.call_key(0, t, t, None, False, None) is None
        for fn in (flash_colsum, flash_colsum_f32, flash_colsum_ext):
            with pytest.raises(ValueError, match="only supports CUDA tensors"):
                fn(t, t)


def _pair(seed, shape=(2, 4, 100, 64), dtype=torch.float16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return tuple(torch.randn(shape, generator=g, device="cuda").to(dtype) for _ in range(2))


def _good(out, q, k, **kw):
    ref = colsum_exact(q, k, **kw)
    rel = 1e-3 if out.dtype == torch.float32 else 2e-3  # one rounding to fp16 on top
    assert out.shape == ref.shape and ((out.double() - ref).abs() <= rel * ref.abs() + 1e-7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_repeated_calls_see_their_own_tensors(dtype):
    for seed in range(4):
        q, k = _pair(seed, dtype=dtype)
        _good(flash_colsum(q, k), q, k)
        _good(flash_colsum_f32(q, k, 0.3), q, k, scale=0.3)
        _good(flash_colsum(q, k, cls_len=2), q, k, cls_len=2)
        _good(flash_colsum_ext(q, k, out_dtype=torch.float32), q, k)
        assert flash_colsum_ext(q, k).dtype == torch.float16
        a, b = flash_colsum(q, k), flash_colsum(k, q)  # results of their own
        assert a.data_ptr() != b.data_ptr()
        _good(a, q, k)


@pytest.mark.gpu
def test_what_the_geometry_does_not_decide():
    shape = (2, 4, 100, 64)
    q, k = _pair(0, shape)
    for _ in range(2):
        flash_colsum(q, k)
    # a base that is not 16-byte aligned
    odd = torch.empty(q.numel() + 8, dtype=torch.float16, device="cuda")[1:1 + q.numel()].view(shape)
    odd.copy_(q)
    assert odd.stride() == q.stride() and odd.data_ptr() % 16 != 0
    _good(flash_colsum(odd, k), q, k)
    # the other operand elsewhere
    with pytest.raises(ValueError):
        flash_colsum(q, k.cpu())
    with pytest.raises(ValueError):
        flash_colsum(q.cpu(), k)
    # another stream
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        out = flash_colsum(q, k)
    s.synchronize()
    _good(out, q, k)
    # fp32: out of fp16's range after a call that was not, not finite, and in range again
    q32, k32 = _pair(1, shape, torch.float32)
    for _ in range(2):
        _good(flash_colsum(q32, k32), q32, k32)
    big = q32.clone()
    big[0, 1, 7] *= 1e6
    _good(flash_colsum_f32(big, k32, 1e-5), big, k32, scale=1e-5)
    _good(flash_colsum_f32(q32, k32, 1e-5), q32, k32, scale=1e-5)
    _good(flash_colsum_f32(big, k32, 1e-5), big, k32, scale=1e-5)
    big[0, 0, 0, 0] = float("nan")
    with pytest.raises(ValueError, match="NaN"):
        flash_colsum_f32(big, k32, 1e-5)
    neg = torch._neg_view(q32)
    _good(flash_colsum(neg, k32), -q32, k32)


@pytest.mark.gpu
def test_repeated_call_in_a_graph():
    q, k = _pair(2)
    for _ in range(3):
        eager = flash_colsum(q, k)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = flash_colsum(q, k)
    for i in range(4):
        q.copy_(q.flip(2))
        g.replay()
        assert torch.equal(out, flash_colsum(q, k))
    assert eager.shape == out.shape


class _Counted:
    """The library, with a count of its calls."""

    def __init__(self, lib):
        self.lib, self.n = lib, {}

    def __getattr__(self, name):
        fn = getattr(self.lib, name)

        def call(*args):
            self.n[name] = self.n.get(name, 0) + 1
            return fn(*args)

        return call


@pytest.mark.gpu
@pytest.mark.parametrize("fn", [flash_colsum, flash_colsum_f32])
def test_operands_beyond_fp16_are_computed_once_more_only(fn, monkeypatch):
    """fp32 operands that leave fp16's range: one rounding, one discarded computation and that of the split operands, also on
    repeated calls; a geometry is remembered by calls that stayed inside the range."""
    q, k = _pair(3, (2, 3, 90, 64), torch.float32)
    big = q.clone()
    big[1, 2, 5] *= 1e6
    counted = _Counted(_hip.lib())
    monkeypatch.setattr(_hip, "_lib", counted)
    monkeypatch.setattr(_hip._tls, "known", {}, raising=False)

    def calls(a):
        counted.n.clear()
        _good(fn(a, k, 1e-5), a, k, scale=1e-5)
        return counted.n.get("fcs_round_f16", 0), counted.n["fcs_colsum_call"]

    for a, n, known in [(big, (1, 2), 0), (big, (1, 2), 0), (q, (1, 1), 1), (q, (1, 1), 1), (big, (1, 2), 0), (big, (1, 2), 0), (q, (1, 1), 1)]:
        assert calls(a) == n and len(_hip._tls.known) == known


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(2, 4, 100, 64), (2, 4, 100, 36)])  # (36 channels are padded, by a copy)
def test_pending_negations(shape, dtype):
    """A view whose negation torch has put off, as the first call of a geometry and as a repeated one."""
    q, k = _pair(4, shape, dtype)
    for _ in range(2):
        for a, b in ((torch._neg_view(q), k), (q, torch._neg_view(k)), (torch._neg_view(q), torch._neg_view(k))):
            assert a.is_neg() or b.is_neg()
            _good(flash_colsum(a, b), a.resolve_neg(), b.resolve_neg())
            t = a.transpose(1, 2).contiguous().transpose(1, 2) if not a.is_neg() else torch._neg_view(q.transpose(1, 2).contiguous()).transpose(1, 2)
            _good(flash_colsum(t, b), t.resolve_neg(), b.resolve_neg())
        _good(flash_colsum(q, k), q, k)
