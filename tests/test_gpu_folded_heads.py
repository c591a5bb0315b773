"""Grouped key heads whose rows are laid end to end, in calls large enough that the plan does so (every call here asserts
it): heads that end inside a 32-row fragment, a wave or a row block, each storage order of Q, the pre-scaled operand,
rows beyond the unstabilised range, and the exact size of the workspace."""
import ctypes
import re

import pytest
import torch

pytestmark = pytest.mark.gpu


def _plan(q, k, kw):
    from flash_colsum import _hip

    kw = dict(kw)
    t = _hip.plan_description(tuple(q.shape), tuple(k.shape), causal=kw.get("is_causal", False), cls_n=kw.get("cls_len"), k_past=kw.get("k_past"),
                              scale=kw.get("scale"), bf16=q.dtype == torch.bfloat16)
    m = re.search(r"rowstream_kernel<\d+,\d+,\d+,\w+,(\w+)(,true)?>", t)
    return m[1] == "true", m[2] is not None  # pre-scaled, folded


def _check(q, k, kw, prescaled=False, folded=True):
    from flash_colsum import flash_colsum_ext
    from oracle import colsum_ext_exact

    print("folded heads", tuple(q.shape), q.stride(), tuple(k.shape), q.dtype, kw, flush=True)
    assert _plan(q, k, kw) == (prescaled, folded)
    out = flash_colsum_ext(q, k, out_dtype=torch.float32, **kw).double()
    # the oracle takes one batch entry at a time: float64 scores of all of them would not be small
    ref = torch.cat([colsum_ext_exact(q[b:b + 1], k[b:b + 1], **kw) for b in range(q.shape[0])]).double()
    # the bar of every kernel of this package, and 2^-126 for probabilities that fp32 flushes to zero
    err = (out - ref).abs()
    assert torch.isfinite(out).all()
    assert (err <= 1e-4).all() and (err <= 1e-3 * ref.abs() + 2.0 ** -126).all(), err.max()


def _strided(shape, layout, gen, dtype):
    b, h, s, d = shape
    full = {"tokens": (b, s, h, d), "padded rows": (b, h, s, d + 8), "sliced heads": (b, 2 * h, s, d)}[layout]
    x = torch.randn(full, generator=gen, device="cuda").to(dtype)
    return {"tokens": lambda: x.transpose(1, 2), "padded rows": lambda: x[..., :d], "sliced heads": lambda: x[:, ::2]}[layout]()


@pytest.mark.parametrize("group,q_len", [(2, 1), (8, 1), (3, 31), (4, 33), (8, 16), (5, 64), (2, 64)])
@pytest.mark.parametrize("causal", [True, False])
def test_up_to_64_rows(group, q_len, causal):
    q_len = q_len if causal else max(q_len, 5)  # fewer rows of a non-causal call have a kernel of their own
    gen = torch.Generator(device="cuda").manual_seed(group * 1000 + q_len)
    for dtype, d, hk in [(torch.bfloat16, 128, 2), (torch.float16, 64, 3), (torch.float16, 40, 2), (torch.bfloat16, 192, 2)]:
        s_k = 2051
        b = -(-257 // (hk * group * 9))
        q, k = (torch.randn((b, h, s, d), generator=gen, device="cuda").to(dtype) for h, s in ((hk * group, q_len), (hk, s_k)))
        _check(q, k, {"is_causal": causal})


@pytest.mark.parametrize("group,q_len", [(2, 65), (4, 100), (8, 127), (2, 128), (3, 96)])
@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 128), (torch.float16, 64), (torch.bfloat16, 256)])
def test_65_to_128_rows(group, q_len, dtype, d):
    gen = torch.Generator(device="cuda").manual_seed(group * 1000 + q_len + d)
    hk, s_k = 2, 4200
    b = -(-(512 if d > 128 else 2560) // (hk * group * 17))
    q, k = (torch.randn((b, h, s, d), generator=gen, device="cuda").to(dtype) for h, s in ((hk * group, q_len), (hk, s_k)))
    # (the pre-scaled operand needs 16384 averaged rows)
    for kw in [{"is_causal": True}, {"is_causal": False}]:
        _check(q, k, kw)


@pytest.mark.parametrize("group,q_len", [(2, 1), (16, 8), (4, 32), (17, 7), (2, 64)])
def test_one_unit_per_batch_entry(group, q_len):
    """All rows of a key head in one unit: means written by the column pass itself."""
    gen = torch.Generator(device="cuda").manual_seed(group + q_len)
    for d, s_k, b in [(64, 70, 1), (128, 300, 3), (256, 1000, 2)]:
        q, k = (torch.randn((b, h, s, d), generator=gen, device="cuda").half() for h, s in ((group, q_len), (1, s_k)))
        for kw in [{"is_causal": True}, {"is_causal": True, "k_past": 3}, {"is_causal": True, "scale": 4.0}]:
            _check(q, k, kw)


@pytest.mark.parametrize("layout", ["tokens", "padded rows", "sliced heads"])
def test_storage_orders(layout):
    gen = torch.Generator(device="cuda").manual_seed(4)
    for dtype, d, hk, group, q_len in [(torch.bfloat16, 128, 2, 4, 33), (torch.float16, 64, 2, 8, 16), (torch.float16, 200, 2, 3, 64)]:
        b = -(-257 // (hk * group * 9))
        for kw in [{"is_causal": True}, {"is_causal": False}, {"is_causal": True, "cls_len": 5, "k_past": 2060}]:
            _check(_strided((b, hk * group, q_len, d), layout, gen, dtype), _strided((b, hk, 2060, d), layout, gen, dtype), kw)


@pytest.mark.parametrize("kw", [{"k_past": 70}, {"k_past": 2013}, {"k_past": 2040, "cls_len": 21}, {"scale": -0.1}, {"scale": 4.0}])
def test_masks_and_stabilised_rows(kw):
    gen = torch.Generator(device="cuda").manual_seed(5)
    for group, q_len in [(4, 50), (3, 30), (8, 7)]:
        s_k = 2100
        seen = min(s_k, kw.get("k_past", s_k - q_len) + min(q_len, kw.get("cls_len", q_len)))
        b = -(-257 // (2 * group * -(-seen // 256)))
        q, k = (torch.randn((b, h, s, 64), generator=gen, device="cuda").half() for h, s in ((2 * group, q_len), (2, s_k)))
        _check(q, k, {"is_causal": True, **kw})


@pytest.mark.parametrize("q_len", [64, 100])
@pytest.mark.parametrize("kw", [{"is_causal": True}, {"is_causal": True, "k_past": 2513}, {"is_causal": False}, {"is_causal": True, "scale": -0.125}])
def test_pre_scaled_operand(q_len, kw):
    """fp16, 64-wide heads, 16384 rows or more: whole stages on Q * c rounded to fp16, the rest on the raw operand.  Then a row
    whose scores leave the range of that form."""
    gen = torch.Generator(device="cuda").manual_seed(q_len)
    q, k = (torch.randn((1, h, s, 64), generator=gen, device="cuda").half() for h, s in ((256, q_len), (32, 3000)))
    _check(q, k, kw, prescaled=True)
    q[0, 77, q_len // 2] *= 60
    _check(q, k, kw, prescaled=True)


def test_exact_workspace():
    """The call writes nothing behind the bytes that fcs_workspace_bytes() names, in a shape where the rows laid end to end
    need more than the heads on their own."""
    from flash_colsum import _hip
    from oracle import colsum_ext_exact

    b, h, hk, s_q, s_k, d = 4, 32, 8, 1, 32768, 128
    gen = torch.Generator(device="cuda").manual_seed(6)
    q, k = (torch.randn((b, n, s, d), generator=gen, device="cuda").half() for n, s in ((h, s_q), (hk, s_k)))
    assert _plan(q, k, {"is_causal": True}) == (False, True)
    n = _hip.workspace_bytes(True, b, h, s_q, s_k, d)
    guard = 1 << 20
    ws = torch.full((n + guard,), 0xA5, dtype=torch.uint8, device="cuda")
    out = torch.empty((b, s_k), dtype=torch.float32, device="cuda")
    c = _hip._Call()
    c.struct_bytes, c.dtype, c.causal = ctypes.sizeof(_hip._Call), 0, 1
    c.B, c.Hq, c.Hk, c.Sq, c.Sk, c.D = b, h, hk, s_q, s_k, d
    c.cls_n, c.k_past, c.scale = -1, s_k - s_q, d ** -0.5
    c.q_strides, c.k_strides = _hip._I64x4(*q.stride()), _hip._I64x4(*k.stride())
    c.q, c.k, c.out, c.out_f16 = q.data_ptr(), k.data_ptr(), out.data_ptr(), None
    c.ws, c.ws_bytes, c.hip_stream = ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream
    print("exact workspace", n, flush=True)
    assert _hip.lib().fcs_colsum_call(ctypes.byref(c)) == 0
    torch.cuda.synchronize()
    assert (ws[n:] == 0xA5).all()
    ref = colsum_ext_exact(q, k, is_causal=True).double()
    assert ((out.double() - ref).abs() <= 1e-3 * ref).all()


@pytest.mark.parametrize("group,q_len,d,dtype", [(8, 128, 64, torch.bfloat16), (4, 100, 128, torch.float16), (8, 33, 128, torch.bfloat16), (5, 16, 64, torch.float16),
                                                 (8, 7, 256, torch.float16), (2, 120, 256, torch.bfloat16)])
def test_one_row_beyond_the_range(group, q_len, d, dtype):
    """A row whose scores leave the unstabilised range makes the waves that hold its head redo their sums with the maximum
    subtracted and take the two-constant form of the column pass; the block's other waves keep theirs.  The row lies at
    the edges of heads, of waves and of blocks."""
    gen = torch.Generator(device="cuda").manual_seed(group * 100 + q_len)
    hk, s_k = 2, 4200
    b = -(-(257 if q_len <= 64 else 512 if d > 128 else 2560) // (hk * group * 16))
    q, k = (torch.randn((b, h, s, d), generator=gen, device="cuda").to(dtype) for h, s in ((hk * group, q_len), (hk, s_k)))
    rows = group * q_len
    for at in [[0], [q_len - 1, q_len], [63 % rows], [64 % rows], [127 % rows, 256 % rows], [511 % rows], [rows - 1], list(range(0, rows, 64))]:
        x = q.clone()
        for v in at:
            x[0, v // q_len, v % q_len] *= 60
            x[-1, hk * group - 1 - v // q_len, v % q_len] *= -40
        for causal in (True, False):
            _check(x, k, {"is_causal": causal})
