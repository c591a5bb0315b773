"""Single-pass path with 64 query rows per wave (up to 1024 keys).  Error bar as everywhere: max 1e-4, element-wise
relative 1e-3, of the fp32 means against float64."""
import ctypes
import re

import pytest
import torch

from flash_colsum import _hip, flash_colsum_ext
from oracle import colsum_ext_exact

pytestmark = pytest.mark.gpu


def _tiles(q, k, kw):
    t = _hip.plan_description(tuple(q.shape), tuple(k.shape), bf16=q.dtype == torch.bfloat16, cls_n=kw.get("cls_len", -1), scale=kw.get("scale"))
    m = re.match(r"fcs_tall_kernel<\d,\d,(\d)", t)
    return int(m[1]) if m else 0


def _check(q, k, kw, tiles):
    print("tall tiles", tuple(q.shape), q.stride(), tuple(k.shape), q.dtype, kw, flush=True)
    assert _tiles(q, k, kw) == tiles
    got = flash_colsum_ext(q, k, out_dtype=torch.float32, **kw)
    ref = torch.cat([colsum_ext_exact(q[b:b + 1], k[b:b + 1], **kw) for b in range(q.shape[0])])
    err = (got.double() - ref).abs()
    assert torch.isfinite(got).all()
    assert (err <= 1e-4).all() and (err <= 1e-3 * ref + 1e-12).all(), (err.max().item(), (err / ref).max().item())
    assert torch.equal(got, flash_colsum_ext(q, k, out_dtype=torch.float32, **kw))  # fixed order of additions


def _make(b, h, hk, q_len, k_len, d, dtype, layout="heads", seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def one(n, s):
        if layout == "tokens":
            return torch.randn((b, s, n, d), generator=g, device="cuda").to(dtype).transpose(1, 2)
        return torch.randn((b, n, s, d), generator=g, device="cuda").to(dtype)
    return one(h, q_len), one(hk, k_len)


# first and last length of each number of tiles, a last key tile of one key, waves without a key of their own
LENGTHS = [(449, 128, 2), (512, 128, 2), (385, 96, 2), (480, 72, 2), (513, 128, 3), (545, 128, 3), (768, 128, 3), (737, 120, 3),
           (769, 128, 4), (801, 80, 4), (897, 128, 4), (1023, 104, 4), (1024, 128, 4)]


@pytest.mark.parametrize("s,d,tiles", LENGTHS)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_lengths(s, d, tiles, dtype):
    q, k = _make(6, 8, 8, s, s, d, dtype, layout="tokens" if s % 2 else "heads", seed=s)
    _check(q, k, {}, tiles)


@pytest.mark.parametrize("q_len,cls_len", [(33, None), (64, None), (65, None), (300, 34), (300, 129), (1, None)])
@pytest.mark.parametrize("hk", [1, 3, 12])
def test_rows_and_key_heads(q_len, cls_len, hk):
    """Row blocks that end inside 64 rows, rows that are not averaged, and units that do or do not change the key head."""
    for k_len, d, tiles in [(500, 128, 2), (700, 88, 3), (1000, 128, 4)]:
        # (65 rows, two blocks or three of 32: from 384 blocks on)
        q, k = _make(16 if q_len == 65 else 12, 12, hk, q_len, k_len, d, torch.float16, seed=q_len)
        if q_len == 1:
            tiles = 0  # 32 averaged rows or fewer
        _check(q, k, {"cls_len": cls_len} if cls_len else {}, tiles)


@pytest.mark.parametrize("which", ["row", "head", "keys", "scale"])
@pytest.mark.parametrize("s,d,tiles", [(512, 128, 2), (700, 72, 3), (1000, 128, 4)])
def test_rows_out_of_range(which, s, d, tiles):
    """Row blocks of either order of the key tiles that leave the unstabilised range, between such that do not."""
    q, k = _make(2, 9, 3, s, s, d, torch.float16, layout="tokens", seed=3)
    kw = {}
    if which == "row":
        q[:, 3, 200] *= 60
    elif which == "head":
        q[1, 4] *= -30
    elif which == "keys":
        k[:, 1, s - 40:] *= 40
    else:
        kw = {"scale": -0.7}
    _check(q, k, kw, tiles)


def test_scales():
    q, k = _make(4, 8, 8, 600, 600, 128, torch.bfloat16, seed=4)
    for scale in (0.0, -0.05, 0.3):
        _check(q, k, {"scale": scale}, 3)


@pytest.mark.parametrize("s,d", [(897, 64), (1000, 64), (1024, 64), (800, 8), (993, 48), (1024, 32)])
@pytest.mark.parametrize("hk", [16, 4])
def test_up_to_64_channels(s, d, hk):
    """Keys that stay in the ring through a key head's row blocks; operands that are not pre-scaled."""
    for dtype, kw in [(torch.bfloat16, {}), (torch.float16, {"scale": 0.3})]:
        q, k = _make(3, 16, hk, s, s, d, dtype, layout="tokens" if s % 2 else "heads", seed=s + d)
        _check(q, k, kw, 4)
        q[:, 5, s // 2] *= 60
        k[1, hk - 1, -1] *= 50
        _check(q, k, kw, 4)


def _check_causal(q, k, kw):
    t = _hip.plan_description(tuple(q.shape), tuple(k.shape), causal=True, bf16=q.dtype == torch.bfloat16, cls_n=kw.get("cls_len", -1),
                              k_past=kw.get("k_past"), scale=kw.get("scale"))
    assert re.match(r"fcs_tall_kernel<\d,\d,%d,\w+,\w+,true>" % max(2, -(-k.shape[2] // 256)), t), t
    print("causal tall tiles", tuple(q.shape), q.stride(), tuple(k.shape), q.dtype, kw, flush=True)
    got = flash_colsum_ext(q, k, is_causal=True, out_dtype=torch.float32, **kw)
    ref = torch.cat([colsum_ext_exact(q[b:b + 1], k[b:b + 1], is_causal=True, **kw) for b in range(q.shape[0])])
    err = (got.double() - ref).abs()
    assert torch.isfinite(got).all()
    # (2^-126: probabilities that fp32 flushes to zero)
    assert (err <= 1e-4).all() and (err <= 1e-3 * ref.abs() + 2.0 ** -126).all(), (err.max().item(), (err / ref).max().item())
    assert torch.equal(got, flash_colsum_ext(q, k, is_causal=True, out_dtype=torch.float32, **kw))


# prompts (square), windows, diagonals that start at and between tile edges, last tiles of one key, more rows than keys
CAUSAL = [(300, 300, None), (257, 257, None), (512, 512, None), (700, 700, None), (769, 769, None), (1024, 1024, None), (33, 1000, None), (1, 900, None),
          (16, 520, None), (64, 1024, None), (130, 600, 31), (65, 600, 32), (200, 993, 500), (300, 700, 0), (300, 700, 5000), (900, 400, 0), (400, 400, 7),
          # 32 rows per wave: five to eight tiles
          (1025, 1025, None), (1280, 1280, None), (1500, 1500, None), (1537, 1537, None), (2048, 2048, None), (128, 2048, None), (1, 1100, None),
          (33, 1793, None), (500, 1700, 31), (300, 1300, 1290), (100, 2000, 0)]


@pytest.mark.parametrize("q_len,k_len,k_past", CAUSAL)
@pytest.mark.parametrize("d,dtype", [(64, torch.float16), (128, torch.bfloat16), (40, torch.bfloat16), (96, torch.float16)])
def test_causal(q_len, k_len, k_past, d, dtype):
    q, k = _make(1, 6, 6, q_len, k_len, d, dtype, layout="tokens" if k_len % 2 else "heads", seed=q_len + d)
    _check_causal(q, k, {} if k_past is None else {"k_past": k_past})


@pytest.mark.parametrize("which", ["row", "keys", "scale", "cls_len", "units"])
@pytest.mark.parametrize("s,d", [(400, 64), (700, 72), (1000, 128), (1100, 64), (1400, 48), (1600, 104), (2000, 128)])
def test_causal_rows_out_of_range_and_units(which, s, d):
    """Row blocks that leave the unstabilised range; several heads and row blocks per workgroup, there and back."""
    h = 9 if which != "units" else 360 if s <= 1792 else 27  # (longer prompts of many heads run in two passes)
    q, k = _make(1, h, h // 3, s, s, d, torch.float16, seed=5)
    kw = {}
    if which == "row":
        q[:, 3, [0, 70, s - 1]] *= 60
    elif which == "keys":
        k[:, 1, 5:s // 2] *= 40
    elif which == "scale":
        kw = {"scale": -0.7}
    elif which == "cls_len":
        kw = {"cls_len": 150}
    _check_causal(q, k, kw)


@pytest.mark.parametrize("q_len,k_len,d,cls_len,causal", [(1024, 1024, 96, 96, False), (600, 600, 128, 65, False), (900, 1000, 128, 127, False), (1000, 1000, 64, 70, False),
                                                          (700, 1700, 128, 5, False), (400, 400, 64, 33, True), (1024, 1024, 128, 63, True), (1500, 1500, 72, 40, True)])
def test_rows_that_are_not_averaged_are_not_read(q_len, k_len, d, cls_len, causal):
    """NaN and infinities in the rows behind the averaged ones, the first of them in the same row block."""
    q, k = _make(1 if causal else 12, 16 if causal else 32, 16, q_len, k_len, d, torch.bfloat16, seed=q_len)
    kw = {"cls_len": cls_len, "is_causal": causal}
    t = _hip.plan_description(tuple(q.shape), tuple(k.shape), causal=causal, bf16=True, cls_n=cls_len)
    print("rows not averaged", tuple(q.shape), tuple(k.shape), kw, t, flush=True)
    assert t.startswith("fcs_tall_kernel<")
    want = flash_colsum_ext(q, k, out_dtype=torch.float32, **kw)
    q[:, ::2, cls_len:] = float("nan")
    q[:, 1::2, cls_len:] = float("inf")
    assert torch.isfinite(want).all() and torch.equal(flash_colsum_ext(q, k, out_dtype=torch.float32, **kw), want)


def _means_of_seen(q, k, scale, k_past, rows):
    """float64 means whose probabilities are 0, and not what a NaN makes of them, at keys that a row does not see."""
    s = q[:, :, :rows].double() @ k.double().transpose(2, 3) * scale
    seen = torch.arange(k.shape[2], device=q.device)[None, :] <= k_past + torch.arange(rows, device=q.device)[:, None]
    e = torch.where(seen, torch.exp(s - torch.where(seen, s, -torch.inf).amax(3, keepdim=True)), 0.0)
    return torch.where(seen, e / e.sum(3, keepdim=True), 0.0).mean((1, 2))


@pytest.mark.parametrize("q_len,k_len,d,k_past,cls_len", [(805, 805, 96, 0, None), (400, 400, 64, 0, 70), (58, 1282, 128, 844, None), (1000, 1427, 120, 427, 49),
                                                          (33, 978, 48, 548, 12), (1100, 1100, 128, 0, 700), (737, 707, 72, 193, 464), (1, 2048, 128, 700, None)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["row", "key", "keys that no row sees"])
def test_causal_not_a_number_stays_where_it_is_seen(q_len, k_len, d, k_past, cls_len, value, where):
    q, k = _make(1, 4, 4, q_len, k_len, d, torch.bfloat16, seed=k_len)
    rows = q_len if cls_len is None else cls_len
    last = k_past + rows  # the first key that no averaged row sees
    if where == "row":
        q[:, 1, rows // 3] = value
    elif where == "key":
        k[:, 2, k_past + rows // 2] = value
    elif last < k_len:
        k[:, :, last:] = value
    print(where, value, tuple(q.shape), tuple(k.shape), k_past, cls_len, flush=True)
    t = _hip.plan_description(tuple(q.shape), tuple(k.shape), causal=True, bf16=True, k_past=k_past, cls_n=rows)
    assert t.startswith("fcs_tall_kernel<")
    got = flash_colsum_ext(q, k, is_causal=True, k_past=k_past, cls_len=cls_len, out_dtype=torch.float32).double()
    ref = _means_of_seen(q, k, d ** -0.5, k_past, rows)
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and (got[:, last:] == 0).all()
    fine = ~torch.isnan(ref)
    assert ((got - ref).abs()[fine] <= 1e-4).all() and ((got - ref).abs()[fine] <= 1e-3 * ref[fine] + 1e-12).all()


@pytest.mark.parametrize("h,q_len,k_len,d,causal", [(8, 100, 1000, 128, True), (4, 700, 700, 64, True), (16, 1300, 1300, 96, True), (4, 300, 1700, 96, False)])
def test_query_rows_stored_backwards(h, q_len, k_len, d, causal):
    """The C entry point takes query rows of a negative stride: these calls had been served by the two passes, which do."""
    q, k = _make(1, h, h, q_len, k_len, d, torch.float16, seed=k_len)
    back = q.flip(2).contiguous()
    i64x4 = ctypes.c_int64 * 4
    ws = torch.empty(_hip.workspace_bytes(causal, 1, h, q_len, k_len, d), dtype=torch.uint8, device="cuda")
    out = torch.empty(1, k_len, device="cuda")
    assert _hip.plan_description(tuple(q.shape), tuple(k.shape), causal=causal).startswith("fcs_tall_kernel<")
    last_row = back.data_ptr() + (q_len - 1) * d * 2  # row r of head i is at last_row + 2 (i q_len d - r d)
    print("backwards", tuple(q.shape), tuple(k.shape), causal, flush=True)
    rc = _hip.lib().fcs_colsum_general(0, int(causal), last_row, k.data_ptr(), out.data_ptr(), None, ws.data_ptr(), ws.numel(), 1, h, h, q_len, k_len, d, -1,
                                       max(0, k_len - q_len) if causal else 0, i64x4(h * q_len * d, q_len * d, -d, 1), i64x4(*k.stride()),
                                       ctypes.c_float(d ** -0.5), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(out, flash_colsum_ext(q, k, is_causal=causal, out_dtype=torch.float32))


@pytest.mark.parametrize("b,h,s,d,dtype,causal", [(8, 16, 1024, 128, torch.bfloat16, False), (4, 24, 1000, 96, torch.float16, False), (16, 16, 1000, 32, torch.bfloat16, False),
                                                  (2, 24, 1800, 96, torch.float16, False), (4, 12, 2048, 128, torch.bfloat16, False), (1, 64, 600, 64, torch.float16, True),
                                                  (1, 48, 300, 128, torch.bfloat16, True), (1, 40, 1000, 128, torch.float16, True), (1, 40, 1500, 64, torch.float16, True),
                                                  (1, 30, 2040, 72, torch.float16, True)])
@pytest.mark.parametrize("every", [1, 3])
def test_units_out_of_range_between_others(b, h, s, d, dtype, causal, every):
    """A row block outside the unstabilised range takes the ring for itself: the units behind it, of the same head and of the next
    one, find it as they expect it."""
    q, k = _make(b, h, h, s, s, d, dtype, seed=s)
    for i in range(0, h, every):
        q[:, i, (37 * i) % s::128] *= 40
    print("units out of range", tuple(q.shape), dtype, causal, every, flush=True)
    assert _hip.plan_description(tuple(q.shape), tuple(k.shape), causal=causal, bf16=dtype == torch.bfloat16).startswith("fcs_tall_kernel<")
    got = flash_colsum_ext(q, k, is_causal=causal, out_dtype=torch.float32).double()
    ref = torch.cat([colsum_ext_exact(q[i:i + 1], k[i:i + 1], is_causal=causal) for i in range(b)])
    err = (got - ref).abs()
    # (2^-126: probabilities that fp32 flushes to zero)
    assert torch.isfinite(got).all() and (err <= 1e-4).all() and (err <= 1e-3 * ref + 2.0 ** -126).all(), (err.max(), (err / ref).max())
