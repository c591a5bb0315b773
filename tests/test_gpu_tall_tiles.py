"""Single-pass path with 64 query rows per wave (up to 1024 keys).  Error bar as everywhere: max 1e-4, element-wise
relative 1e-3, of the fp32 means against float64."""
import re

import pytest
import torch

from flash_colsum import _hip, flash_colsum_ext
from oracle import colsum_ext_exact

pytestmark = pytest.mark.gpu


def _tiles(q, k, kw):
    t = _hip.plan_description(tuple(q.shape), tuple(k.shape), bf16=q.dtype == torch.bfloat16, cls_n=kw.get("cls_len", -1), scale=kw.get("scale"))
    m = re.match(r"fcs_tall_kernel<\d,(\d)", t)
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
        q, k = _make(12, 12, hk, q_len, k_len, d, torch.float16, seed=q_len)
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


@pytest.mark.parametrize("s,d", [(865, 64), (1000, 64), (1024, 64), (800, 8), (993, 48), (1024, 32)])
@pytest.mark.parametrize("hk", [16, 4])
def test_up_to_64_channels(s, d, hk):
    """Keys that stay in the ring through a key head's row blocks; operands that are not pre-scaled."""
    for dtype, kw in [(torch.bfloat16, {}), (torch.float16, {"scale": 0.3})]:
        q, k = _make(3, 16, hk, s, s, d, dtype, layout="tokens" if s % 2 else "heads", seed=s + d)
        _check(q, k, kw, 4)
        q[:, 5, s // 2] *= 60
        k[1, hk - 1, -1] *= 50
        _check(q, k, kw, 4)
