"""Single-pass path: nine and ten key tiles per wave (64-wide heads, up to 2560 keys), and small calls whose keys are split over
more waves.  Error bar as everywhere: max 1e-4, element-wise relative 1e-3, of the fp32 means against float64."""
import re

import pytest
import torch

from flash_colsum import _hip, flash_colsum_ext
from oracle import colsum_ext_exact

pytestmark = pytest.mark.gpu


def _variant(q, k, kw):
    t = _hip.plan_description(tuple(q.shape), tuple(k.shape), bf16=q.dtype == torch.bfloat16, cls_n=kw.get("cls_len", -1), scale=kw.get("scale"))
    m = re.match(r"fcs_fused_kernel<(\d+),(\d+),(true|false),(\d),(true|false),(true|false)", t)
    return (int(m[2]), int(m[4]), m[6] == "true") if m else t


def _check(q, k, kw, variant):
    print(tuple(q.shape), tuple(k.shape), q.dtype, kw, flush=True)
    assert _variant(q, k, kw) == variant
    got = flash_colsum_ext(q, k, out_dtype=torch.float32, **kw)
    ref = torch.cat([colsum_ext_exact(q[b:b + 1], k[b:b + 1], **kw) for b in range(q.shape[0])])
    err = (got.double() - ref).abs()
    assert torch.isfinite(got).all()
    assert err.max().item() <= 1e-4 and (err / ref.abs().clamp_min(1e-12)).max().item() <= 1e-3, (err.max().item(), (err / ref).max().item())
    assert torch.equal(got, flash_colsum_ext(q, k, out_dtype=torch.float32, **kw))  # fixed order of additions


def _make(b, h, hk, q_len, k_len, d, dtype, layout="heads", seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    def one(n, s):
        if layout == "tokens":
            return torch.randn((b, s, n, d), generator=g, device="cuda").to(dtype).transpose(1, 2)
        return torch.randn((b, n, s, d), generator=g, device="cuda").to(dtype)
    return one(h, q_len), one(hk, k_len)


# (key groups, tiles): first and last length of each, and a last key tile of one key
WIDE = [(24, 513, 2, 9), (24, 545, 2, 9), (24, 576, 2, 9), (32, 577, 2, 10), (32, 608, 2, 10), (32, 640, 2, 10),
        (8, 1025, 4, 9), (8, 1152, 4, 9), (8, 1153, 4, 10), (8, 1280, 4, 10), (1, 2049, 8, 9), (2, 2304, 8, 9), (1, 2305, 8, 10), (2, 2559, 8, 10),
        (1, 2560, 8, 10)]


@pytest.mark.parametrize("b,s,kg,tiles", WIDE)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_nine_and_ten_tiles(b, s, kg, tiles, dtype):
    q, k = _make(b, 16, 16, s, s, 64, dtype, layout="tokens" if s % 2 else "heads")
    _check(q, k, {}, (tiles, kg, dtype == torch.float16 and s <= 2048))


@pytest.mark.parametrize("which", ["row", "head", "keys"])
@pytest.mark.parametrize("b,s,kg,tiles", [(32, 577, 2, 10), (8, 1100, 4, 9), (2, 2500, 8, 10)])
def test_rows_out_of_range(b, s, kg, tiles, which):
    """Units of either order whose rows leave the unstabilised range, between units that do not."""
    q, k = _make(b, 16, 16, s, s, 64, torch.float16, seed=1)
    if which == "row":
        q[:, 3, 200] *= 60
    elif which == "head":
        q[:, 5] *= 40
    else:
        k[:, 7, s - 40:] *= 50
    _check(q, k, {}, (tiles, kg, s <= 2048))


@pytest.mark.parametrize("std", [1.0, 2.5, 3.5, 5.0])
@pytest.mark.parametrize("b,h,s", [(1, 16, 2300), (2, 8, 2560), (1, 8, 2049)])
def test_logits_beyond_2048_keys_are_not_rounded(b, h, s, std):
    """More than 2048 keys take the operand as it is whatever the number of pairs: rows of widely spread logits (row sums of 2^20 and
    more) had it when such calls ran in two passes.  Bound: an fp32 score of up to 6 std is off by 1e-6 of itself at most, and with
    it its exponential; a mean adds 16000 and more of them, of either sign.  With Q * c rounded to fp16 it is 6.5e-6 at std 1
    and 2e-4 at std 3.5."""
    g = torch.Generator(device="cuda").manual_seed(int(10 * std))
    q, k = ((torch.randn((b, h, s, 64), generator=g, device="cuda") * std ** 0.5).half() for _ in range(2))
    print((b, h, s), std, flush=True)
    assert _variant(q, k, {})[1:] == (8, False)
    ref = torch.cat([colsum_ext_exact(q[i:i + 1], k[i:i + 1]) for i in range(b)])
    got = flash_colsum_ext(q, k, out_dtype=torch.float32)
    assert ((got.double() - ref).abs() / ref).max().item() <= 3e-6


@pytest.mark.parametrize("kw", [{"scale": -0.1}, {"scale": 0.3}, {"cls_len": 300}])
@pytest.mark.parametrize("s,kg", [(2100, 8), (2400, 8)])
def test_beyond_2048_keys(s, kg, kw):
    """Grouped heads (key tiles kept from one query head to the next), other scales, fewer rows than keys."""
    tiles = 9 if s <= 2304 else 10
    q, k = _make(2, 16, 4, s, s, 64, torch.float16, seed=2)
    _check(q, k, kw, (tiles, kg, False))
    q, k = _make(3, 2, 1, 150, s, 64, torch.bfloat16, seed=3)
    _check(q, k, {k_: v for k_, v in kw.items() if k_ != "cls_len"}, (tiles, kg, False))


@pytest.mark.parametrize("b,h,s,d,tiles", [(2, 4, 512, 64, 2), (1, 8, 289, 64, 2), (1, 8, 600, 64, 3), (1, 16, 1024, 64, 4), (1, 8, 512, 128, 2),
                                           (3, 12, 33, 128, 1), (1, 4, 100, 80, 1), (2, 6, 400, 32, 2), (1, 6, 600, 96, 3), (8, 8, 197, 128, 2)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_small_calls_split_over_more_waves(b, h, s, d, tiles, dtype):
    """One to four tiles per wave; key groups without any key among them."""
    q, k = _make(b, h, h, s, s, d, dtype, seed=4)
    _check(q, k, {}, (tiles, 0, True))
    q[:, 0, s // 2] *= 60
    _check(q, k, {}, (tiles, 0, True))
