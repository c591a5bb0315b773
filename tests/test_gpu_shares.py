"""Two-pass path: workgroups whose equal share of a pass crosses into other row blocks, units, key chunks, heads and batch
entries, or ends inside one (GPU).  Error bar as everywhere: max 1e-4, element-wise relative 1e-3, of the fp32 means against float64."""
import ctypes

import pytest
import torch

from flash_colsum import _hip, flash_colsum_ext
from oracle import colsum_ext_exact

pytestmark = pytest.mark.gpu


def _check(got, ref):
    err = (got.double() - ref).abs()
    assert err.max().item() <= 1e-4 and (err / ref.abs().clamp_min(1e-12)).max().item() <= 1e-3, (err.max().item(), (err / ref).max().item())


def _call(b, h, hk, q_len, k_len, d, dtype=torch.float16, causal=True, seed=0, prepare=None, **kw):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randn(b, h, q_len, d, generator=g, device="cuda")
    k = torch.randn(b, hk, k_len, d, generator=g, device="cuda")
    if prepare:
        prepare(q, k)
    q, k = q.to(dtype), k.to(dtype)
    print((b, h, hk, q_len, k_len, d, dtype, causal, kw), flush=True)
    return flash_colsum_ext(q, k, is_causal=causal, out_dtype=torch.float32, **kw), colsum_ext_exact(q, k, is_causal=causal, **kw), q, k


# several row blocks per share and several shares per row block; a last key stage of one key; head dims of every kernel width
SHAPES = [(1, 12, 12, 2400, 2400, 128, True), (1, 8, 8, 4097, 4097, 64, True), (3, 5, 5, 1537, 1537, 64, True), (1, 16, 4, 2600, 3000, 80, True),
          (1, 12, 12, 4500, 4500, 64, False), (2, 7, 7, 2305, 2305, 128, False), (1, 6, 6, 2900, 2900, 256, True), (40, 3, 3, 200, 2113, 48, False),
          (2, 24, 24, 513, 700, 64, True)]


@pytest.mark.parametrize("b,h,hk,q_len,k_len,d,causal", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_shares_that_cross(b, h, hk, q_len, k_len, d, causal, dtype):
    t = _hip.plan_description((b, h, q_len, d), (b, hk, k_len, d), causal=causal, bf16=dtype == torch.bfloat16)
    assert "places" in t
    got, ref, q, k = _call(b, h, hk, q_len, k_len, d, dtype, causal)
    _check(got, ref)
    assert torch.equal(got, flash_colsum_ext(q, k, is_causal=causal, out_dtype=torch.float32))  # fixed order of additions


@pytest.mark.parametrize("d,h,s", [(64, 16, 3000), (128, 8, 2500)])
@pytest.mark.parametrize("which", ["one_row", "late_keys", "one_head"])
def test_rows_out_of_range_in_some_parts(d, h, s, which):
    """A part of a row block that leaves the unstabilised range is redone while the next one's rows and stages are on their way;
    the parts of a row are then of both kinds."""
    def scale_up(q, k):
        if which == "one_row":
            q[:, 0, 777] *= 40.0
        elif which == "late_keys":
            k[:, :, s - 300:] *= 30.0
        else:
            q[:, h // 2] *= 25.0
    got, ref, _, _ = _call(1, h, h, s, s, d, prepare=scale_up)
    _check(got, ref)


def test_rows_that_see_nothing_and_few_averaged_rows():
    # k_past well below K_len - Q_len: the last chunks are seen by no row, their means are 0
    got, ref, _, _ = _call(2, 6, 6, 1100, 9000, 64, k_past=100)
    _check(got, ref)
    assert (got[:, 1200:] == 0).all()
    got, ref, _, _ = _call(1, 16, 16, 3000, 3000, 64, cls_len=1030)
    _check(got, ref)


def _static(q, k):
    b, h, s, d = q.shape
    out = torch.empty(b, s, device="cuda")
    strides = (ctypes.c_int64 * 4)(*q.stride())
    rc = _hip.lib().fcs_colsum_noncausal_f16_static(
        ctypes.c_void_p(q.data_ptr()), ctypes.c_void_p(k.data_ptr()), ctypes.c_void_p(out.data_ptr()), None, b, h, s, d, strides, strides,
        ctypes.c_float(d ** -0.5), -1, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    return out


@pytest.mark.parametrize("b,h,s,d", [(352, 23, 27, 256), (568, 14, 2, 72), (172, 47, 13, 200), (64, 8, 1537, 96), (256, 1, 1700, 80)])
def test_static_scratch_without_room_for_slabs(b, h, s, d):
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k = (torch.randn(b, h, s, d, generator=g, device="cuda").half() for _ in range(2))
    out, usual = _static(q, k), flash_colsum_ext(q, k, is_causal=False, out_dtype=torch.float32)
    # the same terms in another grouping: up to 47 x 13 of them (the last two: a single pass otherwise)
    assert ((out - usual).abs() <= 2e-6 * usual).all()


def test_static_scratch_lays_out_what_the_usual_plan_does_not_fit():
    """Accepted before the parts of row blocks had workspace of their own: 12 heads of 55565 keys."""
    b, h, s, d = 1, 12, 55565, 64
    assert _hip.workspace_bytes(False, b, h, s, s, d) > 8 << 20
    g = torch.Generator(device="cuda").manual_seed(1)
    q = torch.randn(b, h, s, d, generator=g, device="cuda").half()
    k = torch.randn(b, h, s, d, generator=g, device="cuda").half()
    out = _static(q, k)
    usual = flash_colsum_ext(q, k, is_causal=False, out_dtype=torch.float32)
    assert ((out - usual).abs() <= 2e-6 * usual).all()  # the same terms in another grouping: 12 x 109 fp32 partial sums


@pytest.mark.parametrize("scale", [1e-45, 5e-39, 2e-38, 1e-37, 9e-31, 1.1e-30, 1e-20, -2e-38, 0.0])
@pytest.mark.parametrize("d,dtype,causal", [(64, torch.float16, True), (64, torch.float16, False), (128, torch.float16, False), (64, torch.bfloat16, True),
                                            (200, torch.bfloat16, True)])
def test_scales_next_to_zero(d, dtype, causal, scale):
    """Every row is uniform; log2(row sum) / scale is beyond fp32 for the first of them."""
    got, ref, _, _ = _call(1, 4, 4, 4096, 4100, d, dtype, causal, scale=scale)
    _check(got, ref)


def test_scale_next_to_zero_on_scores_next_to_the_largest():
    """bf16 scores of standard deviation 2^124, a scale of 2^-125: logits of one half."""
    got, ref, _, _ = _call(1, 4, 4, 40, 4096, 64, torch.bfloat16, True, scale=2.0 ** -125, prepare=lambda q, k: (q.mul_(2.0 ** 61), k.mul_(2.0 ** 60)))
    assert ref.max() / ref.median() > 1.1
    _check(got, ref)


@pytest.mark.parametrize("d", [8, 40, 56, 72, 96, 120, 136, 200, 248])
@pytest.mark.parametrize("causal", [True, False])
def test_channels_past_the_head_dim_are_not_read(d, causal):
    """Heads narrower than the kernels are compiled for, in rows that go on with NaN: whole key stages and the last one."""
    g = torch.Generator(device="cuda").manual_seed(d)
    wide = [torch.full((2, 3, s, 256), float("nan"), device="cuda", dtype=torch.float16) for s in (700, 2900 if not causal else 1000)]
    q, k = (w[..., :d] for w in wide)
    for t in (q, k):
        t.copy_(torch.randn(t.shape, generator=g, device="cuda"))
    print((d, causal), flush=True)
    got = flash_colsum_ext(q, k, is_causal=causal, out_dtype=torch.float32)
    _check(got, colsum_ext_exact(q.contiguous(), k.contiguous(), is_causal=causal))
