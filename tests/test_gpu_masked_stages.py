"""Two-pass path: the stages of 64 keys that not every row of a wave sees run in loops of their own, pipelined from stage to
stage where a wave holds 32 rows (up to 128 rows per head, and 256-wide heads), key fragment by key fragment where it
holds 64.  Sizes at their edges: the first masked stage is the first of the stream, of the ring's slots, the last; one,
two or many of them; a wave that sees none; a last stage with 1 .. 64 keys; the stages behind a pre-scaled prefix."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(b, h, q_len, s_k, d, dtype, kw, seed):
    from flash_colsum import flash_colsum_ext
    from oracle import colsum_ext_exact

    g = torch.Generator().manual_seed(seed)
    q = torch.randn((b, h, q_len, d), generator=g).to(dtype).cuda()
    k = torch.randn((b, h, s_k, d), generator=g).to(dtype).cuda()
    print("masked stages", b, h, q_len, s_k, d, dtype, kw, flush=True)
    out = flash_colsum_ext(q, k, out_dtype=torch.float32, **kw).double()
    ref = colsum_ext_exact(q, k, **kw).double()
    # the bar of every kernel of this package: 1e-4 absolute, 1e-3 of the value.  A probability below the normal range of
    # fp32 (2^-126) may be flushed to zero, so a mean of them is off by that much at most
    assert torch.isfinite(out).all()
    err = (out - ref).abs()
    assert (err <= 1e-4).all() and (err <= 1e-3 * ref.abs() + 2.0 ** -126).all(), err.max()


@pytest.mark.parametrize("d", [64, 128, 200])
@pytest.mark.parametrize("k_past", [0, 1, 63, 64, 130, 191, 192, 255, 257, 320])
def test_where_the_diagonal_starts(d, k_past):
    for q_len in (1, 33, 128, 129, 300):
        _check(1, 2, q_len, k_past + q_len, d, torch.float16, {"is_causal": True, "k_past": k_past}, k_past + q_len)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("tail", [1, 31, 32, 33, 63, 64])
def test_last_stage_without_a_diagonal(d, tail):
    for q_len in (64, 128, 200):
        _check(1, 1, q_len, 2048 + tail, d, torch.bfloat16, {}, tail + q_len)


@pytest.mark.parametrize("q_len,s_k,k_past", [(128, 700, 572), (128, 513, 256), (128, 640, 383), (256, 900, 260), (64, 1000, 936)])
def test_stages_behind_a_pre_scaled_prefix(q_len, s_k, k_past):
    from flash_colsum import _hip

    h = 16384 // q_len
    assert "true> grid" in _hip.plan_description((1, h, q_len, 64), (1, h, s_k, 64), causal=True, k_past=k_past)
    _check(1, h, q_len, s_k, 64, torch.float16, {"is_causal": True, "k_past": k_past}, s_k)


def test_rows_beyond_the_unstabilised_range():
    """Scores of several hundred: the maximum and the shifted sweep of the row pass, the two-constant form of the column pass."""
    for q_len, d in [(70, 64), (128, 128), (100, 256), (200, 64)]:
        _check(1, 2, q_len, 400, d, torch.float16, {"is_causal": True, "scale": 4.0}, d + q_len)


@pytest.mark.parametrize("d,dtype,q_len", [(64, torch.bfloat16, 512), (64, torch.float16, 200), (128, torch.float16, 512), (128, torch.bfloat16, 250), (128, torch.float16, 128),
                                           (256, torch.float16, 128), (256, torch.bfloat16, 300)])
@pytest.mark.parametrize("causal", [True, False])
def test_one_row_beyond_the_range_in_each_wave(d, dtype, q_len, causal):
    """A row whose scores leave the unstabilised range makes its block redo its sums with the maximum subtracted and its unit
    take the two-constant form of the column pass, whichever wave (32 or 64 rows each) holds it."""
    from flash_colsum import flash_colsum_ext
    from oracle import colsum_ext_exact

    g = torch.Generator(device="cuda").manual_seed(d + q_len)
    q = torch.randn((1, 6, q_len, d), generator=g, device="cuda").to(dtype)
    k = torch.randn((1, 2, 2500, d), generator=g, device="cuda").to(dtype)
    for rows in [[0], [31, 33], [64], [127], [q_len - 1], [q_len // 2, 5], list(range(0, q_len, 32))]:
        x = q.clone()
        x[0, 1, rows] *= 60
        x[0, 4, rows[0]] *= -40
        print("one row", d, dtype, q_len, causal, rows, flush=True)
        out = flash_colsum_ext(x, k, is_causal=causal, out_dtype=torch.float32).double()
        ref = colsum_ext_exact(x, k, is_causal=causal).double()
        err = (out - ref).abs()
        assert torch.isfinite(out).all() and (err <= 1e-4).all() and (err <= 1e-3 * ref.abs() + 2.0 ** -126).all(), err.max()
