"""Grouped key heads on the two-pass path: the rows of a key head's query heads are laid end to end.  Sizes where the
numbering can go wrong: one row per head, heads that end inside a 32-row fragment, a wave or a row block, the last
row count that is folded and the first that is not, keys masked differently for rows of different heads."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(q, k, kw, what):
    from flash_colsum import flash_colsum_ext
    from oracle import colsum_ext_exact

    out = flash_colsum_ext(q.cuda(), k.cuda(), out_dtype=torch.float32, **kw).cpu().double()
    ref = colsum_ext_exact(q.cuda(), k.cuda(), **kw).cpu().double()
    # the bar of every kernel of this package: 1e-4 absolute, 1e-3 of the value
    assert torch.isfinite(out).all(), what
    assert ((out - ref).abs() <= 1e-4).all() and ((out - ref).abs() <= 1e-3 * ref.abs()).all(), (what, (out - ref).abs().max())


@pytest.mark.parametrize("group,q_len", [(2, 1), (8, 1), (3, 31), (4, 33), (8, 16), (5, 64), (2, 128), (2, 129), (8, 100), (3, 300), (2, 511), (2, 512)])
@pytest.mark.parametrize("causal", [True, False])
def test_rows_of_grouped_heads(group, q_len, causal):
    for dtype, d, hk, b in [(torch.bfloat16, 128, 2, 2), (torch.float16, 64, 1, 3), (torch.float16, 40, 2, 1), (torch.bfloat16, 192, 1, 1)]:
        g = torch.Generator().manual_seed(group * 1000 + q_len + d)
        for s_k in (2051, 2900):  # beyond the single-pass kernels
            q = torch.randn((b, hk * group, q_len, d), generator=g).to(dtype)
            k = torch.randn((b, hk, s_k, d), generator=g).to(dtype)
            print("grouped rows", group, q_len, causal, dtype, d, s_k, flush=True)
            _check(q, k, {"is_causal": causal}, (group, q_len, causal, dtype, d, s_k))


@pytest.mark.parametrize("kw", [{"is_causal": True, "k_past": 0}, {"is_causal": True, "k_past": 37}, {"is_causal": True, "cls_len": 21},
                                {"is_causal": True, "k_past": 5000}, {"is_causal": True, "scale": -0.1}, {"is_causal": True, "scale": 4.0}])
def test_masks_and_stabilised_rows_of_grouped_heads(kw):
    """Short pasts (most tiles masked, each row at its own key), a mean over the first rows, scores that leave the
    unstabilised range (scale 4)."""
    g = torch.Generator().manual_seed(5)
    for group, q_len, s_k in [(4, 50, 300), (3, 100, 100), (8, 7, 1000), (2, 200, 129)]:
        q = torch.randn((2, 2 * group, q_len, 64), generator=g).half()
        k = torch.randn((2, 2, s_k, 64), generator=g).half()
        print("grouped masks", group, q_len, s_k, kw, flush=True)
        _check(q, k, kw, (group, q_len, s_k, kw))
