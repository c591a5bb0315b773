"""Two-pass path, one piece per workgroup: the stages that all rows of a block see are streamed backwards, the others behind them.  Where that part
ends relative to stages, chunks and waves; batches, which stay on the two-pass path at any length.  Error bar as everywhere: max 1e-4,
element-wise relative 1e-3, of the fp32 means against float64."""
import pytest
import torch

from flash_colsum import _hip, flash_colsum_ext
from oracle import colsum_ext_exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dtype", [(64, torch.bfloat16), (128, torch.float16), (80, torch.bfloat16), (256, torch.float16)])
@pytest.mark.parametrize("q_len,k_len,k_past", [(128, 1000, 0), (128, 1000, 63), (128, 1000, 64), (100, 1000, 447), (64, 1500, 1436), (128, 1536, 1400),
                                                (33, 777, 744), (128, 640, 5000), (1, 900, 899), (1, 2500, 1300)])
def test_where_the_backwards_part_ends(q_len, k_len, k_past, d, dtype):
    g = torch.Generator(device="cuda").manual_seed(k_past + d)
    q, k = (torch.randn((2, h, s, d), generator=g, device="cuda").to(dtype) for h, s in ((4, q_len), (4, k_len)))
    t = _hip.plan_description(tuple(q.shape), tuple(k.shape), causal=True, k_past=k_past, bf16=dtype == torch.bfloat16)
    print(tuple(q.shape), tuple(k.shape), k_past, dtype, t, flush=True)
    assert "colstream" in t
    for rows in (None, 0):  # then with rows beyond the unstabilised range
        if rows is not None:
            q[:, 1, rows] *= 60
        got = flash_colsum_ext(q, k, is_causal=True, k_past=k_past, out_dtype=torch.float32).double()
        ref = torch.cat([colsum_ext_exact(q[b:b + 1], k[b:b + 1], is_causal=True, k_past=k_past) for b in range(2)])
        err = (got - ref).abs()
        # (2^-126: probabilities that fp32 flushes to zero)
        assert torch.isfinite(got).all() and (err <= 1e-4).all() and (err <= 1e-3 * ref.abs() + 2.0 ** -126).all(), err.max()
