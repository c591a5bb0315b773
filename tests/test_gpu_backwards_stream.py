"""Two-pass path, one piece per workgroup: the stages that all rows of a block see are streamed backwards, the others behind them.  Where that part
ends relative to stages, chunks and waves; batches, which stay on the two-pass path at any length.  Error bar as everywhere: max 1e-4,
element-wise relative 1e-3, of the fp32 means against float64."""
import re

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
    assert "one piece each" in t.split("fcs_colstream_kernel")[1]  # else it streams forwards
    for rows in (None, 0):  # then with rows beyond the unstabilised range
        if rows is not None:
            q[:, 1, rows] *= 60
        got = flash_colsum_ext(q, k, is_causal=True, k_past=k_past, out_dtype=torch.float32).double()
        ref = torch.cat([colsum_ext_exact(q[b:b + 1], k[b:b + 1], is_causal=True, k_past=k_past) for b in range(2)])
        err = (got - ref).abs()
        # (2^-126: probabilities that fp32 flushes to zero)
        assert torch.isfinite(got).all() and (err <= 1e-4).all() and (err <= 1e-3 * ref.abs() + 2.0 ** -126).all(), err.max()


# every kernel with such workgroups: blocks of 128, 256 and 512 rows, rows laid end to end, chunks of 9 to 18 stages: rings of three and four slots wrap
WRAPS = [("128,1,4", 1, 64, 64, 128, 9000, 128), ("128,1,4", 4, 16, 16, 100, 4100, 128), ("128,2,4", 4, 16, 16, 200, 4100, 128), ("128,2,8", 4, 4, 4, 600, 4100, 128),
         ("128,2,8,fold", 4, 32, 8, 100, 9000, 128), ("256,1,4", 4, 8, 8, 100, 4100, 256), ("256,1,8", 2, 8, 2, 400, 4100, 256), ("256,1,8,fold", 4, 16, 4, 100, 7000, 256),
         ("64,1,4", 2, 32, 32, 100, 4100, 64), ("64,2,4", 4, 16, 4, 200, 4100, 64), ("64,2,8", 8, 2, 2, 600, 4100, 64), ("64,2,8,fold", 2, 64, 16, 100, 9000, 64)]


def _k_past(kernel, b, h, hk, q_len, k_len, d, stages, off):
    """The largest k_past that leaves `stages` stages and `off` keys of a chunk to the first row, and its column pass."""
    for k_past in range(k_len - 1, 1000, -1):
        t = _hip.plan_description((b, h, q_len, d), (b, hk, k_len, d), causal=True, k_past=k_past, bf16=True).split(" + ")[1]
        name, fold, chunk = re.match(r"fcs_colstream_kernel<(\d+,\d,\d),true,false(,true)?> .* chunks of (\d+) keys, one piece each", t).groups()
        if kernel == name + (",fold" if fold else "") and (k_past - off) % int(chunk) == 64 * stages:
            return k_past, t
    raise AssertionError(kernel)


@pytest.mark.parametrize("kernel,b,h,hk,q_len,k_len,d", WRAPS)
@pytest.mark.parametrize("stages", [2, 3, 4, 5, 7])
def test_rings_wrap(kernel, b, h, hk, q_len, k_len, d, stages):
    """Row 0 sees `stages` whole stages of a chunk, but for a key, and one key more."""
    g = torch.Generator(device="cuda").manual_seed(stages)
    q, k = (torch.randn((b, n, s, d), generator=g, device="cuda").to(torch.bfloat16) for n, s in ((h, q_len), (hk, k_len)))
    for off in (-2, -1, 0):
        k_past, plan = _k_past(kernel, b, h, hk, q_len, k_len, d, stages, off)
        print(tuple(q.shape), tuple(k.shape), k_past, plan, flush=True)
        got = flash_colsum_ext(q, k, is_causal=True, k_past=k_past, out_dtype=torch.float32).double()
        for i in range(b):
            ref = colsum_ext_exact(q[i:i + 1], k[i:i + 1], is_causal=True, k_past=k_past)[0]
            err = (got[i] - ref).abs()
            assert torch.isfinite(got[i]).all() and (err <= 1e-4).all() and (err <= 1e-3 * ref + 2.0 ** -126).all(), (i, err.max())
