"""Top-k and threshold selection at the sizes where the kernels change: entries per lane (1024 lanes hold 1, 2, 4, ...
32 each, longer rows are re-read), words per thread of the sort, rows whose keys share all, many or no leading bits.
The reference is a stable sort of the same values, so the comparison is exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(kind, b, s, gen):
    x = torch.rand((b, s), generator=gen)
    if kind == "narrow":      # a few thousand distinct values around 1e-4: long common prefix, many ties
        x = 1e-4 + (x * 4096).round() * 2.0 ** -37
    elif kind == "wide":      # both signs, every exponent
        x = (x - 0.5) * torch.exp2(torch.randint(-120, 120, (b, s), generator=gen).float())
    elif kind == "constant":
        x = torch.full((b, s), 0.25)
    return x


@pytest.mark.parametrize("kind", ["uniform", "narrow", "wide", "constant"])
@pytest.mark.parametrize("s", [1, 63, 65, 1024, 1025, 2049, 4096, 8191, 16385, 32768, 32769, 41001])
def test_topk_and_threshold_sizes(kind, s):
    from flash_colsum import _hip

    gen = torch.Generator().manual_seed(s)
    x = _rows(kind, 2, s, gen)
    print(kind, s, flush=True)
    order = torch.sort(x, dim=1, descending=True, stable=True).indices
    for k in sorted({k for k in (1, 2, 63, 64, 65, 1000, 1024, 1025, 2048, 2049, 4096, s // 2, s) if 1 <= k <= s}):
        want = order[:, :k]
        if k <= _hip.TOPK_SORT_MAX:
            val, idx = _hip.topk_f32(x.cuda(), k, sorted=True)
            assert torch.equal(idx.cpu(), want) and torch.equal(val.cpu(), x.gather(1, want)), k
        asc = want.sort(dim=1).values
        val, idx = _hip.topk_f32(x.cuda(), k, sorted=False)
        assert torch.equal(idx.cpu(), asc) and torch.equal(val.cpu(), x.gather(1, asc)), k
    tau = float(x[0, s // 3])
    idx, cnt = _hip.threshold_f32(x.cuda(), tau)
    for r in range(2):
        want = (x[r] >= tau).nonzero().view(-1)
        assert cnt[r].item() == want.numel() and torch.equal(idx[r, : want.numel()].cpu(), want)


@pytest.mark.parametrize("s", [2 ** 31 - 8193, 2 ** 31 - 1])
def test_longest_rows(s):
    """Rows whose length, rounded up to whole sweeps of the workgroup (8192 entries), reaches or passes 2^31."""
    from flash_colsum import _hip

    print("longest rows", s, flush=True)
    x = torch.rand((1, s), device="cuda")
    at = torch.tensor([0, 12345, 2 ** 30 + 1, s - 8192, s - 1], device="cuda")
    x[0, at] = torch.tensor([2.0, 3.0, 5.0, 4.0, 6.0], device="cuda")
    val, idx = _hip.topk_f32(x, 5, sorted=True)
    assert val.tolist() == [[6.0, 5.0, 4.0, 3.0, 2.0]] and torch.equal(idx[0], at[[4, 2, 3, 1, 0]])
    idx, cnt = _hip.threshold_f32(x, 2.0)
    assert cnt.item() == 5 and torch.equal(idx[0, :5], at)


@pytest.mark.parametrize("k", [64, 65, 513, 1024, 1025, 2048, 4095, 4096])
@pytest.mark.parametrize("shape", ["full", "crowded", "outlier", "outliers", "spread"])
def test_order_by_counting(shape, k):
    """More than 64 taken entries are ordered by counting in 2048 bins between the smallest and the largest of them (without
    those of one wave where they lie far above the others), unless a bin holds more than 64."""
    from flash_colsum import _hip

    print(shape, k, flush=True)
    gen = torch.Generator().manual_seed(k)
    if shape in ("full", "crowded"):  # bins of 2^10 keys, each with 64 or 65 entries; the row is taken whole
        m = 64 if shape == "full" else 65
        n = torch.arange(k)
        bits = 0x3F000000 + (n // m) * 1024 + n % m
        bits[-1] = 0x3F000000 + 2 ** 21 - 1
        x = bits[torch.randperm(k, generator=gen)].to(torch.int32).view(torch.float32)[None]
    else:
        x = torch.randn((3, 2 * k), generator=gen)
        if shape != "spread":  # all but the outliers, of one wave or of two, lie close together
            x = 1.0 + 1e-3 * x
            x[:, [0, 1] if shape == "outlier" else [0, -1]] = 3e38
    order = torch.sort(x, dim=1, descending=True, stable=True).indices[:, :k]
    val, idx = _hip.topk_f32(x.cuda(), k, sorted=True)
    assert torch.equal(idx.cpu(), order) and torch.equal(val.cpu(), x.gather(1, order))
