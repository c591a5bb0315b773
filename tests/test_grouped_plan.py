"""Which calls with grouped key heads lay the rows of a key head's query heads end to end (no GPU needed)."""
from flash_colsum import _hip


def test_grouped_rows_fill_row_blocks():
    d = _hip.plan_description
    # 4 query heads x 64 rows per key head: one block of 256 rows instead of four of 128 half empty ones
    t = d((4, 32, 64, 128), (4, 8, 8192, 128), causal=True, bf16=True)
    assert "fcs_rowstream_kernel<128,2,4,true,false,true> grid 1 x 16 x 32" in t and "fcs_colstream_kernel<128,2,4,true,false,true>" in t, t
    # full blocks of 512 rows, and ungrouped heads, stay head by head
    assert "fcs_rowstream_kernel<128,2,8,false,false> grid 1 x" in d((1, 32, 512, 128), (1, 8, 8192, 128), causal=True)
    assert "fcs_rowstream_kernel<128,1,4,false,false> " in d((1, 8, 64, 128), (1, 8, 8192, 128), causal=True)
    # the single-pass kernels are unchanged by grouping
    assert d((2, 8, 577, 64), (2, 2, 577, 64)) == d((2, 8, 577, 64), (2, 8, 577, 64))


def test_workspace_serves_every_number_of_key_heads():
    """fcs_workspace_bytes() does not know the number of key heads: a multiple of 256, never less than what the
    ungrouped call needs, still linear in the sizes."""
    for b, h, sq, sk, d in [(1, 64, 1, 32768, 128), (4, 32, 64, 8192, 128), (2, 12, 300, 5000, 64), (1, 60, 511, 3000, 256)]:
        n = _hip.workspace_bytes(True, b, h, sq, sk, d)
        assert n > 0 and n % 256 == 0
        assert n <= 64 * b * h * (sq + 1024) + 4 * 4096 * (b * sk + 1024) + (1 << 20)
