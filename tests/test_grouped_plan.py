"""Which calls with grouped key heads lay the rows of a key head's query heads end to end, and what workspace that takes
(no GPU needed).  fcs_plan.h is plain host arithmetic: it is compiled here on its own, so that the plan of a given
number of key heads can be looked at next to what fcs_workspace_bytes() promises for all of them."""
import ctypes
import os
import random
import subprocess

import pytest

from flash_colsum import _hip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_SOURCE = """
#include "fcs_plan.h"
// out: fold, total, where the row statistics and the column slabs begin and where the last one written ends
extern "C" int plan(int causal, int B, int H, int Hk, int Sq, int Sk, int D, int cls_n, int k_past, long *out)
{
    fcs::Plan p;
    if (!fcs::make_plan(p, causal, B, H, Hk, Sq, Sk, D, cls_n, k_past)) return 0;
    const bool two_pass = !(p.fewrows || p.small || p.fused);
    out[0] = p.fold;
    out[1] = (long)p.total;
    const long blocks = (long)B * p.v_heads * p.n_qblk;
    out[2] = (long)p.off_lse; out[3] = (long)p.off_partial;
    out[4] = out[2] + (two_pass ? 8L * p.k1_waves * p.qw * (blocks + (p.r_whole ? 0 : p.r_blocks - 1)) : 0);
    out[5] = out[3] + 4L * (!two_pass ? (long)p.n_partials * B * Sk : p.c_direct ? 0 : ((long)p.c_blocks + (long)B * p.c_nchunks - 1) * p.c_chunk);
    return 1;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, lib = d / "plan.cpp", d / "libplan.so"
    src.write_text(_SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "flash-colsum_amd", "csrc"), "-o", str(lib), str(src)], check=True)
    fn = ctypes.CDLL(str(lib)).plan

    def call(causal, b, h, hk, sq, sk, d, cls_n=-1, k_past=None):
        out = (ctypes.c_long * 6)()
        ok = fn(int(causal), b, h, hk, sq, sk, d, cls_n, (max(0, sk - sq) if k_past is None else k_past) if causal else 0, out)
        return dict(zip(("fold", "total", "stats", "slabs", "stats_end", "slabs_end"), out)) if ok else None

    return call


def test_grouped_rows_fill_row_blocks():
    d = _hip.plan_description
    # 4 query heads x 64 rows per key head: one block of 256 rows instead of four of 128 half empty ones
    t = d((4, 32, 64, 128), (4, 8, 8192, 128), causal=True, bf16=True)
    assert "fcs_rowstream_kernel<128,2,4,true,false,true> grid 512, shares of 8 places, one piece each" in t and "fcs_colstream_kernel<128,2,4,true,false,true>" in t, t
    # full blocks of 512 rows, and ungrouped heads, stay head by head
    assert "fcs_rowstream_kernel<128,2,8,false,false> grid 256, " in d((1, 32, 512, 128), (1, 8, 8192, 128), causal=True)
    assert "fcs_rowstream_kernel<128,1,4,false,false> " in d((1, 8, 64, 128), (1, 8, 8192, 128), causal=True)
    # the single-pass kernels are unchanged by grouping
    assert d((2, 8, 577, 64), (2, 2, 577, 64)) == d((2, 8, 577, 64), (2, 8, 577, 64))


@pytest.mark.parametrize("d,q_len,b,h,hk,s_k,kw,folds", [
    # up to 64 rows: more than 256 blocks of 256 keys, whatever the head dim
    (64, 64, 1, 32, 8, 2048, {}, False), (64, 64, 1, 32, 8, 2049, {}, True), (128, 4, 4, 32, 8, 300, {}, False), (256, 33, 4, 32, 8, 600, {}, True),
    # 65 .. 128 rows: 2560 of them, 512 for heads wider than 128
    (128, 65, 1, 32, 8, 20224, {}, False), (128, 65, 1, 32, 8, 20225, {}, True), (64, 128, 4, 32, 8, 4864, {}, False), (64, 128, 4, 32, 8, 4865, {}, True),
    (136, 128, 4, 32, 8, 768, {}, False), (136, 128, 4, 32, 8, 769, {}, True), (64, 129, 8, 64, 8, 30000, {}, False),
    # one unit per batch entry: no slabs
    (64, 8, 1, 16, 1, 300, {}, True), (64, 8, 1, 17, 1, 300, {}, False), (128, 64, 3, 2, 1, 40, {}, True), (64, 1, 1, 2, 2, 300, {}, False),
    # what counts are the keys that some row sees, and the rows that are averaged
    (128, 64, 4, 32, 8, 8192, {"k_past": 0}, False), (128, 64, 4, 32, 8, 8192, {"k_past": 449}, True), (128, 64, 4, 32, 8, 8192, {"k_past": 448}, False),
    (128, 300, 4, 32, 8, 8192, {"cls_n": 20}, True), (64, 64, 1, 32, 8, 2304, {"causal": False}, True),
])
def test_which_calls_are_laid_end_to_end(plan, d, q_len, b, h, hk, s_k, kw, folds):
    kw = dict(kw)
    causal = kw.pop("causal", True)
    p = plan(causal, b, h, hk, q_len, s_k, d, **kw)
    assert (p["fold"] > 1) == folds and p["fold"] in (1, h // hk), p


def test_workspace_serves_every_number_of_key_heads(plan):
    """fcs_workspace_bytes() knows neither the number of key heads nor k_past: it is at least what the plan of any of them
    needs, a multiple of 256, and still linear in the sizes."""
    rng = random.Random(11)
    shapes = [(True, 1, 64, 1, 32768, 128), (True, 4, 32, 64, 8192, 128), (True, 2, 12, 300, 5000, 64), (True, 1, 60, 511, 3000, 256),
              (True, 4, 32, 1, 32768, 128), (True, 4, 32, 100, 32768, 128)]
    for _ in range(300):
        causal = rng.random() < 0.7
        shapes.append((causal, rng.choice([1, 2, 3, 8]), rng.choice([1, 2, 6, 8, 12, 32, 64]), rng.choice([1, 2, 31, 64, 65, 100, 128, 129, 600]),
                       rng.choice([1, 40, 300, 2049, 5000, 30000]), rng.choice([64, 96, 128, 200])))
    grouped_needs_more = 0
    for causal, b, h, sq, sk, d in shapes:
        n = _hip.workspace_bytes(causal, b, h, sq, sk, d)
        assert n > 0 and n % 256 == 0
        assert n <= 64 * b * h * (sq + 1024) + 4 * 4096 * (b * sk + 1024) + (1 << 20)
        alone = plan(causal, b, h, h, sq, sk, d)["total"]
        for hk in [x for x in range(1, h + 1) if h % x == 0]:
            for k_past in {0, 17, sk // 2, max(0, sk - sq), sk} if causal else {0}:
                p = plan(causal, b, h, hk, sq, sk, d, k_past=k_past)
                assert p["total"] <= n, (causal, b, h, hk, sq, sk, d, k_past)
                grouped_needs_more += p["total"] > alone
                # the parts lie one behind the other inside the total, each 256-byte aligned
                assert p["stats"] % 256 == 0 and p["slabs"] % 256 == 0
                assert p["stats"] <= p["stats_end"] <= p["slabs"] <= p["slabs_end"] <= p["total"]
    assert grouped_needs_more > 0  # else the shapes above would not show a bound that forgets the grouped layouts


def test_narrow_heads_beyond_1536_keys(plan):
    """In one pass, but for many heads of few rows each; what fcs_workspace_bytes() promises holds for both."""
    d = _hip.plan_description
    for b, h, hk, q_len, s_k, dim, one in [(8, 16, 16, 2000, 2000, 96, True), (8, 32, 32, 256, 1600, 120, True), (16, 32, 32, 256, 1600, 120, False), (32, 32, 32, 127, 1600, 120, True),
                                           (32, 32, 32, 512, 1600, 112, False), (32, 32, 32, 513, 1600, 112, True), (32, 32, 32, 256, 1600, 88, False),
                                           (32, 32, 32, 300, 1600, 96, True), (32, 32, 32, 256, 1536, 120, True), (32, 32, 8, 128, 1600, 96, False), (32, 32, 8, 128, 1600, 80, True),
                                           (16, 32, 8, 128, 1600, 96, True), (32, 32, 16, 32, 1600, 120, True), (32, 32, 8, 32, 1600, 72, False), (32, 32, 8, 129, 1600, 120, True)]:
        t = d((b, h, q_len, dim), (b, hk, s_k, dim))
        assert t.startswith("fcs_tall_kernel<" if one else "fcs_rowstream_kernel<128,"), (b, h, hk, q_len, s_k, dim, t)
    rng = random.Random(12)
    for _ in range(200):
        b, h, sq, sk, dim = rng.choice([1, 8, 32, 64, 300]), rng.choice([4, 12, 32]), rng.choice([1, 33, 128, 256, 512, 700]), rng.randint(1500, 2050), rng.choice([72, 88, 96, 120])
        n = _hip.workspace_bytes(False, b, h, sq, sk, dim)
        for hk in [x for x in range(1, h + 1) if h % x == 0]:
            assert plan(False, b, h, hk, sq, sk, dim)["total"] <= n, (b, h, hk, sq, sk, dim)
    # the static scratch holds the slabs of one pass where it does not hold the row statistics of two
    rc = _hip.lib().fcs_colsum_noncausal_f16_static(None, None, None, None, 487, 19, 1884, 104, None, None, ctypes.c_float(0.1), 153, None)
    assert _hip.lib().fcs_strerror(rc) == b"a required pointer is NULL"


@pytest.mark.parametrize("b,h,q_len,s_k,d,tall", [
    # 65 .. 128 channels: a generation of 64-row blocks for one and a half of 32-row ones
    (4, 12, 132, 762, 128, False), (8, 4, 484, 484, 128, True), (3, 12, 219, 713, 128, False), (8, 12, 147, 753, 128, False), (12, 6, 255, 578, 80, True),
    (9, 24, 69, 598, 96, True), (8, 4, 448, 448, 128, False), (8, 16, 1024, 1024, 128, True), (64, 16, 32, 1024, 128, False),
    # up to 64: more than one block per head, and below 897 keys more than six
    (31, 32, 50, 900, 48, False), (31, 32, 65, 897, 48, True), (40, 8, 153, 806, 48, False), (8, 12, 785, 785, 32, True), (64, 16, 896, 896, 64, False), (64, 16, 897, 897, 64, True),
    (64, 16, 768, 768, 32, False), (64, 16, 385, 769, 32, True), (64, 16, 384, 769, 32, False), (8, 8, 512, 1000, 64, False)])
def test_which_calls_take_64_rows_per_wave(b, h, q_len, s_k, d, tall):
    t = _hip.plan_description((b, h, q_len, d), (b, h, s_k, d), bf16=True)
    assert t.startswith("fcs_tall_kernel<" if tall else "fcs_fused_kernel<"), t
