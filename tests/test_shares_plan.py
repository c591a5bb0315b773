"""Two-pass path: the equal shares that its workgroups take of a pass's stages (no GPU needed).  fcs_plan.h is plain host
arithmetic: it is compiled here on its own, and the walk of every workgroup is followed as the kernels do it."""
import ctypes
import os
import random
import subprocess

import pytest

from flash_colsum import _hip

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_SOURCE = r"""
#include <algorithm>
#include <map>
#include <set>
#include <vector>
#include "fcs_plan.h"
using namespace fcs;

// keys of a row block's rows [v0, v1) that at least one of them sees
static int seen(const Plan &p, int v1)
{
    if (!p.causal) return p.Sk;
    const long rows = p.fold > 1 ? p.q_rows : std::min(v1, p.q_rows);
    return (int)std::min<long>(p.Sk, p.k_past + rows);
}

// 0: every stage is in exactly one share, and what the shares leave behind fits the workspace; else the check that failed
extern "C" int check(int causal, int B, int H, int Hk, int Sq, int Sk, int D, int cls_n, int k_past, int tight, long *two_pass)
{
    Plan p;
    *two_pass = 0;
    if (!make_plan(p, causal, B, H, Hk, Sq, Sk, D, cls_n, k_past, tight)) return 1;
    if (p.fewrows || p.small || p.fused) return 0;
    *two_pass = 1;
    const long heads = (long)B * p.v_heads;
    // the tightest layout: the row statistics alone
    if (tight < 0 && (!p.c_direct || p.total != align256((size_t)8 * heads * p.rows_pad))) return 25;
    if (tight > 0 && (!p.r_whole || p.c_chunk > std::min(tight, 32) * kStageKeys)) return 26;

    // pass 1
    const int rows1 = p.k1_waves * p.qw;
    std::vector<std::set<long>> sets(heads * p.n_qblk);
    std::vector<int> done1(heads * p.n_qblk);
    for (long share = 0; share < p.r_blocks; ++share) {
        int pos = (int)share * p.r_seg, left = std::min(p.r_seg, p.r_len - pos), bx = 0;
        if (left <= 0) return 2;
        long bh = p.r_by_head.quot(pos, pos);
        if (p.r_line.step == 0) bx = p.r_by_block.quot(pos);
        else for (int sum = 0; pos >= (sum += p.r_line.n(bx) + p.r_line.start); ++bx) {}
        for (int at = pos - p.r_line.places(bx); left > p.r_line.start || at >= 0; at = 0) {
            if (bh >= heads || bx >= p.n_qblk) return 3;
            const int first = std::max(0, at - p.r_line.start), past = std::min(p.r_line.n(bx), at + left - p.r_line.start);
            const long i = bh * p.n_qblk + bx, set = p.r_whole ? i : share + i;
            if (past <= first || done1[i] != first) return 4;  // in order, none left out
            done1[i] = past;
            sets[i].insert(set);
            if ((size_t)(set + 1) * rows1 * 8 > p.off_partial) return 5;
            left -= p.r_line.n(bx) + p.r_line.start - at;
            if (left <= p.r_line.start) break;
            if (++bx == p.n_qblk) { bx = 0; ++bh; }
        }
    }
    std::set<long> all;
    for (long i = 0; i < heads * p.n_qblk; ++i) {
        if ((long)done1[i] * p.r_unit * 64 < seen(p, (int)(i % p.n_qblk + 1) * rows1)) return 6;
        // the sets as the column pass looks for them
        long w0 = 0, parts = 1;
        if (!p.r_whole) {
            const int start = (int)(i / p.n_qblk) * p.r_line.places(p.n_qblk) + p.r_line.places((int)(i % p.n_qblk)) + p.r_line.start;
            w0 = p.r_by_seg.quot(start);
            parts = p.r_by_seg.quot(start + p.r_line.n((int)(i % p.n_qblk)) - 1) - w0 + 1;
        }
        if ((long)sets[i].size() != parts || *sets[i].begin() != w0 + i || *sets[i].rbegin() != w0 + i + parts - 1) return 7;
        for (long s : sets[i]) if (!all.insert(s).second) return 8;  // a single writer each
    }

    // column pass
    const int rows2 = 32 * p.c_nb * p.c_waves, cs = p.c_cs;
    if (p.c_chunk > col_chunk_max(p.Dp, p.c_waves) || p.c_cs * p.c_unit * kStageKeys != p.c_chunk) return 10;
    std::vector<std::set<long>> slabs((long)B * p.c_nchunks);
    std::set<long> numbers;
    std::vector<int> done2((long)B * p.c_nchunks * p.v_heads * p.c_nrb);
    for (long share = 0; share < p.c_blocks; ++share) {
        long b;
        int cx, h = 0, rb = 0, at = 0, left = 0x7fffffff;
        if (p.c_direct) {
            b = p.c_by_chunks.quot((int)share, cx);
        } else {
            int pos = (int)share * p.c_seg;
            left = std::min(p.c_seg, p.c_len - pos);
            if (left <= 0) return 11;
            // the line in order: batch entry, chunk, head, row block
            b = p.c_by_batch.quot(pos, pos);
            for (cx = 0; pos >= p.v_heads * p.c_line.chunk_places(p.c_nrb, cs, cx + 1); ++cx) {}
            pos -= p.v_heads * p.c_line.chunk_places(p.c_nrb, cs, cx);
            const int per_h = p.c_line.chunk_places(p.c_nrb, cs, cx + 1) - p.c_line.chunk_places(p.c_nrb, cs, cx);
            for (; pos >= per_h; ++h) pos -= per_h;
            for (;; ++rb) {
                const int n = p.c_line.between(rb, cx * cs, cx * cs + cs), len = n > 0 ? n + p.c_line.start : 0;
                if (pos < len) break;
                pos -= len;
            }
            at = pos;
            // the kernel's three ways to the same place
            int k_cx, k_h, k_rb;
            if (p.c_one) {  // chunks of a unit side by side: another place, and the share that belongs there
                long k_b = p.by_heads.quot(p.c_by_blocks.quot(p.c_by_chunks.quot((int)share, k_cx), k_rb), k_h);
                const long number = ((k_b * (int)p.c_by_chunks.d + k_cx) * p.v_heads + k_h) * p.c_nrb + k_rb;
                if (number < 0 || number >= p.c_blocks || !numbers.insert(number).second) return 20;
                // that share, by the line: its slab is the one that the walk below gives it
                int q = (int)number * p.c_seg, q_cx, q_h, q_rb;
                const long q_b = p.c_by_batch.quot(q, q);
                q_rb = q % p.c_nrb, q_h = q / p.c_nrb % p.v_heads, q_cx = q / p.c_nrb / p.v_heads;
                if (p.c_seg != 1 || p.c_line.start || q_b != k_b || q_cx != k_cx || q_h != k_h || q_rb != k_rb) return 21;
            } else if (p.c_unit > 1) {
                const long k_b = p.c_by_chunks.quot(p.by_heads.quot(p.c_by_blocks.quot((int)share * p.c_seg, k_rb), k_h), k_cx);
                if (k_b != b || k_cx != cx || k_h != h || k_rb != rb || at != 0) return 22;
            } else {
                p.c_by_batch.quot((int)share * p.c_seg, pos);
                k_cx = std::min(p.c_by_chunks.quot(pos), p.c_every - (p.c_every * cs > p.c_line.n(0) ? 1 : 0));
                int pairs = k_cx * p.c_nrb, steps = 0;
                for (;; ++k_cx, ++steps) {
                    pairs += p.c_line.sees(p.c_nrb, cs, k_cx);
                    if (pos < p.v_heads * (p.c_line.sum(p.c_nrb, (k_cx + 1) * cs) + pairs * p.c_line.start)) break;
                }
                if (k_cx != cx || pairs != p.c_line.pairs(p.c_nrb, cs, cx + 1, p.c_every)) return 23;
                // only chunks that not every row block sees to its end are walked over
                if (steps > (p.c_line.last - p.c_line.n(0)) / cs + 1) return 24;
            }
        }
        for (;;) {
            if (b >= B || cx >= p.c_nchunks) return 12;
            const long chunk = b * p.c_nchunks + cx;
            bool any = p.c_direct;
            for (; left > 0 && h < p.v_heads; at = 0, rb = (rb + 1 == p.c_nrb) ? 0 : rb + 1, h += (rb == 0)) {
                const int n = p.c_line.between(rb, cx * cs, cx * cs + cs);
                if (n <= 0) continue;
                const int first = std::max(0, at - p.c_line.start), past = std::max(0, std::min(n, at + std::min(left, 0x3fffffff) - p.c_line.start));
                left -= n + p.c_line.start - at;
                if (past <= first) break;
                int &d = done2[(chunk * p.v_heads + h) * p.c_nrb + rb];
                if (d != first) return 13;
                d = past;
                any = true;
            }
            if (!any) return 19;  // a chunk is entered for at least one stage
            slabs[chunk].insert(share + chunk);
            if (!p.c_direct && p.off_partial + (size_t)(share + chunk + 1) * p.c_chunk * 4 > p.total) return 14;
            if (p.c_direct || left <= p.c_line.start) break;
            h = rb = at = 0;
            do {
                if (++cx == p.c_nchunks) { cx = 0; ++b; }
            } while (cx * cs >= p.c_line.last);
        }
    }
    all.clear();
    for (long chunk = 0; chunk < (long)B * p.c_nchunks; ++chunk) {
        const int cx = (int)(chunk % p.c_nchunks);
        for (int h = 0; h < p.v_heads; ++h)
            for (int rb = 0; rb < p.c_nrb; ++rb) {
                const int end = std::min(seen(p, (rb + 1) * rows2), std::min(Sk, (cx + 1) * p.c_chunk));
                if ((long)(cx * cs + done2[(chunk * p.v_heads + h) * p.c_nrb + rb]) * p.c_unit * 64 < end) return 15;
            }
        if (p.c_direct) continue;
        // the slabs as the final reduction looks for them
        const int before = p.c_line.chunk_places(p.c_nrb, cs, cx), len = (p.c_line.chunk_places(p.c_nrb, cs, cx + 1) - before) * p.v_heads;
        const int start = (int)(chunk / p.c_nchunks) * (int)p.c_by_batch.d + before * p.v_heads;
        const long w0 = p.c_by_seg.quot(start + p.c_line.start), n = len > 0 ? p.c_by_seg.quot(start + len - 1) - w0 + 1 : 0;
        if ((long)slabs[chunk].size() != n || n > p.n_partials) return 16;
        if (n && (*slabs[chunk].begin() != w0 + chunk || *slabs[chunk].rbegin() != w0 + chunk + n - 1)) return 17;
        for (long s : slabs[chunk]) if (!all.insert(s).second) return 18;
    }
    return 0;
}

// The longest workgroup of each pass over their mean, in stages, and the workgroups.  Row blocks are looked at as the walks above do.
extern "C" int balance(int causal, int B, int H, int Sq, int Sk, int D, double *out)
{
    Plan p;
    if (!make_plan(p, causal, B, H, H, Sq, Sk, D, -1, causal ? std::max(0, Sk - Sq) : 0) || p.fewrows || p.small || p.fused) return 0;
    const int rows1 = p.k1_waves * p.qw, rows2 = 32 * p.c_nb * p.c_waves;
    double most = 0, all = 0;
    for (long share = 0; share < p.r_blocks; ++share) {
        int pos = (int)share * p.r_seg, left = std::min(p.r_seg, p.r_len - pos), bx = 0;
        p.r_by_head.quot(pos, pos);
        if (p.r_line.step == 0) bx = p.r_by_block.quot(pos);
        else for (int sum = 0; pos >= (sum += p.r_line.n(bx) + p.r_line.start); ++bx) {}
        double mine = 0;
        for (int at = pos - p.r_line.places(bx); left > 0; at = 0) {
            const int first = std::max(0, at - p.r_line.start), past = std::min(p.r_line.n(bx), at + left - p.r_line.start);
            const long end = ceil_div(seen(p, (bx + 1) * rows1), kStageKeys);
            mine += std::max(0L, std::min((long)past * p.r_unit, end) - (long)first * p.r_unit);
            left -= p.r_line.n(bx) + p.r_line.start - at;
            if (++bx == p.n_qblk) bx = 0;
        }
        most = std::max(most, mine);
        all += mine;
    }
    out[0] = most * p.r_blocks / all;
    out[1] = p.r_blocks;
    most = all = 0;
    for (long share = 0; share < p.c_blocks; ++share) {
        int cx, h = 0, rb = 0, at = 0, left = 0x7fffffff, cs = p.c_cs;
        if (p.c_direct) {
            p.c_by_chunks.quot((int)share, cx);
        } else {
            int pos = (int)share * p.c_seg;
            left = std::min(p.c_seg, p.c_len - pos);
            p.c_by_batch.quot(pos, pos);
            for (cx = 0; pos >= p.v_heads * p.c_line.chunk_places(p.c_nrb, cs, cx + 1); ++cx) {}
            pos -= p.v_heads * p.c_line.chunk_places(p.c_nrb, cs, cx);
            const int per_h = p.c_line.chunk_places(p.c_nrb, cs, cx + 1) - p.c_line.chunk_places(p.c_nrb, cs, cx);
            for (; pos >= per_h; ++h) pos -= per_h;
            for (;; ++rb) {
                const int n = p.c_line.between(rb, cx * cs, cx * cs + cs), len = n > 0 ? n + p.c_line.start : 0;
                if (pos < len) break;
                pos -= len;
            }
            at = pos;
        }
        double mine = 0;
        for (;;) {
            for (; left > 0 && h < p.v_heads; at = 0, rb = (rb + 1 == p.c_nrb) ? 0 : rb + 1, h += (rb == 0)) {
                const int n = p.c_direct ? 1 : p.c_line.between(rb, cx * cs, cx * cs + cs);
                if (n <= 0) continue;
                const int first = std::max(0, at - p.c_line.start), past = std::max(0, std::min(n, at + std::min(left, 0x3fffffff) - p.c_line.start));
                const long end = ceil_div(seen(p, (rb + 1) * rows2), kStageKeys), from = ((long)cx * cs + first) * p.c_unit;
                mine += std::max(0L, std::min(((long)cx * cs + past) * p.c_unit, end) - from);
                left -= n + p.c_line.start - at;
            }
            if (p.c_direct || left <= p.c_line.start) break;
            h = rb = at = 0;
            cx = (cx + 1) * cs >= p.c_line.last ? 0 : cx + 1;
        }
        most = std::max(most, mine);
        all += mine;
    }
    out[2] = most * p.c_blocks / all;
    out[3] = p.c_blocks;
    return 1;
}
"""


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    d = tmp_path_factory.mktemp("shares")
    src, lib = d / "shares.cpp", d / "libshares.so"
    src.write_text(_SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "flash-colsum_amd", "csrc"), "-o", str(lib), str(src)], check=True)
    dll = ctypes.CDLL(str(lib))
    fn = dll.check

    def call(causal, b, h, hk, sq, sk, d, cls_n, k_past, tight=0):
        two_pass = ctypes.c_long()
        return fn(int(causal), b, h, hk, sq, sk, d, cls_n, k_past, tight, ctypes.byref(two_pass)), two_pass.value

    call.dll = dll
    return call


@pytest.mark.parametrize("seed", range(4))
def test_every_stage_is_in_one_share(check, seed):
    rng = random.Random(seed)
    fixed = [(False, 1, 16, 16, 8192, 8192, 64, -1, 0), (False, 1, 16, 16, 9289, 9289, 64, -1, 0), (True, 1, 32, 32, 4096, 4096, 128, -1, 0),
             (True, 1, 32, 32, 512, 65536, 128, -1, 65024), (True, 4, 32, 8, 64, 8192, 128, -1, 8128), (True, 1, 8, 8, 512, 4096, 256, -1, 3584),
             (True, 257, 1, 1, 128, 250, 64, -1, 122), (True, 3, 5, 1, 1, 1, 64, -1, 0), (True, 1, 2, 2, 20000, 300, 128, -1, 0),
             (True, 1, 8, 8, 1024, 262144, 128, -1, 261120), (True, 1, 3, 3, 1100, 90000, 64, -1, 50000), (True, 1, 1, 1, 65536, 65536, 64, -1, 0),
             (False, 300, 3, 3, 5, 3000, 64, -1, 0), (True, 2, 3, 3, 700, 5000, 200, 100, 10)]
    shapes, n_two_pass = fixed if seed == 0 else [], 0
    for _ in range(400):
        causal = rng.random() < 0.75
        hk = rng.choice([1, 2, 3, 8, 12])
        sq = rng.choice([1, 2, 63, 64, 65, 128, 129, 256, 257, 511, 512, 513, 700, 1025, rng.randint(1, 9000)])
        sk = rng.choice([1, 40, 64, 65, 300, 2047, 2049, rng.randint(1, 12000), rng.randint(1, 40000)])
        shapes.append((causal, rng.choice([1, 1, 2, 3, 8, 40, 300]), hk * rng.choice([1, 1, 2, 4, 8]), hk, sq, sk, rng.choice([64, 80, 128, 200]),
                       rng.choice([-1, -1, -1, 20, 300]), rng.choice([max(0, sk - sq), max(0, sk - sq), 0, sk // 2, sk])))
    for s in shapes:
        rc, two_pass = check(*s)
        assert rc == 0, (rc, s)
        n_two_pass += two_pass
        if not s[0]:  # the layouts for a given workspace
            for tight in (32, 16, 8, 4, 2, 1, -1):
                assert check(*s[:3], s[2], *s[4:], tight)[0] == 0, (tight, s)
    assert n_two_pass > 100


@pytest.mark.parametrize("b,h,s,d", [(352, 23, 27, 256), (446, 18, 12, 256), (157, 51, 17, 128), (568, 14, 2, 72), (467, 17, 1, 96), (172, 47, 13, 200),
                                     (1, 12, 55565, 64), (64, 1, 16384, 256)])
def test_static_scratch_takes_calls_whose_row_statistics_fit(b, h, s, d):
    """8 MiB hold them in each of these; slabs beside them do not fit in most.  The size is looked at before the pointers."""
    lib = _hip.lib()
    rc = lib.fcs_colsum_noncausal_f16_static(None, None, None, None, b, h, s, d, None, None, ctypes.c_float(0.1), -1, None)
    assert lib.fcs_strerror(rc) == b"a required pointer is NULL"
    rc = lib.fcs_colsum_noncausal_f16_static(None, None, None, None, 2 * b, 2 * h, s, d, None, None, ctypes.c_float(0.1), -1, None)
    assert b"static scratch" in lib.fcs_strerror(rc)


@pytest.mark.parametrize("b,h,s,d", [(32, 16, 1537, 96), (64, 8, 1537, 96), (256, 1, 1700, 96), (192, 2, 2000, 80), (256, 2, 2016, 120), (512, 1, 1600, 72)])
def test_static_scratch_takes_narrow_heads_beyond_1536_keys(b, h, s, d):
    """The single pass that serves them otherwise does not fit, the two passes do; and so wherever the row statistics fit."""
    static = _hip.lib().fcs_colsum_noncausal_f16_static
    assert _hip.workspace_bytes(False, b, h, s, s, d) > 8 << 20
    assert static(None, None, None, None, b, h, s, d, None, None, ctypes.c_float(0.1), -1, None) == -1  # the size is looked at before the pointers
    rng = random.Random(s)
    for _ in range(100):
        s2, h2 = rng.randint(1537, 2016), rng.choice([1, 2, 3, 8])
        b2 = (8 << 20) // (8 * h2 * -(-s2 // 512) * 512)  # rows in blocks of up to 512
        assert static(None, None, None, None, b2, h2, s2, d, None, None, ctypes.c_float(0.1), -1, None) == -1, (b2, h2, s2, d)


def test_shares_of_uneven_row_blocks_are_equal():
    """The triangle of a prompt against itself: 32 heads x (8 + 16 + .. + 64) stages over 256 workgroups."""
    t = _hip.plan_description((1, 32, 4096, 128), (1, 32, 4096, 128), causal=True)
    assert "grid 256, shares of 38 places + " in t and "grid 256, shares of 39 places" in t, t


@pytest.mark.parametrize("h,q_len,k_len,d,places", [(8, 4096, 65536, 64, 256), (4, 2048, 65536, 128, 64), (16, 2048, 32768, 64, 128), (12, 1000, 65536, 128, 96)])
def test_almost_equal_row_blocks_stay_whole(h, q_len, k_len, d, places):
    """The last rows of a long context: whole units of 32 stages per workgroup, two to eight of them."""
    t = _hip.plan_description((1, h, q_len, d), (1, h, k_len, d), causal=True)
    assert f"grid 256, shares of {places} places, chunks of 2048 keys" in t, t
    # ... and not where the longest is much longer than the others
    t = _hip.plan_description((1, 12, 4096, 128), (1, 12, 12288, 128), causal=True)
    assert "shares of 66 places" in t, t


@pytest.mark.parametrize("h,q_len,k_len,d", [(32, 4096, 4096, 128), (1, 65536, 65536, 64), (64, 1 << 20, 1 << 20, 128)])
def test_long_lines_have_equal_shares(check, h, q_len, k_len, d):
    """Up to 2^31 places: no workgroup has more than a few percent above the mean (1.75 times it with whole row blocks of a million
    rows in static runs)."""
    out = (ctypes.c_double * 4)()
    assert check.dll.balance(1, 1, h, q_len, k_len, d, out)
    assert out[0] <= 1.15 and out[2] <= 1.2 and out[1] <= 512 and out[3] <= 512, list(out)


def test_lines_beyond_the_limit_are_handed_out_by_the_hardware(check):
    """4.3e9 places: a workgroup per row block of uneven ones, which the hardware starts one after the other."""
    t = _hip.plan_description((1, 64, 1 << 21, 128), (1, 64, 1 << 21, 128), causal=True)
    assert f"grid {64 * 4096}, shares of {1 << 15} places, one piece each" in t and "direct" in t, t
    assert check(True, 1, 64, 64, 1 << 17, 1 << 17, 64, -1, 0)[0] == 0
