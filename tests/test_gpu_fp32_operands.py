"""fp32 operands: rounded to fp16 in one pass with the range test.  The result is that of the same operands rounded by torch
beforehand, bit for bit, whatever the storage order, the element count modulo the kernel's 8-element pieces and its steps of
1024 pieces; a value beyond the range anywhere takes the other route."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _f32(q, k, **kw):
    from flash_colsum import flash_colsum_f32

    return flash_colsum_f32(q, k, **kw)


@pytest.mark.parametrize("b,h,s,d", [(1, 1, 1, 1), (1, 1, 3, 5), (1, 3, 7, 9), (2, 4, 33, 8), (1, 2, 511, 20), (1, 4, 2048, 2), (3, 5, 577, 64), (2, 16, 1025, 64)])
@pytest.mark.parametrize("layout", ["heads", "tokens", "gaps", "offset"])
def test_rounded_operands(b, h, s, d, layout):
    g = torch.Generator().manual_seed(s * 10 + d)
    x = []
    for _ in range(2):
        if layout == "tokens":
            x.append(torch.randn((b, s, h, d), generator=g).cuda().transpose(1, 2))
        elif layout == "gaps":  # rows with space between them
            x.append(torch.randn((b, h, s, d + 3), generator=g).cuda()[..., :d])
        elif layout == "offset":  # base not 16-byte aligned
            x.append(torch.randn((b * h * s * d + 1,), generator=g).cuda()[1:].view(b, h, s, d))
        else:
            x.append(torch.randn((b, h, s, d), generator=g).cuda())
    print("fp32 operands", b, h, s, d, layout, flush=True)
    q, k = x
    for kw in [{}, {"cls_len": 1}]:
        assert torch.equal(_f32(q, k, **kw), _f32(q.half(), k.half(), **kw)), (b, h, s, d, layout, kw)
    if b == 1:
        assert torch.equal(_f32(q, k, is_causal=True), _f32(q.half(), k.half(), is_causal=True))


@pytest.mark.parametrize("where", [0, 7, 8, 8191, 8192, -1])
@pytest.mark.parametrize("operand", ["q", "k"])
def test_one_value_beyond_the_range(where, operand):
    """The first and last element, the edges of a piece and (of Q; K's: below) of a workgroup's step; then an in-range call:
    no stale flag."""
    g = torch.Generator().manual_seed(3)
    q, k = (torch.randn((1, 3, 301, 25), generator=g).cuda() for _ in range(2))
    clean = _f32(q, k)
    hurt = {"q": q, "k": k}
    t = hurt[operand].clone()
    hurt[operand] = t
    for value in [float("-inf")] + [float("nan")] * (operand == "q"):
        t.view(-1)[where] = value
        with pytest.raises(ValueError, match="NaN or infinite"):
            _f32(hurt["q"], hurt["k"])
    t.view(-1)[where] = 65504.0
    assert torch.equal(_f32(hurt["q"], hurt["k"], scale=1e-6), _f32(hurt["q"].half(), hurt["k"].half(), scale=1e-6))
    t.view(-1)[where] = -65505.0  # would round to -65504: still the other route, whose operands keep 16 bits
    from oracle import colsum_exact

    ref = colsum_exact(hurt["q"].double(), hurt["k"].double(), scale=1e-6)
    got = _f32(hurt["q"], hurt["k"], scale=1e-6).double()
    assert ((got - ref).abs() <= 1e-3 * ref.abs()).all()
    assert torch.equal(_f32(q, k), clean)


def test_negation_that_torch_has_put_off():
    """A tensor with torch's negative bit holds the opposite of what its storage says: it is resolved before the kernel reads it."""
    g = torch.Generator().manual_seed(5)
    q, k = (torch.randn((1, 3, 301, 64), generator=g).cuda() for _ in range(2))
    lazy = torch._neg_view(q)
    assert lazy.is_neg()
    assert torch.equal(_f32(lazy, k), _f32((-q).half(), k.half()))


def test_step_edges_of_the_second_operand():
    """K's pieces are counted behind Q's: the last and first element on either side of each edge of a workgroup's step."""
    g = torch.Generator().manual_seed(6)
    q, k = (torch.randn((1, 3, 301, 25), generator=g).cuda() for _ in range(2))
    behind_q = (q.numel() + 7) // 8
    edges = [8 * (p - behind_q) for p in range(1024, behind_q + (k.numel() + 7) // 8, 1024) if p > behind_q]
    assert len(edges) == 3
    for e in [e + d for e in edges for d in (-1, 0, 7, 8)]:
        x = k.clone()
        x.view(-1)[e] = float("inf")
        with pytest.raises(ValueError, match="NaN or infinite"):
            _f32(q, x)
        x.view(-1)[e] = 65504.0
        assert torch.equal(_f32(q, x, scale=1e-6), _f32(q.half(), x.half(), scale=1e-6))


@pytest.mark.parametrize("more", [-8, 0, 3])
def test_more_elements_than_one_walk_of_the_grid(more):
    """4096 workgroups take 1024 pieces of 8 elements each; from there on they walk.  Bit for bit torch's rounding, and a value
    out of range in the very last element is seen."""
    from flash_colsum import _hip

    g = torch.Generator(device="cuda").manual_seed(7)
    n0 = 8 * 1024 * 1500 + 5
    n1 = 8 * 1024 * 4096 - (n0 + 7) // 8 * 8 + more
    x = [torch.randn((n,), generator=g, device="cuda") * 100 for n in (n0, n1)]
    y = [torch.full((n,), -1.0, dtype=torch.float16, device="cuda") for n in (n0, n1)]
    flag = torch.zeros((1,), dtype=torch.int32, device="cuda")

    def rounded():
        stream = torch.cuda.current_stream().cuda_stream
        print("rounding", n0, n1, flush=True)
        assert _hip.lib().fcs_round_f16(x[0].data_ptr(), y[0].data_ptr(), n0, x[1].data_ptr(), y[1].data_ptr(), n1, flag.data_ptr(), stream) == 0
        return flag.item()

    assert rounded() == 0 and all(torch.equal(b, a.half()) for a, b in zip(x, y))
    x[1][-1] = -65505.0
    assert rounded() == 1 and torch.equal(y[1][:-1], x[1][:-1].half())


def test_range_is_reported_before_the_head_dim():
    """A head dim that the library refuses and values beyond the range at once: the range is named, as for every other storage
    and type of fp32 operands; values within it leave the head dim."""
    for value, error, text in [(1e6, ValueError, "beyond fp16's range"), (float("inf"), ValueError, "NaN or infinite"), (1.0, RuntimeError, "head dim")]:
        q, k = (torch.full((1, 2, 40, 264), 0.5).cuda() for _ in range(2))
        k[0, 1, 3, 5] = value
        with pytest.raises(error, match=text):
            _f32(q, k)
