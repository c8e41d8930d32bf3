"""Operands whose rows lie closer together than a row is long: a gradient broadcast over the
sequence (stride 0, what `o.sum(dim=2)` hands the backward), rows that overlap, and the
stride of a dimension of one entry, which may be anything.  Results are those of the same
values laid out one row after the other."""

import math

import pytest
import torch

from helpers import GRAD_RTOL, c_backward, c_backward_varlen, cu_from_lens, np64, oracle_bwd, randn, rel_err
from oracle import attention as orc

pytestmark = pytest.mark.gpu

# per gradient, against float64: fp16's bound, and four times it for bf16, whose P and dS have
# three mantissa bits less but whose products add up the same way
RTOL = {torch.float16: GRAD_RTOL, torch.bfloat16: 4 * GRAD_RTOL}


def rows(shape, seed, dim, step):
    """Normal values of `shape` whose entries along `dim` are `step` elements apart, the
    other dimensions (the last one aside) apart from each other."""
    n, d = shape[dim], shape[-1]
    strides, size = [0] * len(shape), (n - 1) * step + d
    strides[dim], strides[-1] = step, 1
    for i in reversed(range(len(shape) - 1)):
        if i != dim:
            strides[i], size = size, size * shape[i]
    return randn((size,), seed).as_strided(shape, strides)


def same(got, want):
    for i, (g, w) in enumerate(zip(got, want)):
        assert torch.equal(g, w), f"output {i}: max difference {float((g.float() - w.float()).abs().max())}"


# One grid that the GPU is not filled by (head dims 128 and 256 split its key tiles) and one
# that fills it.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [32, 64, 96, 128, 256])
@pytest.mark.parametrize("B,Hq,Hkv,N,causal", [(2, 4, 2, 300, True), (4, 16, 16, 513, False)])
def test_gradient_of_a_sum_over_the_sequence(B, Hq, Hkv, N, causal, d, dtype):
    from flash_attn_legacy import flash_attention
    q, k, v = (randn((B, h, N, d), i).to(dtype).requires_grad_(True) for i, h in enumerate((Hq, Hkv, Hkv)))
    w = randn((B, Hq, d), 3).to(dtype)
    o = flash_attention(q, k, v, is_causal=causal)
    seen = []
    o.register_hook(lambda g: seen.append(g.stride()))
    (o.sum(dim=2) * w).sum().backward()
    assert seen[0][2] == 0                      # the backward did get a broadcast gradient
    do = w.unsqueeze(2).expand(B, Hq, N, d)
    for name, x, ref in zip(("dq", "dk", "dv"), (q, k, v), oracle_bwd(q, k, v, do, d ** -0.5, causal)):
        assert rel_err(x.grad, ref) <= RTOL[dtype], name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [32, 64, 96, 128, 256])
def test_packed_gradient_of_a_sum_over_the_tokens(d, dtype):
    from flash_attn_legacy import flash_attn_varlen_func
    lens, hq, hkv = [1, 33, 300, 129], 4, 2
    cu, total = cu_from_lens(lens), sum(lens)
    q, k, v = (randn((total, h, d), i).to(dtype).requires_grad_(True) for i, h in enumerate((hq, hkv, hkv)))
    w = randn((hq, d), 3).to(dtype)
    (flash_attn_varlen_func(q, k, v, cu, cu, 300, 300, causal=True).sum(0) * w).sum().backward()
    do = w.expand(total, hq, d)
    c = cu.cpu().numpy()
    ref = orc.varlen_bwd(np64(q), np64(k), np64(v), np64(do), c, c, d ** -0.5, True)
    for name, x, r in zip(("dq", "dk", "dv"), (q, k, v), ref):
        assert rel_err(x.grad, torch.from_numpy(r)) <= RTOL[dtype], name


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("d", [32, 64, 96, 128, 256])
@pytest.mark.parametrize("short", [0, 0.5])
def test_short_rows(short, d, causal):
    from flash_attn_legacy import hip_ext
    B, Hq, Hkv, N, step = 2, 4, 2, 197, int(short * d)
    scale = 1 / math.sqrt(d)
    dense = [randn((B, h, N, d), i) for i, h in enumerate((Hq, Hkv, Hkv, Hq))]
    for which in range(4):                      # q, k, v, dO in turn
        x = list(dense)
        x[which] = rows(x[which].shape, 10 + which, 2, step)
        y = [t.contiguous() for t in x]
        o, lse = hip_ext.forward(*x[:3], scale, causal)
        same((o, lse), hip_ext.forward(*y[:3], scale, causal))
        same(hip_ext.backward(x[3], *x[:3], o, lse, scale, causal),
             hip_ext.backward(y[3], *y[:3], o, lse, scale, causal))


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("short", [0, 0.5])
def test_short_rows_packed(short, d):
    from flash_attn_legacy import hip_ext
    lens, hq, hkv, step = [70, 0, 1, 130], 4, 2, int(short * d)
    cu, total, scale = cu_from_lens(lens), sum(lens), 1 / math.sqrt(d)
    tail = (cu, cu, max(lens), max(lens), scale, True)
    dense = [randn((total, h, d), i) for i, h in enumerate((hq, hkv, hkv, hq))]
    for which in range(4):
        x = list(dense)
        x[which] = rows(x[which].shape, 10 + which, 0, step)
        y = [t.contiguous() for t in x]
        o, lse = hip_ext.forward_varlen(*x[:3], *tail)
        same((o, lse), hip_ext.forward_varlen(*y[:3], *tail))
        same(hip_ext.backward_varlen(x[3], *x[:3], o, lse, *tail),
             hip_ext.backward_varlen(y[3], *y[:3], o, lse, *tail))


@pytest.mark.parametrize("layout", ["bshd", "bhsd"])
@pytest.mark.parametrize("short", [0, 0.5])
def test_short_rows_decode(short, layout):
    from flash_attn_legacy import hip_ext
    B, Hq, Hkv, S, d = 3, 8, 2, 150, 64
    shape, dim = ((B, S, Hkv, d), 1) if layout == "bshd" else ((B, Hkv, S, d), 2)
    q, lens = randn((B, Hq, d), 0), torch.tensor([150, 1, 77], dtype=torch.int32, device="cuda")
    for which in range(2):
        x = [randn(shape, 1), randn(shape, 2)]
        x[which] = rows(shape, 3, dim, int(short * d))
        same(hip_ext.decode(q, *x, lens, 0.125, cache_layout=layout, return_lse=True),
             hip_ext.decode(q, *(t.contiguous() for t in x), lens, 0.125, cache_layout=layout, return_lse=True))


@pytest.mark.parametrize("d", [64, 128, 256])
def test_stride_of_a_single_row(d):
    from flash_attn_legacy import hip_ext
    B, Hq, Hkv, scale = 2, 4, 2, 1 / math.sqrt(d)
    y = [randn((B, h, 1, d), i) for i, h in enumerate((Hq, Hkv, Hkv, Hq))]
    x = [t.as_strided(t.shape, (t.stride(0), d, 8, 1)) for t in y]
    o, lse = hip_ext.forward(*y[:3], scale, True)
    same(hip_ext.forward(*x[:3], scale, True), (o, lse))
    same(hip_ext.backward(x[3], *x[:3], o, lse, scale, True), hip_ext.backward(y[3], *y[:3], o, lse, scale, True))
    lens = torch.ones(B, dtype=torch.int32, device="cuda")
    same(hip_ext.decode(y[0][:, :, 0], x[1], x[2], lens, scale, cache_layout="bhsd", return_lse=True),
         hip_ext.decode(y[0][:, :, 0], y[1], y[2], lens, scale, cache_layout="bhsd", return_lse=True))


# Q of the forward is read where it is: also the next item's by workgroups that walk several,
# in batches that fill the GPU and in packed sequences.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("short", [0, 0.5])
def test_short_query_rows_of_several_items(short, causal):
    from flash_attn_legacy import hip_ext
    d, scale, step = 128, 128 ** -0.5, int(short * 128)
    q = rows((2, 16, 4032, d), 0, 2, step)
    k, v = randn((2, 4, 4032, d), 1), randn((2, 4, 4032, d), 2)
    same(hip_ext.forward(q, k, v, scale, causal), hip_ext.forward(q.contiguous(), k, v, scale, causal))
    lens = [1 + 37 * i % 400 for i in range(70)]
    cu, total = cu_from_lens(lens), sum(lens)
    q, k, v = rows((total, 8, d), 3, 0, step), randn((total, 2, d), 4), randn((total, 2, d), 5)
    tail = (cu, cu, max(lens), max(lens), scale, causal)
    same(hip_ext.forward_varlen(q, k, v, *tail), hip_ext.forward_varlen(q.contiguous(), k, v, *tail))


# O of the backward is: an output of equal rows, as one broadcast over the sequence.
@pytest.mark.parametrize("d", [32, 64, 96, 128, 256])
def test_broadcast_output(d):
    from flash_attn_legacy import hip_ext
    B, Hq, Hkv, N, scale = 2, 4, 2, 197, 1 / math.sqrt(d)
    q, k, do = randn((B, Hq, N, d), 0), randn((B, Hkv, N, d), 1), randn((B, Hq, N, d), 2)
    v = randn((B, Hkv, 1, d), 3).expand(B, Hkv, N, d).contiguous()       # so every row of O is V's
    _, lse = hip_ext.forward(q, k, v, scale, False)
    o = v[:, :, :1].repeat_interleave(Hq // Hkv, 1).expand(B, Hq, N, d)
    assert o.stride(2) == 0
    same(c_backward(do, q, k, v, o, lse, scale, False), c_backward(do, q, k, v, o.contiguous(), lse, scale, False))
    same(hip_ext.backward(do, q, k, v, o, lse, scale, False),
         hip_ext.backward(do, q, k, v, o.contiguous(), lse, scale, False))


# The library itself, without the binding's copies: head dim 256's backward reads such rows
# where they are, on whole and on split key tiles and in packed sequences.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("short", [0, 0.5])
@pytest.mark.parametrize("B,Hq,Hkv,N", [(1, 8, 2, 260), (8, 16, 16, 385)])
def test_library_reads_short_rows_at_head_dim_256(B, Hq, Hkv, N, short, causal):
    from flash_attn_legacy import hip_ext
    d, scale = 256, 1 / 16
    dense = [randn((B, h, N, d), i) for i, h in enumerate((Hq, Hkv, Hkv, Hq))]
    for which in range(4):
        x = list(dense)
        x[which] = rows(x[which].shape, 10 + which, 2, int(short * d))
        y = [t.contiguous() for t in x]
        o, lse = hip_ext.forward(*y[:3], scale, causal)
        same(c_backward(x[3], *x[:3], o, lse, scale, causal), c_backward(y[3], *y[:3], o, lse, scale, causal))


@pytest.mark.parametrize("short", [0, 0.5])
def test_library_reads_short_rows_packed_at_head_dim_256(short):
    from flash_attn_legacy import hip_ext
    lens, hq, hkv, d, scale = [70, 0, 1, 300], 4, 2, 256, 1 / 16
    cu, total = cu_from_lens(lens), sum(lens)
    dense = [randn((total, h, d), i) for i, h in enumerate((hq, hkv, hkv, hq))]
    for which in range(4):
        x = list(dense)
        x[which] = rows(x[which].shape, 10 + which, 0, int(short * d))
        y = [t.contiguous() for t in x]
        o, lse = hip_ext.forward_varlen(*y[:3], cu, cu, 300, 300, scale, True)
        same(c_backward_varlen(x[3], *x[:3], o, lse, cu, cu, 300, 300, scale, True),
             c_backward_varlen(y[3], *y[:3], o, lse, cu, cu, 300, 300, scale, True))
