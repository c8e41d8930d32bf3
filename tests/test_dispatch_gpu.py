"""Every row of every head, O and the natural-log L, for sizes on both sides of the rules
that choose a kernel or a work order by problem size."""

import pytest
import torch

from helpers import (FWD_ATOL, GRAD_RTOL, c_backward, c_backward_varlen, max_abs, oracle_bwd, oracle_fwd, randn,
                     rel_err)

pytestmark = pytest.mark.gpu


def check_forward(B, Hq, Hkv, Nq, Nk, d, causal):
    from flash_attn_legacy import hip_ext
    q, k, v = randn((B, Hq, Nq, d), 0), randn((B, Hkv, Nk, d), 1), randn((B, Hkv, Nk, d), 2)
    scale = d ** -0.5
    o, lse = hip_ext.forward(q, k, v, scale, causal)
    ref_o, ref_l = oracle_fwd(q, k, v, scale, causal)
    assert torch.isfinite(o).all()
    assert max_abs(o, ref_o) <= FWD_ATOL
    assert max_abs(lse, ref_l) <= FWD_ATOL


# Causal grids by workgroup count (128 query rows each): two per CU at most (264, 348), more
# (704, 675, and 288 at one per CU for head_dim 256); heads that divide by 8 and that do not;
# a last tile of one row.
@pytest.mark.parametrize("B,Hq,Hkv,N,d", [
    (8, 11, 11, 300, 64),
    (3, 29, 29, 400, 64),
    (8, 22, 11, 385, 32),
    (5, 27, 9, 520, 96),
    (4, 24, 8, 300, 256),
])
def test_causal_order(B, Hq, Hkv, N, d):
    check_forward(B, Hq, Hkv, N, N, d, True)


# head_dim 128 where the pipelined grid would leave CUs idle or end in a nearly empty round:
# 128-row workgroups.  GQA ratios 7, 4 and 1; one, two and several query tiles, the last of
# one row and of 128; fewer workgroups than CUs, up to two per CU and more; Nq != Nk.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk", [
    (1, 28, 4, 333, 333),
    (2, 8, 8, 130, 517),
    (9, 32, 8, 129, 129),
    (5, 28, 4, 257, 192),
    (3, 16, 16, 640, 640),
    (20, 16, 4, 64, 65),
])
def test_head_dim_128_small_grid(B, Hq, Hkv, Nq, Nk, causal):
    check_forward(B, Hq, Hkv, Nq, Nk, 128, causal)


# ... and where the pipelined persistent grid stays the faster one: one full round of 256
# pairs of query tiles (odd and even tile counts; four heads per workgroup and 256 rows of
# one head; Nq != Nk; a negative scale).
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,sign,causal", [
    (2, 16, 4, 4032, 4032, 1, True),
    (2, 16, 4, 4032, 4032, -1, True),
    (2, 16, 16, 3840, 3840, 1, True),
    (2, 16, 8, 4090, 4090, 1, False),
    (2, 16, 4, 4032, 5000, 1, False),
    (2, 16, 4, 4096, 3000, 1, True),
])
def test_head_dim_128_full_grid(B, Hq, Hkv, Nq, Nk, sign, causal):
    from flash_attn_legacy import hip_ext
    from test_fwd_gpu import check_groups
    q, k, v = randn((B, Hq, Nq, 128), 3), randn((B, Hkv, Nk, 128), 4), randn((B, Hkv, Nk, 128), 5)
    scale = sign * 128 ** -0.5
    o, lse = hip_ext.forward(q, k, v, scale, causal)
    check_groups(o, lse, q, k, v, scale, causal, [(b, g) for b in range(B) for g in range(Hkv)])


# Head dim 64 at 16 key tiles and more on up to 512 workgroups: the pipelined loop.  Whole and
# partial last key tiles and query tiles, the three lengths around 16 tiles, waves without
# rows, unequal lengths, GQA; a negative scale and values that move the row's reference max.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,mul", [
    (2, 16, 16, 960, 960, 1),
    (2, 16, 8, 961, 961, 1),
    (1, 32, 8, 1025, 1024, 1),
    (2, 16, 4, 1000, 1087, -1),
    (1, 33, 11, 1700, 993, 12),
    (8, 16, 16, 40, 1100, 12),
])
def test_head_dim_64_long_tiles(B, Hq, Hkv, Nq, Nk, mul, causal, dtype):
    from flash_attn_legacy import hip_ext
    q, k, v = (randn((B, h, n, 64), i).to(dtype) for i, (h, n) in enumerate([(Hq, Nq), (Hkv, Nk), (Hkv, Nk)]))
    scale = mul * 64 ** -0.5
    o, lse = hip_ext.forward(q, k, v, scale, causal)
    ref_o, ref_l = oracle_fwd(q, k, v, scale, causal)
    # P and O are rounded to fp16 once each: 2^-11 * sum(P |V|) + 2^-11 |O| <= 2^-10 max |V|
    # (scores of a scale of 12 concentrate P on few keys, so |O| comes near max |V|); to bf16
    # 2^-8 each; L is fp32
    top = float(v.abs().max())
    bound = 2 ** -7 * top if dtype == torch.bfloat16 else FWD_ATOL if abs(mul) == 1 else 2 ** -10 * top
    assert max_abs(o, ref_o) <= bound
    assert max_abs(lse, ref_l) <= FWD_ATOL


def check_gradients(B, Hq, Hkv, Nq, Nk, d, causal, sign=1):
    from flash_attn_legacy import hip_ext
    q, k, v, do = (randn(s, i) for i, s in enumerate(
        [(B, Hq, Nq, d), (B, Hkv, Nk, d), (B, Hkv, Nk, d), (B, Hq, Nq, d)]))
    scale = sign * d ** -0.5
    o, lse = hip_ext.forward(q, k, v, scale, causal)
    got = hip_ext.backward(do, q, k, v, o, lse, scale, causal)
    again = hip_ext.backward(do, q, k, v, o, lse, scale, causal)
    for name, g, g2, ref in zip(("dq", "dk", "dv"), got, again, oracle_bwd(q, k, v, do, scale, causal)):
        assert torch.isfinite(g).all(), name
        assert rel_err(g, ref) <= GRAD_RTOL, name
        assert torch.equal(g, g2), name + " differs between two runs"


# head_dim 256 backward: edges of the 32-row items and key tiles, of the 128-key and
# 128-row workgroups, of the causal pairing (odd and even tile counts), GQA, Nq != Nk with
# key tiles that no query sees, a negative scale; bitwise equal over two runs.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,sign", [
    (1, 2, 2, 1, 1, 1),
    (2, 4, 2, 31, 33, 1),
    (1, 4, 4, 129, 127, 1),
    (1, 4, 1, 300, 300, 1),
    (2, 6, 2, 96, 417, -1),
    (1, 2, 1, 545, 64, 1),
])
def test_head_dim_256_backward(B, Hq, Hkv, Nq, Nk, sign, causal):
    check_gradients(B, Hq, Hkv, Nq, Nk, 256, causal, sign)


# Pipelined backward on small grids, where each key tile's items are cut into runs whose sums a
# second kernel adds: runs that start inside a head, key tiles of one run only (the last
# causal ones), a last key tile of one key, MQA and GQA; and a call with too few queries for
# its keys to be worth cutting.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,d", [
    (1, 8, 1, 257, 257, 128),
    (1, 28, 4, 333, 333, 128),
    (2, 16, 4, 512, 385, 128),
    (1, 12, 3, 100, 200, 128),
    (1, 8, 2, 260, 260, 256),
    (1, 6, 1, 515, 129, 256),
    (1, 4, 1, 64, 2000, 128),
])
def test_backward_runs(B, Hq, Hkv, Nq, Nk, d, causal):
    check_gradients(B, Hq, Hkv, Nq, Nk, d, causal)


# The same through the library with less workspace: what the call cannot do without (no runs),
# room for some of the runs, and fal_bwd_workspace_best's.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,Nq,Nk,d", [(1, 28, 4, 333, 333, 128), (1, 6, 1, 515, 129, 256)])
def test_backward_runs_by_workspace(B, Hq, Hkv, Nq, Nk, d, causal):
    from flash_attn_legacy import hip_ext
    q, k, v, do = (randn(s, i) for i, s in enumerate(
        [(B, Hq, Nq, d), (B, Hkv, Nk, d), (B, Hkv, Nk, d), (B, Hq, Nq, d)]))
    scale = d ** -0.5
    o, lse = hip_ext.forward(q, k, v, scale, causal)
    with pytest.raises(RuntimeError, match="workspace needs") as e:
        c_backward(do, q, k, v, o, lse, scale, causal, workspace_bytes=0)
    need = int(str(e.value).split("needs ")[1].split()[0])
    best = hip_ext._lib.fal_bwd_workspace_best(B, Hq, Hkv, Nq, Nk, d, int(causal))
    slot = 128 * d * 2 * 4                      # one workgroup's sums
    assert best >= need + 2 * slot              # the call does cut its key tiles
    ref = oracle_bwd(q, k, v, do, scale, causal)
    for room in (0, slot, (best - need) // 2, best - need):
        got = c_backward(do, q, k, v, o, lse, scale, causal, workspace_bytes=need + room)
        for name, g, r in zip(("dq", "dk", "dv"), got, ref):
            assert rel_err(g, r) <= GRAD_RTOL, (name, room)
    same = hip_ext.backward(do, q, k, v, o, lse, scale, causal)
    assert all(torch.equal(a, b) for a, b in zip(got, same))       # (the binding gives the best)


# At most 128 MB of workspace for the runs' sums, also where more would be of use.
@pytest.mark.parametrize("d", [128, 256])
def test_backward_runs_workspace_bound(d):
    from flash_attn_legacy import hip_ext
    lib, sizes = hip_ext._lib, []
    for Hq, Hkv in ((8, 1), (32, 8), (16, 16), (128, 1)):
        for N in (300, 1024, 2048, 4096, 8192, 16384, 32768):
            for causal in (0, 1):
                need = lib.fal_bwd_workspace_size(1, Hq, N, d) - (min(Hq * N * d * 4, 128 << 20) if d == 256 else 0)
                sizes.append(lib.fal_bwd_workspace_best(1, Hq, Hkv, N, N, d, causal) - need)
    assert max(sizes) > 64 << 20 and max(sizes) <= 128 << 20 and min(sizes) >= 0


# Token-major operands, each its own [B, N, H, d] tensor or all slices of one fused projection,
# on the pipelined backward: grids that split their key tiles and grids that do not.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,N,d", [
    (1, 8, 2, 260, 256),
    (8, 16, 16, 385, 256),
    (1, 28, 4, 333, 128),
    (8, 16, 16, 385, 128),
])
def test_backward_token_major(B, Hq, Hkv, N, d, fused, causal, dtype):
    from flash_attn_legacy import hip_ext
    rows = lambda h, seed: randn((B, N, h, d), seed).to(dtype).transpose(1, 2)
    q, k, v = (torch.split(rows(Hq + 2 * Hkv, 0), [Hq, Hkv, Hkv], 1) if fused else
               [rows(h, i) for i, h in enumerate((Hq, Hkv, Hkv))])
    do, scale = rows(Hq, 3), d ** -0.5
    o, lse = hip_ext.forward(q, k, v, scale, causal)
    got = hip_ext.backward(do, q, k, v, o, lse, scale, causal)
    dense = hip_ext.backward(*(t.contiguous() for t in (do, q, k, v)), o, lse, scale, causal)
    rtol = 4e-2 if dtype == torch.bfloat16 else GRAD_RTOL          # (three mantissa bits less)
    for name, g, g2, ref in zip(("dq", "dk", "dv"), got, dense, oracle_bwd(q, k, v, do, scale, causal)):
        assert torch.equal(g, g2), name
        assert rel_err(g, ref) <= rtol, name


# Packed backward on the pipelined kernels: head_dim 256 always, head_dim 128 from 768 key
# tiles (times KV heads) of sequences of 512 keys on average.  Sequences that end inside a
# query item or key tile, of one row, without queries or keys, in an order that the work
# lists change; GQA, where one head's rows of the row-value array are followed by the next's.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("lens_q,lens_k,hq,hkv,d", [
    ([1, 33, 300, 129], [1, 33, 300, 129], 4, 2, 256),
    ([70, 0, 130, 515, 31], [140, 33, 0, 257, 128], 4, 1, 256),
    ([515, 1201, 64, 700, 641], [515, 1201, 64, 700, 641], 32, 32, 128),
    ([600, 0, 1100, 70], [1, 900, 2200, 3100], 32, 16, 128),
])
def test_packed_backward_pipelined(lens_q, lens_k, hq, hkv, d, causal, dtype):
    from test_varlen_gpu import bwd_check
    if dtype == torch.float16:
        bwd_check(lens_q, lens_k, hq, hkv, d, causal)
    else:
        bwd_check(lens_q, lens_k, hq, hkv, d, causal, dtype=dtype, rtol=4e-2)   # (three mantissa bits less)


# fal_bwd_varlen_workspace_size knows the query heads only, and with them may expect the other
# dK/dV kernel than the call (which goes by the KV heads) takes: its size covers both.
@pytest.mark.parametrize("nq,nk", [(16, 98048), (1, 71680)])
def test_packed_backward_few_queries_many_keys(nq, nk):
    from test_varlen_gpu import bwd_check
    bwd_check([nq], [nk], 2, 1, 128, False)


# No query rows: every dK and dV row is written, as zeros.
@pytest.mark.parametrize("d", [32, 64, 96, 128, 256])
def test_backward_without_queries(d):
    B, Hq, Hkv, Nk = 2, 4, 2, 300
    k, v, one = randn((B, Hkv, Nk, d), 0), randn((B, Hkv, Nk, d), 1), randn((B, Hq, 1, d), 2)
    lse = torch.zeros((B, Hq, 1), device="cuda")
    _, dk, dv = c_backward(one, one, k, v, one, lse, 0.1, False, nq=0)
    assert not dk.any() and not dv.any()
    cu_q, cu_k = torch.zeros(3, dtype=torch.int32, device="cuda"), torch.tensor([0, 100, 300], dtype=torch.int32, device="cuda")
    one = randn((1, Hq, d), 2)
    _, dk, dv = c_backward_varlen(one, one, k[0].transpose(0, 1), v[0].transpose(0, 1), one, lse[0], cu_q, cu_k, 0, 200,
                                  0.1, False, total_q=0)
    assert not dk.any() and not dv.any()


# More sequences than a 32-bit step between two heads' rows of the row-value array can count
# (4 million query tiles), at head_dim 256 with grouped heads: sequences of one query row and
# two keys, a sample of them against fp32.
def test_packed_backward_millions_of_sequences():
    from flash_attn_legacy import hip_ext
    seqs, hq, hkv, d = (1 << 22) + 1000, 2, 1, 256
    rnd = lambda rows, h, seed: torch.randn((rows, h, d), dtype=torch.float16, device="cuda",
                                            generator=torch.Generator(device="cuda").manual_seed(seed))
    q, do, k, v = rnd(seqs, hq, 0), rnd(seqs, hq, 1), rnd(2 * seqs, hkv, 2), rnd(2 * seqs, hkv, 3)
    cu_q = torch.arange(seqs + 1, dtype=torch.int32, device="cuda")
    tail = (cu_q, 2 * cu_q, 1, 2, 0.0625, False)
    o, lse = hip_ext.forward_varlen(q, k, v, *tail)
    dq, dk, dv = hip_ext.backward_varlen(do, q, k, v, o, lse, *tail)
    s = torch.cat([torch.arange(500), torch.arange(seqs - 500, seqs), torch.arange(0, seqs, 997)]).cuda()
    pick = lambda t: t[s].float()
    keys = lambda t: torch.stack([t[2 * s, 0], t[2 * s + 1, 0]], 1).float()
    fq, fdo, fk, fv = pick(q), pick(do), keys(k), keys(v)            # [n, heads, d], [n, keys, d]
    dot = lambda a, b: (a[:, :, None] * b[:, None]).sum(-1)          # [n, heads, keys]
    p = torch.softmax(dot(fq, fk) * 0.0625, -1)
    dp = dot(fdo, fv)
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * 0.0625
    assert rel_err(dq[s], (ds[..., None] * fk[:, None]).sum(2)) <= GRAD_RTOL
    assert rel_err(keys(dk), (ds[..., None] * fq[:, :, None]).sum(1)) <= GRAD_RTOL
    assert rel_err(keys(dv), (p[..., None] * fdo[:, :, None]).sum(1)) <= GRAD_RTOL
