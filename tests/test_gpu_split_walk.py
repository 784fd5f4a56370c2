"""The forward on problems with few rows, where the steps of a list are shared by groups of waves: one
case per split, each at sizes where it can go wrong -- lists of more than 64 slots, of fewer steps
than groups and of none, ragged last blocks, PARTIAL tiles as bytes and as bits, a last block whose
steps behind the diagonal or the sequence are dropped.  Against the fp32 oracle with its bars (the
error of a split is that of the operator: rounded weights and results)."""
import pytest
import torch

import omni_attn_capi
from helpers import compare_with_oracle, random_block_metadata
from oracle.dense_oracle import attention_dense_fp32, dense_mask_from_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("D,QB,KB,H,S", [
    (32, 64, 128, 9, 128), (64, 128, 64, 1, 4480), (128, 128, 128, 3, 384), (128, 64, 64, 5, 192),  # 32 rows, 4 groups
    (32, 128, 128, 40, 512), (64, 64, 64, 33, 512), (128, 64, 128, 52, 512),                         # 64 rows, 2 groups
    (128, 128, 64, 20, 512),                                                                         # 64 rows, 4 groups
    (128, 128, 128, 13, 2048)])                                                                      # 128 rows, 2 groups
def test_split_walks(dtype, D, QB, KB, H, S, gpu_device):
    gen = torch.Generator().manual_seed(D + QB + S)
    q, k, v = (torch.randn(1, H, S, D, generator=gen).to(dtype) for _ in range(3))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, 1, H, S // QB, S // KB, QB, KB, p_empty=0.15, shuffle=True)
    # one head causal as a builder lists it, so that the last slot of every list is the diagonal
    for qb in range(S // QB):
        n = ((qb + 1) * QB + KB - 1) // KB
        nb[0, 0, qb] = n
        idx[0, 0, qb, :n] = torch.arange(n, dtype=torch.int32)
        tys[0, 0, qb, :n] = 1
    dev = lambda t: t.to(gpu_device).contiguous()
    qd, kd, vd, nbd, idxd, tysd, pidxd, pmd = (dev(t) for t in (q, k, v, nb, idx, tys, pidx, pm))
    for seqlen in (S, S - QB - 13 if S > QB else S - 13):
        dense = dense_mask_from_blocks(nb, idx, tys, QB, KB, S, S, pidx, pm, seqlen_orig=seqlen)
        ro, rl = attention_dense_fp32(q, k, v, dense)
        outs = []
        for bits in (None, omni_attn_capi.pack_partial_masks(pmd)):
            o = torch.full_like(qd, float("nan"))
            lse = torch.full(qd.shape[:3], float("nan"), dtype=torch.float32, device=gpu_device)
            omni_attn_capi.fwd(qd, kd, vd, o, lse, nbd, idxd, tysd, QB, KB, seqlen, pidxd,
                               pmd if bits is None else None, partial_bits=bits)
            torch.cuda.synchronize()
            compare_with_oracle(o, lse, ro, rl, dtype, f"seqlen {seqlen}, {'bytes' if bits is None else 'bits'}")
            outs.append((o, lse))
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("D,QB,KB,H,S", [(32, 64, 64, 5, 4480), (128, 64, 64, 1, 8384), (64, 64, 128, 3, 448)])
def test_lone_waves(D, QB, KB, H, S, gpu_device):
    """Lists of up to 131 slots for waves that walk alone (live slots of several chunks moved together), and
    lists of fewer steps than groups."""
    test_split_walks(torch.float16, D, QB, KB, H, S - S % KB, gpu_device)


@pytest.mark.parametrize("D,QB,KB,H,S", [
    (32, 128, 64, 2, 1024), (64, 64, 64, 1, 4480), (128, 128, 128, 1, 1152),   # 32 rows, 4 groups
    (32, 128, 64, 40, 512), (64, 64, 64, 33, 512), (128, 64, 128, 52, 512),    # 64 rows, 2 groups
    (128, 128, 64, 20, 512),                                                   # 64 rows, 4 groups
    (128, 128, 64, 13, 2048)])                                                 # 128 rows, 2 groups
def test_rows_outside_the_list_never_reach_the_output(D, QB, KB, H, S, gpu_device):
    """Windows that leave out the first keys, with lists of every length modulo the groups: what the keys and
    values of blocks that are not listed hold (infinities, NaNs) changes no bit of the result."""
    gen = torch.Generator().manual_seed(D + QB + S)
    q, k, v = (torch.randn(1, H, S, D, generator=gen).half().to(gpu_device) for _ in range(3))
    Tq, Tk = S // QB, S // KB
    nb = torch.zeros(1, H, Tq, dtype=torch.int32)
    idx, tys = (torch.zeros(1, H, Tq, Tk, dtype=torch.int32) for _ in range(2))
    for qb in range(Tq):
        last = min(((qb + 1) * QB - 1) // KB, Tk - 1)
        n = max(0, min(last, 1 + qb % 9))  # of the blocks 1 .. last; CAUSAL cuts the last one
        nb[:, :, qb] = n
        idx[:, :, qb, :n] = torch.arange(last - n + 1, last + 1, dtype=torch.int32)
        tys[:, :, qb, :n] = 1
    seqlen = S - 13
    args = (nb.to(gpu_device), idx.to(gpu_device), tys.to(gpu_device), QB, KB, seqlen)
    results = []
    for bad in (None, float("inf"), float("nan")):
        if bad is not None:
            k[:, :, :KB] = bad
            v[:, :, :KB] = bad
        o = torch.full_like(q, float("nan"))
        lse = torch.full(q.shape[:3], float("nan"), dtype=torch.float32, device=gpu_device)
        omni_attn_capi.fwd(q, k, v, o, lse, *args)
        torch.cuda.synchronize()
        results.append((o, lse))
    assert torch.isfinite(results[0][0]).all()
    for o, lse in results[1:]:
        assert torch.equal(o, results[0][0]) and torch.equal(lse, results[0][1])


@pytest.mark.parametrize("softcap", [0.0, 5.0])
@pytest.mark.parametrize("D,QB,KB,H,S", [
    (32, 64, 128, 9, 128), (64, 128, 64, 1, 4480), (128, 128, 128, 3, 384), (64, 64, 64, 5, 192),  # 32 rows / keys, 4 groups
    (32, 128, 128, 40, 512), (64, 64, 128, 36, 512), (128, 64, 64, 20, 512), (128, 128, 64, 20, 512),  # 64 rows / keys, 2
    (64, 128, 128, 18, 2048)])
def test_split_walks_backward(softcap, D, QB, KB, H, S, gpu_device):
    """The backward of such problems: gradients against autograd through the dense oracle, at the bars of
    the other backward tests; rows and keys behind the sequence get zeros."""
    from oracle.dense_oracle import attention_dense_grads
    from test_gpu_backward import check_grads, run_fwd_bwd
    dtype = torch.bfloat16 if D == 128 else torch.float16
    gen = torch.Generator().manual_seed(D + QB + S + 1)
    q, k, v, dout = (torch.randn(1, H, S, D, generator=gen).to(dtype) for _ in range(4))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, 1, H, S // QB, S // KB, QB, KB, p_empty=0.15, shuffle=True)
    for seqlen in (S, S - QB - 13 if S > QB else S - 13):
        got = run_fwd_bwd(q, k, v, dout, nb, idx, tys, QB, KB, seqlen, pidx, pm, device=gpu_device, softcap=softcap)
        dense = dense_mask_from_blocks(nb, idx, tys, QB, KB, S, S, pidx, pm, seqlen_orig=seqlen)
        check_grads(got[:3], attention_dense_grads(q, k, v, dense, dout, softcap=softcap), dtype, f"seqlen {seqlen}")


@pytest.mark.parametrize("H,S", [(10, 2048), (12, 1500)])
def test_slabs_walked_together_with_different_masks(H, S, gpu_device):
    """A batch of which one element attends everything, in a launch whose slabs form one group: every query
    block is computed exactly once, whichever order the lists' lengths give."""
    from omni_attn_torch import create_omni_block_mask_from_prefix_lengths, omni_attention_forward
    gen = torch.Generator().manual_seed(H)
    B, D = 4, 32
    q, k, v = (torch.randn(B, H, S, D, generator=gen).half() for _ in range(3))
    prefix = torch.arange(1, S + 1).repeat(B, 1)
    prefix[1] = S
    prefix[2, :300] = 300
    m = create_omni_block_mask_from_prefix_lengths(prefix.to(gpu_device), H, S, S, 128, 128)
    o, lse = omni_attention_forward(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), m)
    allow = torch.arange(S).view(1, 1, S) < prefix.unsqueeze(-1)
    ro, rl = attention_dense_fp32(q, k, v, allow.unsqueeze(1))
    compare_with_oracle(o, lse, ro, rl, torch.float16, f"H={H} S={S}")


@pytest.mark.parametrize("H,S", [(10, 600), (16, 300)])
def test_backward_of_slabs_walked_together_with_different_masks(H, S, gpu_device):
    """As above for the backward: 5 slabs per XCD in one group, and 14 in two."""
    from omni_attn_torch import create_omni_block_mask_from_prefix_lengths, omni_attention
    from oracle.dense_oracle import attention_dense_grads
    from test_gpu_backward import check_grads
    gen = torch.Generator().manual_seed(H + 1)
    B, D = (4, 32) if H == 10 else (7, 32)
    q, k, v, dout = (torch.randn(B, H, S, D, generator=gen).half() for _ in range(4))
    prefix = torch.arange(1, S + 1).repeat(B, 1)
    prefix[1] = S
    prefix[2, :150] = 150
    m = create_omni_block_mask_from_prefix_lengths(prefix.to(gpu_device), H, S, S, 64, 64)
    leaves = [t.to(gpu_device).requires_grad_(True) for t in (q, k, v)]
    got = torch.autograd.grad(omni_attention(*leaves, m), leaves, dout.to(gpu_device))
    allow = (torch.arange(S).view(1, 1, S) < prefix.unsqueeze(-1)).unsqueeze(1).expand(B, H, S, S)
    check_grads(got, attention_dense_grads(q, k, v, allow, dout), torch.float16, f"H={H} S={S}")


@pytest.mark.parametrize("D,B,H,S,copies,QB", [
    (128, 1, 2, 1160, 16, 128), (128, 1, 2, 1610, 12, 128), (128, 1, 1, 2700, 16, 128), (128, 3, 1, 1630, 8, 128),
    (64, 2, 1, 1500, 16, 128), (64, 1, 1, 4400, 16, 128), (32, 2, 1, 1300, 24, 128), (32, 1, 1, 2950, 32, 128),
    (128, 1, 2, 1170, 16, 64), (128, 2, 1, 1500, 12, 64), (64, 2, 1, 1500, 12, 64), (32, 1, 2, 1900, 16, 64),
    (32, 2, 1, 1300, 20, 128), (64, 1, 1, 1300, 37, 64)])
def test_lengths_that_end_inside_a_block(D, B, H, S, copies, QB, gpu_device):
    """Launches that are split because of such a length: 64- and 128-row groups, dQ in 64-row groups at head_dim 32 and 64
    (the test of the rules holds which is which).
    The slabs of a batch element are repeated; the first ones against the oracle, the copies bit for bit."""
    from test_gpu_backward import check_grads, run_fwd_bwd
    from oracle.dense_oracle import attention_dense_grads
    gen = torch.Generator().manual_seed(D + S)
    KB = QB
    n = -(-S // QB) * QB
    q, k, v, dout = (torch.randn(B, H, n, D, generator=gen).to(torch.bfloat16) for _ in range(4))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, B, H, n // QB, n // KB, QB, KB, p_empty=0.5, shuffle=True)
    many = lambda t: t.to(gpu_device).repeat(1, copies, *[1] * (t.dim() - 2)).contiguous()
    got = run_fwd_bwd(*(many(t) for t in (q, k, v, dout)), many(nb), many(idx), many(tys), QB, KB, S, many(pidx), pm,
                      device=gpu_device, softcap=0.0, packed=True)
    for t in got:
        assert torch.equal(t, t[:, :H].repeat(1, copies, *[1] * (t.dim() - 2)))
        assert t.dim() < 4 or (t[:, :, S:] == 0).all()
    dq, dk, dv, o, lse = (t[:, :H] for t in got[:5])
    dense = dense_mask_from_blocks(nb, idx, tys, QB, KB, n, n, pidx, pm, seqlen_orig=S)
    ro, rl = attention_dense_fp32(q, k, v, dense)
    compare_with_oracle(o, lse, ro, rl, torch.bfloat16, f"S={S}")
    check_grads((dq, dk, dv), attention_dense_grads(q, k, v, dense, dout), torch.bfloat16, f"S={S}")
