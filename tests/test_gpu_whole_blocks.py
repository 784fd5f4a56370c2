"""Every instance of the whole-block kernels -- forward, dQ, dK/dV, plain and soft-capped -- on random metadata.
Launches of few rows take the split walks (csrc/omni_attn_split_rules.hpp; tests/test_gpu_split_walk.py), so the
slabs of a small problem are repeated until the launch has more than 2048 32-row tiles: the first copy is
compared with the oracle, the others with the first, bit for bit."""
import pytest
import torch

import omni_attn_capi
from helpers import TOL_LSE, random_block_metadata
from oracle.dense_oracle import attention_dense_fp32, attention_dense_grads, dense_mask_from_blocks
from test_gpu_backward import check_grads, run_fwd_bwd

pytestmark = pytest.mark.gpu

COPIES = 33


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("QB,KB", [(128, 128), (128, 64), (64, 128), (64, 64)])
def test_whole_block_walks(dtype, D, QB, KB, gpu_device):
    """Every slot kind, indices beyond either end, a sequence that ends inside a block with NaN behind it, PARTIAL
    tiles as bytes and as bits, with and without a soft cap.  The output is within its two roundings, of the
    weights and of the result: u (sum p |v| + |o|), u = 2^-8 for bf16 and 2^-11 for fp16 (2 % more, and 1e-6, for
    sums in fp32)."""
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    gen = torch.Generator().manual_seed(9000 + 10 * D + QB + KB // 64)
    B, H, S = 2, 2, 512
    assert B * H * COPIES * S // 32 > 2048
    q, k, v, dout = (torch.randn(B, H, S, D, generator=gen).to(dtype) for _ in range(4))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, B, H, S // QB, S // KB, QB, KB, shuffle=True)
    listed = torch.arange(idx.shape[-1]) < nb.unsqueeze(-1)
    wild = idx.clone()  # clamped to the first and the last block
    wild[listed & (idx == 0)] = -7
    wild[listed & (idx == S // KB - 1)] = 1000
    many = lambda t: t.to(gpu_device).repeat(1, COPIES, *[1] * (t.dim() - 2)).contiguous()
    for seqlen in (S, S - 45):
        operands = [t.clone() for t in (q, k, v, dout)]
        for t in operands:
            t[:, :, seqlen:] = float("nan")
        dense = dense_mask_from_blocks(nb, idx, tys, QB, KB, S, S, pidx, pm, seqlen_orig=seqlen)
        zeroed = [torch.where(torch.isnan(t), torch.zeros_like(t), t) for t in operands]
        args = ([many(t) for t in operands], [many(t) for t in (nb, wild, tys)], many(pidx), pm)
        for softcap in (0.0, 2.0):
            what = f"seqlen={seqlen} softcap={softcap}"
            got = [run_fwd_bwd(*args[0], *args[1], QB, KB, seqlen, args[2], pm, device=gpu_device, softcap=softcap,
                               packed=packed) for packed in (False, True)]
            for bytes_, bits in zip(*got):
                assert torch.equal(bytes_, bits), what
            first = []
            for t in got[0]:
                copies = t.view(B, COPIES, H, *t.shape[2:])
                assert torch.equal(copies, copies[:, :1].expand_as(copies)), what
                first.append(copies[:, 0])
            ro, rl = attention_dense_fp32(*zeroed[:3], dense, softcap=softcap)
            mean_abs, _ = attention_dense_fp32(zeroed[0], zeroed[1], zeroed[2].float().abs(), dense, softcap=softcap)
            o, lse = first[3].float().cpu(), first[4].cpu()
            assert bool(((o - ro).abs() <= unit * (mean_abs + ro.abs()) * 1.02 + 1e-6).all()), what
            assert torch.equal(torch.isinf(lse), torch.isinf(rl)) and not torch.isnan(lse).any(), what
            assert (lse - rl)[~torch.isinf(rl)].abs().max().item() <= TOL_LSE, what
            check_grads(first[:3], attention_dense_grads(*zeroed[:3], dense, zeroed[3], softcap=softcap), dtype, what)
            for t in first[:4]:
                assert (t[:, :, seqlen:] == 0).all(), what


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("gain", [4.0, 12.0])
def test_reference_points_that_move_often(dtype, gain, D, gpu_device):
    """Scores whose running maximum keeps jumping by far more than the slack of the reference point: the rescale
    of O in whole-block walks.  Bars as in test_gpu_parity's test of such scores, whose three slabs are split: rows return
    single V entries, so an ulp of the value more than usual, and the logsumexp relative to its size."""
    from helpers import TOL_O
    gen = torch.Generator().manual_seed(int(gain) * 7 + D)
    H, S, QB, KB, copies = 3, 1536, 128, 128, 15
    assert H * copies * S // 32 > 2048
    q = (torch.randn(1, H, S, D, generator=gen) * gain).to(dtype)
    k, v = (torch.randn(1, H, S, D, generator=gen).to(dtype) for _ in range(2))
    k[:, 1] -= 0.5 * q[:, 1].float().mean(1, keepdim=True).to(dtype)  # head 1: mostly negative scores
    nb, idx, tys, pidx, pm = random_block_metadata(gen, 1, H, S // QB, S // KB, QB, KB, p_empty=0.2, shuffle=True)
    many = lambda t: t.to(gpu_device).repeat(1, copies, *[1] * (t.dim() - 2)).contiguous()
    qd = many(q)
    o = torch.full_like(qd, float("nan"))
    lse = torch.full(qd.shape[:3], float("nan"), dtype=torch.float32, device=gpu_device)
    omni_attn_capi.fwd(qd, many(k), many(v), o, lse, many(nb), many(idx), many(tys), QB, KB, S, many(pidx),
                       pm.to(gpu_device))
    torch.cuda.synchronize()
    for t in (o, lse):
        assert torch.equal(t, t[:, :H].repeat(1, copies, *[1] * (t.dim() - 2)))
    wo, wl = attention_dense_fp32(q, k, v, dense_mask_from_blocks(nb, idx, tys, QB, KB, S, S, pidx, pm))
    o32, l32 = o[:, :H].float().cpu(), lse[:, :H].cpu()
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert ((o32 - wo).abs() - ulp * wo.abs()).max().item() <= TOL_O[dtype]
    empty = torch.isinf(wl)
    assert torch.equal(torch.isinf(l32), empty) and (o32[empty] == 0).all()
    assert ((l32 - wl)[~empty].abs() / wl[~empty].abs().clamp(min=1.0)).max().item() <= TOL_LSE


@pytest.mark.parametrize("S,QB,KB,D", [(500, 128, 128, 128), (450, 128, 64, 64), (500, 64, 128, 32), (390, 64, 64, 128)])
def test_operands_are_read_where_they_lie(S, QB, KB, D, gpu_device):
    """A projection's [B, S, H, D] result against contiguous operands padded by hand: the same bits.  Rows behind
    the operands' own are NaN."""
    import omni_attn_torch as oat
    gen = torch.Generator().manual_seed(S + D)
    B, H = 3, 52
    n = -(-S // QB) * QB
    assert B * H * n // 32 > 2048
    spans = torch.tensor([[[1, 100, 150]], [[1, 7, 60]], [[1, 200, 180]]])
    mask = oat.create_omni_block_mask_from_modality_positions(spans, B, H, n, n, QB, KB, device=gpu_device)
    big = [torch.randn(B, S + 2, H, D, generator=gen).to(torch.bfloat16).to(gpu_device) for _ in range(4)]
    for t in big:
        t[:, S:] = float("nan")
    q, k, v, dout = (t[:, :S].transpose(1, 2) for t in big)
    pads = [torch.nn.functional.pad(t, (0, 0, 0, n - S)).contiguous() for t in (q, k, v, dout)]
    meta = (mask.kv_num_blocks, mask.kv_indices, mask.block_mask_types, QB, KB, S, mask.partial_block_mask_indices,
            mask.partial_block_masks)
    ro, dq, dk, dv = (torch.empty_like(pads[0]) for _ in range(4))
    rl = torch.empty(B, H, n, dtype=torch.float32, device=gpu_device)
    omni_attn_capi.fwd(*pads[:3], ro, rl, *meta)
    omni_attn_capi.bwd(*pads[:3], ro, pads[3], rl, dq, dk, dv, *meta)
    q, k, v = (t.requires_grad_(True) for t in (q, k, v))
    out = oat.omni_attention(q, k, v, mask)
    grads = torch.autograd.grad(out, (q, k, v), dout)
    assert torch.isfinite(out).all() and torch.equal(out, ro[:, :, :S])
    for name, a, b in zip(("dq", "dk", "dv"), grads, (dq, dk, dv)):
        assert torch.equal(a, b[:, :, :S]), name


WHOLE_64_ROW_COPIES = (60, 140)  # of two slabs of 256 rows: 960 and 2240 row tiles


@pytest.mark.parametrize("KB", [64, 128])
@pytest.mark.parametrize("seqlen", [129, 159, 160, 161, 191, 192, 193, 255])
def test_gradients_of_64_row_blocks_at_the_edges_of_their_steps(seqlen, KB, gpu_device):
    """64-row query blocks at head_dim 128 walk their lists by 32 keys in large launches and by 64 in others: sequences that
    end around a step and around a block, every slot kind, NaN behind the sequence.  Two launches, on either side of the
    lines of bwd_dq_step (csrc/omni_attn_split_rules.hpp; tests/test_split_rules.py) and not split."""
    gen = torch.Generator().manual_seed(seqlen + KB)
    H, S, D, QB = 2, 256, 128, 64
    q, k, v, dout = (torch.randn(1, H, S, D, generator=gen).to(torch.bfloat16) for _ in range(4))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, 1, H, S // QB, S // KB, QB, KB, p_empty=0.2, shuffle=True)
    many = lambda t: t.to(gpu_device).repeat(1, copies, *[1] * (t.dim() - 2)).contiguous()
    operands = [t.clone() for t in (q, k, v, dout)]
    for t in operands:
        t[:, :, seqlen:] = float("nan")
    dense = dense_mask_from_blocks(nb, idx, tys, QB, KB, S, S, pidx, pm, seqlen_orig=seqlen)
    zeroed = [torch.where(torch.isnan(t), torch.zeros_like(t), t) for t in operands]
    wanted = attention_dense_grads(*zeroed[:3], dense, zeroed[3])
    for copies in WHOLE_64_ROW_COPIES:
        got = run_fwd_bwd(*(many(t) for t in operands), many(nb), many(idx), many(tys), QB, KB, seqlen, many(pidx), pm,
                          device=gpu_device, softcap=0.0, packed=seqlen % 2 == 0)
        for t in got:
            assert torch.equal(t, t[:, :H].repeat(1, copies, *[1] * (t.dim() - 2)))
        check_grads([t[:, :H] for t in got[:3]], wanted, torch.bfloat16, f"seqlen={seqlen}, copies={copies}")
