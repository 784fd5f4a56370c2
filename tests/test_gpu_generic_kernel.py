"""The scalar-semantics forward for shapes without an MFMA instance (any block size, head_dim up
to 256, as the reference's omni_attn_simple_kernel, attn_naive.cu:189-190 and :305-408), against
both CPU oracles.  Bars: max-abs 2e-3 (fp16) / 1e-2 (bf16) on the output, 1e-3 on the logsumexp."""
import pytest
import torch

import omni_attn_capi
from helpers import compare_with_oracle, random_block_metadata
from oracle.block_walk import attention_block_walk
from oracle.dense_oracle import attention_dense_fp32, dense_mask_from_blocks

pytestmark = pytest.mark.gpu


def run_generic(q, k, v, nb, idx, tys, QB, KB, seqlen, pidx, pm, device, softcap=0.0):
    dev = lambda t: None if t is None else t.to(device).contiguous()
    qd = dev(q)
    o = torch.full_like(qd, float("nan"))
    lse = torch.full(qd.shape[:3], float("nan"), dtype=torch.float32, device=device)
    omni_attn_capi.fwd(qd, dev(k), dev(v), o, lse, dev(nb), dev(idx), dev(tys), QB, KB, seqlen, dev(pidx), dev(pm),
                       generic=True, softcap=softcap)
    torch.cuda.synchronize()
    return o, lse


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("QB,KB,D", [(32, 32, 96), (16, 48, 256), (128, 64, 128), (100, 20, 40), (64, 256, 8)])
def test_generic_kernel_any_block_size_and_head_dim(dtype, QB, KB, D, gpu_device):
    gen = torch.Generator().manual_seed(QB * 1000 + KB * 10 + D)
    B, H = 1, 2
    S = 3 * max(QB, KB) if max(QB, KB) % min(QB, KB) == 0 else QB * KB // 10  # a multiple of both
    assert S % QB == 0 and S % KB == 0
    q, k, v = (torch.randn(B, H, S, D, generator=gen).to(dtype) for _ in range(3))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, B, H, S // QB, S // KB, QB, KB, p_empty=0.2, shuffle=True)
    for seqlen in (S, S - 7):
        o, lse = run_generic(q, k, v, nb, idx, tys, QB, KB, seqlen, pidx, pm, gpu_device)
        dense = dense_mask_from_blocks(nb, idx, tys, QB, KB, S, S, pidx, pm, seqlen_orig=seqlen)
        ro, rl = attention_dense_fp32(q, k, v, dense)
        compare_with_oracle(o, lse, ro, rl, dtype, f"generic vs dense oracle, seqlen={seqlen}")
        wo, wl = attention_block_walk(q, k, v, nb, idx, tys, QB, KB, seqlen, pidx, pm)
        compare_with_oracle(o, lse, wo, wl, dtype, f"generic vs block walk, seqlen={seqlen}")


def test_generic_kernel_agrees_with_the_mfma_kernel_where_both_exist(gpu_device):
    gen = torch.Generator().manual_seed(5)
    B, H, S, D, QB, KB = 1, 2, 512, 64, 128, 64
    q, k, v = (torch.randn(B, H, S, D, generator=gen).to(torch.float16) for _ in range(3))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, B, H, S // QB, S // KB, QB, KB, shuffle=True)
    og, lg = run_generic(q, k, v, nb, idx, tys, QB, KB, S, pidx, pm, gpu_device, softcap=3.0)
    dev = lambda t: t.to(gpu_device).contiguous()
    om = torch.empty_like(og)
    lm = torch.empty_like(lg)
    omni_attn_capi.fwd(dev(q), dev(k), dev(v), om, lm, dev(nb), dev(idx), dev(tys), QB, KB, S, dev(pidx), dev(pm),
                       softcap=3.0)
    torch.cuda.synchronize()
    assert (og.float() - om.float()).abs().max().item() <= 2e-3
    live = ~torch.isinf(lm)
    assert torch.equal(torch.isinf(lg), torch.isinf(lm)) and (lg[live] - lm[live]).abs().max().item() <= 1e-3


def test_simple_wrapper_takes_shapes_the_other_wrappers_refuse(gpu_device):
    import omni_attn_torch as oat
    from omni_attn_torch import create_causal_omni_block_mask
    gen = torch.Generator().manual_seed(6)
    S, D, blk = 192, 80, 32
    q, k, v = (torch.randn(1, 2, S, D, generator=gen).to(torch.float16).to(gpu_device) for _ in range(3))
    mask = create_causal_omni_block_mask(1, 2, S, S, blk, blk, device=gpu_device)
    out = oat.omni_attention_simple(q, k, v, mask)
    ref, _ = attention_dense_fp32(q.cpu(), k.cpu(), v.cpu(), torch.tril(torch.ones(S, S, dtype=torch.bool)))
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-3
    with pytest.raises(ValueError, match="head_dim"):
        oat.omni_attention_shared_kv_swizzle(q, k, v, mask)


@pytest.mark.parametrize("QB,KB,D", [(16, 16, 5), (48, 48, 8), (33, 7, 13), (32, 32, 31), (40, 40, 33), (64, 48, 100),
                                     (16, 32, 129), (128, 128, 161), (32, 64, 224), (48, 16, 250), (16, 16, 193),
                                     (32, 64, 217)])
def test_generic_kernel_edges_of_tiles_and_chunks(QB, KB, D, gpu_device):
    """Head dimensions around the 8-column chunks and 32-column tiles, key blocks that do not fill or
    that straddle a 32-key step, query blocks of a fraction of a 32-row tile.  Tighter than the bars:
    the weights are not rounded before the second product, so the error is the rounding of the
    result (half an ulp of |o| < 4: 2^-10) and fp32 sums of at most 600 terms."""
    gen = torch.Generator().manual_seed(QB * 1000 + KB * 10 + D)
    B, H = 2, 1
    S = 2 * QB * KB if QB * KB < 300 else 3 * max(QB, KB)
    S = -(-S // QB) * QB
    q, k, v = (torch.randn(B, H, S, D, generator=gen).to(torch.float16) for _ in range(3))
    Tk = -(-S // KB)
    nb, idx, tys, pidx, pm = random_block_metadata(gen, B, H, S // QB, Tk, QB, KB, p_empty=0.2, shuffle=True)
    for seqlen in (S, S - 5):
        o, lse = run_generic(q, k, v, nb, idx, tys, QB, KB, seqlen, pidx, pm, gpu_device)
        wo, wl = attention_block_walk(q, k, v, nb, idx, tys, QB, KB, seqlen, pidx, pm)
        assert torch.equal(torch.isinf(lse.cpu()), torch.isinf(wl))
        assert (o.float().cpu() - wo).abs().max().item() <= 2.0 ** -10, (QB, KB, D, seqlen)
        live = ~torch.isinf(wl)
        assert (lse.cpu()[live] - wl[live]).abs().max().item() <= 2e-5


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("QB,KB,D,S", [(16, 16, 5, 80), (32, 32, 64, 160), (48, 48, 96, 144), (128, 128, 161, 256),
                                       (64, 32, 256, 192), (32, 32, 250, 96), (24, 24, 40, 120), (40, 40, 256, 200),
                                       (24, 24, 144, 144), (48, 48, 168, 144), (16, 16, 136, 80), (64, 64, 208, 576),
                                       (48, 48, 131, 336), (20, 20, 194, 100)])
def test_values_of_keys_that_are_not_allowed_never_reach_a_row(dtype, QB, KB, D, S, gpu_device):
    """Infinities, NaNs and large values in V: rows that may not attend to those keys get what
    they get without them, rows that may get the infinity, the NaN or the (finite) average.  A query row
    of NaNs has no score: zeros, and no logsumexp."""
    from omni_attn_torch import create_causal_omni_block_mask
    gen = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(1, 1, S, D, generator=gen).to(dtype) for _ in range(3))
    m = create_causal_omni_block_mask(1, 1, S, S, QB, KB, device="cpu")
    args = (m.kv_num_blocks, m.kv_indices, m.block_mask_types, QB, KB, S, None, None, gpu_device)
    clean, lse0 = run_generic(q, k, v, *args)
    bad = v.clone()
    at_inf, at_nan = S // 2 + 3, S - 6
    bad[..., at_inf, 0] = float("inf")
    bad[..., at_nan, 2] = float("nan")
    o, lse = run_generic(q, k, bad, *args)
    assert (lse - lse0).abs().max().item() <= 2e-5
    # (the second walk sums in another order: an ulp of |o| < 4 apart at the most, and half of one is usual)
    ulp = 2.0 ** -9 if dtype == torch.float16 else 2.0 ** -6
    assert (o - clean).float()[..., :at_inf, :].abs().max().item() <= ulp
    assert bool((o[..., at_inf:, 0] == float("inf")).all()) and bool(o[..., at_nan:, 2].isnan().all())
    rest = (o - clean).float()[..., at_inf:, :]
    rest[..., 0] = 0
    rest[..., at_nan - at_inf:, 2] = 0
    assert rest.abs().max().item() <= ulp
    # a large value as every V is its own average (1e-2: rounding of the result and sums in fp32)
    large = 60000.0 if dtype == torch.float16 else 2.0 ** 116
    o, _ = run_generic(q, k, torch.full_like(v, large), *args)
    assert bool(((o.float() / large - 1).abs() <= 1e-2).all())
    nan_row = q.clone()
    nan_row[..., 7, :] = float("nan")
    o, lse = run_generic(nan_row, k, v, *args)
    assert bool((o[..., 7, :] == 0).all()) and bool(torch.isneginf(lse[..., 7]).all())
    keep = torch.arange(S) != 7
    assert (o - clean).float()[..., keep, :].abs().max().item() <= ulp


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("D", [5, 96, 250, 256])
def test_small_weights_reach_the_result(dtype, D, gpu_device):
    """A row whose largest weight meets a V row of zeros: the result is the sum of weights of 2^-8 down to
    2^-44 of it times large values.  Weights are fp32 numbers and none is dropped, so the error is the
    rounding of the result (half an ulp: 2^-11 or 2^-8 of it, 2^-25 where it is an fp16 subnormal) and that of
    exponents below 64 in fp32 (64 * 2^-23 * ln 2 = 2^-17.5, of the score and of its maximum)."""
    exps = torch.tensor([8.0, 15, 20, 26, 31, 36, 40, 44])  # of key block i, which query block i sees; its first key: 0
    n, blk = exps.numel(), 32
    S = n * blk
    want = -exps.repeat_interleave(blk)
    want[::blk] = 0
    want *= D ** 0.5 / 1.4426950408889634
    q, k, v = torch.zeros(1, 1, S, D), torch.zeros(1, 1, S, D), torch.full((1, 1, S, D), 60000.0)
    v[:, :, ::blk] = 0
    q[..., 0] = 1.0
    q[..., 1] = 2.0 ** -8  # (a score is the sum of two rounded parts)
    k[0, 0, :, 0] = want.to(dtype).float()
    k[0, 0, :, 1] = (want - k[0, 0, :, 0]) * 2.0 ** 8
    q, k, v = (t.to(dtype) for t in (q, k, v))
    nb = torch.ones(1, 1, n, dtype=torch.int32)
    idx = torch.arange(n, dtype=torch.int32).view(1, 1, n, 1)
    at = torch.arange(S)
    block = at // blk
    scores = q.double() @ k.double().transpose(2, 3).contiguous() / D ** 0.5
    ulp, least = (2.0 ** -11, 2.0 ** -25) if dtype == torch.float16 else (2.0 ** -8, 0.0)
    for kind, allow in ((2, block == block.unsqueeze(1)), (1, (block == block.unsqueeze(1)) & (at <= at.unsqueeze(1)))):
        o, _ = run_generic(q, k, v, nb, idx, torch.full_like(idx, kind), blk, blk, S, None, None, gpu_device)
        ref = torch.softmax(scores.masked_fill(~allow, float("-inf")), -1) @ v.double()
        assert bool(((o.double().cpu() - ref).abs() <= ref * (ulp + 2.0 ** -16) + least).all()), kind


@pytest.mark.parametrize("blk", [32, 64, 48], ids=lambda b: f"{b}x{b}")  # 48: steps that cross blocks
@pytest.mark.parametrize("D", [8, 40, 96, 136, 168, 256])
def test_rows_of_keys_and_values_lie_differently(D, blk, gpu_device):
    """Rows read straight to LDS keep an offset per lane for K and for V: another distance between rows of one, the
    other, or both gives the same bits."""
    import omni_attn_torch as oat
    from omni_attn_torch import create_causal_omni_block_mask
    gen = torch.Generator().manual_seed(D + blk)
    S = 3 * 64 - 5  # (the last block is ragged)
    q, k, v = (torch.randn(1, 2, S, D, generator=gen).to(torch.float16).to(gpu_device) for _ in range(3))
    mask = create_causal_omni_block_mask(1, 2, S, S, blk, blk, device=gpu_device)
    rows_apart = lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)
    out = oat.omni_attention_simple(q, k, v, mask)
    ref, _ = attention_dense_fp32(q.cpu(), k.cpu(), v.cpu(), torch.tril(torch.ones(S, S, dtype=torch.bool)))
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-3
    for kk, vv in ((rows_apart(k), v), (k, rows_apart(v)), (rows_apart(k), rows_apart(v))):
        assert torch.equal(oat.omni_attention_simple(q, kk, vv, mask), out)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("QB,KB,D,S", [(16, 16, 136, 69 * 16), (48, 48, 168, 70 * 48), (32, 80, 200, 480), (32, 32, 256, 66 * 32),
                                       (64, 112, 224, 448), (16, 144, 64, 96), (32, 256, 160, 96), (24, 24, 144, 72 * 24),
                                       (40, 40, 256, 200), (16, 16, 165, 69 * 16), (64, 32, 131, 192), (20, 36, 250, 180)])
def test_steps_in_halves_and_tiles_that_keys_and_values_take_in_turn(dtype, QB, KB, D, S, gpu_device):
    """Steps whose halves lie in one block, in two, or in two chunks of a list (more than 64 slots); blocks longer than the
    sequence; eight waves with one tile each, whose rows go to LDS directly, key by key or through registers; peaked rows
    (the rests of fp16 weights).  The result's error is its rounding (half an ulp of |o| < 4) and fp32 sums."""
    gen = torch.Generator().manual_seed(QB * 1000 + KB * 10 + D)
    q, k, v = (torch.randn(1, 1, S, D, generator=gen).to(dtype) for _ in range(3))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, 1, 1, -(-S // QB), -(-S // KB), QB, KB, p_empty=0.1, shuffle=True)
    for seqlen, query in ((S, q), (S - 11, 3 * q)):
        o, lse = run_generic(query, k, v, nb, idx, tys, QB, KB, seqlen, pidx, pm, gpu_device)
        wo, wl = attention_block_walk(query, k, v, nb, idx, tys, QB, KB, seqlen, pidx, pm)
        assert torch.equal(torch.isinf(lse.cpu()), torch.isinf(wl))
        ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
        # (exponents of up to 128 in fp32, in either sum: 2 * 2^-17 of a weight, times |v| < 5)
        assert (o.float().cpu() - wo).abs().max().item() <= ulp + 2.0 ** -13, (QB, KB, D, seqlen)
        live = ~torch.isinf(wl)
        assert (lse.cpu()[live] - wl[live]).abs().max().item() <= 5e-5


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("blk,D", [(32, 40), (64, 96), (32, 120), (64, 136), (32, 168), (64, 208), (32, 256), (48, 40), (16, 208)])
def test_nothing_behind_the_sequence_is_read(dtype, blk, D, gpu_device):
    """Sequences that end in the first or the second half of a step, or between them: NaNs behind them change no bit."""
    from omni_attn_torch import create_causal_omni_block_mask
    gen = torch.Generator().manual_seed(D + blk)
    S = 4 * blk
    q, k, v = (torch.randn(1, 2, S, D, generator=gen).to(dtype) for _ in range(3))
    m = create_causal_omni_block_mask(1, 2, S, S, blk, blk, device="cpu")
    for seqlen in (S, S - 1, S - blk // 2, S - 16, S - 17, 16, 1):
        args = (m.kv_num_blocks, m.kv_indices, m.block_mask_types, blk, blk, seqlen, None, None, gpu_device)
        behind = [t.clone() for t in (k, v)]
        zeros = [t.clone() for t in (k, v)]
        for t in behind:
            t[:, :, seqlen:] = float("nan")
        for t in zeros:
            t[:, :, seqlen:] = 0
        o, lse = run_generic(q, *behind, *args)
        wo, wl = run_generic(q, *zeros, *args)
        assert torch.equal(o, wo) and torch.equal(lse, wl), seqlen
        ref, _ = attention_dense_fp32(q[:, :, :seqlen], k[:, :, :seqlen], v[:, :, :seqlen],
                                      torch.tril(torch.ones(seqlen, seqlen, dtype=torch.bool)))
        assert (o[:, :, :seqlen].float().cpu() - ref).abs().max().item() <= (2e-3 if dtype == torch.float16 else 1e-2), seqlen


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("blk,D", [(16, 40), (48, 96), (80, 120), (16, 136), (48, 208), (16, 256), (32, 96), (32, 208), (24, 96),
                                   (24, 208)])
def test_keys_that_no_slot_names_are_not_read(dtype, blk, D, gpu_device):
    """Lists of an odd number of slots, MASKED ones among them and block 0 in none but those: infinities and NaNs in block 0
    and behind the sequence change no bit (a wave that meets one adds up its list again, in another order)."""
    gen = torch.Generator().manual_seed(D + blk)
    T, H = 9, 2
    S = T * blk
    q, k, v = (torch.randn(1, H, S, D, generator=gen).to(dtype) for _ in range(3))
    nb = torch.full((1, H, T), 7, dtype=torch.int32)
    idx = torch.zeros(1, H, T, T, dtype=torch.int32)
    idx[..., :7] = torch.tensor([1, 0, 3, 4, 5, 6, 8])
    tys = torch.zeros_like(idx)
    tys[..., :7] = torch.tensor([2, 0, 2, 2, 0, 2, 2])
    for seqlen in (S, S - 9):
        args = (nb, idx, tys, blk, blk, seqlen, None, None, gpu_device)
        clean, lse0 = run_generic(q, k, v, *args)
        bad = v.clone()
        bad[:, :, 0:blk, ::3] = float("inf")
        bad[:, :, 0:blk, 1::3] = float("nan")
        bad[:, :, seqlen:] = float("nan")
        o, lse = run_generic(q, k, bad, *args)
        assert torch.isfinite(o).all() and torch.equal(o, clean) and torch.equal(lse, lse0), seqlen


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("blk,D", [(32, 131), (32, 250), (16, 165), (48, 225), (64, 194), (20, 161)])
def test_lists_of_as_many_steps_as_half_of_the_waves(dtype, blk, D, gpu_device):
    """Rows at any alignment beyond 128 columns: up to 128 listed keys leave half of the waves out of the sum at the end.
    Query block i lists i blocks, so that lists end before, at and behind that line.  The result's error is its rounding
    (half an ulp of |o| < 4) and fp32 sums."""
    gen = torch.Generator().manual_seed(D)
    T = 256 // blk
    S = T * blk
    q, k, v = (torch.randn(1, 1, S, D, generator=gen).to(dtype) for _ in range(3))
    nb = torch.arange(T, dtype=torch.int32).view(1, 1, T)
    idx = torch.arange(T, dtype=torch.int32).repeat(T, 1).view(1, 1, T, T)
    tys = torch.full_like(idx, 2)
    o, lse = run_generic(q, k, v, nb, idx, tys, blk, blk, S, None, None, gpu_device)
    wo, wl = attention_block_walk(q, k, v, nb, idx, tys, blk, blk, S, None, None)
    assert torch.equal(torch.isinf(lse.cpu()), torch.isinf(wl))
    assert (o.float().cpu() - wo).abs().max().item() <= (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7) + 2.0 ** -16
    assert (lse.cpu()[..., blk:] - wl[..., blk:]).abs().max().item() <= 2e-5


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("QB,KB,D", [(32, 32, 96), (48, 48, 120), (24, 24, 40), (32, 32, 101), (32, 32, 136), (64, 32, 256), (48, 48, 168),
                                     (16, 16, 208), (40, 40, 256), (24, 24, 144), (32, 32, 131), (48, 48, 165), (64, 64, 250)])
def test_soft_capped_scores_in_every_form(dtype, QB, KB, D, gpu_device):
    """Rows straight to LDS in steps of one block, of halves and by key, and rows at any alignment, up to 128 columns and
    beyond, with scores that reach the cap: the result's error is its rounding and the hyperbolic tangent's."""
    gen = torch.Generator().manual_seed(QB + D)
    S = 7 * max(QB, KB)
    q, k, v = (torch.randn(1, 2, S, D, generator=gen).to(dtype) for _ in range(3))
    nb, idx, tys, pidx, pm = random_block_metadata(gen, 1, 2, S // QB, S // KB, QB, KB, p_empty=0.2, shuffle=True)
    for seqlen in (S, S - 13):
        o, lse = run_generic(q, k, v, nb, idx, tys, QB, KB, seqlen, pidx, pm, gpu_device, softcap=1.5)
        dense = dense_mask_from_blocks(nb, idx, tys, QB, KB, S, S, pidx, pm, seqlen_orig=seqlen)
        ro, rl = attention_dense_fp32(q, k, v, dense, softcap=1.5)
        compare_with_oracle(o, lse, ro, rl, dtype, f"soft-capped, seqlen={seqlen}")
