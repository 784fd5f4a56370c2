"""Performance cases of the block-sparse attention operator: what a program that uses it has it do.

Four kinds of work, each through the public entry points:

  forward   an attention layer without gradients (prefill, evaluation, sampling): the operator
            wrappers of omni_attn_torch on q, k, v and a block mask that the program made before
  train     the differentiable operator, forward and backward, as one attention layer of a
            training step runs it
  simple    the scalar-semantics operator for block sizes and head dimensions outside the
            matrix-core operators' {64, 128} and {32, 64, 128}
  mask      the block mask of a batch from its modality positions: every batch of a mixed
            text / image model has other positions, so its mask is made once per step

A case is a dict of plain values:
  B, H, S, D     batch, heads, tokens (any number: not only multiples of a block), head dimension
  dtype          "float16" or "bfloat16"
  QB, KB         query / key block size of the mask
  layout         "causal"; "interleaved" (text and block-aligned image spans in turn);
                 "unaligned" (image spans of 200 .. 1100 tokens anywhere); "images" (spans of 1024
                 tokens anywhere); "mixed" (another of causal / full / interleaved per batch element)
  layout_seed    which layout of that kind; values of q, k, v come from prepare()'s seed
  rows           "bhsd": q, k, v contiguous; "bshd": the [B, S, H, D] result of a projection, seen
                 as [B, H, S, D], the way a model's attention layer hands them over
  tiles          PARTIAL tiles as "bytes" (the reference's format) or "bits" (packed once per mask)
  lse            the row logsumexp is asked for as well
  softcap        cap of the scores, 0 = none
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "omni-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import omni_attn_torch as oat  # noqa: E402
import transfusion_shim as shim  # noqa: E402


def _case(op, B, H, S, D, dtype, QB=128, KB=128, layout="causal", layout_seed=0, rows="bhsd", tiles="bytes",
          lse=False, softcap=0.0):
    return {"op": op, "B": B, "H": H, "S": S, "D": D, "dtype": dtype, "QB": QB, "KB": KB, "layout": layout,
            "layout_seed": layout_seed, "rows": rows, "tiles": tiles, "lse": lse, "softcap": softcap}


def listed():
    named = [
        # one layer of a small text model, a short prompt: launch latency and the host path
        ("forward_causal_512", _case("forward", 1, 8, 512, 64, "float16")),
        # the block size and shape of the operator's original test grid
        ("forward_blocks64_2048", _case("forward", 1, 8, 2048, 64, "float16", 64, 64, "interleaved")),
        # a prompt of arbitrary length with images anywhere in it, straight from a model's projections
        ("forward_ragged_1237", _case("forward", 2, 16, 1237, 128, "bfloat16", layout="unaligned", rows="bshd",
                                      tiles="bits")),
        # the flagship: interleaved text and images
        ("forward_interleaved_4096", _case("forward", 2, 32, 4096, 128, "bfloat16", layout="interleaved")),
        # images at unaligned offsets: many PARTIAL tiles, unequal blocks, logsumexp for a later merge
        ("forward_unaligned_8192", _case("forward", 1, 16, 8192, 128, "bfloat16", 128, 64, "unaligned", lse=True)),
        # a long multimodal document
        ("forward_long_16384", _case("forward", 1, 32, 16384, 128, "bfloat16", layout="images")),
        # a batch of requests with different masks, half the head dimension
        ("forward_batched_8192", _case("forward", 8, 16, 8192, 64, "float16", layout="mixed")),
        # a layer of a small mixed-modality model in training: ragged length, soft-capped scores
        ("train_softcap_1157", _case("train", 4, 8, 1157, 64, "bfloat16", layout="unaligned", rows="bshd",
                                     tiles="bits", softcap=50.0)),
        # a text model's training step at head_dim 64
        ("train_causal_2048", _case("train", 4, 16, 2048, 64, "float16")),
        # the flagship in training
        ("train_interleaved_4096", _case("train", 2, 32, 4096, 128, "bfloat16", layout="interleaved", tiles="bits")),
        # a head dimension and block size that only the scalar-semantics operator takes
        ("simple_d96_2048", _case("simple", 1, 8, 2048, 96, "float16", 32, 32)),
        # the mask of a training batch
        ("mask_8192", _case("mask", 4, 16, 8192, 0, "int32", layout="unaligned", tiles="bits")),
    ]
    return [dict(case, name=name) for name, case in named]


# What a drawn case may cost: the scores B * H * S * S of the largest listed case of its kind
# (times D for the scalar-semantics operator, whose D goes up to 256).
_LIMIT = {"forward": 32 * 16384 ** 2, "train": 64 * 4096 ** 2, "simple": 8 * 2048 ** 2 * 96}


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["forward"] * 6 + ["train"] * 3 + ["simple", "mask"])
    dtype = rng.choice(["float16", "bfloat16"])
    layout = rng.choice(["causal", "interleaved", "unaligned", "unaligned", "images", "mixed"])
    seed = rng.randrange(1 << 20)
    if op == "mask":
        QB, KB = rng.choice([(128, 128), (128, 128), (128, 64), (64, 64)])
        S = _log_uniform(rng, 1024, 64 * min(QB, KB))
        return _case("mask", rng.randint(2, 4), rng.choice([8, 12, 16]), S, 0, "int32", QB, KB,
                     rng.choice(["interleaved", "unaligned", "images"]), seed, tiles="bits")
    if op == "simple":
        D = rng.choice([8 * rng.randint(2, 32), 8 * rng.randint(2, 32), 8 * rng.randint(2, 32), rng.randint(16, 256)])
        blk = rng.choice([16, 32, 32, 48, 64, 128])
        S, B, H = _log_uniform(rng, 64, 2048), rng.choice([1, 1, 2]), rng.choice([2, 4, 8])
        while B * H * S * S * D > _LIMIT[op]:
            S = S * 3 // 4
        return _case(op, B, H, S, D, dtype, blk, blk, rng.choice(["causal", "unaligned"]), seed)
    D = rng.choice([32, 64, 64, 64, 128, 128, 128, 128])
    QB, KB = rng.choice([(128, 128)] * 4 + [(128, 64), (64, 64)])
    S = _log_uniform(rng, 200, 16384 if op == "forward" else 8192)
    if rng.random() < 0.4:
        S = -(-S // 128) * 128
    B, H = rng.choice([1, 1, 2, 4, 8]), rng.choice([4, 8, 12, 16, 32])
    limit = _LIMIT[op] * (0.7 if layout == "mixed" else 1.0)  # a third of a mixed batch attends everything
    while B * H * S * S > limit:
        if B > 1:
            B //= 2
        elif H > 8:
            H = H * 2 // 3
        else:
            S = S * 3 // 4
    softcap = rng.choice([0.0, 0.0, 50.0]) if op == "train" else rng.choice([0.0] * 5 + [50.0])
    return _case(op, B, H, S, D, dtype, QB, KB, layout, seed, rng.choice(["bhsd", "bshd"]),
                 rng.choice(["bytes", "bits"]), lse=op == "forward" and (softcap > 0 or rng.random() < 0.25),
                 softcap=softcap)


# ---- layouts ---------------------------------------------------------------------------------

def _interleaved(rng, S):
    spans, pos = [], 0
    image = min(1024, max(128, S // 4 // 128 * 128))
    while True:
        pos = -(-(pos + rng.randint(128, 512)) // 128) * 128
        if pos + image > S:
            return spans
        spans.append((pos, image))
        pos += image


def _anywhere(rng, S, count, lo, hi):
    lens = [min(rng.randint(lo, hi), max(1, S // 3)) for _ in range(count)]
    while lens and sum(lens) > S - count - 1:
        lens.pop()
    cuts = sorted(rng.randint(1, S - sum(lens)) for _ in lens)
    spans, shift = [], 0
    for cut, n in zip(cuts, lens):
        if cut + shift + n <= S:
            spans.append((cut + shift, n))
        shift += n
    return spans


def _spans(case, seed):
    """Per batch element: (offset, length) of its image spans, or None where everything attends everything."""
    rng, S, kind = random.Random(seed), case["S"], case["layout"]
    per_batch = []
    for b in range(case["B"]):
        k = ("causal", "full", "interleaved")[b % 3] if kind == "mixed" else kind
        if k == "interleaved":
            per_batch.append(_interleaved(rng, S))
        elif k == "unaligned":
            per_batch.append(_anywhere(rng, S, max(1, S // 1024), 200, 1100))
        elif k == "images":
            per_batch.append(_anywhere(rng, S, max(1, S // 2048), 1024, 1024))
        else:
            per_batch.append(None if k == "full" else [])
    return per_batch


def _positions(per_batch):
    """[B, M, 3] rows of (type, offset, length), zero-length rows where an element has fewer spans."""
    M = max([len(s) for s in per_batch if s] + [1])
    rows = [[[1, o, n] for o, n in (s or [])] for s in per_batch]
    return torch.tensor([r + [[0, 0, 0]] * (M - len(r)) for r in rows], dtype=torch.long)


def _batch_positions(case, seed):
    """Modality positions of one training batch.  The spans of a batch element come from the case's
    layout and sit anywhere in the sequence, moved by whole blocks, so that every batch of a case
    has as many PARTIAL tiles (the returned tile store keeps its shape)."""
    slack = case["S"] // 4 // 128
    per_batch = _spans(dict(case, S=case["S"] - 128 * slack), case["layout_seed"])
    moved = []
    for b, spans in enumerate(per_batch):
        shift = 128 * (seed // (slack + 1) ** b % (slack + 1))
        moved.append([(o + shift, n) for o, n in spans])
    return _positions(moved)


def _prefix(case, device):
    """Allowed-prefix length of every row, [B, S]."""
    per_batch = _spans(case, case["layout_seed"])
    prefix = oat.modality_prefix_lengths(_positions(per_batch).to(device), case["S"]).clamp(max=case["S"])
    for b, s in enumerate(per_batch):
        if s is None:
            prefix[b] = case["S"]
    return prefix


def _block_mask(case, device):
    B, H, S, QB, KB = (case[k] for k in ("B", "H", "S", "QB", "KB"))
    if case["layout"] == "causal":
        mask = oat.create_causal_omni_block_mask(B, H, S, S, QB, KB, device=device)
    elif case["layout"] == "mixed":
        mask = oat.create_omni_block_mask_from_prefix_lengths(_prefix(case, device), H, S, S, QB, KB)
    else:
        mp = _positions(_spans(case, case["layout_seed"])).to(device)
        mask = oat.create_omni_block_mask_from_modality_positions(mp, B, H, S, S, QB, KB, device=device)
    return mask.pack_partial_masks() if case["tiles"] == "bits" else mask


# ---- the cases -------------------------------------------------------------------------------

def prepare(case, seed):
    dev = torch.device("cuda")
    if case["op"] == "mask":
        return {"case": case, "positions": _batch_positions(case, seed).to(dev)}
    B, H, S, D = (case[k] for k in ("B", "H", "S", "D"))
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype = getattr(torch, case["dtype"])

    def operand():
        if case["rows"] == "bshd":
            return torch.randn(B, S, H, D, generator=gen, device=dev).to(dtype).transpose(1, 2)
        return torch.randn(B, H, S, D, generator=gen, device=dev).to(dtype)

    state = {"case": case, "q": operand(), "k": operand(), "v": operand(), "mask": _block_mask(case, dev)}
    if case["op"] == "train":
        state["dout"] = operand()
        state["score_mod"] = shim.softcap_score_mod(case["softcap"]) if case["softcap"] else None
        for name in ("q", "k", "v"):
            state[name].requires_grad_(True)
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "mask":
        m = shim.create_transfusion_block_mask(state["positions"], case["H"], case["S"], case["QB"], case["KB"])
        return {"kv_num_blocks": m.kv_num_blocks, "kv_indices": m.kv_indices, "types": m.block_mask_types,
                "partial_indices": m.partial_block_mask_indices, "partial_masks": m.partial_block_masks,
                "partial_bits": m.partial_block_bits}
    q, k, v, mask = state["q"], state["k"], state["v"], state["mask"]
    if op == "simple":
        return oat.omni_attention_simple(q, k, v, mask)
    if op == "train":
        out = shim.omni_flex_attention(q, k, v, block_mask=mask, score_mod=state["score_mod"])
        return (out,) + torch.autograd.grad(out, (q, k, v), state["dout"])
    if case["lse"]:
        return oat.omni_attention_forward(q, k, v, mask, softcap=case["softcap"])
    return oat.omni_attention_shared_kv_swizzle(q, k, v, mask)


def work(case):
    """One pass: every operand read once and every result written once; two products per allowed
    (query, key) pair forward, five more backward."""
    B, H, S, D = (case[k] for k in ("B", "H", "S", "D"))
    if case["op"] == "mask":
        n = -(-S // max(case["QB"], case["KB"])) * max(case["QB"], case["KB"])
        Tq, Tk = n // case["QB"], n // case["KB"]
        mask = oat.create_omni_block_mask_from_modality_positions(
            _batch_positions(case, 0), B, 1, n, n, case["QB"], case["KB"], device="cpu")
        tiles = 0 if mask.partial_block_masks is None else mask.partial_block_masks.numel()
        return {"bytes": 4.0 * B * H * Tq * (1 + 3 * Tk) + tiles * 1.125, "flops": 0.0}
    pairs = float(H * int(_prefix(case, "cpu").sum()))
    train = case["op"] == "train"
    tensors = 8 if train else 4  # q, k, v, out; and dout, dq, dk, dv
    return {"bytes": 2.0 * tensors * B * H * S * D + (4.0 * B * H * S if case["lse"] else 0.0),
            "flops": (14.0 if train else 4.0) * D * pairs}


def tolerance(case):
    """Results have 16 bits, and weights (and score gradients) are rounded to 16 bits before their
    second product; block masks are whole numbers."""
    if case["op"] == "mask":
        return "exact"
    return {"rel": 1e-2 if case["dtype"] == "bfloat16" else 2e-3}
