"""The native builder of prefix-rule masks against the tensor algebra of the CPU build: whole numbers,
so every field has to be equal.  Sizes at the edges of its loops: more key blocks than a wave, key
blocks that 16 bytes or 32 bits do not divide, ragged lengths, no spans, no PARTIAL tile at all."""
import pytest
import torch

import omni_attn_torch as oat
import transfusion_shim as shim

pytestmark = pytest.mark.gpu

FIELDS = ("kv_num_blocks", "kv_indices", "block_mask_types", "partial_block_mask_indices", "partial_block_masks")


def same_mask(gpu, cpu):
    for name in FIELDS:
        a, b = getattr(cpu, name), getattr(gpu, name)
        assert (a is None) == (b is None), name
        if a is not None:
            assert b.is_cuda and a.dtype == b.dtype and torch.equal(a, b.cpu()), name
    assert (gpu.q_len, gpu.kv_len) == (cpu.q_len, cpu.kv_len)
    assert gpu.has_partial_slots() == bool((cpu.block_mask_types == 3).any())


@pytest.mark.parametrize("S,QB,KB", [(128, 128, 128), (130, 64, 128), (1000, 33, 48), (640, 16, 7), (4500, 128, 64),
                                     (8192, 64, 64)])
def test_builder_equals_the_tensor_algebra(S, QB, KB, gpu_device):
    gen = torch.Generator().manual_seed(S + QB)
    spans = torch.zeros(3, 4, 3, dtype=torch.long)  # element 2 keeps its zero-length spans: text only
    for b in range(2):
        cuts = torch.randperm(S - 1, generator=gen)[:8].sort().values.view(4, 2)
        spans[b, :, 1], spans[b, :, 2] = cuts[:, 0], cuts[:, 1] - cuts[:, 0]
    for mp in (spans, spans[2:], spans[:, :0], torch.tensor([[[1, 0, S]]])):
        B = mp.shape[0]
        args = (mp, B, 3, S, S, QB, KB)
        same_mask(oat.create_omni_block_mask_from_modality_positions(*args, device=gpu_device),
                  oat.create_omni_block_mask_from_modality_positions(*args, device="cpu"))
    prefix = torch.randint(0, S + 40, (2, S), generator=gen)  # any prefixes, falling ones and empty rows too
    same_mask(oat.create_omni_block_mask_from_prefix_lengths(prefix.to(gpu_device), 2, S, S, QB, KB),
              oat.create_omni_block_mask_from_prefix_lengths(prefix, 2, S, S, QB, KB))


def test_packed_tiles_come_with_the_mask(gpu_device):
    mp = torch.tensor([[[1, 37, 90], [1, 200, 141]]])
    m = shim.create_transfusion_block_mask(mp.to(gpu_device), 2, 500, 128, 64)
    bits = m.partial_block_bits.clone()
    m.partial_block_bits = None
    assert torch.equal(m.pack_partial_masks().partial_block_bits, bits)
    assert shim.create_transfusion_block_mask(mp.to(gpu_device), 2, 500, pack=False).partial_block_bits is None


def test_more_query_blocks_than_counts_are_sent_for(gpu_device):
    """9 x 512 query blocks: the number of tiles comes as one word instead of a count per query block."""
    gen = torch.Generator().manual_seed(3)
    spans = torch.zeros(9, 3, 3, dtype=torch.long)
    cuts = torch.randint(0, 8000, (9, 3, 2), generator=gen)
    spans[..., 1], spans[..., 2] = cuts.amin(-1), cuts.amax(-1) - cuts.amin(-1)
    args = (spans, 9, 2, 8192, 8192, 16, 64)
    want = oat.create_omni_block_mask_from_modality_positions(*args, device="cpu")
    for _ in range(2):
        same_mask(oat.create_omni_block_mask_from_modality_positions(*args, device=gpu_device), want)


def test_many_masks_in_a_row(gpu_device):
    """More calls than the counts have tags, of two sizes in turn, so that words of earlier calls are still there."""
    small = torch.tensor([[[1, 37, 90], [1, 200, 141]]])
    large = small.repeat(4, 1, 1)
    sizes = [(small, 500), (large, 3000)]
    want = [shim.create_transfusion_block_mask(mp, 2, S, 128, 128, pack=False).partial_block_masks.shape[0] for mp, S in sizes]
    assert want[0] != want[1] > 0
    sizes = [(mp.to(gpu_device), S) for mp, S in sizes]
    for i in range(4200):
        mp, S = sizes[i % 64 == 0]
        m = shim.create_transfusion_block_mask(mp, 2, S, 128, 128, pack=False)
        assert m.partial_block_masks.shape[0] == want[i % 64 == 0]
