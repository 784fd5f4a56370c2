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


@pytest.mark.parametrize("two_launches", [True, False])
@pytest.mark.parametrize("room", [-2, 0, 3, 1000])
def test_room_for_another_number_of_tiles(two_launches, room, gpu_device):
    """The C calls with a tile store of a fixed size: what it has room for is written, the rest of it is left alone."""
    import ctypes
    import omni_attn_capi as capi
    lib = capi.load_library()
    lib.omni_attn_mask_workspace_bytes.restype = ctypes.c_size_t
    B, H, S, QB, KB = 2, 3, 3000, 128, 64
    spans = torch.tensor([[[1, 37, 90], [1, 200, 1041]], [[1, 700, 1500], [0, 0, 0]]])
    want = oat.create_omni_block_mask_from_modality_positions(spans, B, H, S, S, QB, KB, device="cpu")
    n = want.partial_block_masks.shape[0]
    Tq, Tk = want.kv_indices.shape[2:]
    sp = spans.to(gpu_device)
    i32 = lambda *shape: torch.empty(*shape, dtype=torch.int32, device=gpu_device)
    nb, idx, tys, pidx = i32(B, H, Tq), i32(B, H, Tq, Tk), i32(B, H, Tq, Tk), i32(B, H, Tq, Tk)
    ws = i32(lib.omni_attn_mask_workspace_bytes(B, S, S, QB, KB) // 4)
    posted = torch.zeros(B * Tq, dtype=torch.int32, pin_memory=True)
    tiles = torch.full((n + 1000, QB, KB), 7, dtype=torch.uint8, device=gpu_device)
    bits = torch.full((n + 1000, QB, KB // 32), 7, dtype=torch.int32, device=gpu_device)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    lists = (ptr(nb), ptr(idx), ptr(tys), ptr(pidx))
    if two_launches:
        assert lib.omni_attn_mask_classify_gfx950(ptr(sp), None, ptr(ws), ptr(posted), 5, B, 2, S, S, QB, KB, stream) == 0
        torch.cuda.synchronize()
        assert bool((posted >> 20 == 5).all()) and int((posted & 0xfffff).sum()) == n
        assert lib.omni_attn_mask_finish_gfx950(*lists, ptr(ws), ptr(tiles), ptr(bits), n + room, B, H, S, S, QB, KB,
                                                stream) == 0
    else:
        assert lib.omni_attn_mask_lists_gfx950(ptr(sp), None, *lists, ptr(ws), ptr(posted), 9, B, 2, H, S, S, QB, KB,
                                               stream) == 0
        torch.cuda.synchronize()
        assert posted[:2].tolist() == [n, 9]
        assert lib.omni_attn_mask_tiles_gfx950(ptr(sp), None, ptr(ws), ptr(tiles), ptr(bits), n + room, B, 2, H, S, S, QB,
                                               KB, stream) == 0
    same_mask(oat.OmniBlockMask(nb, idx, tys, Tq * QB, Tk * KB, QB, KB, pidx, tiles[:n].view(torch.bool) if room >= 0 else
                                want.partial_block_masks.to(gpu_device)), want)
    written = min(n + room, n)
    assert torch.equal(tiles[:written].cpu(), want.partial_block_masks[:written].to(torch.uint8))
    assert torch.equal(bits[:written], capi.pack_partial_masks(tiles[:written]))
    assert bool((tiles[written:] == 7).all()) and bool((bits[written:] == 7).all())


@pytest.mark.parametrize("two_launches", [True, False])
@pytest.mark.parametrize("B,S,QB", [(1, 100, 128), (1, 65 * 16, 16), (3, 16 * 341 - 3, 16), (16, 1024, 16), (9, 8191, 16)],
                         ids=["1", "65", "1023", "1024", "4608"])
def test_tiles_are_numbered_over_query_blocks(two_launches, B, S, QB, gpu_device):
    """The C calls at numbers of query blocks on both sides of those that are summed up in place, with runs of query
    blocks that have no tile, and room for a few tiles more than there are."""
    import ctypes
    import omni_attn_capi as capi
    lib = capi.load_library()
    lib.omni_attn_mask_workspace_bytes.restype = ctypes.c_size_t
    H, KB = 2, 64
    gen = torch.Generator().manual_seed(S)
    spans = torch.zeros(B, 2, 3, dtype=torch.long)
    cuts = torch.randint(0, S, (B, 2, 2), generator=gen)
    spans[..., 1], spans[..., 2] = cuts.amin(-1), cuts.amax(-1) - cuts.amin(-1)
    spans[::3] = 0
    want = oat.create_omni_block_mask_from_modality_positions(spans, B, H, S, S, QB, KB, device="cpu")
    tiles_wanted = want.partial_block_masks
    n = 0 if tiles_wanted is None else tiles_wanted.shape[0]
    Tq, Tk = want.kv_indices.shape[2:]
    sp = spans.to(gpu_device)
    i32 = lambda *shape: torch.empty(*shape, dtype=torch.int32, device=gpu_device)
    nb, idx, tys, pidx = i32(B, H, Tq), i32(B, H, Tq, Tk), i32(B, H, Tq, Tk), i32(B, H, Tq, Tk)
    ws = i32(lib.omni_attn_mask_workspace_bytes(B, S, S, QB, KB) // 4)
    posted = torch.zeros(max(2, B * Tq), dtype=torch.int32, pin_memory=True)
    room = min(n + 3, B * Tq * Tk)
    tiles = torch.full((room, QB, KB), 7, dtype=torch.uint8, device=gpu_device)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    lists = (ptr(nb), ptr(idx), ptr(tys), ptr(pidx))
    if two_launches:
        assert lib.omni_attn_mask_classify_gfx950(ptr(sp), None, ptr(ws), ptr(posted), 5, B, 2, S, S, QB, KB, stream) == 0
        assert lib.omni_attn_mask_finish_gfx950(*lists, ptr(ws), ptr(tiles), None, room, B, H, S, S, QB, KB, stream) == 0
        torch.cuda.synchronize()
        assert int((posted[:B * Tq] & 0xfffff).sum()) == n
    else:
        assert lib.omni_attn_mask_lists_gfx950(ptr(sp), None, *lists, ptr(ws), ptr(posted), 9, B, 2, H, S, S, QB, KB,
                                               stream) == 0
        assert lib.omni_attn_mask_tiles_gfx950(ptr(sp), None, ptr(ws), ptr(tiles), None, room, B, 2, H, S, S, QB, KB,
                                               stream) == 0
        torch.cuda.synchronize()
        assert posted[:2].tolist() == [n, 9]
    for got, ref in ((nb, want.kv_num_blocks), (idx, want.kv_indices), (tys, want.block_mask_types)):
        assert torch.equal(got.cpu(), ref.to(torch.int32))
    if n:
        assert torch.equal(pidx.cpu(), want.partial_block_mask_indices)
        assert torch.equal(tiles[:n].cpu(), tiles_wanted.to(torch.uint8))
    else:
        assert bool((pidx == -1).all())
    assert bool((tiles[n:] == 7).all())


@pytest.mark.parametrize("blocks", [512, 513])
def test_counts_and_their_sum(blocks, gpu_device):
    """As many query blocks as send a count each, and one more."""
    spans = torch.tensor([[[1, 37, 900], [1, 2000, 1141], [1, 8000, 100]]])
    args = (spans, 1, 3, blocks * 16, blocks * 16, 16, 128)
    want = oat.create_omni_block_mask_from_modality_positions(*args, device="cpu")
    same_mask(oat.create_omni_block_mask_from_modality_positions(*args, device=gpu_device), want)


def test_lists_that_do_not_fit(gpu_device):
    """A call that finds no memory for its lists, while its first kernel runs, ends with torch's own error, and the next ones
    are whole."""
    spans = torch.tensor([[[1, 37, 900], [1, 2000, 1141]]])
    want = oat.create_omni_block_mask_from_modality_positions(spans, 1, 2, 8192, 8192, 128, 128, device="cpu")
    for _ in range(3):
        with pytest.raises(torch.OutOfMemoryError):
            oat.create_omni_block_mask_from_modality_positions(spans, 1, 20_000_000, 8192, 8192, 128, 128, device=gpu_device)
        same_mask(oat.create_omni_block_mask_from_modality_positions(spans, 1, 2, 8192, 8192, 128, 128, device=gpu_device), want)
