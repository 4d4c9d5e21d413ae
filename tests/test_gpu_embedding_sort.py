"""Sorted scatter-add of the embedding gradient at the sizes where its sort changes form: one
workgroup (up to 4096 lookups), 1, 2 or 4 keys per thread (up to 131 072, 524 288, 1 048 576), three
launches per pass beyond; digits of ten bits for ids of 17 to 20, up to 16 384 lookups and from 131 073 on.  Gradients are small whole numbers, so every sum is exact in fp32 in
any order and the results are compared bit for bit with a float64 sum on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(ffk, n, bag, vocab, dim, index_dtype, grad_dtype, deterministic, skew, seed):
    gen = torch.Generator().manual_seed(seed)
    u = torch.rand(n * bag, generator=gen, dtype=torch.float64)
    ids = (u ** (6.0 if skew else 1.0) * vocab).long()
    # ids outside the table are skipped, wherever they stand
    ids[::97] = vocab + 3
    ids[5::131] = -1
    dy = torch.randint(-4, 5, (n, dim), generator=gen).double()
    inside = (ids >= 0) & (ids < vocab)
    want = torch.ones((vocab, dim), dtype=torch.float64)
    want.index_add_(0, ids[inside], dy.repeat_interleave(bag, 0)[inside])
    got = torch.ones((vocab, dim), device="cuda")
    idx = ids.to(index_dtype).view(n, bag).cuda()
    ffk.embedding_backward(idx, dy.to(grad_dtype).cuda(), got, aggr=ffk.AGGR_SUM, deterministic=deterministic)
    assert torch.equal(got.cpu().double(), want)


@pytest.mark.parametrize("n,bag,vocab,dim", [
    (1, 1, 3, 64),            # one lookup, two-bit keys
    (1024, 1, 255, 64),       # one workgroup, one key per thread, all of it
    (1025, 1, 256, 128),      # four keys per thread; nine-bit keys, two passes
    (1365, 3, 70000, 320),    # 4095 lookups: one short of the workgroup; three passes
    (4097, 1, 70000, 64),     # two launches' worth: a last tile of one key
    (26215, 5, 1000, 64),     # 131 075: two keys per thread
    (131072, 1, 60000, 16),   # one key per thread, every tile full
    (131073, 2, 30000, 16),   # 262 146
    (16384, 32, 50000, 128),  # 524 288: two keys per thread, every tile full
    (524289, 1, 300, 16),     # four keys per thread
    (1048577, 1, 300, 16),    # beyond it
    (5, 1, 70000, 16),        # ten-bit digits: one workgroup
    (16384, 1, 131071, 16),   # sixteen tiles, 17 bits
    (16385, 1, 131072, 16),   # a seventeenth: three passes again; 18 bits
    (131073, 1, 70000, 4),    # scanned: two keys per thread, 17 bits
    (524289, 1, 1000000, 4),  # four, 20 bits
])
@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
def test_sizes_where_the_sort_changes_form(ffk, n, bag, vocab, dim, index_dtype):
    # (up to 8192 lookups only a deterministic call sorts)
    for skew, deterministic in ((False, False), (True, False), (False, True), (True, True)):
        _case(ffk, n, bag, vocab, dim, index_dtype, torch.float32, deterministic, skew, n + bag)


@pytest.mark.parametrize("dim", [4, 64, 68, 128, 256, 260, 512, 1024, 1600])
@pytest.mark.parametrize("grad_dtype", [torch.float32, torch.bfloat16])
def test_row_lengths_bags_and_modes(ffk, dim, grad_dtype):
    # a run that fills whole walkers and workgroups (one id in a third of the lookups), bags and single lookups
    for bag, deterministic in ((1, False), (1, True), (7, False), (7, True)):
        _case(ffk, 1171, bag, 900, dim, torch.int64, grad_dtype, deterministic, True, dim + bag)


@pytest.mark.parametrize("dim", [4, 16, 20, 32, 36, 64, 68, 128, 132, 256, 1600])
@pytest.mark.parametrize("n,bag", [(1, 1), (255, 1), (257, 1), (2049, 1), (683, 3), (70001, 1),
                                   # past 8192 lookups, which are matched and not walked: a last walker of one
                                   # position, a workgroup short of one, of one position more, and bags
                                   (8193, 1), (8447, 1), (8449, 1), (2817, 3)])
def test_walk_at_its_borders(ffk, dim, n, bag):
    """Walkers of 4 to 64 lanes, the last one short; runs that cross walkers and workgroups (half of the lookups are
    three ids) beside rows looked up once."""
    gen = torch.Generator().manual_seed(dim * 3 + n)
    vocab = 5000
    ids = torch.where(torch.rand(n * bag, generator=gen) < 0.5, torch.randint(0, 3, (n * bag,), generator=gen) * 1700,
                      torch.randint(-2, vocab + 2, (n * bag,), generator=gen))
    dy = torch.randint(-4, 5, (n, dim), generator=gen).double()
    inside = (ids >= 0) & (ids < vocab)
    want = torch.ones((vocab, dim), dtype=torch.float64)
    want.index_add_(0, ids[inside], dy.repeat_interleave(bag, 0)[inside])
    for dtype in (torch.float32, torch.bfloat16):
        buf = torch.full((vocab * dim + 128,), 1.0, device="cuda")  # (sums of whole numbers: exact in any order)
        got = buf[64:64 + vocab * dim].view(vocab, dim)
        ffk.embedding_backward(ids.view(n, bag).cuda(), dy.to(dtype).cuda(), got, aggr=ffk.AGGR_SUM)
        assert torch.equal(got.cpu().double(), want)
        assert bool((buf[:64] == 1.0).all()) and bool((buf[64 + vocab * dim:] == 1.0).all())


def _large_table(ffk, vocab, dim, n):
    """n lookups in the first and the last 700 rows."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    ids = torch.randint(vocab - 700, vocab, (n,), generator=gen, device="cuda")
    ids[::2] = torch.randint(0, 700, ((n + 1) // 2,), generator=gen, device="cuda")
    ids[:2] = torch.tensor([vocab - 1, 0], device="cuda")
    dy = torch.randint(-4, 5, (n, dim), generator=gen, device="cuda", dtype=torch.float32)
    got = torch.zeros((vocab, dim), device="cuda")
    ffk.embedding_backward(ids.view(n, 1), dy, got, aggr=ffk.AGGR_SUM)
    small = torch.zeros((1400, dim), device="cuda")
    small.index_add_(0, torch.where(ids < 700, ids, ids - (vocab - 1400)), dy)
    assert torch.equal(got[:700], small[:700]) and torch.equal(got[-700:], small[700:])
    assert not bool(got[700:-700].any())


@pytest.mark.parametrize("n", [3000,   # (rows of 1024 count twice) compared with each other
                               5000])  # sorted, for the kernel with 64-bit offsets
def test_table_beyond_32_bit_offsets(ffk, n):
    """4.4 GB of weight gradient: row offsets past 2^32 bytes."""
    _large_table(ffk, 1100000, 1024, n)


# (0xfffff000 bytes are as far as the walk's offsets reach)
@pytest.mark.parametrize("vocab,n", [(1048575, 5000), (1048576, 5000),        # the weight gradient's, and one row more
                                     (3000, 1048575), (3000, 1048576)])       # the output gradient's
def test_walk_at_the_end_of_its_offsets(ffk, vocab, n):
    _large_table(ffk, vocab, 1024, n)
