"""Sorted scatter-add of the embedding gradient at the sizes where its sort changes form: one
workgroup (up to 4096 lookups), 1, 2 or 4 keys per thread (up to 131 072, 524 288, 1 048 576), three
launches per pass beyond.  Gradients are small whole numbers, so every sum is exact in fp32 in
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
])
@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
def test_sizes_where_the_sort_changes_form(ffk, n, bag, vocab, dim, index_dtype):
    for skew in (False, True):
        _case(ffk, n, bag, vocab, dim, index_dtype, torch.float32, False, skew, n + bag)


@pytest.mark.parametrize("dim", [4, 64, 68, 128, 256, 260, 512, 1024, 1600])
@pytest.mark.parametrize("grad_dtype", [torch.float32, torch.bfloat16])
def test_row_lengths_bags_and_modes(ffk, dim, grad_dtype):
    # a run that fills whole walkers and workgroups (one id in a third of the lookups), bags and single lookups
    for bag, deterministic in ((1, False), (1, True), (7, False), (7, True)):
        _case(ffk, 1171, bag, 900, dim, torch.int64, grad_dtype, deterministic, True, dim + bag)
