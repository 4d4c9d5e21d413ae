"""The scatter-add of bags between the walks of few and of many lookups: numbers of lookups at both ends and just past
them, columns of whole and of part lanes, popular rows, ids that are no rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lookups", [65536 - 4, 65536, 100004, 262144 - 4, 262144])
@pytest.mark.parametrize("dim", [64, 68, 100, 128, 132])
def test_bags(ffk, lookups, dim):
    gen = torch.Generator(device="cuda").manual_seed(dim)
    bag, rows = 4, 5001
    for dtype, index in [(torch.float32, torch.int64), (torch.bfloat16, torch.int32)]:
        print("dim", dim, "lookups", lookups, dtype, flush=True)
        ids = (torch.rand(lookups, device="cuda", generator=gen) ** 6 * (rows + 2)).long() - 1  # popular ones, and -1, rows
        dy = torch.randn(lookups // bag, dim, device="cuda", generator=gen).to(dtype)
        dw0 = torch.randn(rows, dim, device="cuda", generator=gen)
        dw = dw0.clone()
        ffk.embedding_backward(ids.to(index).view(-1, bag), dy, dw, aggr=ffk.AGGR_AVG)
        valid = (ids >= 0) & (ids < rows)
        g = dy.double().repeat_interleave(bag, 0)[valid] / bag
        want = dw0.double().index_add(0, ids[valid], g)
        size = dw0.double().abs().index_add(0, ids[valid], g.abs())
        # float32 sums of `times` terms in any order, one scaled by 1 / bag: a rounding each
        times = torch.bincount(ids[valid], minlength=rows).double()[:, None] + 3
        err = (dw.double() - want).abs()
        assert bool((err <= times * 2.0 ** -24 * size).all()), float((err / size).max())
