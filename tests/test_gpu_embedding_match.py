"""The scatter-add of few lookups: numbers of them around a wave's, a workgroup's and the most that are taken,
rows looked up so often that several waves share them, ids that are no rows, every width's lanes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def ids_of(kind, n, rows, gen):
    if kind == "one":
        return torch.full((n,), rows - 1, dtype=torch.int64, device="cuda")
    if kind == "once":
        return torch.randperm(max(n, rows), device="cuda", generator=gen)[:n] % rows
    if kind == "pairs":  # 32 and 33 of each, spread out: the most one wave takes, and one more
        return (torch.arange(n, device="cuda") % max(1, n // 33)).long()
    return (torch.rand(n, device="cuda", generator=gen) ** 6 * (rows + 2)).long() - 1  # popular ones, and -1, rows


@pytest.mark.parametrize("kind", ["one", "once", "pairs", "some"])
@pytest.mark.parametrize("dim", [4, 16, 20, 64, 128, 132, 256, 512, 516, 1056])
def test_few_lookups(ffk, kind, dim):
    gen = torch.Generator(device="cuda").manual_seed(dim)
    most = 8192 // -(-dim // 512)
    for n, bag in [(1, 1), (15, 1), (16, 4), (17, 1), (255, 5), (256, 1), (257, 1), (1055, 5), (most - 1, 1), (most, 8), (most + 1, 1)]:
        n -= n % bag
        rows = max(2, n // 3) if kind != "once" else n + 5
        ids = ids_of(kind, n, rows, gen)
        for dtype, index in [(torch.float32, torch.int64), (torch.bfloat16, torch.int32)]:
            print(kind, "dim", dim, "lookups", n, "bag", bag, dtype, flush=True)
            dy = torch.randn(n // bag, dim, device="cuda", generator=gen).to(dtype)
            dw0 = torch.randn(rows, dim, device="cuda", generator=gen)
            dw = dw0.clone()
            aggr = {} if bag == 1 else {"aggr": ffk.AGGR_AVG}
            ffk.embedding_backward(ids.to(index).view(-1, bag) if bag > 1 else ids.to(index), dy, dw, **aggr)
            valid = (ids >= 0) & (ids < rows)
            g = dy.double().repeat_interleave(bag, 0)[valid] / bag
            want = dw0.double().index_add(0, ids[valid], g)
            size = dw0.double().abs().index_add(0, ids[valid], g.abs())
            # float32 sums of `times` terms in any order, one scaled by 1 / bag: a rounding each
            times = torch.bincount(ids[valid], minlength=rows).double()[:, None] + 3
            err = (dw.double() - want).abs()
            assert bool((err <= times * 2.0 ** -24 * size).all()), float((err / size).max())


@pytest.mark.parametrize("lookups,dim", [(300, 64), (2000, 128), (8192, 256)])
def test_calls_without_scratch_add_to_one_table_side_by_side(ffk, lookups, dim):
    """Atomics: two streams that add to the same rows at a time lose nothing.  Whole numbers, exact in float32."""
    gen = torch.Generator(device="cuda").manual_seed(lookups)
    rows, calls = lookups // 3, 40  # three lookups a row: what one wave would load, add to and store back
    ids = [torch.randint(0, rows, (lookups,), device="cuda", generator=gen) for _ in range(2)]
    dy = [torch.randint(-4, 5, (lookups, dim), device="cuda", generator=gen).float() for _ in range(2)]
    dw = torch.zeros(rows, dim, device="cuda")
    want = calls * sum(torch.zeros(rows, dim, device="cuda").index_add_(0, i, g) for i, g in zip(ids, dy))
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(calls):
        for s, i, g in zip(streams, ids, dy):
            with torch.cuda.stream(s):
                ffk.embedding_backward(i, g, dw, workspace=False)
    torch.cuda.synchronize()
    assert torch.equal(dw, want)
