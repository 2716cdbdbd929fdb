"""A negative that is the positive's own entity scores exactly what the positive scores, on both sides: the score products
of the two sides take the same pair with its operands exchanged.  And products with infinite or huge operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dim,batch,negs", [(33, 64, 64), (400, 300, 150), (1024, 1000, 500)])
def test_duplicate_of_the_positive_ties_exactly(pbg, dim, batch, negs):
    print("ties", dim, batch, negs, flush=True)
    g = torch.Generator(device=DEV).manual_seed(dim)
    rows = 40  # every entity many times in a chunk
    w = torch.randn(rows, dim, generator=g, device=DEV)
    lhs, rhs = (torch.randint(0, rows, (batch,), generator=g, device=DEV) for _ in range(2))
    spec = pbg.StepSpec(dim=dim, batch_size=batch, num_workers=1, num_batch_negs=negs, num_uniform_negs=200, operator="none",
                        comparator="dot", loss="softmax")
    runner = pbg.StepRunner(spec, w, torch.ones(rows, device=DEV))
    chunks = -(-batch // negs)
    uni = torch.randint(0, rows, (2, chunks * 200), generator=g, device=DEV)
    lp, rp, ln, rn = runner.forward(lhs, rhs, torch.zeros(1, dtype=torch.long, device=DEV), uni[0], uni[1])
    for ids, pos, neg, draws in ((lhs, lp, ln, uni[0]), (rhs, rp, rn, uni[1])):
        pos, neg = pos.view(batch), neg.view(batch, -1)
        seen = 0
        for e in range(batch):
            c, i = divmod(e, negs)
            cols = torch.cat((ids[c * negs:(c + 1) * negs], draws.view(chunks, 200)[c]))
            same = cols == ids[e]
            same[i] = False  # the positive's own column is masked
            width = len(ids[c * negs:(c + 1) * negs])
            row = torch.cat((neg[e, :width], neg[e, min(negs, batch):]))
            assert torch.equal(row[same], pos[e].expand(int(same.sum())))
            seen += int(same.sum())
        assert seen > batch


@pytest.mark.parametrize("akm,bkm", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_infinite_and_huge_operands(pbg, akm, bkm):
    print("inf", akm, bkm, flush=True)
    batch, m, n, k = 2, 130, 70, 65
    g = torch.Generator(device=DEV).manual_seed(5)
    a, b = torch.randn(batch, m, k, generator=g, device=DEV), torch.randn(batch, n, k, generator=g, device=DEV)
    b[:, :, 3] = 1.0
    a[0, 5, 3] = float("inf")
    a[0, 7, 3] = -float("inf")
    a[1, 129, 3] = float("nan")
    a[1, 8, :] = 0.0
    a[1, 8, 3] = 3.4028e38  # rounds up to an infinite bf16 number
    want = torch.bmm(a.double().cpu(), b.double().cpu().transpose(1, 2).contiguous()).float()
    c0 = torch.randn(batch, m, n, generator=g, device=DEV)
    c = c0.clone()
    ga, gb = a.transpose(1, 2).contiguous() if akm else a, b.transpose(1, 2).contiguous() if bkm else b
    pbg.native.gemm(ga, gb, c, batch, m, n, k, ga.shape[2], gb.shape[2], n, m * k, n * k, m * n, akm, bkm, alpha=1.0, beta=2.0)
    want = want + 2.0 * c0.cpu()
    c = c.cpu()
    assert torch.equal(torch.isnan(c), torch.isnan(want))
    assert torch.equal(torch.isinf(c), torch.isinf(want)) and torch.equal(c[torch.isinf(c)], want[torch.isinf(want)])
    ok = torch.isfinite(want)
    # k + 3 fp32 roundings of sums of at most sum |a b| + 2 |c|
    size = torch.bmm(a.double().nan_to_num(0, 0, 0).abs().cpu(), b.double().abs().cpu().transpose(1, 2).contiguous()) + 2 * c0.double().abs().cpu()
    assert ((c.double() - want.double()).abs()[ok] <= (2.0 ** -24) * (k + 3) * size[ok]).all()
