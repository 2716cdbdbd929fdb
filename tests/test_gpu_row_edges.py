"""Row lengths at which the rank kernel changes its form and the score rows their stride, the product that is added to what is
there at the edges of its tiles, and the corrected softplus / sigmoid."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("loss", ["ranking", "logistic", "softmax"])
@pytest.mark.parametrize("columns", [127, 128, 256, 257, 1024, 1025, 2048, 2049])
def test_ranks_at_row_length_edges(pbg, loss, columns):
    print("ranks", loss, columns, flush=True)
    g = torch.Generator(device=DEV).manual_seed(columns)
    dim, batch, negs, rows = 24, 70, 50, 500
    spec = pbg.StepSpec(dim=dim, batch_size=batch, num_workers=1, num_batch_negs=negs, num_uniform_negs=columns - negs,
                        operator="none", comparator="dot", loss=loss, margin=0.1)
    runner = pbg.StepRunner(spec, torch.randn(rows, dim, generator=g, device=DEV), torch.ones(rows, device=DEV))
    lhs, rhs = (torch.randint(0, rows, (batch,), generator=g, device=DEV) for _ in range(2))
    uni = torch.randint(0, rows, (2, 2 * (columns - negs)), generator=g, device=DEV)
    args = (lhs, rhs, torch.zeros(1, dtype=torch.long, device=DEV), uni[0], uni[1])
    lp, rp, ln, rn = (t.clone() for t in runner.forward(*args))
    lhs_pos, rhs_pos, lhs_rank, rhs_rank, loss_edge, _ = runner.ranks(*args)
    assert torch.equal(lhs_pos, lp) and torch.equal(rhs_pos, rp)
    want = torch.zeros(1, batch, dtype=torch.float64, device=DEV)
    for pos, neg, rank in ((lp, ln, lhs_rank), (rp, rn, rhs_rank)):
        assert torch.equal(rank, (neg >= pos.unsqueeze(2)).sum(2) + 1)
        pos, neg = pos.double(), neg.double()
        if loss == "ranking":
            want += (neg - pos.unsqueeze(2) + 0.1).clamp_min(0).sum(2)
        elif loss == "logistic":
            want += torch.nn.functional.softplus(-pos) + torch.nn.functional.softplus(neg).mean(2)
        else:
            want += torch.logsumexp(torch.cat((pos.unsqueeze(2), neg), 2), 2) - pos
    # per lane at most columns / 64 + 1 additions, six more across the wave, a few roundings of each term: 2^-24 of the sum each;
    # softmax subtracts scores of size max |s| from one another
    size = want.abs() + (0 if loss == "logistic" else torch.maximum(lp.abs(), rp.abs()).double() * (columns if loss == "ranking" else 4))
    assert ((loss_edge.double() - want).abs() <= 2.0 ** -24 * (columns // 64 + 30) * size).all()


@pytest.mark.parametrize("m,n", [(64, 64), (63, 65), (257, 129), (255, 128), (128, 256), (1, 1)])
def test_product_added_at_tile_edges(pbg, m, n):
    print("beta", m, n, flush=True)
    batch, k = 256, 40
    g = torch.Generator(device=DEV).manual_seed(m + n)
    a, b, c0 = (torch.randn(batch, *s, generator=g, device=DEV) for s in ((m, k), (k, n), (m, n)))
    c = c0.clone()
    pbg.native.gemm(a, b, c, batch, m, n, k, k, n, n, m * k, k * n, m * n, 0, 1, alpha=0.5, beta=-1.5)
    want = 0.5 * torch.bmm(a.double(), b.double()) - 1.5 * c0.double()
    size = 0.5 * torch.bmm(a.double().abs(), b.double().abs()) + 1.5 * c0.double().abs()
    # two k steps of six instructions, each rounding and aligning its products; scale, fold and addition
    assert ((c.double() - want).abs() <= 2.0 ** -24 * (2 * 12 + 5) * size).all()


@pytest.mark.parametrize("low,high", [(-1e-2, 1e-2), (-5.0, 5.0), (-20.0, -5.0), (5.0, 80.0), (-80.0, -20.0)])
def test_softplus_and_sigmoid(pbg, low, high):
    print("softplus", low, high, flush=True)
    g = torch.Generator(device=DEV).manual_seed(7)
    z = (torch.rand(64, 4096, generator=g, device=DEV) * (high - low) + low).requires_grad_()
    pos = torch.full((64,), 200.0, device=DEV)
    fn = pbg.losses.LOSS_FUNCTIONS.get_class("logistic")(margin=0.0)
    loss = fn(pos, z, None)
    loss.sum().backward()
    want = torch.sigmoid(z.detach().double()) / 4096
    # the exponential (1 ulp), the reciprocal's and the product's roundings, 1 / n and its product: 2^-23 + 4 * 2^-24
    assert ((z.grad.double() - want).abs() <= 6 * 2.0 ** -24 * want).all()
    total = torch.nn.functional.softplus(z.detach().double(), threshold=1e9).sum() / 4096
    # a lane adds 64 terms, then six and the rows' sums: fp32 additions of positive terms, two ulp each term
    assert abs(float(loss.detach().double().sum()) - float(total)) <= 2.0 ** -24 * 150 * float(total)


@pytest.mark.parametrize("value,softplus,sigmoid", [(float("-inf"), 0.0, 0.0), (float("inf"), float("inf"), 1.0)])
def test_softplus_of_infinities(pbg, value, softplus, sigmoid):
    z = torch.full((1, 64), value, device=DEV, requires_grad=True)
    loss = pbg.losses.LOSS_FUNCTIONS.get_class("logistic")(margin=0.0)(torch.full((1,), 200.0, device=DEV), z, None)
    loss.sum().backward()
    assert float(loss.detach().sum()) == softplus
    assert torch.equal(z.grad * 64, torch.full_like(z, sigmoid))
