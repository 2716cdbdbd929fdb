"""Calls that report to the host: the id check on every route of the step, and the sums of a ranking evaluation."""
import pytest
import torch

DEV = "cuda:0"
pytestmark = pytest.mark.gpu

# one shape per place that looks at the ids: the chunk kernel, the row-id kernel of many chunks (with and without an
# operator whose step runs beside the update), the sliced, streaming and staged routes, and max_norm, which writes first
ROUTES = [
    dict(dim=100, batch_size=1000, num_workers=1),
    dict(dim=100, batch_size=1000, num_workers=8),
    dict(dim=64, batch_size=1000, num_workers=8, operator="translation"),
    dict(dim=200, batch_size=300, num_workers=4),
    dict(dim=400, batch_size=300, num_workers=2, num_uniform_negs=400, operator="complex_diagonal", dynamic=True, num_relations=5),
    dict(dim=64, batch_size=700, num_workers=1, num_batch_negs=300, num_uniform_negs=7, loss="softmax"),
    dict(dim=32, batch_size=100, num_workers=1, max_norm=0.5),
]


def make(pbg, fields, rows=500):
    spec = pbg.StepSpec(**fields)
    gen = torch.Generator().manual_seed(3)
    w = (torch.randn(rows, spec.dim, generator=gen) * 0.3).to(DEV)
    g = torch.rand(rows, generator=gen).to(DEV)
    names = {"complex_diagonal": ("real", "imag"), "translation": ("translation",), "none": ()}[spec.operator]
    width = spec.dim // 2 if spec.operator == "complex_diagonal" else spec.dim
    ops = [{n: torch.randn(spec.num_relations, width, generator=gen).to(DEV) for n in names} for _ in range(4)]
    for sums in (ops[1], ops[3]):
        for t in sums.values():
            t.abs_()
    lhs_ops = ops[2:] if spec.dynamic else [{}, {}]
    runner = pbg.StepRunner(spec, w, g, None, None, ops[0], ops[1], *lhs_ops)
    k, b = spec.num_workers, spec.batch_size
    ids = [torch.randint(0, rows, (k * b,), generator=gen) for _ in range(2)]
    ids.append(torch.randint(0, spec.num_relations, (k * b if spec.dynamic else k,), generator=gen))
    ids += [torch.randint(0, rows, (k, spec.num_chunks, spec.num_uniform_negs), generator=gen) for _ in range(2)]
    return runner, [i.to(DEV) for i in ids], [w, g, *(t for op in ops for t in op.values())]


@pytest.mark.parametrize("fields", ROUTES)
def test_checked_step(pbg, fields):
    """Any id outside what it indexes raises IndexError and changes nothing; with ids in range the call does what the
    unchecked one does, and its statistics on the host are those the device tensors hold."""
    runner, ids, state = make(pbg, fields)
    rows = runner.w_lhs.shape[0]
    before = [t.clone() for t in state]
    for which, at, value in ((0, 0, rows), (1, -1, -1), (2, -1, runner.spec.num_relations), (3, 0, rows + 7), (4, -1, -5)):
        bad = [t.clone() for t in ids]
        bad[which].view(-1)[at] = value
        with pytest.raises(IndexError):
            runner.train_stats(*bad, check_ids=True)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(before, state)), (which, value)
    loss, _, viol = (a.copy() for a in runner.train_stats(*ids, check_ids=True))
    after = [t.clone() for t in state]
    for t, old in zip(state, before):
        t.copy_(old)
    runner.train(*ids)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(after, state))
    assert loss.tolist() == runner.loss_out.tolist() and viol.tolist() == runner.violators_out.tolist()


@pytest.mark.parametrize("batch,workers", [(1, 1), (257, 1), (300, 7), (16641, 1)])
def test_rank_sums(pbg, batch, workers):
    """Around one thread's, one block's and all blocks' share: the sums are those of ranks()' outputs.  The whole
    numbers are equal; loss and reciprocals are float32 values added in float64 (error below 1e-12 relative)."""
    runner, ids, _ = make(pbg, dict(dim=16, batch_size=batch, num_workers=workers, num_batch_negs=20, num_uniform_negs=15))
    loss, sides = runner.rank_sums(*ids, auc_samples=1000, auc_seed=5)
    _, _, lr, rr, le, hits = runner.ranks(*ids, auc_samples=1000, auc_seed=5)
    assert loss == pytest.approx(float(le.double().sum()), rel=1e-12)
    for side, rank, hit in zip(sides, (lr, rr), hits.tolist()):
        assert side[0] == int(rank.sum()) and side[5] == hit
        assert side[1] == pytest.approx(float(rank.float().reciprocal().double().sum()), rel=1e-12)
        assert side[2:5] == [int((rank <= n).sum()) for n in (1, 10, 50)]
    ids[3].view(-1)[-1] = runner.w_lhs.shape[0]
    with pytest.raises(IndexError):
        runner.rank_sums(*ids)
