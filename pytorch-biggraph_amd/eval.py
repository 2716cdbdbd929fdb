"""Ranking evaluation of a batch (reference: torchbiggraph/eval.py:43-86,
util.py:420-428, stats.py:16-17).  The scores come from
MultiRelationEmbedder.forward, i.e. from pbg_model_forward on the GPU; the
metrics are a handful of reductions over [B] and [B, N] tensors."""
from statistics import mean

import numpy as np
import torch

from .batching import AbstractBatchProcessor
from .edgelist import EdgeList
from .model import MultiRelationEmbedder, Scores
from .stats import Stats


def average_of_sums(*tensors: torch.Tensor) -> float:
    """stats.py:16-17."""
    return mean(t.sum().item() for t in tensors)


def compute_randomized_auc(pos_: torch.Tensor, neg_: torch.Tensor, num_samples: int) -> float:
    """Probability that a randomly chosen positive scores higher than a randomly
    chosen negative, from num_samples random pairs (util.py:420-428)."""
    pos_, neg_ = pos_.reshape(-1), neg_.reshape(-1)
    dev = pos_.device
    diff = (pos_[torch.randint(len(pos_), (num_samples,), device=dev)]
            > neg_[torch.randint(len(neg_), (num_samples,), device=dev)])
    return float(diff.float().mean())


def _sum_of_reciprocals(rank: torch.Tensor) -> float:
    """The float32 reciprocals, added in float64 and rounded once: the same sum in whatever order it is formed."""
    return rank.float().reciprocal().double().sum().float().item()


def ranking_stats(sides, loss: float, count: int) -> Stats:
    """The sums RankingEvaluator reports for `count` edges (eval.py:57-81).
    sides: (pos [n], neg [n, N]) per side; a side without negatives is skipped.
    Rank = 1 + number of negatives scoring at least as high as the positive."""
    ranks, aucs = [], []
    for pos, neg in sides:
        if neg.nelement() > 0:
            ranks.append((neg >= pos.unsqueeze(1)).sum(1) + 1)
            aucs.append(compute_randomized_auc(pos, neg, count))
    return Stats(
        loss=float(loss),
        pos_rank=average_of_sums(*ranks),
        mrr=mean(_sum_of_reciprocals(rank) for rank in ranks),
        r1=average_of_sums(*(rank.le(1) for rank in ranks)),
        r10=average_of_sums(*(rank.le(10) for rank in ranks)),
        r50=average_of_sums(*(rank.le(50) for rank in ranks)),
        auc=count * sum(aucs) / len(aucs),  # averaged over count at the end
        count=count,
    )


def ranking_stats_from_sums(sides, loss: float, count: int, auc_samples: int) -> Stats:
    """The same sums from StepRunner.rank_sums: one (ranks, reciprocals, <= 1, <= 10, <= 50, auc hits) per side that
    has negatives."""
    sides = [(ranks, float(np.float32(reciprocals)), *rest) for ranks, reciprocals, *rest in sides]
    pos_rank, mrr, r1, r10, r50, hits = (sum(column) / len(column) for column in zip(*sides))
    return Stats(loss=loss, pos_rank=pos_rank, mrr=mrr, r1=r1, r10=r10, r50=r50, auc=count * hits / auc_samples, count=count)


class RankingEvaluator(AbstractBatchProcessor):
    """eval.py:43-86: rank of each positive among its negatives (ties count
    against the positive), MRR, hits@1/10/50 and a randomized AUC, averaged over
    the sides that have negatives; sums over the batch, to be divided by count."""

    def _process_one_batch(self, model: MultiRelationEmbedder, batch_edges: EdgeList) -> Stats:
        # Without a score filter (the _adjust_scores hook) nothing needs the [B, N] score matrices: ranks,
        # loss and the AUC count come from one call, summed on the device.
        if type(self)._adjust_scores is RankingEvaluator._adjust_scores and len(batch_edges) > 0:
            count = len(batch_edges)
            kind = batch_edges.get_relation_type_as_scalar() if batch_edges.has_scalar_relation_type() else 0
            loss, sides = model.rank_sums(batch_edges, loss=self.loss_fn.loss_name, margin=self.loss_fn.fused_margin,
                                          relation_weight=float(self.relation_weights[kind]), auc_samples=count,
                                          auc_seed=int(torch.randint(0, 2**62, (1,))))
            return ranking_stats_from_sums(sides, loss, count, count)
        with torch.no_grad():
            scores, _ = model(batch_edges)
        self._adjust_scores(scores, batch_edges)
        loss = self.calc_loss(scores, batch_edges)
        return ranking_stats(((scores.lhs_pos, scores.lhs_neg), (scores.rhs_pos, scores.rhs_neg)), float(loss),
                             len(batch_edges))

    def _adjust_scores(self, scores: Scores, batch_edges: EdgeList) -> None:
        """Hook for a filtered evaluator (eval.py:82-86)."""
