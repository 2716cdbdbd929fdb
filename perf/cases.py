"""Performance cases: the work a user of this framework has it do, with sizes, inputs and the least it costs.

A case is a dict of plain values; `kind` says which entry point it goes through:

  step         StepRunner.train: one call of `workers` lock-step batches (forward, loss, backward, both optimizers)
  trainer      Trainer.process_one_batch on one EdgeList: the reference's per-batch loop, statistics read on the host
  evaluator    RankingEvaluator.process_one_batch: ranks of a batch's edges among batch and uniform negatives
  epoch        BucketLoop.train_epoch: every bucket of a partitioned graph, partitions swapped from pinned host memory
  repartition  the `_C` helpers as partition-wise training uses them: permutation, its inverse, the shuffle of a
               partition's rows and Adagrad sums, the split of the bucket's edges

Tables are those of a run under way: entries of a size that gives scores of order one, Adagrad sums of order one,
relation parameters near the identity.  `skew` is s in P(entity of rank r) ~ r^-s (0: uniform), ranks assigned to
entities by a random permutation; `rel_skew` the same for relation types.
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

pbg = load_package()
DEVICE = "cuda:0"
LR = 0.1
MARGIN = 0.1


# --- cases ------------------------------------------------------------------
def step_case(name=None, **fields):
    case = dict(kind="step", dim=100, batch=1000, workers=1, batch_negs=50, uniform_negs=50, entities=100_000, tables=1,
                operator="none", comparator="dot", loss="ranking", relations=1, dynamic=False, skew=0.0, rel_skew=0.0,
                n3=0.0, half=False)
    assert set(fields) <= set(case)
    case.update(fields)
    if name is not None:
        case["name"] = name
    return case


def listed():
    social = dict(dim=100, batch=1000, batch_negs=50, uniform_negs=50, entities=100_000, operator="none", comparator="dot",
                  loss="ranking")
    return [
        # One batch through the plugin-level trainer, as code written against the reference's Trainer drives it:
        # the smallest call, where launches, host work and the read-back of the statistics count.
        dict(name="trainer-batch", kind="trainer", dim=100, batch=1000, batch_negs=50, uniform_negs=50, entities=100_000,
             operator="none", comparator="dot", loss="ranking", skew=0.75),
        # Strictly sequential training of a social graph: one batch per call.
        step_case("social-sequential", workers=1, **social),
        # The same with 64 batches per call: the headline workload.
        step_case("social-64", workers=64, **social),
        # One bucket of a 4 x 4 partitioned knowledge base (two resident 10.4M-row partitions, TransE), hot entities.
        step_case("wiki-translation-l2", workers=64, entities=10_413_058, tables=2, operator="translation", comparator="l2",
                  skew=1.8),
        # The FB15k example as configured: ComplEx, one relation per edge, 1000 uniform negatives, N3 regularizer.
        step_case("fb15k-complex", dim=400, workers=64, uniform_negs=1000, entities=14_951, operator="complex_diagonal",
                  loss="softmax", relations=1345, dynamic=True, skew=1.1, rel_skew=1.1, n3=1e-3),
        # A social graph at dim 1024 with wide shared negatives and large batches: the matrix-product-bound case.
        step_case("livejournal-softmax", dim=1024, batch=10_000, workers=8, batch_negs=1000, uniform_negs=100,
                  entities=4_847_571, loss="softmax", skew=0.75),
        # The same under half_precision.
        step_case("livejournal-softmax-half", dim=1024, batch=10_000, workers=8, batch_negs=1000, uniform_negs=100,
                  entities=4_847_571, loss="softmax", skew=0.75, half=True),
        # The LiveJournal example as configured: the default comparator and negatives on wide rows.
        step_case("livejournal-cos", dim=1024, workers=64, entities=4_847_571, comparator="cos", skew=0.75),
        # RESCAL-like: a matrix per relation, mixed batches.
        step_case("linear-logistic", dim=256, batch=2000, workers=64, batch_negs=100, uniform_negs=100, entities=2_000_000,
                  operator="linear", comparator="cos", loss="logistic", relations=500, dynamic=True, rel_skew=1.2),
        # Evaluation with the configuration's default 1000 + 1000 candidates (forward only).
        dict(name="evaluate-ranks", kind="evaluator", dim=400, batch=10_000, batch_negs=1000, uniform_negs=1000, entities=1_000_000,
             operator="none", comparator="dot", loss="softmax", skew=0.75),
        # A whole pass over a partitioned graph whose edges and partitions live in host memory.
        dict(name="bucket-epoch", kind="epoch", dim=100, batch=1000, workers=64, batch_negs=50, uniform_negs=50, partitions=4,
             rows=100_000, edges=200_000, resident=3, operator="translation", comparator="l2", loss="ranking", relations=1,
             eval_fraction=0.0, skew=0.75),
        # What a partition and a bucket go through before they are split over sub-partitions.
        dict(name="repartition", kind="repartition", rows=10_413_058, dim=100, edges=20_000_000, parts=8, skew=1.0),
    ]


def log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw_once(rng):
    family = rng.choice(("narrow", "narrow", "wide", "relations", "contraction", "linear", "trainer", "evaluator", "epoch", "repartition"))
    loss = rng.choice(("ranking", "softmax", "logistic"))
    if family == "narrow":  # a chunk's rows fit a compute unit: social and TransE graphs
        return step_case(dim=rng.choice((64, 100, 128, log_int(rng, 32, 128))), batch=log_int(rng, 250, 4000), workers=log_int(rng, 1, 64),
                         batch_negs=rng.randint(20, 60), uniform_negs=rng.randint(20, 60), entities=log_int(rng, 10_000, 10_000_000),
                         tables=rng.choice((1, 2)), operator=rng.choice(("none", "translation", "diagonal")),
                         comparator=rng.choice(("dot", "cos", "l2")), loss=loss, skew=rng.choice((0.0, 0.75, 1.8)))
    if family == "wide":  # the default negatives on rows wider than that
        return step_case(dim=rng.choice((200, 400, 1024, 4 * log_int(rng, 33, 256))), batch=log_int(rng, 250, 2000), workers=log_int(rng, 4, 64),
                         batch_negs=rng.randint(20, 50), uniform_negs=rng.randint(20, 50), entities=log_int(rng, 10_000, 4_000_000),
                         operator=rng.choice(("none", "translation")), comparator=rng.choice(("dot", "cos", "l2")), loss=loss,
                         skew=rng.choice((0.0, 0.75)))
    if family == "relations":  # many relation types, many uniform negatives
        return step_case(dim=rng.choice((128, 200, 256, 400)), batch=log_int(rng, 250, 2000), workers=log_int(rng, 2, 64), batch_negs=rng.randint(20, 60),
                         uniform_negs=log_int(rng, 150, 1000), entities=log_int(rng, 10_000, 1_000_000),
                         operator=rng.choice(("complex_diagonal", "diagonal")), loss=rng.choice(("softmax", "ranking")),
                         relations=log_int(rng, 10, 2000), dynamic=rng.random() < 0.6, skew=1.1, rel_skew=1.1)
    if family == "contraction":  # large chunks
        half = rng.random() < 0.3
        return step_case(dim=rng.choice((128, 256, 400, 1024, log_int(rng, 100, 1024))), batch=log_int(rng, 1000, 10_000), workers=log_int(rng, 1, 8),
                         batch_negs=log_int(rng, 150, 1000), uniform_negs=rng.choice((0, 50, 100, rng.randint(1, 200))),
                         entities=log_int(rng, 10_000, 4_000_000), comparator=rng.choice(("dot", "cos") if half else ("dot", "cos", "l2")),
                         loss=rng.choice(("softmax", "logistic")), skew=0.75, half=half)
    if family == "linear":
        return step_case(dim=rng.choice((64, 100, 128, 200, 256)), batch=log_int(rng, 500, 2000), workers=log_int(rng, 4, 64),
                         batch_negs=rng.randint(50, 100), uniform_negs=rng.randint(50, 100), entities=log_int(rng, 10_000, 2_000_000),
                         operator="linear", comparator=rng.choice(("dot", "cos")), loss=rng.choice(("softmax", "logistic")),
                         relations=log_int(rng, 10, 500), dynamic=rng.random() < 0.7, rel_skew=1.2)
    if family == "trainer":
        return dict(kind="trainer", dim=rng.choice((64, 100, 200, 400, log_int(rng, 32, 400))), batch=log_int(rng, 100, 4000), batch_negs=rng.randint(20, 60),
                    uniform_negs=rng.randint(20, 60), entities=log_int(rng, 10_000, 1_000_000),
                    operator=rng.choice(("none", "translation", "diagonal", "complex_diagonal")), comparator=rng.choice(("dot", "cos")), loss=loss,
                    skew=0.75)
    if family == "evaluator":
        return dict(kind="evaluator", dim=rng.choice((100, 128, 400, 1024, log_int(rng, 64, 1024))), batch=log_int(rng, 500, 10_000), batch_negs=log_int(rng, 100, 1000),
                    uniform_negs=log_int(rng, 100, 1000), entities=log_int(rng, 10_000, 1_000_000), operator=rng.choice(("none", "translation", "diagonal")),
                    comparator=rng.choice(("dot", "cos")), loss=loss, skew=0.75)
    if family == "epoch":
        return dict(kind="epoch", dim=rng.choice((64, 100, log_int(rng, 32, 128))), batch=log_int(rng, 500, 2000), workers=rng.choice((16, 64)), batch_negs=rng.randint(20, 60),
                    uniform_negs=rng.randint(20, 60), partitions=rng.randint(2, 4), rows=log_int(rng, 20_000, 150_000), edges=log_int(rng, 50_000, 250_000),
                    resident=rng.choice((2, 3)), operator=rng.choice(("none", "translation", "diagonal")), comparator=rng.choice(("dot", "cos", "l2")), loss=loss,
                    relations=rng.choice((1, 1, rng.randint(2, 40))), eval_fraction=rng.choice((0.0, 0.0, 0.05)), skew=0.75)
    return dict(kind="repartition", rows=log_int(rng, 100_000, 10_000_000), dim=rng.choice((64, 100, 128, 400, log_int(rng, 32, 512))),
                edges=log_int(rng, 1_000_000, 20_000_000), parts=rng.choice((2, 4, 8)), skew=rng.choice((0.0, 1.0)))


#: no drawn case costs more than the largest listed one
MOST_FLOPS = 1.1e12
MOST_BYTES = 9.5e9
MOST_TABLE = 20e9


def draw(rng):
    while True:
        case = draw_once(rng)
        if case.get("operator") == "complex_diagonal":
            case["dim"] -= case["dim"] % 2
        w = work(case)
        rows = case.get("rows", case.get("entities", 0)) * case.get("tables", 1)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES and 4.0 * rows * case["dim"] <= MOST_TABLE:
            return case


# --- inputs -----------------------------------------------------------------
class Source:
    """Random inputs on the GPU, from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(int(seed))

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.gen, device=DEVICE).mul_(scale)

    def positive(self, *shape):
        """Adagrad sums: 0.5 ... 1.5."""
        return torch.rand(*shape, generator=self.gen, device=DEVICE).add_(0.5)

    def ids(self, n, count, skew):
        if skew == 0.0:
            return torch.randint(0, count, (n,), generator=self.gen, device=DEVICE)
        a = 1.0 - skew
        u = torch.rand(n, generator=self.gen, device=DEVICE, dtype=torch.float64)
        rank = torch.exp(u * math.log(count)) if abs(a) < 1e-9 else ((count ** a - 1.0) * u + 1.0) ** (1.0 / a)
        rank = (rank.floor().long() - 1).clamp_(0, count - 1)
        return torch.randperm(count, generator=self.gen, device=DEVICE)[rank]


def entry_scale(case):
    """Entries that make a score of two random rows of order one."""
    return case["dim"] ** (-0.25 if case["comparator"] == "dot" else -0.5)


def operator_parameters(case, src):
    """Parameters of the case's operator near the identity, and their Adagrad sums."""
    r, d = case["relations"], case["dim"]
    if case["operator"] == "none":
        return {}, {}
    if case["operator"] == "complex_diagonal":
        p = {"real": 1.0 + src.normal(r, d // 2, scale=0.1), "imag": src.normal(r, d // 2, scale=0.1)}
    elif case["operator"] == "translation":
        p = {"translation": src.normal(r, d, scale=0.1 * entry_scale(case))}
    elif case["operator"] == "diagonal":
        p = {"diagonal": 1.0 + src.normal(r, d, scale=0.1)}
    else:
        p = {"linear_transformation": torch.eye(d, device=DEVICE) + src.normal(r, d, d, scale=0.1 / math.sqrt(d))}
    return p, {k: src.positive(*v.shape) for k, v in p.items()}


def prepare(case, seed):
    return {"step": prepare_step, "trainer": prepare_trainer, "evaluator": prepare_evaluator, "epoch": prepare_epoch,
            "repartition": prepare_repartition}[case["kind"]](case, seed)


def prepare_step(case, seed):
    src = Source(seed)
    k, b, d = case["workers"], case["batch"], case["dim"]
    w = [src.normal(case["entities"], d, scale=entry_scale(case)) for _ in range(case["tables"])]
    g = [src.positive(case["entities"]) for _ in range(case["tables"])]
    rhs_op, rhs_sum = operator_parameters(case, src)
    lhs_op, lhs_sum = operator_parameters(case, src) if case["dynamic"] else ({}, {})
    spec = pbg.StepSpec(dim=d, batch_size=b, num_workers=k, num_batch_negs=case["batch_negs"], num_uniform_negs=case["uniform_negs"],
                        operator=case["operator"], dynamic=case["dynamic"], num_relations=case["relations"], comparator=case["comparator"],
                        loss=case["loss"], margin=MARGIN, lr=LR, regularization_coef=case["n3"], half_precision=case["half"])
    runner = pbg.StepRunner(spec, w[0], g[0], w[1] if len(w) > 1 else None, g[1] if len(g) > 1 else None, rhs_op, rhs_sum, lhs_op, lhs_sum)
    calls = []  # a bucket's edges, cut into calls
    for _ in range(2):
        lhs, rhs = src.ids(k * b, case["entities"], case["skew"]), src.ids(k * b, case["entities"], case["skew"])
        rel = src.ids(k * b if case["dynamic"] else k, case["relations"], case["rel_skew"])
        if case["dynamic"]:
            rel = rel.view(k, b).sort(dim=1).values.reshape(-1)
        calls.append((lhs, rhs, rel))
    state = {"w_" + str(i): t for i, t in enumerate(w)}
    state.update({"g_" + str(i): t for i, t in enumerate(g)})
    for name, params in (("rhs", rhs_op), ("rhs_sum", rhs_sum), ("lhs", lhs_op), ("lhs_sum", lhs_sum)):
        state.update({name + "_" + key: t for key, t in params.items()})
    return {"kind": "step", "runner": runner, "calls": calls, "count": 0, "seed": int(seed) << 24, "edges": float(b), "n3": case["n3"] != 0,
            "trained": state}


def build_model(case, src):
    d = case["dim"]
    weight = torch.nn.Parameter(src.normal(case["entities"], d, scale=entry_scale(case)))
    rhs_op = pbg.operators.instantiate_operator(case["operator"], pbg.types.Side.RHS, 0, d).to(DEVICE)
    with torch.no_grad():
        for p in rhs_op.parameters():
            p.add_(src.normal(*p.shape, scale=0.1 * entry_scale(case)))
    model = pbg.model.MultiRelationEmbedder(
        d, [pbg.config.RelationSchema(name="follows", lhs="user", rhs="user", operator=case["operator"])], {"user": pbg.config.EntitySchema()},
        case["batch_negs"], case["uniform_negs"], False, False, [None], [rhs_op], pbg.model.COMPARATORS.get_class(case["comparator"])())
    for side in (pbg.types.Side.LHS, pbg.types.Side.RHS):
        model.set_embeddings("user", side, weight)
    loss_fn = pbg.losses.LOSS_FUNCTIONS.get_class(case["loss"])(margin=MARGIN)
    return model, weight, loss_fn


def edge_lists(case, src, count):
    entities = pbg.entitylist.EntityList
    rel = torch.tensor(0)
    return [pbg.edgelist.EdgeList(entities.from_tensor(src.ids(case["batch"], case["entities"], case["skew"])),
                                  entities.from_tensor(src.ids(case["batch"], case["entities"], case["skew"])), rel) for _ in range(count)]


def prepare_trainer(case, seed):
    src = Source(seed)
    model, weight, loss_fn = build_model(case, src)
    train = pbg.train
    relation = list(model.parameters())
    relation = [p for p in relation if p is not weight]
    trainer = train.Trainer(train.make_optimizer(relation, False, LR), loss_fn, [1.0])
    optimizer = train.make_optimizer([weight], True, LR)
    trainer.partitioned_optimizers[("user", 0)] = optimizer
    sums = optimizer.state[weight]["sum"]
    sums.copy_(src.positive(*sums.shape))
    batches = edge_lists(case, src, 4)
    trained = {"w": weight.detach(), "g": sums}
    trained.update({"op_%d" % i: p.detach() for i, p in enumerate(relation)})
    torch.manual_seed(int(seed))  # the uniform negatives are drawn with torch's generator
    return {"kind": "trainer", "model": model, "trainer": trainer, "batches": batches, "count": 0, "trained": trained}


def prepare_evaluator(case, seed):
    src = Source(seed)
    model, _, loss_fn = build_model(case, src)
    evaluator = pbg.eval.RankingEvaluator(loss_fn, [1.0])
    batches = edge_lists(case, src, 2)
    torch.manual_seed(int(seed))
    return {"kind": "evaluator", "model": model, "evaluator": evaluator, "batches": batches, "count": 0}


def prepare_epoch(case, seed):
    src = Source(seed)
    loops, parts, rows, n = pbg.bucket_loop, case["partitions"], case["rows"], case["edges"]
    store = loops.PartitionStore()
    for p in range(parts):
        store.add(("user", p), src.normal(rows, case["dim"], scale=entry_scale(case)).cpu(), src.positive(rows).cpu())
    edges = {}
    for i in range(parts):
        for j in range(parts):
            edges[loops.Bucket(i, j)] = tuple(t.cpu() for t in (src.ids(n, rows, case["skew"]), src.ids(n, rows, case["skew"]),
                                                               src.ids(n, case["relations"], 0.75 if case["relations"] > 1 else 0.0)))
    rhs_op, rhs_sum = operator_parameters(case, src)
    loop = loops.BucketLoop(store, edges, lhs_entity="user", rhs_entity="user", nparts_lhs=parts, nparts_rhs=parts, dim=case["dim"],
                            batch_size=case["batch"], num_workers=case["workers"], num_batch_negs=case["batch_negs"],
                            num_uniform_negs=case["uniform_negs"], operator=case["operator"], comparator=case["comparator"], loss=case["loss"],
                            margin=MARGIN, lr=LR, num_relations=case["relations"], rhs_op=rhs_op, rhs_op_sum=rhs_sum,
                            resident_partitions=case["resident"], eval_fraction=case["eval_fraction"], seed=int(seed) % 65536)
    trained = {"w_%d" % p: store.tables[("user", p)] for p in range(parts)}
    trained.update({"g_%d" % p: store.sums[("user", p)] for p in range(parts)})
    trained.update({"op_" + k: v for k, v in rhs_op.items()})
    return {"kind": "epoch", "loop": loop, "trained": trained}


def prepare_repartition(case, seed):
    src = Source(seed)
    rows, n = case["rows"], case["edges"]
    lhs, rhs = src.ids(n, rows, case["skew"]), src.ids(n, rows, case["skew"])
    out = [torch.empty_like(lhs) for _ in range(3)]
    return {"kind": "repartition", "rows": rows, "parts": case["parts"], "seed": int(seed) & 0xFFFFFF, "table": src.normal(rows, case["dim"]),
            "sums": src.positive(rows), "edges": (lhs, rhs, torch.zeros_like(lhs)), "out": out}


# --- one pass ---------------------------------------------------------------
def run(state):
    return {"step": run_step, "trainer": run_trainer, "evaluator": run_evaluator, "epoch": run_epoch,
            "repartition": run_repartition}[state["kind"]](state)


def run_step(state):
    runner = state["runner"]
    i = state["count"]
    state["count"] = i + 1
    lhs, rhs, rel = state["calls"][i % len(state["calls"])]
    runner.train(lhs, rhs, rel, uniform_seed=state["seed"] + i)  # the step draws its uniform negatives, a fresh seed per call
    out = {"loss": runner.loss_out, "violators_per_edge": runner.violators_out / state["edges"], **state["trained"]}
    if state["n3"]:
        out["reg"] = runner.reg_out
    return out


def run_trainer(state):
    i = state["count"]
    state["count"] = i + 1
    stats = state["trainer"].process_one_batch(state["model"], state["batches"][i % len(state["batches"])])
    return {"stats": stats.average().to_dict(), **state["trained"]}


def run_evaluator(state):
    i = state["count"]
    state["count"] = i + 1
    stats = state["evaluator"].process_one_batch(state["model"], state["batches"][i % len(state["batches"])])
    return stats.average().to_dict()


def run_epoch(state):
    stats = state["loop"].train_epoch()
    out = {"edges": np.array([s.num_edges for s in stats]), "loss": np.array([s.loss for s in stats]),
           "violators_per_edge": np.array([(s.violators_lhs / s.num_edges, s.violators_rhs / s.num_edges) for s in stats])}
    for when in ("eval_before", "eval_after"):
        held = [getattr(s, when) for s in stats]
        if all(h is not None for h in held):
            out[when] = {name: np.array([h.average().metrics[name] for h in held]) for name in held[0].metrics}
    return {**out, **state["trained"]}


def run_repartition(state):
    helpers, (lhs, rhs, rel), out, rows = pbg._C, state["edges"], state["out"], state["rows"]
    perm = helpers.randperm(rows, 8, state["seed"])
    inverse = helpers.reverse_permutation(perm, 8)
    helpers.shuffle(state["table"], perm, 8)
    helpers.shuffle(state["sums"], perm, 8)
    split = helpers.sub_bucket(lhs, rhs, rel, [rows], [perm], [rows], [inverse], out[0], out[1], out[2], state["parts"], state["parts"], 8, False)
    sizes = np.array([len(v[0]) for v in split.values()])
    return {"perm": perm, "inverse": inverse, "table": state["table"], "sums": state["sums"], "lhs": out[0], "rhs": out[1], "rel": out[2],
            "sizes": sizes}


# --- the least a pass costs -------------------------------------------------
def distinct(draws, count, skew):
    """Expected number of different ids among `draws` draws of Source.ids."""
    if skew == 0.0:
        return count * -math.expm1(-draws / count)
    edges = np.unique(np.floor(np.geomspace(1, count + 1, 2000)))  # ranks [edges[i], edges[i + 1]) share a probability
    a = 1.0 - skew
    cdf = np.log(edges) / math.log(count + 1) if abs(a) < 1e-9 else (edges ** a - 1.0) / ((count + 1) ** a - 1.0)
    size = np.diff(edges)
    return float(np.sum(size * -np.expm1(-draws * np.diff(cdf) / size)))


def step_work(case, workers, batch, tables=1):
    """(bytes, flops) of training `workers` batches: the distinct table rows and Adagrad sums read and written, the
    ids read, the relations' parameters; three products (scores, two gradients) of both sides, six per operated row
    and value pair for a linear operator."""
    d, u = case["dim"], case["uniform_negs"]
    p = min(case["batch_negs"], batch)
    chunks = -(-batch // p)
    relations, dynamic = case.get("relations", 1), case.get("dynamic", False)
    rows = 0.0
    for side in range(tables):
        ends = workers * batch * (2 if tables == 1 else 1)
        negs = workers * chunks * u * (2 if tables == 1 else 1)
        named = distinct(ends, case["entities"], case["skew"])
        rows += named + (case["entities"] - named) * -math.expm1(-negs / case["entities"])
    nbytes = rows * (8 * d + 8) + workers * batch * (24 if dynamic else 16)
    flops = 3 * 2.0 * workers * (batch * d + 2.0 * chunks * p * (p + u) * d)
    kinds = distinct(workers * batch if dynamic else workers, relations, case.get("rel_skew", 0.0)) * (2 if dynamic else 1)
    size = {"none": 0, "linear": d * d}.get(case["operator"], d)
    nbytes += kinds * size * 16
    if case["operator"] == "linear":
        flops += 3 * 2.0 * workers * (2 * batch if dynamic else batch + chunks * u) * d * d
    return nbytes, flops


def work(case):
    kind, d = case["kind"], case["dim"]
    if kind == "step":
        nbytes, flops = step_work(case, case["workers"], case["batch"], case["tables"])
    elif kind == "trainer":
        nbytes, flops = step_work(case, 1, case["batch"])
    elif kind == "evaluator":
        p = min(case["batch_negs"], case["batch"])
        chunks = -(-case["batch"] // p)
        u = case["uniform_negs"]
        rows = min(case["entities"], distinct(2 * case["batch"], case["entities"], case["skew"]) + distinct(2 * chunks * u, case["entities"], 0.0))
        nbytes, flops = rows * 4 * d + 16 * case["batch"], 2.0 * (case["batch"] * d + 2.0 * chunks * p * (p + u) * d)
    elif kind == "epoch":
        # per bucket: both partitions' touched rows trained, the edges uploaded; per pass every partition up and down once
        buckets, parts = case["partitions"] ** 2, case["partitions"]
        b, f = step_work(dict(case, entities=case["rows"]), max(1, case["edges"] // case["batch"]), case["batch"], 2)
        nbytes, flops = buckets * (b + 24 * case["edges"]) + 2 * parts * case["rows"] * (4 * d + 4), buckets * f
    else:
        # permutation and inverse written, rows and sums moved, per edge three ids read and written and two places looked up
        nbytes, flops = case["rows"] * (8 + 16 + 8 * d + 8 + 8) + case["edges"] * (48 + 16), 0.0
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "repartition":
        return "exact"
    if case["kind"] == "evaluator":
        return {"rel": 1e-4}  # a score within rounding of the positive's changes a rank by one, and with it hits and AUC counts
    if case.get("half"):
        # float16 products (2^-11 each): a gradient entry differs by about 1e-3, an update by lr times that
        return {"rel": 2e-3, "max": 0.1}
    if case["loss"] == "ranking":
        # 32-bit sums; a hinge argument within rounding of zero adds or leaves out one negative's row (about one pair in
        # 1e7), which moves the two rows it belongs to by up to lr times a row's size
        return {"rel": 1e-4, "max": 0.5}
    # 32-bit sums, 1e-5; the counts of violators tie as ranks do
    return {"rel": 1e-4, "max": 4e-3}
