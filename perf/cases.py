"""The calls that this package's speed is judged by.

A case is one call of a public metric (or a forward and its gradients), described by plain
values: the metric, the data type, whether gradients are taken, and the sizes.  The listed ones
are the benchmark's configurations and ordinary calls of the same metrics at small, middle and
ragged sizes; ``draw`` gives more of the same ranges.

Keys of a case: ``metric``; ``dtype`` of the points; ``grad`` (take both gradients for a given
upstream gradient); ``b`` (0: two-dimensional points), ``n``, ``m`` (0: the points against
themselves), ``d`` (hausdorff: ``n`` and ``m`` clouds of ``d`` points in space); ``arg`` (p of
minkowski, k of the neighbour mask, the share of set bits of the boolean metrics, 0 where there
is none).
"""
import torch

import torchpairwise as tp

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "bool": torch.bool}
PRODUCTS = ("euclidean", "cosine")
BOOLEAN = ("hamming", "jaccard")


def _case(metric, dtype, grad, b, n, m, d, arg=0.0, name=None):
    case = {"metric": metric, "dtype": dtype, "grad": grad, "b": b, "n": n, "m": m, "d": d, "arg": arg}
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # one training step's contrastive loss over a mini-batch of embeddings: launches and host
        # time count, not arithmetic
        _case("cosine", "fp32", True, 0, 64, 64, 128, name="cosine_minibatch_grad"),
        # a few query vectors against a codebook of an odd size and width (vector quantisation)
        _case("euclidean", "fp32", False, 0, 37, 1003, 50, name="euclidean_codebook"),
        # the headline configuration: the full distance matrix of two 16k point sets
        _case("euclidean", "fp32", False, 0, 16384, 16384, 128, name="euclidean_16k"),
        # batched metric learning with gradients, in both of the matrix cores' types
        _case("euclidean", "fp32", True, 8, 8192, 8192, 256, name="euclidean_batched_grad"),
        _case("cosine", "bf16", True, 8, 8192, 8192, 256, name="cosine_batched_grad_bf16"),
        # an L1 loss between two sets of ordinary, odd sizes
        _case("manhattan", "fp32", True, 0, 3001, 1999, 100, name="manhattan_odd_grad"),
        # the general-p configuration: the largest of the non-product kernels
        _case("minkowski", "fp32", True, 0, 16384, 16384, 128, 3.0, name="minkowski3_16k_grad"),
        # an RBF kernel matrix with gradients (kernel regression, MMD losses) at an odd width
        _case("rbf", "fp32", True, 0, 4096, 4000, 90, name="rbf_kernel_grad"),
        # the boolean configuration: long fingerprints, all pairs
        _case("jaccard", "bool", False, 0, 32768, 32768, 1024, 0.1, name="jaccard_32k"),
        # short structural keys, a library of an odd size searched by an ordinary batch
        _case("hamming", "bool", False, 0, 2000, 30011, 166, 0.3, name="hamming_keys"),
        # a k-nearest-neighbour graph of one point set
        _case("knn_mask", "fp32", False, 0, 10007, 0, 96, 10, name="knn_graph"),
        # directed Hausdorff between all pairs of two batches of large point clouds, as a loss
        _case("hausdorff", "fp32", True, 0, 16, 16, 65536, name="hausdorff_clouds_grad"),
    ]


def _size(rng, low, high):
    """A size between low and high, even over its logarithm; every other one a multiple of 32."""
    v = int(round(low * (high / low) ** rng.random()))
    return min(high, -(-v // 32) * 32) if rng.random() < 0.5 and low >= 32 else v


def draw(rng):
    metric = rng.choice(["euclidean", "cosine", "euclidean", "cosine", "manhattan", "minkowski", "rbf",
                         "hamming", "jaccard", "knn_mask", "hausdorff"])
    if metric in PRODUCTS:
        # to the batched configuration's sizes; its work bounds the product of them
        dtype, grad, b = rng.choice(["fp32", "bf16"]), rng.random() < 0.5, rng.choice([0, 0, 2, 8])
        d = _size(rng, 32, 512)
        n, m = _size(rng, 32, 16384), _size(rng, 32, 16384)
        while max(1, b) * n * m * d > 8 * 8192 * 8192 * 256:
            n, m = -(-n // 2), -(-m // 2)
        return _case(metric, dtype, grad, b, n, m, d)
    if metric in ("manhattan", "minkowski", "rbf"):
        grad, b, d = rng.random() < 0.5, rng.choice([0, 0, 4]), _size(rng, 8, 256)
        n, m = _size(rng, 32, 16384), _size(rng, 32, 16384)
        p = rng.choice([1.5, 3.0]) if metric == "minkowski" else 0.0
        # a fractional power costs a logarithm and an exponential where p = 3 costs products
        while max(1, b) * n * m * d > 16384 * 16384 * (16 if p == 1.5 else 128):
            n, m = -(-n // 2), -(-m // 2)
        return _case(metric, "fp32", grad, b, n, m, d, p)
    if metric in BOOLEAN:
        n, m = _size(rng, 64, 32768), _size(rng, 64, 32768)
        return _case(metric, "bool", False, 0, n, m, _size(rng, 32, 2048), rng.choice([0.1, 0.3, 0.5]))
    if metric == "knn_mask":
        n = _size(rng, 300, 16384)
        return _case(metric, "fp32", False, 0, n, 0, _size(rng, 16, 256), rng.choice([1, 5, 10, 20]))
    clouds = rng.choice([1, 4, 8, 16])
    return _case("hausdorff", "fp32", rng.random() < 0.5, 0, clouds, rng.choice([1, clouds]), _size(rng, 256, 65536))


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    b, n, m, d = (case[k] for k in ("b", "n", "m", "d"))
    if case["metric"] == "hausdorff":  # n and m clouds of d points in space, the second set shifted
        x1 = torch.rand(n, d, 3, generator=g, device="cuda")
        x2 = torch.rand(m, d, 3, generator=g, device="cuda").add_(0.05)
        return x1, x2, torch.randn(n, m, generator=g, device="cuda") if case["grad"] else None
    lead = (b,) if b else ()
    if case["dtype"] == "bool":
        x1 = torch.rand(n, d, generator=g, device="cuda") < case["arg"]
        x2 = torch.rand(m, d, generator=g, device="cuda") < case["arg"]
        return x1, x2, None
    dtype = DTYPES[case["dtype"]]
    x1 = torch.randn(*lead, n, d, generator=g, device="cuda").to(dtype)
    x2 = torch.randn(*lead, m, d, generator=g, device="cuda").to(dtype) if m else None
    gout = torch.randn(*lead, n, m, generator=g, device="cuda").to(dtype) if case["grad"] else None
    return x1, x2, gout


def prepare(case, seed):
    x1, x2, gout = _inputs(case, seed)
    if case["grad"]:
        x1.requires_grad_()
        x2.requires_grad_()
    return {"metric": case["metric"], "arg": case["arg"], "x1": x1, "x2": x2, "gout": gout}


def _call(metric, arg, x1, x2):
    if metric == "minkowski":
        return tp.minkowski_distances(x1, x2, arg)
    if metric == "rbf":
        return tp.rbf_kernel(x1, x2)
    if metric == "knn_mask":
        return tp.k_neighbors_mask(x1, x2, int(arg))
    if metric == "hausdorff":
        return tp.directed_hausdorff_distances(x1, x2)[0]
    return getattr(tp, metric + "_distances")(x1, x2)


def run(state):
    x1, x2, gout = state["x1"], state["x2"], state["gout"]
    out = _call(state["metric"], state["arg"], x1, x2)
    if gout is None:
        return {"out": out}
    g1, g2 = torch.autograd.grad(out, (x1, x2), gout)
    return {"out": out.detach(), "grad1": g1, "grad2": g2}


def work(case):
    metric, b, n, m, d = case["metric"], max(1, case["b"]), case["n"], case["m"], case["d"]
    passes = 3 if case["grad"] else 1  # a forward and a pass of the same size for each gradient
    if metric == "hausdorff":
        # the inputs once (and the gradients); a nearest-point search cannot do without a test
        # of each point, eight operations a test
        points = (n + m) * d * 3
        return {"bytes": 4.0 * points * (2 if case["grad"] else 1) + 8.0 * n * m, "flops": 8.0 * n * m * d}
    m = m or n
    e = {"fp32": 4, "bf16": 2, "bool": 1}[case["dtype"]]
    inputs, pairs = b * (n + (m if case["m"] else 0)) * d * e, b * n * m
    if metric == "knn_mask":
        return {"bytes": float(inputs + pairs), "flops": 2.0 * pairs * d}
    if metric in BOOLEAN:
        return {"bytes": float(inputs + 4 * pairs), "flops": 2.0 * pairs * d}
    per = {"minkowski": 4.0, "rbf": 3.0}.get(metric, 2.0)
    return {"bytes": float(inputs * (2 if case["grad"] else 1) + e * pairs * (2 if case["grad"] else 1)),
            "flops": per * passes * pairs * d}


def tolerance(case):
    metric = case["metric"]
    if metric == "knn_mask":
        # two neighbours whose distances round alike may swap: a few of n * n mask bytes
        return {"rel": 0.0, "max": 0.0, "differ": 1e-5}
    if metric in BOOLEAN or metric == "hausdorff":
        return "exact"  # counts and one quotient; a selection of the given points
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.1}
    # sums over the features and, for gradients, over the pairs, in 32 bits
    return {"rel": 1e-5, "max": 1e-3}


def _exact_block(case, x1, x2):
    """The metric of rows x1 against x2, both in 64 bits."""
    metric = case["metric"]
    if metric == "euclidean":
        sq = x1.square().sum(1)[:, None] + x2.square().sum(1)[None, :] - 2 * (x1 @ x2.T)
        return sq.clamp_min(0).sqrt()
    if metric == "cosine":
        return 1 - (x1 @ x2.T) / (x1.norm(dim=1)[:, None] * x2.norm(dim=1)[None, :])
    if metric == "hamming":
        eq = x1 @ x2.T + (1 - x1) @ (1 - x2).T
        return (x1.shape[1] - eq) / x1.shape[1]
    if metric == "jaccard":
        both = x1 @ x2.T
        either = x1.sum(1)[:, None] + x2.sum(1)[None, :] - both
        return torch.where(either > 0, (either - both) / either.clamp_min(1), torch.zeros_like(either))
    diff = (x1[:, None, :] - x2[None, :, :]).abs()
    if metric == "manhattan":
        return diff.sum(-1)
    if metric == "minkowski":
        p = case["arg"]
        return diff.pow(p).sum(-1).pow(1 / p)
    return (diff.square().sum(-1) * (-1.0 / x1.shape[1])).exp()  # rbf


def exact(case, seed):
    if case["metric"] in ("knn_mask", "hausdorff"):
        return None
    x1, x2, gout = _inputs(case, seed)
    lead, (n, d), m = max(1, case["b"]), x1.shape[-2:], x2.shape[-2]
    x1, x2 = x1.view(lead, n, d), x2.view(lead, m, d)
    # rows at a time: 2^26 differences of the sum metrics, 2^28 entries of the others
    direct = case["metric"] in ("manhattan", "minkowski", "rbf")
    rows = max(1, min(n, (2 ** 26 // (m * d)) if direct else (2 ** 28 // m)))
    out = torch.empty(lead, n, m, dtype=torch.float64, device="cuda")
    if case["grad"]:
        gout = gout.view(lead, n, m)
        g1 = torch.empty(lead, n, d, dtype=torch.float64, device="cuda")
        g2 = torch.zeros(lead, m, d, dtype=torch.float64, device="cuda")
    for i in range(lead):
        whole = x2[i].double().requires_grad_(case["grad"])
        for r in range(0, n, rows):
            part = x1[i, r:r + rows].double().requires_grad_(case["grad"])
            got = _exact_block(case, part, whole)
            out[i, r:r + rows] = got.detach()
            if case["grad"]:
                a, c = torch.autograd.grad(got, (part, whole), gout[i, r:r + rows].double())
                g1[i, r:r + rows] = a
                g2[i] += c
    shape = (lambda t: t) if case["b"] else (lambda t: t[0])
    if not case["grad"]:
        return {"out": shape(out)}
    return {"out": shape(out), "grad1": shape(g1), "grad2": shape(g2)}
