"""The calls that the framework's speed is measured on: every public operator over the sizes its users bring.

A case is a plain dict.  ``op`` names the operator:

* ``cdist``: ``kermac.cdist(a, b, p=p)``, ``M`` x ``N`` distances of ``K``-dimensional points, ``L`` batch entries;
* ``kernel``: ``kermac.run_kernel`` of one descriptor (``kernel``), optionally of a set against itself (``self``) with
  a regularised diagonal, and optionally with one bandwidth per batch entry on shared points (``L`` > 1);
* ``product``: the same kernel matrix contracted with ``O`` columns of coefficients;
* ``gradient``: ``kermac.cdist_grad``, ``O`` x ``N`` x ``M`` results, contraction over ``K`` centres.

``layout`` is the storage of the operands and the result: ``"torch"`` as torch allocates them (``[M, K]``, the result
returned by the call), ``"panel"`` with the points contiguous (``[K, M]``, handed over as ``.t()`` views, the result
written into a buffer that the caller keeps), as in the reference's benchmark.
"""
import math

import torch

import kermac_amd as kermac

_DIFF, _POW = kermac.InnerOperator.DIFF, kermac.PowerType

_DESCRIPTORS = {
    "laplace_l1": kermac.kernel_descriptor_laplace_l1,
    "laplace_l2": kermac.kernel_descriptor_laplace_l2,
    "gaussian": kermac.KernelDescriptor(_DIFF, _POW.SQUARE, _POW.NOOP, kermac.KernelType.GAUSSIAN),
    "linear": kermac.kernel_descriptor_mma,
}


def listed():
    return [
        # A small Euclidean distance matrix (1024 points against 1024): bound by latency and launches.
        dict(name="cdist_p2_small", op="cdist", p=2.0, L=1, M=1024, N=1024, K=64, layout="panel"),
        # Several kernels on the same few-feature data in one call, as in examples/broadcast_kernel.py: store-bound.
        dict(name="kernel_two_bandwidths", op="kernel", kernel="laplace_l2", L=2, M=10000, N=10000, K=6, layout="torch", self=True),
        # An ordinary Euclidean distance matrix on image-sized features, no size a multiple of a tile.
        dict(name="cdist_p2_medium", op="cdist", p=2.0, L=1, M=2000, N=2000, K=784, layout="torch"),
        # The reference's benchmark for p = 2.
        dict(name="cdist_p2_large", op="cdist", p=2.0, L=1, M=30000, N=30000, K=1024, layout="panel"),
        # The training matrix of a kernel machine: a set against itself with a regularised diagonal.
        dict(name="kernel_training_set", op="kernel", kernel="gaussian", L=1, M=10000, N=10000, K=784, layout="torch", self=True),
        # An ordinary Manhattan distance matrix of ragged size.
        dict(name="cdist_p1_medium", op="cdist", p=1.0, L=1, M=3000, N=2900, K=2048, layout="torch"),
        # The reference's headline benchmark.
        dict(name="cdist_p1_large", op="cdist", p=1.0, L=1, M=30000, N=30000, K=1024, layout="panel"),
        # A fractional norm at the default size of examples/cdist.py, one batch entry.
        dict(name="cdist_p1.3", op="cdist", p=1.3, L=1, M=10000, N=10000, K=1024, layout="torch"),
        # The gradient of a Laplace kernel machine (average gradient outer product), 16 outputs.
        dict(name="gradient_p1", op="gradient", p=1.0, L=1, M=8192, N=512, O=16, K=8192, layout="torch"),
        # The default call of examples/cdist_grad.py.
        dict(name="gradient_p2", op="gradient", p=2.0, L=2, M=10000, N=768, O=16, K=10000, layout="torch"),
        # Kernel matrix times coefficients for four batches of points against shared centres, matrix never stored.
        dict(name="product_laplace_batched", op="product", kernel="laplace_l1", L=4, M=16384, N=16384, K=256, O=32, layout="panel"),
        # Prediction: a batch of new points against all training points, 10 classes.
        dict(name="product_prediction", op="product", kernel="gaussian", L=1, M=1000, N=60000, K=784, O=10, layout="torch"),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


# A rough price per elementary term, in arbitrary units in which the reference's headline benchmark costs about 28:
# it only keeps drawn cases below the largest listed one.
def _price(case):
    terms = float(case["L"]) * case["M"] * case["N"] * case["K"]
    if case["op"] == "gradient":
        return 1e-11 * terms * (8 + case["O"])
    fractional = case["op"] == "cdist" and case["p"] not in (1.0, 2.0)
    return terms * (2.5e-10 if fractional else 4e-11) + 4e-9 * case["L"] * case["M"] * case["N"]


def _rows(rng, low, high):
    """A number of points: any size, or one of the round ones that users like."""
    n = _log_int(rng, low, high)
    return n if rng.random() < 0.6 or n < 64 else n // 64 * 64


def draw(rng):
    """Another call of the same operators: sizes over the whole range, odd ones among them."""
    while True:
        op = rng.choice(("cdist", "cdist", "kernel", "product", "gradient"))
        layout = rng.choice(("torch", "panel"))
        if op == "gradient":
            case = dict(op=op, p=rng.choice((1.0, 2.0)), L=rng.choice((1, 1, 2)), M=_rows(rng, 200, 12000), N=_rows(rng, 16, 1024),
                        O=rng.choice((1, 4, 10, 16, 32)), K=_rows(rng, 200, 12000), layout="torch")
        else:
            case = dict(op=op, L=rng.choice((1, 1, 1, 2, 4)), M=_rows(rng, 256, 30000), N=_rows(rng, 256, 30000),
                        K=_rows(rng, 6, 4096), layout=layout)
            if op == "cdist":
                case["p"] = rng.choice((1.0, 2.0, 2.0, 1.3))
            elif op == "kernel":
                case["kernel"] = rng.choice(("laplace_l1", "laplace_l2", "gaussian", "linear"))
                if rng.random() < 0.4:
                    case["self"], case["N"] = True, case["M"]
            else:
                case["kernel"], case["O"] = rng.choice(("laplace_l1", "laplace_l2", "gaussian")), rng.choice((1, 10, 32))
        if _price(case) <= 25.0 and float(case["L"]) * case["M"] * case["N"] <= 4e8:
            return case


def _bandwidth(case):
    """About the distance of two points, so that the kernel's values are neither all zero nor all one."""
    kernel, K = case["kernel"], case["K"]
    if kernel == "laplace_l1":
        return 1.128 * K
    if kernel == "gaussian":
        return math.sqrt(K)        # of the squared distance: exp(-d^2 / (2 bandwidth^2))
    return math.sqrt(2.0 * K)


def prepare(case, seed):
    """The tensors (and the result's buffer, with ``layout`` "panel") that a user's program holds before the call."""
    device = torch.device("cuda")
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, device=device, generator=gen)

    L, M, N, K = case["L"], case["M"], case["N"], case["K"]
    batch = (L,) if L > 1 else ()
    if case["op"] == "gradient":
        spread = N ** -0.5
        return dict(case=case, a=torch.rand(*batch, K, M, device=device, generator=gen), b=normal(*batch, N, K) * spread,
                    c=normal(*batch, case["O"], K), d=normal(*batch, N, M) * spread)

    panel = case["layout"] == "panel"

    def points(rows, *lead):
        return normal(*lead, K, rows).transpose(-1, -2) if panel else normal(*lead, rows, K)

    state = dict(case=case)
    shared = case["op"] == "kernel" and L > 1       # one kernel per bandwidth on shared points
    state["a"] = points(M) if shared else points(M, *batch)
    if case.get("self"):
        state["b"] = state["a"]
    else:
        # the centres of a product are shared by the batch
        state["b"] = points(N) if shared or case["op"] == "product" else points(N, *batch)
    state["out"] = None
    if case["op"] == "product":
        state["coefficients"] = normal(*batch, N, case["O"])
    elif panel:
        state["out"] = torch.empty(L, N, M, device=device).transpose(-1, -2)
    if case["op"] != "cdist":
        bandwidth = _bandwidth(case)
        if shared:
            state["bandwidth"] = torch.tensor([bandwidth * (1 + i) for i in range(L)], device=device)
        else:
            state["bandwidth"] = bandwidth
    return state


def run(state):
    case = state["case"]
    if case["op"] == "cdist":
        return kermac.cdist(state["a"], state["b"], out=state["out"], p=case["p"])
    if case["op"] == "gradient":
        return kermac.cdist_grad(state["a"], state["b"], state["c"], state["d"], p=case["p"])
    options = {}
    if case["kernel"] != "linear":
        options["bandwidth"] = state["bandwidth"]
        if case.get("self"):
            options["regularization"] = 1e-3
    if case["op"] == "product":
        options["coefficients"] = state["coefficients"]
    return kermac.run_kernel(_DESCRIPTORS[case["kernel"]], state["a"], state["b"], out=state["out"], **options)


def work(case):
    L, M, N, K = case["L"], case["M"], case["N"], case["K"]
    terms = L * M * N * K
    if case["op"] == "gradient":
        O = case["O"]
        # p = 1: the sign of each difference, its product with a and O multiply-adds; p = 2 factors into products
        flops = terms * (2 * O + (3 if case["p"] == 1.0 else 0))
        return {"bytes": 4 * L * (K * M + N * K + O * K + N * M + O * N * M), "flops": flops}
    # squared differences and products need one multiply-add per term; other powers subtract, raise and add
    squares = case.get("p") == 2.0 or case.get("kernel") in ("laplace_l2", "gaussian", "linear")
    flops = terms * (2 if squares else 3)
    if case.get("self"):
        flops //= 2
    shared = case["op"] == "kernel" and L > 1
    read = (1 if shared else L) * M * K + (0 if case.get("self") else (1 if shared or case["op"] == "product" else L) * N * K)
    if shared:
        flops //= L
    if case["op"] == "product":
        O = case["O"]
        return {"bytes": 4 * (read + L * O * (M + N)), "flops": flops + 2 * L * M * N * O}
    return {"bytes": 4 * (read + L * M * N), "flops": flops}


def tolerance(case):
    """About four times the error of today's kernels against float64, which grows with the length of the fp32 sums:
    4.8e-7 for distances at K = 1024, 1.0e-6 for gradients at K = 8192, 1.1e-6 for products with one column (the sum over
    centres cancels); the largest single error is four to five times the 2-norm one, and up to 20 times where a kernel's
    exponential amplifies it."""
    rel = (4e-6 if case["op"] == "product" else 4e-7) + 6e-8 * math.sqrt(case["K"])
    return {"rel": rel, "max": 8 * rel}
