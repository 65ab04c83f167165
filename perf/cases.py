"""The measured work of a program that serves quantized models with this package.

Each case is one pass through the public entry points as a model's MLP or projection calls them.
Five kinds of work, over the ranges that ``draw`` spans:

* ``decode``: the MLPs of a model's layers on one token (or a small batch of them), each one
  ``affine_mlp`` call over weights kept in the code layout that the tuner picks when the model is
  loaded (``metile_amd.tuning``), replayed from a HIP graph as a serving loop does.
* ``mlp``: one layer's ``affine_mlp`` called eagerly on a batch of sequences or on a prompt, over
  stored (MLX) or repacked codes.
* ``linear``: one quantized projection: ``QuantizedLinear`` (a model's layer after ``quantize_mlp``),
  ``CompressedDownWeight`` (an INT8 down projection), ``affine_qmv`` or the fused ``affine_swiglu``
  over stored weights; 4 and 8 bits, groups of 32 to 128, both activation types.
* ``dense``: a 16-bit MLP through ``mlx_dense_swiglu`` and ``mlx_dense_residual_qmv``, up to 128 rows.
* ``load``: quantizing a projection when a model is loaded (``QuantizedLinear.from_linear``).

Weights follow the recipe of the benchmark (codes uniform, scale |N(0, 1)| * 0.02 for 4 bits and
* 0.002 for 8, bias -8 or -128 scales); activations are N(0, 1). Shapes are those of the benchmark,
the tests and the reference's published tables: MLPs of 896 x 4864, 1536 x 8960, 2048 x 8192,
3584 x 18944, 4096 x 14336 and 5120 x 17408, and generic ones between them.
"""

import math

import torch

import metile_amd as mt
from metile_amd import tuning

MLPS = ((896, 4864), (1536, 8960), (2048, 8192), (3584, 18944), (4096, 14336), (5120, 17408))
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
MOST_FLOPS = 2 * 2048 * 4096 * 14336  # of the largest listed case


def listed():
    return [
        # one projection of a decode step called eagerly: the smallest call there is
        dict(name="qmv-1row", kind="linear", entry="qmv", rows=1, k=1536, n=8960, bits=4, group=64,
             dtype="bf16", residual=False),
        # the headline: the MLPs of a 28-layer model on one token
        dict(name="decode-1row", kind="decode", rows=1, hidden=1536, inter=8960, layers=28,
             dtype="bf16"),
        # the same model serving eight sequences at once
        dict(name="decode-8rows", kind="decode", rows=8, hidden=1536, inter=8960, layers=28,
             dtype="bf16"),
        # a batch of 48 sequences, one layer
        dict(name="mlp-48rows", kind="mlp", rows=48, hidden=1536, inter=8960, dtype="bf16",
             packed=True),
        # a prompt of odd length through one layer
        dict(name="mlp-prompt-333", kind="mlp", rows=333, hidden=1536, inter=8960,
             dtype="bf16", packed=False),
        # an 8-bit SwiGLU of a small model in float16, groups of 128, a few tokens to verify at once
        dict(name="swiglu-int8-5rows", kind="linear", entry="swiglu", rows=5, k=896, n=4864, bits=8,
             group=128, dtype="f16", residual=False),
        # an 8-bit projection of a large model, sixteen sequences
        dict(name="int8-16rows", kind="linear", entry="compressed", rows=16, k=5120, n=17408, bits=8,
             group=64, dtype="bf16", residual=False),
        # the up projection on a 512-token prompt
        dict(name="prefill-512", kind="linear", entry="module", rows=512, k=1536, n=8960, bits=4,
             group=64, dtype="bf16", residual=False),
        # the down projection of a large model on a 2048-token prompt
        dict(name="prefill-2048", kind="linear", entry="module", rows=2048, k=14336, n=4096, bits=4,
             group=64, dtype="f16", residual=False),
        # a 16-bit MLP on one token, and on a large ragged batch
        dict(name="dense-1row", kind="dense", rows=1, hidden=2048, inter=8192, dtype="bf16"),
        dict(name="dense-100rows", kind="dense", rows=100, hidden=2048, inter=8192, dtype="bf16"),
        # one projection of a large model quantized while loading
        dict(name="load", kind="load", k=4096, n=14336, bits=4, group=64, dtype="bf16"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _mlp_shape(rng, most):
    """(hidden, inter) of a model with at most ``most`` weights a projection, or a generic one."""
    if rng.random() < 0.65:
        return rng.choice([s for s in MLPS if s[0] * s[1] <= most])
    while True:
        hidden, inter = 64 * _log(rng, 8, 80), 64 * _log(rng, 24, 300)
        if hidden < inter and hidden * inter <= most:
            return hidden, inter


def draw(rng):
    kind = rng.choice(("decode", "mlp", "mlp", "linear", "linear", "linear", "dense", "load"))
    dtype = rng.choice(("bf16", "bf16", "f16"))
    if kind == "decode":
        hidden, inter = _mlp_shape(rng, 4096 * 14336)
        layers = max(1, min(28, 28 * 1536 * 8960 // (hidden * inter)))
        return dict(kind=kind, rows=_log(rng, 1, 32), hidden=hidden, inter=inter, layers=layers,
                    dtype=dtype)
    if kind == "mlp":
        hidden, inter = _mlp_shape(rng, 4096 * 14336)
        most = min(2048, MOST_FLOPS // (6 * hidden * inter))
        return dict(kind=kind, rows=_log(rng, 1, most), hidden=hidden, inter=inter, dtype=dtype,
                    packed=rng.random() < 0.5)
    hidden, inter = _mlp_shape(rng, 5120 * 17408)
    if kind == "dense":
        return dict(kind=kind, rows=_log(rng, 1, 128), hidden=hidden, inter=inter, dtype=dtype)
    down = rng.random() < 0.5
    k, n = (inter, hidden) if down else (hidden, inter)
    bits = rng.choice((4, 4, 8))
    group = rng.choice((64, 64, 128, 32 if bits == 8 else 64))
    group = group if k % group == 0 else 64
    if kind == "load":
        return dict(kind=kind, k=k, n=n, bits=bits, group=group, dtype=dtype)
    entry = rng.choice(("qmv", "swiglu", "module", "module") if bits == 4
                       else ("qmv", "swiglu", "compressed"))
    if entry == "swiglu":
        k, n = hidden, inter
        group = group if k % group == 0 else 64
    cost = 2 * k * n * (2 if entry == "swiglu" else 1)
    most = min(2048 if entry == "module" else 512, MOST_FLOPS // cost)
    return dict(kind=kind, entry=entry, rows=_log(rng, 1, most), k=k, n=n, bits=bits, group=group,
                dtype=dtype, residual=entry == "qmv" and rng.random() < 0.5)


# ---- inputs --------------------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activations(gen, rows, width, dtype):
    return torch.randn(rows, width, generator=gen, device="cuda").to(dtype)


def _affine(gen, k, n, bits, group, dtype):
    words = torch.randint(-2**31, 2**31, (n, k * bits // 32), generator=gen, device="cuda",
                          dtype=torch.int64).to(torch.int32)
    coef, zero = (0.02, 8.0) if bits == 4 else (0.002, 128.0)
    scales = (torch.randn(n, k // group, generator=gen, device="cuda").abs() * coef).to(dtype)
    return words, scales, (scales.float() * -zero).to(dtype)


def _inputs(case, seed):
    """Activations, residual and weights of a case (before any preparation of the weights)."""
    gen = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    kind = case["kind"]
    if kind == "load":
        return (torch.randn(case["n"], case["k"], generator=gen, device="cuda") * 0.02).to(dtype)
    if kind == "dense":
        h, i = case["hidden"], case["inter"]
        weights = [(torch.randn(n, k, generator=gen, device="cuda") * 0.02).to(dtype)
                   for n, k in ((i, h), (i, h), (h, i))]
        return (_activations(gen, case["rows"], h, dtype), _activations(gen, case["rows"], h, dtype),
                weights)
    if kind in ("decode", "mlp"):
        h, i = case["hidden"], case["inter"]
        layers = []
        for _ in range(case.get("layers", 1)):
            layers.append((_activations(gen, case["rows"], h, dtype),
                           _activations(gen, case["rows"], h, dtype),
                           [_affine(gen, k, n, 4, 64, dtype)
                            for k, n in ((h, i), (h, i), (i, h))]))
        return layers
    weights = [_affine(gen, case["k"], case["n"], case["bits"], case["group"], dtype)
               for _ in range(2 if case["entry"] == "swiglu" else 1)]
    x = _activations(gen, case["rows"], case["k"], dtype)
    res = _activations(gen, case["rows"], case["n"], dtype) if case["residual"] else None
    return x, res, weights


def _packed(triple):
    words, scales, biases = triple
    return mt.affine_repack(words, bits=4), scales, biases


def _mlp(x, res, gate, up, down):
    return mt.affine_mlp(x, gate, up, down, residual=res)


def _keep_layouts(layers):
    """Each stage's weights in the layout that the tuner's plan for these rows reads fastest,
    decided on the first layer (all have its shape)."""
    calls = []
    layout = None
    for x, res, mlx in layers:
        packed = [_packed(t) for t in mlx]
        if layout is None:
            stage = {"repacked": (*packed[0], *packed[1]), "mlx": (*mlx[0], *mlx[1])}
            first = tuning.ensure_qmv_layout(x, stage, group_size=64, bits=4)
            hidden = mt.affine_swiglu(x, *stage[first])
            second = tuning.ensure_qmv_layout(hidden, {"repacked": packed[2], "mlx": mlx[2]},
                                              group_size=64, bits=4)
            layout = (first, first, second)
        calls.append((x, res, *(p if kept == "repacked" else m
                                for p, m, kept in zip(packed, mlx, layout))))
    return calls


def prepare(case, seed):
    kind = case["kind"]
    data = _inputs(case, seed)
    if kind == "load":
        linear = torch.nn.Linear(case["k"], case["n"], bias=False, device="meta")
        linear.weight = torch.nn.Parameter(data, requires_grad=False)
        return dict(kind=kind, linear=linear, bits=case["bits"], group=case["group"])
    if kind == "dense":
        x, res, weights = data
        gate, up, down = (mt.DenseWeight.from_torch(w) for w in weights)
        return dict(kind=kind, x=x, res=res, gate=gate, up=up, down=down.native_weight)
    if kind == "mlp":
        x, res, (gate, up, down) = data[0]
        if case["packed"]:
            gate, up, down = (_packed(t) for t in (gate, up, down))
        return dict(kind=kind, call=(x, res, gate, up, down))
    if kind == "decode":
        calls = _keep_layouts(data)
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):  # once outside capture: the stream's workspace
            for call in calls:
                _mlp(*call)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            outs = [_mlp(*call) for call in calls]
        return dict(kind=kind, graph=graph, outs=outs, calls=calls)
    x, res, weights = data
    entry, options = case["entry"], dict(group_size=case["group"], bits=case["bits"])
    state = dict(kind=kind, entry=entry, x=x, res=res, weights=weights, options=options)
    if entry == "module":
        state["module"] = mt.QuantizedLinear(*weights[0], **options)
    elif entry == "compressed":
        state["module"] = mt.CompressedDownWeight(*weights[0], (case["n"], case["k"]), "affine8",
                                                  case["group"])
    return state


def run(state):
    kind = state["kind"]
    if kind == "decode":
        state["graph"].replay()
        return state["outs"]
    if kind == "mlp":
        return _mlp(*state["call"])
    if kind == "dense":
        hidden = mt.mlx_dense_swiglu(state["x"], state["gate"], state["up"], autotune=False)
        return hidden, mt.mlx_dense_residual_qmv(hidden, state["down"], state["res"],
                                                 autotune=False)
    if kind == "load":
        q = mt.QuantizedLinear.from_linear(state["linear"], group_size=state["group"],
                                           bits=state["bits"])
        return q.weight, q.packed, q.scales, q.biases
    if state["entry"] == "swiglu":
        gate, up = state["weights"]
        return mt.affine_swiglu(state["x"], *gate, *up, **state["options"])
    if state["entry"] == "qmv":
        return mt.affine_qmv(state["x"], *state["weights"][0], residual=state["res"],
                             **state["options"])
    return state["module"](state["x"])


# ---- what a pass cannot do without ----------------------------------------------------------------


def _weight_bytes(k, n, bits, group):
    return n * k * bits // 8 + 4 * n * (k // group)


def work(case):
    kind = case["kind"]
    if kind == "load":
        k, n = case["k"], case["n"]
        q = _weight_bytes(k, n, case["bits"], case["group"])
        return {"bytes": 2 * k * n + q + n * k * case["bits"] // 8, "flops": 4 * k * n}
    if kind == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        nproj = 2 if case["entry"] == "swiglu" else 1
        return {"bytes": nproj * _weight_bytes(k, n, case["bits"], case["group"])
                + 2 * m * (k + n * (2 if case["residual"] else 1)),
                "flops": 2 * m * k * n * nproj}
    m, h, i = case["rows"], case["hidden"], case["inter"]
    layers = case.get("layers", 1)
    weights = 3 * 2 * h * i if kind == "dense" else 2 * _weight_bytes(h, i, 4, 64) + _weight_bytes(
        i, h, 4, 64)
    hidden = 2 * m * i if kind == "dense" else 0  # an output of the dense pair
    return {"bytes": layers * (weights + 3 * 2 * m * h + hidden),
            "flops": layers * 6 * m * h * i}


# ---- correctness -----------------------------------------------------------------------------------


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    # One projection rounds once, so another order of its fp32 sums flips a few roundings by one
    # last place (2^-7 of the value at most in bf16, 2^-10 in f16). An MLP rounds its hidden
    # activation in between, and those flips travel through the down projection. Measured between
    # this package's own plans (other kernels, other K splits): relative errors up to 7e-5 for one
    # projection in either type, 9e-4 (bf16) and 8e-5 (f16) for an MLP; largest differences up to
    # 1.2e-2 and 1.7e-3.
    bf16 = case["dtype"] == "bf16"
    if case["kind"] == "linear":
        return {"rel": 3e-4, "max": 0.03 if bf16 else 0.004}
    return {"rel": 3e-3 if bf16 else 4e-4, "max": 0.04 if bf16 else 0.008}


def _dequantize(triple, bits, group):
    words, scales, biases = triple
    shifts = torch.arange(0, 32, bits, device=words.device, dtype=torch.int64)
    codes = (words.to(torch.int64)[..., None] >> shifts) & ((1 << bits) - 1)
    codes = codes.reshape(words.shape[0], -1).double()
    s = scales.double().repeat_interleave(group, 1)
    return codes.mul_(s).add_(biases.double().repeat_interleave(group, 1))


def exact(case, seed):
    kind = case["kind"]
    if kind == "load":
        return None  # bytes
    data = _inputs(case, seed)
    silu = torch.nn.functional.silu
    if kind == "dense":
        x, res, weights = data
        gate, up, down = (w.double() for w in weights)
        hidden = silu(x.double() @ gate.T) * (x.double() @ up.T)
        return hidden, hidden @ down.T + res.double()
    if kind in ("decode", "mlp"):
        outs = []
        for x, res, (gate, up, down) in data:
            xd = x.double()
            hidden = silu(xd @ _dequantize(gate, 4, 64).T) * (xd @ _dequantize(up, 4, 64).T)
            outs.append(hidden @ _dequantize(down, 4, 64).T + res.double())
        return outs if kind == "decode" else outs[0]
    x, res, weights = data
    projected = [x.double() @ _dequantize(w, case["bits"], case["group"]).T for w in weights]
    if case["entry"] == "swiglu":
        return silu(projected[0]) * projected[1]
    return projected[0] if res is None else projected[0] + res.double()
