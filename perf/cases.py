"""What a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values with a "kind":

  train       a short training run of the byte-level GPT through the engine: a chunk of steps, its losses, the weights
  train16     the same of the width-16 network that an engine created from the plain Config trains
  gradient    one fixed batch through the engine: logits, losses and, unless it only evaluates, the flat gradient
  text        bytes predicted one after another over a sliding window, as the sampling loop of a host program does
  projection  one linear layer through the operator entries: forward, input gradient, weight gradient
  mlp         an MLP block through the operator entries: up + GELU, down + residual, and all four gradients
  attention   causal attention through the operator entries: forward, then the recompute backward

prepare() makes a case's inputs from the seed and what a program keeps (an engine, weights, buffers, workspaces); run()
is one pass through the public entry points.
"""
import math

import numpy as np
import torch

from turbogpt_amd.bridge import Config, ModelConfig, Native, check, library

BF16 = torch.bfloat16
VOCAB = 256


def listed():
    return [
        # The reference's own network and default trainer shape (batch 2560 of context 4): thousands of steps of well
        # under a millisecond each, so launches and latency count.
        dict(name="train16-default", kind="train16", depth=4, context=4, batch=2560, inflight=1, steps=16),
        # Its smallest shape class at full depth and context, with batches in flight on stale weights.
        dict(name="train16-inflight", kind="train16", depth=8, context=8, batch=16, inflight=4, steps=16),
        # A model for a laptop-sized corpus: 2048 tokens a step, many short launches.
        dict(name="train-d256", kind="train", d_model=256, depth=4, ffn=1024, context=256, batch=8, inflight=1, steps=16),
        # Widths and token counts that no large tile divides.
        dict(name="train-d640-odd", kind="train", d_model=640, depth=6, ffn=1920, context=384, batch=5, inflight=1, steps=16),
        # The headline workload.
        dict(name="train-d768", kind="train", d_model=768, depth=12, ffn=3072, context=1024, batch=16, inflight=1, steps=16),
        # The long-context workload: attention over 4096 positions, 302 million parameters.
        dict(name="train-d1024-long", kind="train", d_model=1024, depth=24, ffn=4096, context=4096, batch=4, inflight=1, steps=8),
        # Gradients of a given batch, for a program with an optimizer or a check of its own.
        dict(name="gradient-d256", kind="gradient", d_model=256, depth=4, ffn=1024, context=256, batch=8, backward=True),
        # Sampling from the headline model while it trains: the engine has its training shape.
        dict(name="text-d768", kind="text", d_model=768, depth=12, ffn=3072, context=1024, batch=16, bytes=8),
        # The QKV projection of the headline model in a program with its own layer loop.
        dict(name="projection-qkv", kind="projection", tokens=16384, inputs=768, outputs=2304, transposed=True),
        # An MLP with an odd number of tokens and no transposed weight copies.
        dict(name="mlp-odd", kind="mlp", tokens=1920, width=640, hidden=1920, transposed=False),
        # Attention of the headline model.
        dict(name="attention-t1024", kind="attention", batch=16, heads=12, context=1024),
        # Attention of the small model: few, short sequences.
        dict(name="attention-small", kind="attention", batch=8, heads=4, context=256),
    ]


def _spread(rng, low, high, step=1):
    """A multiple of `step` from low to high, spread over the logarithm."""
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high, max(low, int(round(value / step)) * step))


def _draw_model(rng, most_flops_per_token_pass):
    while True:
        d = 128 * rng.randint(1, 8)
        shape = dict(d_model=d, depth=_spread(rng, 1, 24), ffn=rng.choice([2, 3, 4, 4]) * d,
                     context=_spread(rng, 128, 4096, 128), batch=_spread(rng, 1, 16))
        if shape["batch"] * shape["context"] <= 16384 and _step_flops(shape) <= most_flops_per_token_pass:
            return shape


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(["train", "train", "train16", "gradient", "text", "projection", "mlp", "attention"])
    if kind == "train16":
        context = rng.choice([4, 8])
        batch = 16 // context * _spread(rng, 2, 2560 * context // 16)
        return dict(kind=kind, depth=rng.choice([4, 8]), context=context, batch=batch,
                    inflight=rng.choice([1, 1, 2, 4, 8]), steps=_spread(rng, 8, 64))
    if kind == "train":
        case = dict(kind=kind, **_draw_model(rng, 1.2e13), inflight=1, steps=_spread(rng, 4, 16))
        if case["batch"] * case["context"] <= 4096:
            case["inflight"] = rng.choice([1, 1, 2])
        return case
    if kind == "gradient":
        return dict(kind=kind, **_draw_model(rng, 4e12), backward=rng.choice([True, True, False]))
    if kind == "text":
        return dict(kind=kind, **_draw_model(rng, 1.2e13), bytes=_spread(rng, 4, 16))
    if kind == "projection":
        unit = rng.choice([128, 192])
        return dict(kind=kind, tokens=_spread(rng, 128, 16384, 128), inputs=unit * rng.randint(1, 3072 // unit),
                    outputs=128 * rng.randint(1, 24), transposed=rng.choice([True, False]))
    if kind == "mlp":
        d = 128 * rng.randint(1, 8)
        return dict(kind=kind, tokens=_spread(rng, 128, 16384, 128), width=d, hidden=rng.choice([2, 3, 4]) * d,
                    transposed=rng.choice([True, False]))
    while True:
        case = dict(kind=kind, batch=_spread(rng, 1, 16), heads=rng.randint(1, 16), context=_spread(rng, 128, 8192, 128))
        if case["batch"] * case["context"] <= 16384:
            return case


# ---- inputs ----------------------------------------------------------------------------------------------------------


def _generator(seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    return generator


def _normal(generator, *shape, scale=1.0):
    return (torch.randn(*shape, device="cuda", generator=generator) * scale).to(BF16)


def _zipf_bytes(generator, n, exponent=1.1):
    weights = torch.arange(1, VOCAB + 1, device="cuda", dtype=torch.float64) ** -exponent
    cdf = torch.cumsum(weights / weights.sum(), 0)
    draws = torch.rand(n, device="cuda", generator=generator, dtype=torch.float64)
    return torch.searchsorted(cdf, draws).clamp_(max=VOCAB - 1).to(torch.uint8).cpu().numpy()


class _Engine(Native):
    """An engine that gives its device memory back with its last reference."""

    handle = None

    def __del__(self):
        self.close()


def _model(case, seed, inflight=1):
    return ModelConfig(d_model=case["d_model"], ffn=case["ffn"], depth=case["depth"], context=case["context"],
                       batch=case["batch"], inflight=inflight, learning_rate=3e-4, beta1=0.9, beta2=0.95,
                       weight_decay=0.1, clip=1.0, seed=seed)


def _model_weights(case, generator):
    """N(0, 0.02) matrices, those that write to the residual stream scaled by 1/sqrt(2 depth), unit norms."""
    d, f, depth = case["d_model"], case["ffn"], case["depth"]
    parts = []

    def matrix(rows, cols, scale=0.02):
        parts.append(torch.randn(rows * cols, device="cuda", generator=generator) * scale)

    def norm():
        parts.append(torch.ones(d, device="cuda"))
        parts.append(torch.zeros(d, device="cuda"))

    inner = 0.02 / math.sqrt(2 * depth)
    matrix(VOCAB, d)
    matrix(case["context"], d)
    for _ in range(depth):
        norm()
        matrix(3 * d, d)
        matrix(d, d, inner)
        norm()
        matrix(f, d)
        matrix(d, f, inner)
    norm()
    matrix(VOCAB, d)
    return torch.cat(parts).cpu().numpy()


def _width16_weights(case, generator):
    """N(0, 0.08) matrices and unit scales in the network's flat order."""
    parts = []

    def matrix(n):
        parts.append(torch.randn(n, device="cuda", generator=generator) * 0.08)

    def scale():
        parts.append(torch.ones(16, device="cuda"))

    matrix(VOCAB * 16)
    for _ in range(case["depth"]):
        scale()
        matrix(48 * 16 + 16 * 16)
        scale()
        matrix(3 * 48 * 16)
    scale()
    matrix(VOCAB * 16)
    return torch.cat(parts).cpu().numpy()


def prepare(case, seed):
    generator = _generator(seed)
    kind = case["kind"]
    if kind == "train16":
        engine = _Engine(Config(depth=case["depth"], context=case["context"], batch=case["batch"],
                                inflight=case["inflight"], seed=seed))
        engine.set_weights(_width16_weights(case, generator))
        engine.set_onecycle(488282)
        engine.set_data(_zipf_bytes(generator, 1 << 20))
        return dict(kind=kind, engine=engine, steps=case["steps"])
    if kind == "train":
        engine = _Engine(_model(case, seed, case["inflight"]))
        engine.set_weights(_model_weights(case, generator))
        engine.set_data(_zipf_bytes(generator, 1 << 22))
        return dict(kind=kind, engine=engine, steps=case["steps"])
    if kind in ("gradient", "text"):
        engine = _Engine(_model(case, seed))
        engine.set_weights(_model_weights(case, generator))
        if kind == "gradient":
            stream = _zipf_bytes(generator, case["batch"] * case["context"] + 1)
            shape = (case["batch"], case["context"])
            return dict(kind=kind, engine=engine, backward=case["backward"], x=stream[:-1].reshape(shape),
                        y=stream[1:].reshape(shape))
        return dict(kind=kind, engine=engine, bytes=case["bytes"], context=case["context"],
                    text=_zipf_bytes(generator, case["context"] + case["bytes"]))
    if kind == "projection":
        m, k, n = case["tokens"], case["inputs"], case["outputs"]
        return dict(kind=kind, m=m, k=k, n=n, x=_normal(generator, m, k), w=_layer_weight(generator, n, k, case),
                    dy=_normal(generator, m, n), y=_empty(m, n), dx=_empty(m, k), dw=_empty(n, k, dtype=torch.float32),
                    workspace=_bytes(library().tgk_gemm_wgrad_workspace(m, n, k)))
    if kind == "mlp":
        m, d, f = case["tokens"], case["width"], case["hidden"]
        need = max(library().tgk_gemm_wgrad_workspace(m, f, d), library().tgk_gemm_wgrad_workspace(m, d, f))
        return dict(kind=kind, m=m, d=d, f=f, x=_normal(generator, m, d), residual=_normal(generator, m, d),
                    up=_layer_weight(generator, f, d, case), down=_layer_weight(generator, d, f, case),
                    dy=_normal(generator, m, d), u=_empty(m, f), a=_empty(m, f), y=_empty(m, d), du=_empty(m, f),
                    dx=_empty(m, d), dup=_empty(f, d, dtype=torch.float32), ddown=_empty(d, f, dtype=torch.float32),
                    workspace=_bytes(need))
    b, h, t = case["batch"], case["heads"], case["context"]
    return dict(kind=kind, b=b, h=h, t=t, qkv=_normal(generator, b * t, 3 * 64 * h), do=_normal(generator, b * t, 64 * h),
                o=_empty(b * t, 64 * h), lse=_empty(b, h, t, dtype=torch.float32), dqkv=_empty(b * t, 3 * 64 * h),
                workspace=_bytes(library().tgk_attn_bwd_workspace(b, h, t)))


def _empty(*shape, dtype=BF16):
    return torch.empty(*shape, device="cuda", dtype=dtype)


def _bytes(n):
    return torch.empty(max(n, 16), device="cuda", dtype=torch.uint8)


def _layer_weight(generator, rows, cols, case):
    """A weight [Out][In] and, where the program keeps one for its input gradients, the transposed copy."""
    weight = _normal(generator, rows, cols, scale=cols ** -0.5)
    return weight, weight.t().contiguous() if case["transposed"] else None


# ---- one pass --------------------------------------------------------------------------------------------------------


def _forward(stream, m, n, k, x, weight, y, residual=None, gelu=None):
    check(library().tgk_gemm_fwd(stream, m, n, k, x.data_ptr(), k, weight[0].data_ptr(), k, y.data_ptr(), n,
                                 residual.data_ptr() if residual is not None else None, n if residual is not None else 0,
                                 gelu.data_ptr() if gelu is not None else None, n if gelu is not None else 0))


def _input_gradient(stream, m, n, k, dy, weight, dx, gelu_pre=None):
    pre, ld = (gelu_pre.data_ptr(), k) if gelu_pre is not None else (None, 0)
    if weight[1] is not None:
        check(library().tgk_gemm_dgrad_t(stream, m, n, k, dy.data_ptr(), n, weight[1].data_ptr(), n, dx.data_ptr(), k, pre, ld))
    else:
        check(library().tgk_gemm_dgrad(stream, m, n, k, dy.data_ptr(), n, weight[0].data_ptr(), k, dx.data_ptr(), k, pre, ld))


def _weight_gradient(stream, m, n, k, dy, x, dw, workspace):
    check(library().tgk_gemm_wgrad(stream, m, n, k, dy.data_ptr(), n, x.data_ptr(), k, dw.data_ptr(), k, 0,
                                   workspace.data_ptr(), workspace.numel()))


def run(s):
    kind = s["kind"]
    if kind in ("train", "train16"):
        s["engine"].train(s["steps"])
        losses = s["engine"].training_losses(s["steps"])
        return losses, s["engine"].weights()
    if kind == "gradient":
        return s["engine"].batch(s["x"], s["y"], backward=s["backward"])
    if kind == "text":
        return np.stack([s["engine"].predict(s["text"][i:i + s["context"]]) for i in range(s["bytes"])])
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "projection":
        m, n, k = s["m"], s["n"], s["k"]
        _forward(stream, m, n, k, s["x"], s["w"], s["y"])
        _input_gradient(stream, m, n, k, s["dy"], s["w"], s["dx"])
        _weight_gradient(stream, m, n, k, s["dy"], s["x"], s["dw"], s["workspace"])
        return s["y"], s["dx"], s["dw"]
    if kind == "mlp":
        m, d, f = s["m"], s["d"], s["f"]
        _forward(stream, m, f, d, s["x"], s["up"], s["u"], gelu=s["a"])
        _forward(stream, m, d, f, s["a"], s["down"], s["y"], residual=s["residual"])
        _weight_gradient(stream, m, d, f, s["dy"], s["a"], s["ddown"], s["workspace"])
        _input_gradient(stream, m, d, f, s["dy"], s["down"], s["du"], gelu_pre=s["u"])
        _weight_gradient(stream, m, f, d, s["du"], s["x"], s["dup"], s["workspace"])
        _input_gradient(stream, m, f, d, s["du"], s["up"], s["dx"])
        return s["u"], s["a"], s["y"], s["du"], s["dx"], s["dup"], s["ddown"]
    b, h, t = s["b"], s["h"], s["t"]
    width = 64 * h
    qkv, dqkv = s["qkv"].data_ptr(), s["dqkv"].data_ptr()
    check(library().tgk_attn_fwd(stream, b, h, t, 64, qkv, qkv + 2 * width, qkv + 4 * width, 3 * width, s["o"].data_ptr(),
                                 width, s["lse"].data_ptr(), 0.125))
    check(library().tgk_attn_bwd(stream, b, h, t, 64, qkv, qkv + 2 * width, qkv + 4 * width, 3 * width, s["o"].data_ptr(),
                                 width, s["lse"].data_ptr(), s["do"].data_ptr(), width, dqkv, dqkv + 2 * width,
                                 dqkv + 4 * width, 3 * width, 0.125, s["workspace"].data_ptr(), s["workspace"].numel()))
    return s["o"], s["lse"], s["dqkv"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------


def _matrix_parameters(case):
    d, f = case["d_model"], case["ffn"]
    return case["depth"] * (4 * d * d + 2 * d * f) + VOCAB * d  # with the head


def _parameters(case):
    d = case["d_model"]
    return _matrix_parameters(case) + VOCAB * d + case["context"] * d + (4 * case["depth"] + 2) * d


def _attention_flops(batch, heads, context):
    return 4.0 * batch * heads * context * context * 64 / 2  # forward, the causal half


def _forward_flops(case, batch):
    return (2.0 * batch * case["context"] * _matrix_parameters(case) +
            case["depth"] * _attention_flops(batch, case["d_model"] // 64, case["context"]))


def _step_flops(case):
    tokens = case["batch"] * case["context"]
    return (6.0 * tokens * _matrix_parameters(case) +
            3.5 * case["depth"] * _attention_flops(case["batch"], case["d_model"] // 64, case["context"]))


def work(case):
    kind = case["kind"]
    if kind == "train16":
        matrices = case["depth"] * (4 * 16 * 16 + 3 * 48 * 16) + VOCAB * 16
        parameters = matrices + VOCAB * 16 + (2 * case["depth"] + 1) * 16
        tokens = case["batch"] * case["context"]
        return dict(flops=6.0 * tokens * matrices * case["steps"],
                    bytes=case["steps"] * (24 * parameters + 2 * tokens) + 4 * parameters)
    if kind == "train":  # weights, momentum and variance read and written every step
        return dict(flops=_step_flops(case) * case["steps"],
                    bytes=case["steps"] * (24 * _parameters(case) + 2 * case["batch"] * case["context"]) + 4 * _parameters(case))
    if kind == "gradient":
        tokens = case["batch"] * case["context"]
        flops = _step_flops(case) if case["backward"] else _forward_flops(case, case["batch"])
        return dict(flops=flops, bytes=(2 + 4 * case["backward"]) * _parameters(case) + (2 + 4 * VOCAB) * tokens)
    if kind == "text":  # one sequence's forward pass for each byte
        return dict(flops=_forward_flops(case, 1) * case["bytes"],
                    bytes=case["bytes"] * (2 * _parameters(case) + case["context"] + 4 * VOCAB))
    if kind == "projection":
        m, k, n = case["tokens"], case["inputs"], case["outputs"]
        return dict(flops=6.0 * m * k * n, bytes=2 * (2 * m * k + 2 * m * n + n * k) + 4 * n * k)
    if kind == "mlp":
        m, d, f = case["tokens"], case["width"], case["hidden"]
        return dict(flops=12.0 * m * d * f, bytes=2 * (5 * m * d + 3 * m * f + 2 * d * f) + 4 * 2 * d * f)
    b, h, t = case["batch"], case["heads"], case["context"]
    return dict(flops=3.5 * _attention_flops(b, h, t), bytes=2 * b * t * h * 64 * 8 + 4 * b * h * t)


def tolerance(case):
    """About four times what another correct computation of the same pass was measured to differ by."""
    kind = case["kind"]
    if kind == "train16":
        # The same steps with the gradient's sums in another order (the batch's sequences permuted): weights 2e-9 in the
        # synchronous case; 6e-4 (largest 9.5e-3) with batches in flight, where a near tie of the arg-max attention falls
        # the other way.
        return {"rel": 3e-3, "max": 5e-2}
    if kind == "train":
        # Against the same steps in fp32 with library operators: weights 7e-4 to 2.2e-3 (largest 0.08), losses 2e-4 to
        # 8e-3 (the first Adam steps of a deep model amplify rounding), 12 layers most.
        return {"rel": 2e-2, "max": 0.3}
    if kind in ("gradient", "text"):
        # Against fp32: logits 7e-3 at 4 layers and 9.3e-3 at 12 (largest 0.03), gradient 1.8e-3 (largest 0.04).
        return {"rel": 2e-2, "max": 0.15}
    if kind == "attention":
        # Against fp64: output 2.0e-3, gradients 2.4e-3; single elements that nearly cancel 0.11.
        return {"rel": 1e-2, "max": 0.4}
    # Against fp64: outputs 1.7e-3 (a bf16 rounding) to 2.9e-3 (a product of rounded factors), largest 0.014.
    return {"rel": 1e-2, "max": 6e-2}
