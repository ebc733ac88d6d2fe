"""What a program that trains with this package asks of it, as measurable cases.

The package's work is the optimizer step and what surrounds it, so a case is one of the calls that a
training loop makes, over the parameter list of a model:

* ``step``: ``optimizer.step()`` of Adam/AdamW without mixed precision, in float32, float64 or float16;
* ``train``: one iteration from the micro-batches' gradients on: ``accumulate_grads`` (what a backward pass
  hands over), the AMP/clip/AdamW update by one of its three call sequences, ``zero_grad()``;
* ``norm``: the gradient norm that a loop logs;
* ``gather``: gradients kept from step to step: ``zero_grad(set_to_none=False)``, several micro-batches,
  a clip, and the clipped gradients read by the program (its own update rule, a reduction);
* ``refresh``: the low-precision copy of the weights that evaluation or export uses, brought up to date.

Lists come from ``namitorch_amd.param_lists`` (the GPT-2 and Llama layouts at the sizes the benchmark uses and at
smaller ones), a plain classifier, and one flat tensor.
"""

from __future__ import annotations

import gc
import math

import torch

import namitorch_amd as nt
from namitorch_amd.param_lists import gpt2_shapes, llama7b_shapes, numel, total_params

# A program that shares the GPU with PyTorch has the package's launches follow PyTorch's current stream.
nt.runtime.set_stream_provider(lambda device: torch.cuda.current_stream(device).cuda_stream)

_TORCH = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32, "float64": torch.float64}
_SIZE = {"float16": 2, "bfloat16": 2, "float32": 4, "float64": 8}
_LR, _BETAS, _DECAY, _SCALE, _STEP = 3e-4, (0.9, 0.999), 0.1, 65536.0, 10


def listed():
    return [
        # The smallest call there is in earnest: a classifier of six tensors, 26 thousand weights. Launch and host cost.
        {"name": "step_classifier", "kind": "step", "list": "mlp", "d": 128, "layers": 2, "dtype": "float32"},
        # One flat parameter (a flattened or sharded model): the benchmark's 4 Mi elements.
        {"name": "step_flat_4m", "kind": "step", "list": "flat", "d": 4194304, "layers": 1, "dtype": "float32"},
        # The headline: GPT-2 124M in float32.
        {"name": "step_gpt2_124m", "kind": "step", "list": "gpt2", "d": 768, "layers": 12, "vocab": 50257, "ctx": 1024,
         "dtype": "float32"},
        # Double precision (numerical studies, gradient checks of a whole model), with Adam's coupled decay.
        {"name": "step_adam_f64", "kind": "step", "list": "gpt2", "d": 384, "layers": 6, "vocab": 5003, "ctx": 512,
         "dtype": "float64", "adam": True},
        # Pure half precision: weights, gradients and moments in float16.
        {"name": "step_half", "kind": "step", "list": "gpt2", "d": 512, "layers": 8, "vocab": 10007, "ctx": 512,
         "dtype": "float16"},
        # A small model's AMP iteration: fresh float16 gradients every step, fused_step with a clip.
        {"name": "train_amp_small", "kind": "train", "list": "gpt2", "d": 256, "layers": 4, "vocab": 5003, "ctx": 256,
         "dtype": "float16", "state": "float32", "amp": True, "path": "fused", "micro": 1},
        # The same for GPT-2 124M.
        {"name": "train_amp_gpt2", "kind": "train", "list": "gpt2", "d": 768, "layers": 12, "vocab": 50257, "ctx": 1024,
         "dtype": "float16", "state": "float32", "amp": True, "path": "fused", "micro": 1},
        # The reference's call sequence (unscale_, clip, step, update) on a Llama-shaped list, bfloat16, two
        # micro-batches of which the last is deferred into the step.
        {"name": "train_api_llama", "kind": "train", "list": "llama", "d": 1024, "layers": 8, "vocab": 32000, "ctx": 2752,
         "dtype": "bfloat16", "state": "float32", "amp": True, "path": "api", "micro": 2, "defer": True},
        # The largest: GPT 1.3B, bfloat16 model, gradients and moments, float32 master, clip at 1.0, no scaler.
        {"name": "train_clip_gpt_1p3b", "kind": "train", "list": "gpt2", "d": 2048, "layers": 24, "vocab": 50304,
         "ctx": 2048, "dtype": "bfloat16", "state": "bfloat16", "amp": False, "path": "api", "micro": 1},
        # The L1 norm of the gradients, logged beside the L2 norm that clipping already gives.
        {"name": "norm_l1", "kind": "norm", "list": "gpt2", "d": 512, "layers": 8, "vocab": 10007, "ctx": 512,
         "dtype": "float32", "p": 1.0},
        # Gradients kept and read: two micro-batches into zeroed bfloat16 gradients, clipped, read.
        {"name": "gather_clip_gpt2", "kind": "gather", "list": "gpt2", "d": 768, "layers": 12, "vocab": 50257,
         "ctx": 1024, "dtype": "bfloat16", "micro": 2},
        # The bfloat16 copy of float32 weights for evaluation.
        {"name": "refresh_llama", "kind": "refresh", "list": "llama", "d": 1024, "layers": 8, "vocab": 32000, "ctx": 2752,
         "dtype": "float32", "to": "bfloat16"},
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "train", "train", "train", "norm", "gather", "refresh"])
    case = {"kind": kind, "list": rng.choice(["mlp", "gpt2", "gpt2", "llama"] + (["flat"] if kind != "train" else []))}
    if case["list"] == "flat":
        case.update(d=_spread(rng, 1000, 40_000_000), layers=1)
    elif case["list"] == "mlp":
        case.update(d=_spread(rng, 20, 1500), layers=rng.randint(1, 6))
    else:
        case.update(d=_spread(rng, 40, 1000), layers=rng.randint(1, 12), vocab=_spread(rng, 200, 50000))
        case["ctx"] = _spread(rng, 16, 1024) if case["list"] == "gpt2" else 8 * case["d"] // 3 + rng.randint(0, 7)
    # Views into one buffer without padding (bucketed gradients): odd sizes then leave tensors unaligned.
    case["pack"] = rng.random() < 0.2
    if kind == "step":
        case.update(dtype=rng.choice(["float32", "float32", "float64", "float16"]), adam=rng.random() < 0.3)
    elif kind == "train":
        case.update(dtype=rng.choice(["float16", "bfloat16"]), state=rng.choice(["float32", "bfloat16"]),
                    amp=rng.random() < 0.6, path=rng.choice(["fused", "api", "step"]), micro=rng.randint(1, 2))
        case["defer"] = case["micro"] == 2 and rng.random() < 0.5
    elif kind == "norm":
        case.update(dtype=rng.choice(["float32", "float16", "bfloat16"]), p=rng.choice([1.0, 2.0, 3.0, math.inf]))
    elif kind == "gather":
        case.update(dtype=rng.choice(["float32", "float16", "bfloat16"]), micro=rng.randint(1, 3))
    else:
        case.update(dtype="float32", to=rng.choice(["float16", "bfloat16", "float64"]))
    return case


def _shapes(case):
    d, layers = case["d"], case["layers"]
    if case["list"] == "flat":
        return [(d,)]
    if case["list"] == "mlp":
        widths = [64] + [d] * layers + [10]
        return [shape for a, b in zip(widths, widths[1:]) for shape in ((a, b), (b,))]
    if case["list"] == "gpt2":
        return gpt2_shapes(vocab=case["vocab"], ctx=case["ctx"], d=d, layers=layers)
    return llama7b_shapes(vocab=case["vocab"], d=d, layers=layers, ffn=case["ctx"])


# ---- one flat buffer per role, the tensors as views of it -----------------------------------------
class _Arena:
    """Where each tensor of a list lies in a flat buffer: starts on multiples of `align` elements."""

    def __init__(self, shapes, align):
        self.shapes, self.starts, self.total = shapes, [], 0
        for shape in shapes:
            self.starts.append(self.total)
            self.total += -(-numel(shape) // align) * align

    def views(self, flat):
        return [flat[start:start + numel(shape)].view(shape) for start, shape in zip(self.starts, self.shapes)]

    def normal(self, seed, salt, dtype, sigma, square=False):
        """A buffer of normal values, zero between the tensors; with `square`, of second moments that average several
        steps' squares (so none is far below the others, as none is in a run)."""
        generator = torch.Generator(device="cuda").manual_seed(1_000_003 * seed + salt)
        kind = torch.float64 if dtype == "float64" else torch.float32
        flat = torch.zeros(self.total, dtype=_TORCH[dtype], device="cuda")
        for view in self.views(flat):
            values = torch.randn(view.shape, generator=generator, dtype=kind, device="cuda").mul_(sigma)
            view.copy_(values.square_().mul_(0.75).add_(0.25 * sigma * sigma) if square else values)
        return flat


def _arenas(case):
    """(model and gradients, optimizer state): state starts on multiples of 256, as the optimizer lays it out."""
    shapes = _shapes(case)
    return _Arena(shapes, 1 if case.get("pack") else 64), _Arena(shapes, 256)


def _sigma(case):
    # Gradients as the benchmark draws them; float16 ones under the loss scale, or large enough for float16 moments.
    if case["kind"] == "step" and case["dtype"] == "float16":
        return 0.1
    return 1e-3 * (_SCALE if case.get("amp") else 1.0)


def _inputs(case, seed):
    model, state = _arenas(case)
    kind, dtype = case["kind"], case["dtype"]
    sigma = _sigma(case)
    real = sigma / _SCALE if case.get("amp") else sigma
    given = {"incoming": [model.normal(seed, 100 + k, dtype, sigma) for k in range(case.get("micro", 1))]}
    if kind == "refresh":
        return {"weights": model.normal(seed, 1, dtype, 0.02)}
    if kind == "step":
        given["param"] = model.normal(seed, 1, dtype, 0.02)
        given["exp_avg"] = state.normal(seed, 2, dtype, real / 3)
        given["exp_avg_sq"] = state.normal(seed, 3, dtype, real, square=True)
    elif kind == "train":
        given["master"] = state.normal(seed, 1, "float32", 0.02)
        given["param"] = torch.zeros(model.total, dtype=_TORCH[dtype], device="cuda")
        for view, master in zip(model.views(given["param"]), state.views(given["master"])):
            view.copy_(master)
        given["exp_avg"] = state.normal(seed, 2, case["state"], real / 3)
        given["exp_avg_sq"] = state.normal(seed, 3, case["state"], real, square=True)
    return given


def _tensors(arena, flat):
    return [nt.Tensor._from_storage(nt.DeviceArray.wrap(view)) for view in arena.views(flat)]


def _parameters(arena, flat):
    """Parameters over a program's own device memory (a Parameter built from an array copies it)."""
    made = []
    for view in arena.views(flat):
        parameter = nt.Parameter.__new__(nt.Parameter)
        nt.Tensor._initialize(parameter, nt.DeviceArray.wrap(view), True)
        made.append(parameter)
    return made


def _groups(params):
    """Weight decay on matrices only, as the training runner groups them."""
    groups = [{"params": [p for p in params if p.ndim >= 2], "weight_decay": _DECAY},
              {"params": [p for p in params if p.ndim < 2], "weight_decay": 0.0}]
    return [group for group in groups if group["params"]]


def _eps(case):
    return 1e-4 if case["kind"] == "step" and case["dtype"] == "float16" else 1e-8


def _optimizer(case, params, state, given):
    """The optimizer in the middle of a run: moments (and masters) filled, `_STEP` steps taken."""
    options = dict(lr=_LR, betas=_BETAS, eps=_eps(case))
    if case["kind"] == "train":
        names = ("exp_avg", "exp_avg_sq", "master")
        moment = nt.bfloat16 if case["state"] == "bfloat16" else None
        optimizer = nt.optim.AdamW(_groups(params), master_weights=True, state_dtype=moment, **options)
    else:
        names = ("exp_avg", "exp_avg_sq")
        optimizer = (nt.optim.Adam if case.get("adam") else nt.optim.AdamW)(_groups(params), **options)
    buffers = [_tensors(state, given[name]) for name in names]
    for parameter, values in zip(params, zip(*buffers)):
        optimizer.state[id(parameter)] = {**dict(zip(names, values)), "step": _STEP}
    return optimizer


def _room(case):
    """Two allocators share the card: before a list of many gigabytes is built, what earlier lists left behind goes
    back to the device (reading a version settles the steps whose outcome the host has not read yet)."""
    if total_params(_shapes(case)) > 500_000_000:
        nt.Tensor(0.0, device="cuda:0")._version
        gc.collect()
        nt.runtime.empty_cache(0)
        torch.cuda.empty_cache()


def prepare(case, seed):
    _room(case)
    given = _inputs(case, seed)
    model, state = _arenas(case)
    kind = case["kind"]
    held = {"case": case, "given": given}
    if kind == "refresh":
        held["copy"] = torch.zeros(model.total, dtype=_TORCH[case["to"]], device="cuda")
        held["pairs"] = list(zip(_tensors(model, held["copy"]), _tensors(model, given["weights"])))
        return held
    if kind in ("norm", "gather"):
        given["param"] = torch.zeros(model.total, dtype=_TORCH[case["dtype"]], device="cuda")
    params = held["params"] = _parameters(model, given["param"])
    held["incoming"] = [_tensors(model, flat) for flat in given["incoming"]]
    if kind in ("step", "norm"):
        for parameter, gradient in zip(params, held["incoming"][0]):
            parameter.grad = gradient
    if kind == "gather":
        held["grads"] = torch.zeros_like(given["param"])
        for parameter, gradient in zip(params, _tensors(model, held["grads"])):
            parameter.grad = gradient
        held["optimizer"] = nt.optim.AdamW(params, master_weights=True)
        held["max_norm"] = _max_norm(case, model)
    if kind in ("step", "train"):
        held["optimizer"] = _optimizer(case, params, state, given)
    if kind == "train":
        held["scaler"] = nt.GradScaler(init_scale=_SCALE) if case["amp"] else None
        held["loss"] = nt.Tensor._from_storage(nt.DeviceArray.wrap(torch.ones((), device="cuda")))
    return held


def _max_norm(case, model):
    """A bound that the gradients exceed by about a half (so the clip is applied), but 1.0 while training."""
    if case["kind"] == "train":
        return 1.0
    return 0.7 * _sigma(case) * math.sqrt(case["micro"] * sum(map(numel, model.shapes)))


def _accumulate(held, params):
    last = len(held["incoming"]) - 1
    for k, gradients in enumerate(held["incoming"]):
        nt.accumulate_grads(params, gradients, defer=bool(held["case"].get("defer")) and k == last > 0)


def _train(held):
    case, params, optimizer, scaler = held["case"], held["params"], held["optimizer"], held["scaler"]
    if scaler is not None:
        scaler.scale(held["loss"])
    _accumulate(held, params)
    norm = None
    if case["path"] == "fused":
        nt.amp.fused_step(optimizer, scaler, max_norm=1.0)
    elif case["path"] == "api":
        if scaler is None:
            nt.optim.clip_grad_norm_(params, 1.0)
            optimizer.step()
        else:
            if scaler.unscale_(optimizer):
                norm = nt.optim.clip_grad_norm_(params, 1.0).item()     # the runner logs it
            scaler.step(optimizer)
            scaler.update()
    elif scaler is None:
        optimizer.step()
    else:
        scaler.step(optimizer)
        scaler.update()
    optimizer.zero_grad()
    given = held["given"]
    outputs = {name: given[name] for name in ("param", "master", "exp_avg", "exp_avg_sq")}
    if norm is not None:
        outputs["norm"] = norm
    return outputs


def run(held):
    case, given = held["case"], held["given"]
    kind = case["kind"]
    if kind == "step":
        held["optimizer"].step()
        return {name: given[name] for name in ("param", "exp_avg", "exp_avg_sq")}
    if kind == "train":
        return _train(held)
    if kind == "norm":
        return nt.optim.get_grad_norm(held["params"], norm_type=case["p"]).item()
    if kind == "gather":
        params = held["params"]
        held["optimizer"].zero_grad(set_to_none=False)
        _accumulate(held, params)
        norm = nt.optim.clip_grad_norm_(params, held["max_norm"])
        for parameter in params:
            parameter.grad.detach()                                     # the program reads each gradient
        return {"grads": held["grads"], "norm": norm.item()}
    for copy, weights in held["pairs"]:
        copy.copy_(weights)
    return held["copy"]


def work(case):
    n, kind, size = total_params(_shapes(case)), case["kind"], _SIZE[case["dtype"]]
    if kind == "step":
        return {"bytes": 7 * size * n, "flops": 16 * n}
    if kind == "train":
        moments = _SIZE[case["state"]]
        # Each micro-batch's gradients read; master and moments read and written; the model copy written.
        return {"bytes": (size * case["micro"] + 2 * 4 + 4 * moments + size) * n, "flops": (20 + case["micro"]) * n}
    if kind == "norm":
        return {"bytes": size * n, "flops": 3 * n}
    if kind == "gather":
        return {"bytes": (case["micro"] + 1) * size * n, "flops": (4 + case["micro"]) * n}
    return {"bytes": (size + _SIZE[case["to"]]) * n, "flops": n}


def tolerance(case):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "refresh":
        return "exact"                                   # one correct rounding per value
    if kind == "norm":
        return {"rel": 1e-12}                            # sums in 64 bits
    if dtype == "float64":
        return {"rel": 1e-14}
    if kind == "step" and dtype == "float32":
        return {"rel": 2e-6}
    # Outputs of 16-bit types (half a unit in the last place is 2e-4 and 1.7e-3 over all values), norms of such gradients.
    return {"rel": 1e-2 if "bfloat16" in (dtype, case.get("state")) else 1e-3}


# ---- the same in 64 bits, tensor by tensor (the largest list would not fit the card all at once) ---------------
def _wide_grads(case, model, given):
    """Each tensor's gradient: the micro-batches' sum, unscaled."""
    for parts in zip(*(model.views(flat) for flat in given["incoming"])):
        total = sum(part.double() for part in parts)
        yield total / _SCALE if case.get("amp") else total


def _wide_norm(grads, p=2.0):
    if math.isinf(p):
        return max(float(g.abs().max()) for g in grads)
    return sum(float(g.abs().pow(p).sum()) for g in grads) ** (1 / p)


def _wide_step(case, g, p, m, v):
    """Adam/AdamW's step `_STEP + 1` on one tensor, in place."""
    step = _STEP + 1
    decay = _DECAY if g.dim() >= 2 else 0.0
    if case.get("adam"):
        g = g + decay * p
    m.mul_(_BETAS[0]).add_(g, alpha=1 - _BETAS[0])
    v.mul_(_BETAS[1]).add_(g * g, alpha=1 - _BETAS[1])
    update = (m / (1 - _BETAS[0] ** step)) / ((v / (1 - _BETAS[1] ** step)).sqrt() + _eps(case))
    if not case.get("adam"):
        p.mul_(1 - _LR * decay)
    p.sub_(update, alpha=_LR)


def exact(case, seed):
    given = _inputs(case, seed)
    model, state = _arenas(case)
    kind = case["kind"]
    if kind == "refresh":
        return given["weights"].double()
    if kind == "norm":
        return _wide_norm(_wide_grads(case, model, given), case["p"])
    outputs, coefficient = {}, 1.0
    if kind == "gather" or (kind == "train" and case["path"] != "step"):
        norm = _wide_norm(_wide_grads(case, model, given))
        coefficient = min(1.0, _max_norm(case, model) / (norm + 1e-6))
        if kind == "gather" or (case["path"] == "api" and case["amp"]):
            outputs["norm"] = norm
    if kind == "gather":
        outputs["grads"] = torch.zeros(model.total, dtype=torch.float64, device="cuda")
        for view, gradient in zip(model.views(outputs["grads"]), _wide_grads(case, model, given)):
            view.copy_(gradient.mul_(coefficient))
        return outputs
    for name in ("exp_avg", "exp_avg_sq"):
        outputs[name] = given.pop(name).double()
    weights, at = ("param", model) if kind == "step" else ("master", state)
    outputs[weights] = given.pop(weights).double()
    lists = (at.views(outputs[weights]), state.views(outputs["exp_avg"]), state.views(outputs["exp_avg_sq"]))
    for gradient, *tensors in zip(_wide_grads(case, model, given), *lists):
        _wide_step(case, gradient.mul_(coefficient), *tensors)
    if kind == "train":
        given.clear()
        outputs["param"] = torch.zeros(model.total, dtype=torch.float64, device="cuda")
        for view, wide in zip(model.views(outputs["param"]), state.views(outputs["master"])):
            view.copy_(wide)
    return outputs
