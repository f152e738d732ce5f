"""The optimizer-step workloads whose speed this repository is judged by.

Each case is one call sequence a training program makes with this package:

  step   set_optimizer_lr, GradScaler.unscale_, clip_grad_norm_, AdamW.step and
         GradScaler.update over one parameter set, either eagerly or as a
         replayed HIP graph (capturable=True)
  clip   clip_grad_norm_ over parameters that no AdamW of this package owns:
         the gradients are scaled in place
  norm   mgopt_grad_norm_noalloc of the C ABI over one flat gradient buffer

Parameters, gradients and saved optimizer state are made as flat buffers whose
tensors start on 512-byte boundaries, as torch's caching allocator places
separate tensors.  The optimizer resumes from a saved state (non-zero moments,
step 1,000), so every pass is a step in the middle of a training run; a
replayed step starts a new run with one eager step instead.
"""

from __future__ import annotations

import ctypes
import importlib
import math
import os

import torch

mg = importlib.import_module("minigpt-train-infra_amd")
paramsets = importlib.import_module("minigpt-train-infra_amd.paramsets")

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
CODES = {"f32": 0, "f16": 1, "bf16": 2}         # include/mgopt.h
ALIGN = 512                                     # bytes between tensor starts
SCALE = 65536.0                                 # loss scale of the scaled cases
SIGMA = 1e-2                                    # unscaled gradient standard deviation
RESUME_STEP = 1000
MAX_STEPS, WARMUP, LR, MIN_LR = 100_000, 100, 3e-4, 3e-5
BETAS, EPS, DECAY, MAX_NORM = (0.9, 0.95), 1e-8, 0.1, 1.0
SHOWN_LARGE, SHOWN_SMALL = 9, 3                 # tensors whose optimizer state is returned


# ----------------------------------------------------------------- the cases


def _step(name, shapes, param, grad, **more):
    """A whole optimizer step.  scaler: a GradScaler drives it; replay: as a
    captured HIP graph; layout: AdamW's state_layout; writeback: the clipped
    gradients are stored back into .grad."""
    case = {"kind": "step", "param": param, "grad": grad, "scaler": False, "replay": False, "layout": "rows",
            "writeback": False, **shapes, **more}
    return {"name": name, **case} if name else case


def _gpt(vocab, block, n_layer, n_embd):
    return {"family": "gpt", "vocab": vocab, "block": block, "n_layer": n_layer, "n_embd": n_embd}


def _uniform(total, tensors):
    return {"family": "uniform", "total": total, "tensors": tensors}


def _ragged(tensors, total, sizes_seed):
    return {"family": "ragged", "tensors": tensors, "total": total, "sizes_seed": sizes_seed}


def _qwen(n_layer):
    return {"family": "qwen", "n_layer": n_layer}


def listed():
    return [
        # the MiniGPT configuration the reference trains (0.8M parameters), fp32 without a loss scale:
        # the smallest step a user takes, where launches and host time count
        _step("tiny_fp32", _gpt(96, 128, 4, 128), "f32", "f32"),
        # the same model with fp16 gradients and a GradScaler, the step captured once and replayed
        _step("tiny_fp16_replay", _gpt(96, 128, 4, 128), "f32", "f16", scaler=True, replay=True),
        # a few million elements in a handful of equal tensors: adapters, heads, one layer of a small model
        _step("uniform_4m_fp32", _uniform(4_194_304, 16), "f32", "f32"),
        # a small language model (39M parameters, half of them in the embedding), bf16 with fp32 masters
        _step("gpt_4x512_bf16", _gpt(50304, 1024, 4, 512), "bf16", "bf16"),
        # GPT-2-small, fp32 parameters, fp16 gradients, GradScaler: the mixed-precision run of the reference's loop
        _step("gpt2_small_fp16", _gpt(50304, 1024, 12, 768), "f32", "f16", scaler=True),
        # the same set entirely in fp32, contiguous state, for a program that reads .grad after the step
        _step("gpt2_small_writeback", _gpt(50304, 1024, 12, 768), "f32", "f32", layout="separate", writeback=True),
        # GPT-1.3B in bf16 with fp32 masters
        _step("gpt_1p3b_bf16", _gpt(50304, 1024, 24, 2048), "bf16", "bf16"),
        # the Qwen3-8B shapes with 8 of their 36 layers (2.8B parameters), bf16 with masters and a GradScaler:
        # a large model, and one GPU's share of a sharded larger one
        _step("qwen3_8_layers_bf16", _qwen(8), "bf16", "bf16", scaler=True),
        # 20,000 tensors of log-uniform odd sizes, fp32 parameters, fp16 gradients, GradScaler
        _step("ragged_20k_fp16", _ragged(20_000, 2_500_000_000, 5), "f32", "f16", scaler=True),
        # gradient clipping for a model another optimizer steps
        {"name": "clip_gpt2_small_bf16", "kind": "clip", "grad": "bf16", **_gpt(50304, 1024, 12, 768)},
        # the norm of one flat gradient buffer, for callers that may not allocate
        {"name": "norm_flat_16m_bf16", "kind": "norm", "grad": "bf16", "total": 16_777_259},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes over the whole range, no dearer than the largest listed one."""
    kind = rng.choices(("step", "clip", "norm"), (0.75, 0.15, 0.1))[0]
    grad = rng.choice(("f32", "f16", "bf16"))
    if kind == "norm":
        return {"kind": kind, "grad": grad, "total": _log_uniform(rng, 100_000, 1_000_000_000)}
    family = rng.choices(("gpt", "uniform", "ragged"), (0.5, 0.25, 0.25))[0]
    if family == "gpt":
        shapes = _gpt(_log_uniform(rng, 65, 50304), rng.choice((128, 256, 1000, 1024, 2048)), rng.randint(1, 24),
                      8 * _log_uniform(rng, 8, 256))
    elif family == "uniform":
        k = _log_uniform(rng, 1, 500)
        shapes = _uniform(max(k, _log_uniform(rng, 200_000, 600_000_000)), k)
    else:
        n = _log_uniform(rng, 20, 10_000)
        shapes = _ragged(n, min(1_500_000_000, n * _log_uniform(rng, 3_000, 300_000)), rng.randint(0, 9999))
    if kind == "clip":
        return {"kind": kind, "grad": grad, **shapes}
    param, grad = rng.choice((("f32", "f32"), ("f32", "f16"), ("f32", "bf16"), ("bf16", "bf16"), ("f16", "f16")))
    scaler, replay = grad == "f16" or rng.random() < 0.3, rng.random() < 0.15
    # written-back gradients are the next pass's input, so only without a loss scale to take off again
    return _step(None, shapes, param, grad, scaler=scaler, replay=replay, layout=rng.choice(("rows",) * 4 + ("separate",)),
                 writeback=not (scaler or replay) and rng.random() < 0.4)


# ---------------------------------------------------------------- the inputs


def _shapes(case):
    """Tensor shapes, those with weight decay (two and more dimensions) first, and how many have it."""
    if case["family"] == "gpt":
        got = paramsets.minigpt_shapes(case["vocab"], case["block"], case["n_layer"], case["n_embd"])
    elif case["family"] == "qwen":
        got = paramsets.qwen3_shapes(n_layer=case["n_layer"])
    elif case["family"] == "uniform":
        got = paramsets.uniform_shapes(case["total"], case["tensors"])
    else:
        got = paramsets.ragged_shapes(case["tensors"], total=case["total"], seed=case["sizes_seed"])
    decay = [s for _, s in got if len(s) >= 2]
    return decay + [s for _, s in got if len(s) < 2], len(decay)


def _numel(case):
    return case["total"] if case["kind"] == "norm" else sum(math.prod(s) for s in _shapes(case)[0])


class _Flat:
    """Tensors of the given shapes in one flat buffer, 512-byte aligned, zero between them."""

    def __init__(self, shapes, dtype):
        pad = ALIGN // 2                        # elements of the narrowest type, so that all types share offsets
        self.offsets, end = [], 0
        for s in shapes:
            self.offsets.append(end)
            end += -(-math.prod(s) // pad) * pad
        self.shapes, self.dtype, self.total = shapes, dtype, end

    def views(self, flat):
        return [flat[o : o + math.prod(s)].view(s) for o, s in zip(self.offsets, self.shapes)]

    def normal(self, gen, sigma):
        flat = torch.empty(self.total, dtype=self.dtype, device=DEV).normal_(0.0, sigma, generator=gen)
        return self._clear(flat)

    def squares(self, gen, size):
        flat = torch.empty(self.total, dtype=self.dtype, device=DEV).uniform_(0.5 * size, 1.5 * size, generator=gen)
        return self._clear(flat)

    def _clear(self, flat):
        gaps = [flat[o + n : e] for o, n, e in zip(self.offsets, map(math.prod, self.shapes),
                                                  self.offsets[1:] + [self.total]) if o + n < e]
        if gaps:
            torch._foreach_zero_(gaps)
        return flat


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _inputs(case, seed):
    """The flat buffers of a case, the same for the same seed."""
    gen = _generator(seed)
    if case["kind"] == "norm":
        return {"grad": torch.empty(case["total"], dtype=DTYPES[case["grad"]], device=DEV).normal_(0.0, SIGMA, generator=gen)}
    shapes, _ = _shapes(case)
    scale = SCALE if case.get("scaler") else 1.0
    out = {"grad": _Flat(shapes, DTYPES[case["grad"]]).normal(gen, SIGMA * scale)}
    if case["kind"] == "clip":
        return out
    f32 = _Flat(shapes, torch.float32)
    out["exp_avg"], out["exp_avg_sq"] = f32.normal(gen, 1e-4), f32.squares(gen, 1e-8)
    weight = f32.normal(gen, 0.02)
    if case["param"] == "f32":
        out["weight"] = weight
    else:
        out["master"], out["weight"] = weight, weight.to(DTYPES[case["param"]])
    return out


def _lr(step):
    return mg.cosine_lr(RESUME_STEP + step, LR, MIN_LR, WARMUP, MAX_STEPS)


def _shown(shapes):
    """The tensors whose optimizer state a step returns: the largest and the smallest."""
    order = sorted(range(len(shapes)), key=lambda i: -math.prod(shapes[i]))
    return order if len(order) <= SHOWN_LARGE + SHOWN_SMALL else order[:SHOWN_LARGE] + order[-SHOWN_SMALL:]


# ------------------------------------------------------------------ prepare


def _library():
    lib = ctypes.CDLL(os.path.join(os.getcwd(), "minigpt-train-infra_amd", "_build", "libmgopt.so"))
    vp = ctypes.c_void_p
    lib.mgopt_grad_norm_noalloc.argtypes = [vp, ctypes.c_int32, ctypes.c_int64, vp, ctypes.c_double, vp, vp, vp, vp]
    lib.mgopt_last_error.restype = ctypes.c_char_p
    return lib


def prepare(case, seed):
    bufs = _inputs(case, seed)
    if case["kind"] == "norm":
        out = torch.zeros(3, dtype=torch.float32, device=DEV)
        return {"kind": "norm", "lib": _library(), "grad": bufs["grad"], "code": CODES[case["grad"]], "out": out}
    shapes, n_decay = _shapes(case)
    if case["kind"] == "clip":
        flat = _Flat(shapes, DTYPES[case["grad"]])
        weight = flat.normal(_generator(seed + 1), 0.02)
        params = [torch.nn.Parameter(w) for w in flat.views(weight)]
        for p, g in zip(params, flat.views(bufs["grad"])):
            p.grad = g
        return {"kind": "clip", "params": params, "grad": bufs["grad"]}

    f32 = _Flat(shapes, torch.float32)
    params = [torch.nn.Parameter(w) for w in f32.views(bufs["weight"])]
    groups = [{"params": params[:n_decay], "weight_decay": DECAY}, {"params": params[n_decay:], "weight_decay": 0.0}]
    opt = mg.AdamW([g for g in groups if g["params"]], lr=LR, betas=BETAS, eps=EPS, state_layout=case["layout"],
                   writeback_grads=case["writeback"], capturable=case["replay"])
    if not case["replay"]:
        saved = opt.state_dict()
        step = torch.tensor(float(RESUME_STEP))
        masters = f32.views(bufs["master"]) if "master" in bufs else [None] * len(shapes)
        for i, (m, v, w) in enumerate(zip(f32.views(bufs["exp_avg"]), f32.views(bufs["exp_avg_sq"]), masters)):
            saved["state"][i] = {"step": step, "exp_avg": m, "exp_avg_sq": v}
            if w is not None:
                saved["state"][i]["master_param"] = w
        opt.load_state_dict(saved)
    grads = f32.views(bufs["grad"])
    if case["grad"] == case["param"]:
        for p, g in zip(params, grads):
            p.grad = g
    else:
        opt.set_grad_source(grads)
    scaler = None
    if case["scaler"]:
        scaler = mg.GradScaler("cuda", init_scale=SCALE)
        scaler.scale(torch.ones((), device=DEV))
    out = {"weight": bufs["weight"]}
    state = {"kind": "step", "params": params, "opt": opt, "scaler": scaler, "step": 0, "out": out, "graph": None}
    if case["replay"]:
        _one_step(state)                        # the eager step that capture needs
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            out["norm"] = _launches(state)
        state["graph"] = graph
    if scaler is not None:
        out["scale"], out["tracker"] = scaler._scale, scaler._growth_tracker
    if case["writeback"]:
        out["grad"] = bufs["grad"]
    for i in _shown(shapes):
        for key, value in opt.state[params[i]].items():
            out[f"{key}.{i}"] = value
    return state


# ---------------------------------------------------------------------- run


def _launches(state):
    opt, scaler = state["opt"], state["scaler"]
    if scaler is not None:
        scaler.unscale_(opt)
    norm = mg.clip_grad_norm_(state["params"], MAX_NORM)
    if scaler is not None:
        scaler.step(opt)
        scaler.update()
    else:
        opt.step()
    return norm


def _one_step(state):
    mg.set_optimizer_lr(state["opt"], _lr(state["step"]))
    state["step"] += 1
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        state["out"]["norm"] = _launches(state)


def run(state):
    if state["kind"] == "norm":
        out = state["out"].data_ptr()
        grad = state["grad"]
        rc = state["lib"].mgopt_grad_norm_noalloc(grad.data_ptr(), state["code"], grad.numel(), None, MAX_NORM, out,
                                                  out + 4, out + 8, torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError(state["lib"].mgopt_last_error().decode())
        return {"norm_coef_found": state["out"]}
    if state["kind"] == "clip":
        return {"norm": mg.clip_grad_norm_(state["params"], MAX_NORM), "grad": state["grad"]}
    _one_step(state)
    return state["out"]


# --------------------------------------------------- work, tolerance, oracle


def work(case):
    n = _numel(case)
    g = BYTES[case["grad"]]
    if case["kind"] == "norm":
        return {"bytes": n * g, "flops": 2 * n}
    if case["kind"] == "clip":
        return {"bytes": n * 2 * g, "flops": 3 * n}
    per = g + 24 + (2 if case["param"] != "f32" else 0) + (g if case["writeback"] else 0)
    return {"bytes": n * per, "flops": 20 * n}


def tolerance(case):
    # fp32 results of one correctly rounded evaluation differ from another's by a few units in the last place
    # (6e-8); a 16-bit result may round the other way where the fp32 value lies next to a tie, at most one unit
    # (2**-7 of the value in bf16, 2**-10 in fp16) in few elements.
    narrow = {case["grad"]} if case["kind"] == "clip" or case.get("writeback") else set()
    narrow |= {case["param"]} if case["kind"] == "step" else set()
    if "bf16" in narrow:
        return {"rel": 1e-4, "max": 0.016}
    if "f16" in narrow:
        return {"rel": 2e-5, "max": 0.002}
    return {"rel": 1e-6, "max": 2e-5}


def exact(case, seed):
    """The first pass in fp64 (for a replayed case, the second step: the first ran eagerly before the capture)."""
    bufs = _inputs(case, seed)
    if case["kind"] == "norm":
        norm = math.sqrt(sum(float(part.double().square().sum()) for part in bufs["grad"].split(1 << 26)))
        return {"norm_coef_found": torch.tensor([norm, min(1.0, MAX_NORM / (norm + 1e-6)), 0.0], dtype=torch.float64)}
    shapes, n_decay = _shapes(case)
    flat = _Flat(shapes, torch.float32)
    inv = 1.0 / SCALE if case.get("scaler") else 1.0
    norm = inv * math.sqrt(sum(float(part.double().square().sum()) for part in bufs["grad"].split(1 << 26)))
    coef = min(1.0, MAX_NORM / (norm + 1e-6))
    norm_out = torch.tensor(norm, dtype=torch.float64)
    if case["kind"] == "clip":
        return {"norm": norm_out, "grad": bufs["grad"].double() * coef}

    shown = set(_shown(shapes))
    begun, steps = (0, 2) if case["replay"] else (RESUME_STEP, 1)
    weight = torch.zeros(flat.total, dtype=torch.float64, device=DEV)
    out = {"weight": weight}
    grad = torch.zeros(flat.total, dtype=torch.float64, device=DEV) if case["writeback"] else None
    views = {k: flat.views(b) for k, b in bufs.items()}
    targets = flat.views(weight)
    written = flat.views(grad) if grad is not None else None
    for i in range(len(shapes)):
        p = (views["master"] if "master" in views else views["weight"])[i].double()
        m, v, g = (views[k][i].double() for k in ("exp_avg", "exp_avg_sq", "grad"))
        if not begun:                           # a new run: masters widened from the weights, no moments yet
            p = views["weight"][i].double()
            m, v = torch.zeros_like(m), torch.zeros_like(v)
        u = g * (inv * coef)
        for k in range(1, steps + 1):
            t = begun + k
            lr = _lr(k - 1)
            if i < n_decay:
                p = p * (1.0 - lr * DECAY)
            m = m + (1.0 - BETAS[0]) * (u - m)
            v = v * BETAS[1] + (1.0 - BETAS[1]) * u * u
            bc1, bc2 = 1.0 - BETAS[0] ** t, 1.0 - BETAS[1] ** t
            p = p - (lr / bc1) * m / (v.sqrt() / math.sqrt(bc2) + EPS)
        targets[i].copy_(p)
        if written is not None:
            written[i].copy_(u)
        if i in shown:
            out[f"step.{i}"] = torch.tensor(float(begun + steps), dtype=torch.float64)
            out[f"exp_avg.{i}"], out[f"exp_avg_sq.{i}"] = m, v
            if case["param"] != "f32":
                out[f"master_param.{i}"] = p
    if grad is not None:
        out["grad"] = grad
    if case["scaler"]:
        out["scale"] = torch.tensor(SCALE, dtype=torch.float64)
    out["norm"] = norm_out
    return out
