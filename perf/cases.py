"""The work that users of this framework have it do, as cases that can be timed: training steps, evaluation passes and
text generation through the C ABI of include/llmk_gpt2.h, over the model sizes its descriptors name, both storage types,
the options of the trainer program and sequence lengths that are not multiples of anything.

listed() are the cases to look at one by one, draw() gives more of the same ranges. The library is the one of the working
folder (llm.c_amd/lib), which has to be built.
"""
import ctypes as C
import importlib.util
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

# descriptor -> layers, heads, channels, longest sequence (gpt2_build_from_descriptor)
MODELS = {
    "d6": (6, 6, 384, 1024),
    "d12": (12, 12, 768, 1024),
    "d24": (24, 16, 1024, 1024),
    "d36": (36, 20, 1280, 1024),
    "d48": (48, 25, 1600, 1024),
    "gpt3:c768": (12, 12, 768, 2048),
    "gpt3:c1536": (24, 16, 1536, 2048),     # heads of 96
    "gpt3:c2048": (24, 16, 2048, 2048),     # heads of 128
}
VOCAB, PADDED_VOCAB = 50257, 50304
EOT = 50256
PARAM_NAMES = ("wte", "wpe", "ln1w", "ln1b", "qkvw", "qkvb", "attprojw", "attprojb", "ln2w", "ln2b", "fcw", "fcb",
               "fcprojw", "fcprojb", "lnfw", "lnfb")


# ---- the cases -------------------------------------------------------------------------------------------------------
def _train(model, B, T, precision="bf16", recompute=0, gelu_fusion=3, micro_steps=1):
    return {"kind": "train", "model": model, "B": B, "T": T, "precision": precision, "recompute": recompute,
            "gelu_fusion": gelu_fusion, "micro_steps": micro_steps}


def _validate(model, B, T, precision="bf16"):
    return {"kind": "validate", "model": model, "B": B, "T": T, "precision": precision}


def _generate(model, tokens, precision="bf16"):
    return {"kind": "generate", "model": model, "tokens": tokens, "precision": precision}


def listed():
    return [
        # the smallest step anyone runs on purpose: the shape of the CPU trainer's default run, launches and the optimizer
        dict(_train("d12", 4, 64), name="train_d12_b4_t64"),
        # a debugging model on odd sizes
        dict(_train("d6", 7, 333), name="train_d6_b7_t333"),
        # the trainer program's defaults: -b 4 -t 1024 -r 1 -ge 2
        dict(_train("d12", 4, 1024, recompute=1, gelu_fusion=2), name="train_d12_b4_t1024"),
        # the benchmark configuration
        dict(_train("d12", 64, 1024), name="train_d12_b64_t1024"),
        # gradient accumulation through the four calls of the reference's loop
        dict(_train("d24", 16, 1024, micro_steps=2), name="train_d24_b16_t1024_accum2"),
        # the largest GPT-2 at its published batch, activations recomputed
        dict(_train("d48", 16, 1024, recompute=1, gelu_fusion=2), name="train_d48_b16_t1024"),
        # the GPT-3 sizes: heads of 128 at the full context, heads of 96 on a ragged batch
        dict(_train("gpt3:c2048", 2, 2048), name="train_c2048_b2_t2048"),
        dict(_train("gpt3:c1536", 3, 1000, recompute=2, gelu_fusion=2), name="train_c1536_b3_t1000"),
        # the single-precision library, used to check against the CPU trainer
        dict(_train("d12", 4, 512, precision="fp32"), name="train_fp32_d12_b4_t512"),
        # validation loss: a batch shorter than what training uses, and one of the multiple-choice evaluation's ragged ones
        dict(_validate("d12", 32, 1024), name="validate_d12_b32_t1024"),
        dict(_validate("d24", 5, 777), name="validate_d24_b5_t777"),
        # the trainer's sampling pass: 64 tokens, one at a time
        dict(_generate("d12", 64), name="generate_d12_64"),
    ]


def _between(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("train", "train", "train", "train", "validate", "validate", "generate"))
    if kind == "generate":
        return _generate(rng.choice(("d6", "d12", "d24", "gpt3:c1536")), rng.randint(16, 96), rng.choice(("bf16", "bf16", "bf16", "fp32")))
    fp32 = rng.random() < 0.15
    model = rng.choice(("d6", "d12")) if fp32 else rng.choice(tuple(MODELS))
    longest = MODELS[model][3]
    for _ in range(100):
        T = _between(rng, 48, longest)
        if rng.random() < 0.4:                       # round lengths are what people type
            T = max(64, T // 64 * 64)
        B = _between(rng, 1, 64)
        case = _train(model, B, T) if kind == "train" else _validate(model, B, T)
        # single precision runs at a sixteenth of the rate; heads that are not 64 wide are for few sequences at a time
        scale = 24.0 if fp32 else 1.0
        tokens = 4096 if MODELS[model][2] // MODELS[model][1] != 64 else 65536
        if work(case)["flops"] * scale <= 8e13 and B * T <= tokens:
            break
    else:
        B, T = 1, 64
    precision = "fp32" if fp32 else "bf16"
    if kind == "validate":
        return _validate(model, B, T, precision)
    recompute = rng.choice((0, 0, 1, 2))
    return _train(model, B, T, precision, recompute, rng.choice((0, 2, 3)) if recompute == 0 else rng.choice((0, 2)),
                  rng.choice((1, 1, 2)))


# ---- what a program has in hand ----------------------------------------------------------------------------------------
_package = None


def _library(precision):
    global _package
    if _package is None:
        spec = importlib.util.spec_from_file_location("llmc_amd", os.path.join(os.getcwd(), "llm.c_amd", "__init__.py"))
        _package = importlib.util.module_from_spec(spec)
        sys.modules["llmc_amd"] = _package
        spec.loader.exec_module(_package)
    first = precision not in _package._loaded
    lib = _package.load(precision)
    if first:
        lib.llmk_init(0)
    return lib


class _Memory:
    """Device memory of a model as an array; holds on to the model that owns it."""

    def __init__(self, owner, address, shape, precision):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<i2" if precision == "bf16" else "<f4",
                                         "data": (address, False), "version": 2}


class _Model:
    def __init__(self, case, B, T):
        self.precision = case["precision"]
        self.lib = _library(self.precision)
        self.layers, self.heads, self.channels, self.longest = MODELS[case["model"]]
        self.handle = self.lib.gpt2_create()
        self.lib.gpt2_set_options(self.handle, 1, case.get("recompute", 1), case.get("gelu_fusion", 2))
        header = [20240326, 5 if self.precision == "bf16" else 3, self.longest, VOCAB, self.layers, self.heads, self.channels,
                  PADDED_VOCAB] + [0] * 248
        with tempfile.NamedTemporaryFile(suffix=".bin") as f:      # the shape alone: the weights are written below
            f.write(struct.pack("256i", *header))
            f.flush()
            self.lib.gpt2_build_from_checkpoint(self.handle, f.name.encode(), 0)
        self.parameters = self.lib.gpt2_num_parameters(self.handle)
        self.lib.gpt2_allocate_state(self.handle, B, T)
        self.B, self.T = B, T

    def __del__(self):
        if getattr(self, "handle", None):
            self.lib.gpt2_free(self.handle)
            self.handle = None

    def tensor(self, address, *shape):
        t = torch.as_tensor(_Memory(self, address, shape, self.precision), device="cuda")
        return t.view(torch.bfloat16) if self.precision == "bf16" else t

    def params(self):
        return self.tensor(self.lib.gpt2_params_memory(self.handle), self.parameters)

    def grads(self):
        return self.tensor(self.lib.gpt2_grads_memory(self.handle), self.parameters)

    def fill(self, seed, final_gain=1.0):
        """GPT-2's initial weights: N(0, 0.02), residual projections divided by sqrt(2 L), LayerNorm weights 1, biases 0."""
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        sizes = (C.c_size_t * 16)()
        self.lib.gpt2_param_sizes(self.handle, sizes)
        at, p = 0, self.params()
        for name, n in zip(PARAM_NAMES, sizes):
            part = p[at:at + n]
            at += n
            if name in ("ln1w", "ln2w"):
                part.fill_(1.0)
            elif name == "lnfw":
                part.fill_(final_gain)
            elif name.endswith("b"):
                part.zero_()
            else:
                part.normal_(0.0, 0.02 / math.sqrt(2 * self.layers) if "proj" in name else 0.02, generator=gen)
                if name == "wte":
                    part[VOCAB * self.channels:].zero_()
        torch.cuda.synchronize()


def _tokens(rng, n):
    """n tokens with the frequencies of text: the r-th most common of the vocabulary in proportion to 1 / (r + 2.7)."""
    frequency = 1.0 / (np.arange(1, VOCAB + 1) + 2.7)
    edges = np.cumsum(frequency / frequency.sum())
    rank = np.minimum(np.searchsorted(edges, rng.random_sample(n)), VOCAB - 1)
    return ((rank.astype(np.int64) * 7919) % VOCAB).astype(np.int32)       # common tokens lie all over the vocabulary


def prepare(case, seed):
    rng = np.random.RandomState(seed % (1 << 32))
    if case["kind"] == "generate":
        # the trainer samples with the batch that it trains on allocated: its defaults are 4 x 1024
        model = _Model(case, 4, 1024)
        model.fill(seed, final_gain=6.0)             # a trained model's logits spread over several nats
        return {"case": case, "model": model, "tokens": np.zeros(model.B * model.T, np.int32), "rng": 1337 + 2 * seed}
    B, T = case["B"], case["T"]
    # evaluation runs on the model that is being trained; what it takes is at most the training batch
    model = _Model(case, B, T) if case["kind"] == "train" else _Model(case, B + 1, min(MODELS[case["model"]][3], T + 64))
    model.fill(seed)
    batches = []
    for _ in range(case.get("micro_steps", 1)):
        stream = _tokens(rng, B * T + 1)
        batches.append((np.ascontiguousarray(stream[:-1]), np.ascontiguousarray(stream[1:])))
    return {"case": case, "model": model, "batches": batches, "step": 0}


# ---- one pass ------------------------------------------------------------------------------------------------------------
LR, BETA1, BETA2, EPS, DECAY, CLIP = 3e-4, 0.9, 0.95, 1e-8, 0.1, 1.0


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def run(state):
    case, model = state["case"], state["model"]
    lib, h = model.lib, model.handle
    if case["kind"] == "generate":
        n = case["tokens"]
        rng = C.c_ulonglong(state["rng"])
        lib.gpt2_generate(h, _ptr(state["tokens"]), n, EOT, C.byref(rng))
        # the tokens, and the logits that the last of them was drawn from
        logits = model.tensor(lib.gpt2_output_memory(h) + (n - 2) * PADDED_VOCAB * (2 if model.precision == "bf16" else 4), PADDED_VOCAB)
        return {"tokens": torch.from_numpy(state["tokens"][:n].copy()), "logits": logits[:VOCAB]}
    if case["kind"] == "validate":
        B, T = case["B"], case["T"]
        inputs, targets = state["batches"][0]
        loss = lib.gpt2_validate(h, _ptr(inputs), _ptr(targets), B, T)
        losses = np.ctypeslib.as_array(lib.gpt2_cpu_losses(h), (B * T,)).copy()
        logits = model.tensor(lib.gpt2_output_memory(h), B * T, PADDED_VOCAB)
        return {"loss": loss, "losses": torch.from_numpy(losses), "logits": logits}
    state["step"] += 1
    if case["micro_steps"] == 1:
        loss, norm = C.c_float(), C.c_float()
        inputs, targets = state["batches"][0]
        lib.gpt2_train_step(h, _ptr(inputs), _ptr(targets), LR, BETA1, BETA2, EPS, DECAY, CLIP, state["step"], C.byref(loss),
                            C.byref(norm))
        loss, norm = loss.value, norm.value
    else:
        steps = case["micro_steps"]
        for k, (inputs, targets) in enumerate(state["batches"]):
            lib.gpt2_forward(h, _ptr(inputs), case["B"], case["T"])
            lib.gpt2_backward_and_reduce(h, _ptr(inputs), _ptr(targets), steps, k)
        loss = lib.gpt2_mean_loss(h)
        norm = lib.gpt2_calculate_grad_norm(h)
        scale = CLIP / norm if norm > CLIP else 1.0
        lib.gpt2_update(h, LR, BETA1, BETA2, EPS, DECAY, scale, state["step"], 0)
    return {"loss": loss, "norm": norm, "grads": model.grads(), "params": model.params()}


# ---- what it cannot do without, and how far results may be apart -----------------------------------------------------------
def work(case):
    L, NH, Cc, longest = MODELS[case["model"]]
    X = 2 if case["precision"] == "bf16" else 4
    matrices = L * 12 * Cc * Cc + PADDED_VOCAB * Cc          # weights that every token is multiplied with
    P = matrices + longest * Cc + L * 13 * Cc + 2 * Cc
    if case["kind"] == "generate":
        n = case["tokens"] - 1                               # one token after the other: the weights are read for each
        return {"bytes": float(n * matrices * X), "flops": float(n * 2 * matrices + L * 4 * Cc * (n * (n + 1) // 2))}
    B, T = case["B"], case["T"]
    forward = 2.0 * B * T * matrices + L * 4.0 * Cc * B * (T * (T + 1) // 2)
    if case["kind"] == "validate":
        return {"bytes": float(P * X + B * T * (PADDED_VOCAB * X + 12)), "flops": forward}
    # forward and twice as much backward (attention two and a half times); parameters, gradients and the fp32 state
    backward = 2.0 * 2.0 * B * T * matrices + L * 10.0 * Cc * B * (T * (T + 1) // 2)
    micro = case["micro_steps"]
    return {"bytes": float(P * (3 * X + 24) + micro * B * T * 8), "flops": micro * (forward + backward)}


def tolerance(case):
    """About four times what a run shows against another correct one. Single precision: the batch in reverse order moves the
    gradients by 8e-7 and single updated weights (a first AdamW step has the sign of a gradient near zero) by 3e-4 of their
    root mean square. bf16: against the single-precision library on the same weights the logits are off by 1.3e-2, the
    gradients by 4e-3 to 1.5e-2, single small gradients by up to their root mean square."""
    if case["precision"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}
    if case["kind"] == "train":
        return {"rel": 0.03, "max": 0.99, "differ": 0.0}
    return {"rel": 0.03, "max": 0.3, "differ": 0.0}
