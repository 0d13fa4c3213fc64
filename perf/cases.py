"""What the library is timed on: the calls that training and generation with it consist of.

Every case goes through the Python binding of the C ABI (`deers_amd.rocm`), on torch tensors
that live on the GPU.  Six kinds of work (`case["work"]`):

  train       forward and backward of causal attention, one layer
  prefill     a prompt's keys and values into the KV cache, then attention over the prompt
  decode      one query per sequence against a KV cache
  generate    one token of a GPT: embedding, every block through the few-rows products and the
              appending decode, final norm, LM head
  loss        cross-entropy of a batch of logits with its gradient
  optimizer   gradient norm, read by the host, and an AdamW step over all parameters
  block_ops   the other kernels around attention and the products in a training step: embedding,
              RMSNorm, rotary embedding, squared ReLU, forward and backward
"""
import ctypes
import math

import numpy as np
import torch

from deers_amd import rocm, synth

DTYPES = {"f16": (np.float16, torch.float16, 2), "f32": (np.float32, torch.float32, 4)}
EPS = 1e-5


def listed():
    return [
        # a 6-layer TinyStories model's attention (n_embd 192, 256 tokens): three launches, all latency
        {"name": "train-f32-small", "work": "train", "dtype": "f32", "B": 4, "H": 6, "T": 256, "D": 32},
        # one layer of a GPT-2-small-sized f32 training step
        {"name": "train-f32", "work": "train", "dtype": "f32", "B": 8, "H": 12, "T": 1024, "D": 64},
        # the same layer in half precision: the benchmark's headline workload
        {"name": "train-f16", "work": "train", "dtype": "f16", "B": 8, "H": 12, "T": 1024, "D": 64},
        # long context, wide heads
        {"name": "train-f16-long", "work": "train", "dtype": "f16", "B": 1, "H": 16, "T": 8192, "D": 128},
        # a batch cut to its longest text: no length a multiple of a tile, few heads
        {"name": "train-f16-ragged", "work": "train", "dtype": "f16", "B": 3, "H": 5, "T": 777, "D": 128},
        # 32 prompts of 512 tokens entering their caches
        {"name": "prefill-f16", "work": "prefill", "dtype": "f16", "B": 32, "H": 12, "T": 512, "D": 64,
         "capacity": 768},
        # one conversation: 12 heads cannot fill the GPU without splitting the cache
        {"name": "decode-f16-single", "work": "decode", "dtype": "f16", "B": 1, "H": 12, "L": 1500, "D": 64},
        # a full serving batch on long caches: the benchmark's decode workload
        {"name": "decode-f16-batch", "work": "decode", "dtype": "f16", "B": 32, "H": 12, "L": 4096, "D": 64},
        # a token for 32 sequences of a GPT-2-small-sized model, 600 tokens in
        {"name": "generate-f16", "work": "generate", "dtype": "f16", "B": 32, "layers": 12, "H": 12, "D": 64,
         "vocab": 50257, "pos": 600, "capacity": 768},
        # the loss of a training step over GPT-2's vocabulary
        {"name": "loss-f32", "work": "loss", "dtype": "f32", "rows": 8192, "classes": 50257},
        # clip and AdamW over the same model's 162 M parameters in 74 tensors
        {"name": "optimizer-f32", "work": "optimizer", "dtype": "f32", "layers": 12, "width": 768, "vocab": 50257},
        # what else one block of that step and the embedding launch
        {"name": "block-ops-f32", "work": "block_ops", "dtype": "f32", "B": 8, "T": 1024, "H": 12, "D": 64,
         "vocab": 50257},
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    work = rng.choice(["train", "train", "train", "train", "train", "prefill", "decode", "decode", "generate", "loss",
                       "optimizer", "block_ops"])
    D = rng.choice([32, 64, 64, 128])
    if work == "train":
        dtype = rng.choice(["f16", "f16", "f32"])
        T = _log_int(rng, 64, 8192)
        BH_max = (6e11 if dtype == "f16" else 5e10) / (7.0 * T * T * D)
        H = min(_log_int(rng, 3, 25), max(1, int(BH_max)))
        B = _log_int(rng, 1, max(1, min(32, int(BH_max) // H, 32768 // T)))
        return {"work": work, "dtype": dtype, "B": B, "H": H, "T": T, "D": D}
    if work == "prefill":
        T = _log_int(rng, 16, 4096)
        B = _log_int(rng, 1, max(1, min(32, 16384 // T)))
        return {"work": work, "dtype": "f16", "B": B, "H": rng.randint(4, 16), "T": T, "D": D,
                "capacity": T + rng.randint(1, 512)}
    if work == "decode":
        H = rng.randint(4, 25)
        L = _log_int(rng, 16, 16384)
        B = _log_int(rng, 1, max(1, min(64, int(1e8 / (H * L * D)))))
        return {"work": work, "dtype": "f16", "B": B, "H": H, "L": L, "D": D}
    if work == "generate":
        H, D = rng.choice([(8, 32), (4, 64), (8, 64), (12, 64), (16, 64), (8, 128)])
        pos = _log_int(rng, 16, 1500)
        return {"work": work, "dtype": "f16", "B": rng.choice([1, 2, 3, 5, 8, 16, 24, 32]),
                "layers": rng.randint(2, 12), "H": H, "D": D, "vocab": _log_int(rng, 1024, 50257), "pos": pos,
                "capacity": pos + rng.randint(1, 256)}
    if work == "loss":
        return {"work": work, "dtype": rng.choice(["f32", "f32", "f16"]), "rows": _log_int(rng, 256, 8192),
                "classes": _log_int(rng, 257, 50257)}
    if work == "optimizer":
        return {"work": work, "dtype": "f32", "layers": rng.randint(2, 12),
                "width": 64 * rng.randint(2, 12), "vocab": _log_int(rng, 1024, 50257)}
    T = _log_int(rng, 128, 2048)
    return {"work": work, "dtype": rng.choice(["f32", "f32", "f16"]), "B": _log_int(rng, 1, 8192 // T), "T": T,
            "H": rng.randint(2, 12), "D": rng.choice([32, 64]), "vocab": _log_int(rng, 1024, 50257)}


class _Inputs:
    """Seeded tensors of the case's type on the GPU, and their addresses for the binding."""

    def __init__(self, case, seed):
        rocm.init(0)
        self.np_dtype, self.dtype, _ = DTYPES[case["dtype"]]
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return (torch.randn(*shape, device="cuda", generator=self.gen) * std).to(self.dtype)

    def uniform(self, *shape, bound):
        return ((torch.rand(*shape, device="cuda", generator=self.gen) * 2 - 1) * bound).to(self.dtype)

    def ids(self, n, below):
        return torch.randint(0, below, (n,), device="cuda", generator=self.gen)

    def empty(self, *shape, dtype=None):
        return torch.zeros(*shape, device="cuda", dtype=dtype or self.dtype)


def ptr(t, elements=0):
    return ctypes.c_void_p(t.data_ptr() + elements * t.element_size())


def _rotary(x, T, D):
    cos, sin = synth.rotary_tables(T, D, dtype=x.np_dtype)
    return (torch.from_numpy(np.ascontiguousarray(t)).cuda() for t in (cos, sin))


def _packed(w):
    """A weight [k, n] as the few-rows products stream it: [n/32][k][32]."""
    k, n = w.shape
    out = torch.empty(n // 32, k, 32, device="cuda", dtype=w.dtype)
    rocm.copy_view_raw(np.float16, ptr(w), (32, n, 1), ptr(out), (32 * k, 32, 1), (n // 32, k, 32))
    return out


def _parameter_sizes(case):
    C, V = case["width"], case["vocab"]
    return [V * C] + [C * C, C * C, C * C, C * C, 4 * C * C, 4 * C * C] * case["layers"] + [V * C]


def prepare(case, seed):
    x, s, work = _Inputs(case, seed), {"case": case}, case["work"]
    if work in ("train", "prefill", "decode", "generate"):
        s["scale"] = rocm.default_scale(case["D"])
    if work == "train":
        shape = (case["B"], case["H"], case["T"], case["D"])
        for name in ("q", "k", "v", "do"):
            s[name] = x.normal(*shape)
        for name in ("o", "dq", "dk", "dv"):
            s[name] = x.empty(*shape)
        s["lse"] = x.empty(*shape[:3], dtype=torch.float32)
    elif work == "prefill":
        B, H, T, D = (case[n] for n in "BHTD")
        s["qkv"] = x.normal(B, T, 3 * H * D)
        s["cos"], s["sin"] = _rotary(x, T, D)
        s["qh"] = x.empty(B, H, T, D)
        s["k_cache"], s["v_cache"] = (x.empty(B, H, case["capacity"], D) for _ in range(2))
        s["y"] = x.empty(B, T, H * D)
        s["lse"] = x.empty(B, H, T, dtype=torch.float32)
    elif work == "decode":
        B, H, L, D = (case[n] for n in "BHLD")
        s["q"], s["k_cache"], s["v_cache"] = x.normal(B, H, D), x.normal(B, H, L, D), x.normal(B, H, L, D)
        s["o"] = x.empty(B, H, D)
    elif work == "generate":
        B, H, D, V = case["B"], case["H"], case["D"], case["vocab"]
        C = H * D
        s["wte"], s["ids"], s["lm_head"] = x.normal(V, C), x.ids(B, V), x.uniform(C, V, bound=C ** -0.5)
        cos, sin = synth.rotary_tables(case["capacity"], D, dtype=np.float16)
        s["cos"], s["sin"] = (torch.from_numpy(np.ascontiguousarray(t.reshape(-1, D // 2)[case["pos"]])).cuda()
                              for t in (cos, sin))
        s["blocks"] = []
        for _ in range(case["layers"]):
            weights = {"qkv": x.uniform(C, 3 * C, bound=C ** -0.5), "out": x.uniform(C, C, bound=C ** -0.5),
                       "up": x.uniform(C, 4 * C, bound=C ** -0.5), "down": x.uniform(4 * C, C, bound=(4 * C) ** -0.5)}
            torch.cuda.synchronize()
            block = {n: _packed(w) for n, w in weights.items()}
            block["k"], block["v"] = (x.normal(B, H, case["capacity"], D) for _ in range(2))
            s["blocks"].append(block)
            rocm.sync()
        s["h"], s["qkv"], s["o"], s["u"] = x.empty(B, C), x.empty(B, 3 * C), x.empty(B, C), x.empty(B, 4 * C)
        s["n"], s["logits"] = x.empty(B, C), x.empty(B, V)
    elif work == "loss":
        n, c = case["rows"], case["classes"]
        s["logits"], s["targets"] = x.normal(n, c, std=0.6), x.ids(n, c)
        s["row_lse"], s["loss"] = x.empty(n, dtype=torch.float32), x.empty(1, dtype=torch.float32)
        s["dlogits"] = x.empty(n, c)
    elif work == "optimizer":
        sizes = _parameter_sizes(case)
        total = sum(sizes)
        s["w"], s["grad"] = x.normal(total, std=0.05), x.normal(total, std=1e-3)
        s["m"], s["v"] = x.empty(total), x.empty(total)
        starts = np.concatenate([[0], np.cumsum(sizes)[:-1]]).tolist()
        s["sizes"], s["step"] = sizes, 0
        s["pointers"] = {n: [ptr(s[n], at) for at in starts] for n in ("w", "grad", "m", "v")}
        s["total"] = rocm.DeviceBuffer((1,), np.float32)
    else:
        B, T, H, D, V = (case[n] for n in ("B", "T", "H", "D", "vocab"))
        N, C = B * T, H * D
        s["table"], s["ids"] = x.normal(V, C), x.ids(N, V)
        s["cos"], s["sin"] = _rotary(x, T, D)
        s["u"], s["da"], s["q"], s["dqh"] = x.normal(N, 4 * C), x.normal(N, 4 * C), x.normal(N, C), x.normal(N, C)
        s["dn"], s["residual"] = x.normal(N, C), x.normal(N, C)
        for name in ("x", "n", "qh", "dq", "dx"):
            s[name] = x.empty(N, C)
        s["a"], s["du"], s["dtable"] = x.empty(N, 4 * C), x.empty(N, 4 * C), x.empty(V, C)
    s["np"] = x.np_dtype
    torch.cuda.synchronize()
    return s


def _train(s, c):
    B, H, T, D, dt = c["B"], c["H"], c["T"], c["D"], s["np"]
    rocm.attn_fwd_raw(dt, ptr(s["q"]), ptr(s["k"]), ptr(s["v"]), ptr(s["o"]), ptr(s["lse"]), B, H, T, D, s["scale"])
    rocm.attn_bwd_raw(dt, ptr(s["q"]), ptr(s["k"]), ptr(s["v"]), ptr(s["o"]), ptr(s["lse"]), ptr(s["do"]), ptr(s["dq"]),
                      ptr(s["dk"]), ptr(s["dv"]), B, H, T, D, s["scale"])
    return [s[n] for n in ("o", "lse", "dq", "dk", "dv")]


def _prefill(s, c):
    B, H, T, D, cap, dt = c["B"], c["H"], c["T"], c["D"], c["capacity"], s["np"]
    C = H * D
    bthd, cache = (T * 3 * C, 3 * C, D, 1), (H * cap * D, cap * D, D, 1)
    rocm.rope_fwd_raw(dt, ptr(s["qkv"]), ptr(s["cos"]), ptr(s["sin"]), ptr(s["qh"]), B, T, H, D, x_strides=bthd)
    rocm.rope_fwd_raw(dt, ptr(s["qkv"], C), ptr(s["cos"]), ptr(s["sin"]), ptr(s["k_cache"]), B, T, H, D,
                      x_strides=bthd, y_strides=cache)
    rocm.copy_view_raw(dt, ptr(s["qkv"], 2 * C), (T * 3 * C, D, 3 * C, 1), ptr(s["v_cache"]), cache, (B, H, T, D))
    rocm.attn_fwd_raw(dt, ptr(s["qh"]), ptr(s["k_cache"]), ptr(s["v_cache"]), ptr(s["y"]), ptr(s["lse"]), B, H, T, D,
                      s["scale"], k_strides=cache, v_strides=cache, o_strides=(T * C, D, C, 1))
    return [s["y"], s["lse"], s["k_cache"], s["v_cache"]]


def _decode(s, c):
    rocm.attn_decode_raw(s["np"], ptr(s["q"]), ptr(s["k_cache"]), ptr(s["v_cache"]), ptr(s["o"]), c["B"], c["H"],
                         c["L"], c["D"], s["scale"])
    return s["o"]


def _generate(s, c):
    """The calls of a token step; the pick from the logits is the caller's."""
    B, H, D, V, pos, cap, dt = c["B"], c["H"], c["D"], c["vocab"], c["pos"], c["capacity"], s["np"]
    C = H * D
    h, qkv, o, u = ptr(s["h"]), ptr(s["qkv"]), ptr(s["o"]), ptr(s["u"])
    packed = rocm.LINEAR_W_PACKED

    def linear(prologue, x, k, w, y, n, add, following):
        if following is not None:
            rocm.decode_linear_hint_raw(ptr(following), following.shape[0] * 32, following.shape[1])
        rocm.decode_linear_raw(dt, prologue, EPS, x, k, ptr(w), packed, y, add, B, n, k)

    rocm.index_select_raw(dt, ptr(s["wte"]), ptr(s["ids"]), h, V, B, C)
    blocks = s["blocks"]
    for i, b in enumerate(blocks):
        linear("rms_norm", h, C, b["qkv"], qkv, 3 * C, False, b["out"])
        rocm.attn_decode_append_raw(dt, qkv, ptr(s["qkv"], C), ptr(s["qkv"], 2 * C), (3 * C, D), ptr(s["cos"]),
                                    ptr(s["sin"]), ptr(b["k"]), ptr(b["v"]), (H * cap * D, cap * D, D), o, pos, cap, B,
                                    H, D, s["scale"])
        linear("plain", o, C, b["out"], h, C, True, b["up"])
        linear("rms_norm", h, C, b["up"], u, 4 * C, False, b["down"])
        linear("relu_sq", u, 4 * C, b["down"], h, C, True, blocks[i + 1]["qkv"] if i + 1 < len(blocks) else None)
    rocm.rms_norm_fwd_raw(dt, h, ptr(s["n"]), B, C, EPS)
    rocm.matmul_raw(dt, ptr(s["n"]), (C, 1, 0), ptr(s["lm_head"]), (V, 1, 0), ptr(s["logits"]), 1, B, V, C)
    return [s["logits"], s["h"]] + [b[n][:, :, pos] for b in blocks for n in ("k", "v")]


def _loss(s, c):
    rocm.cross_entropy_fwd_grad_raw(s["np"], ptr(s["logits"]), ptr(s["targets"]), ptr(s["row_lse"]), ptr(s["loss"]),
                                    ptr(s["dlogits"]), c["rows"], c["classes"])
    return [s["loss"], s["row_lse"], s["dlogits"]]


def _optimizer(s, c):
    p = s["pointers"]
    rocm.sum_squares_multi_raw(s["np"], p["grad"], s["sizes"], s["total"].ptr)
    norm = float(s["total"].numpy()[0]) ** 0.5
    s["step"] += 1
    rocm.adamw_step_multi_raw(s["np"], p["w"], p["grad"], p["m"], p["v"], s["sizes"], 3e-4, 0.9, 0.95, 1e-8, 0.1,
                              s["step"], min(1.0, 1.0 / (norm + 1e-6)))
    return [s["w"], s["m"], s["v"], norm]


def _block_ops(s, c):
    B, T, H, D, V, dt = c["B"], c["T"], c["H"], c["D"], c["vocab"], s["np"]
    N, C = B * T, H * D
    rocm.index_select_raw(dt, ptr(s["table"]), ptr(s["ids"]), ptr(s["x"]), V, N, C)
    rocm.rms_norm_fwd_raw(dt, ptr(s["x"]), ptr(s["n"]), N, C, EPS)
    rocm.rope_fwd_raw(dt, ptr(s["q"]), ptr(s["cos"]), ptr(s["sin"]), ptr(s["qh"]), B, T, H, D)
    rocm.relu_sq_fwd_raw(dt, ptr(s["u"]), ptr(s["a"]), N * 4 * C)
    rocm.relu_sq_bwd_raw(dt, ptr(s["u"]), ptr(s["da"]), ptr(s["du"]), N * 4 * C)
    rocm.rope_bwd_raw(dt, ptr(s["dqh"]), ptr(s["cos"]), ptr(s["sin"]), ptr(s["dq"]), B, T, H, D)
    rocm.rms_norm_bwd_add_raw(dt, ptr(s["x"]), ptr(s["dn"]), ptr(s["residual"]), ptr(s["dx"]), N, C, EPS)
    rocm.fill_raw(dt, ptr(s["dtable"]), V * C, 0.0)
    rocm.index_add_raw(dt, ptr(s["dx"]), ptr(s["ids"]), ptr(s["dtable"]), V, N, C)
    return [s[n] for n in ("x", "n", "qh", "a", "du", "dq", "dx", "dtable")]


_RUN = {"train": _train, "prefill": _prefill, "decode": _decode, "generate": _generate, "loss": _loss,
        "optimizer": _optimizer, "block_ops": _block_ops}


def run(state):
    return _RUN[state["case"]["work"]](state, state["case"])


def work(case):
    c, el = case, DTYPES[case["dtype"]][2]
    kind = c["work"]
    if kind == "train":
        heads = c["B"] * c["H"]
        one = heads * c["T"] * c["D"]
        # q, k, v, dO in; O, dQ, dK, dV out; the causal half of 2 + 5 products of T x T x D
        return {"bytes": 8 * one * el + 4 * heads * c["T"], "flops": 7.0 * one * c["T"]}
    if kind == "prefill":
        heads = c["B"] * c["H"]
        one = heads * c["T"] * c["D"]
        return {"bytes": 6 * one * el + 4 * heads * c["T"], "flops": 2.0 * one * c["T"]}
    if kind == "decode":
        row = c["B"] * c["H"] * c["D"]
        return {"bytes": (2.0 * c["L"] + 2) * row * el, "flops": 4.0 * c["L"] * row}
    if kind == "generate":
        C, B = c["H"] * c["D"], c["B"]
        weights = 12.0 * C * C * c["layers"] + C * c["vocab"]
        cache = 2.0 * c["layers"] * B * C * (c["pos"] + 1)
        return {"bytes": (weights + cache + B * (C + c["vocab"])) * el, "flops": 2.0 * B * weights + 2.0 * cache}
    if kind == "loss":
        n = float(c["rows"]) * c["classes"]
        return {"bytes": 2 * n * el + 12 * c["rows"], "flops": 5 * n}
    if kind == "optimizer":
        n = float(sum(_parameter_sizes(c)))
        # the norm has to be known before the first update: gradients are read twice
        return {"bytes": 8 * n * el, "flops": 18 * n}
    N, C = float(c["B"] * c["T"]), float(c["H"] * c["D"])
    # in rows of C: lookup 1 + 1, norm 1 (x again: its mean is known at the row's end) + 1, rotary 2 + 2,
    # activation 8 + 12, norm backward 4, scatter 1 (the rest of it is the table), and the table written once
    return {"bytes": (33 * N * C + c["vocab"] * C) * el + 16 * N, "flops": 80 * N * C}


def tolerance(case):
    half = case["dtype"] == "f16"
    if case["work"] == "train" and half:
        return {"rel": 3e-3, "max": 0.06}  # probabilities and score gradients rounded to f16
    if case["work"] == "generate":
        return {"rel": 1e-2, "max": 0.1}  # a dozen blocks, each rounding its products to f16
    if half:
        return {"rel": 1.5e-3, "max": 0.03}
    return {"rel": 1e-5, "max": 1e-3}
