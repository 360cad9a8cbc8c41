"""Performance cases of the MI355X backend: what is timed, on which inputs,
what it must compute, and how exactly.

Every case is work that a program gives this backend through its public entry
points: the engine over compiled update plans (`DeviceUpdateEngine`) and the
device-pointer kernels of the C-ABI (`include/seeml_hip.h`). Sizes are those
of the repository's own workloads (C1 MLP, C3/C4/C5 decoders: widths 512, 2048
and 4096, MLPs of 1376 to 16384, ranks 8 to 64, head widths 64 and 128, up to
32000 classes), shortened where a case is one layer, and ragged sizes between
them.

  train      one optimizer step of a compiled LoRA update plan: staging, the
             train program, the loss. The engine's main call.
  eval       one batch through the eval program (validation): the loss and
             the class probabilities.
  linear     a dense layer's forward and backward: y = act(x W + b),
             dx = dy W^T, dW = x^T dy.
  linear_q8  a frozen int8 layer: y = act(s x Wq), dx = s dy Wq^T.
  adapter    a LoRA adapter on a layer's output, forward and backward.
  attention  RoPE and causal attention, forward and every backward primitive.
  loss       softmax cross-entropy over the head's logits, or KL distillation
             against a teacher's, forward and backward.
  norm_act   the bandwidth-bound part of a gated MLP block: norm, activation,
             gate product, forward and backward, and the residual sum.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.getcwd()
if os.path.join(_ROOT, "see-ml_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "see-ml_amd"))

from seeml_amd import DeviceUpdateEngine, PROGRAM_EVAL, configs, lib, planner  # noqa: E402

_DEV = "cuda:0"
_ACTS = {"none": 0, "relu": 1, "gelu": 2, "silu": 3}


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # The smallest update: a 256-512-256 MLP on 32 rows. Launch latency.
        dict(name="train_mlp_b32", kind="train", model="mlp", batch=32, d_in=256, hidden=512,
             d_out=256, rank=8),
        # One block of the d_model-2048 decoder (RMSNorm, SwiGLU, rank 16 on
        # q/k/v/o) with its embedding and head, 4 sequences of 512.
        dict(name="train_decoder_d2048", kind="train", model="decoder", norm="rms", mlp="swiglu",
             vocab=8192, dim=2048, layers=1, heads=16, ffn=5504, seq=512, seqs=4, rank=16,
             targets="wq wk wv wo"),
        # A LayerNorm/GELU decoder, rank 64 on every product, sequences whose
        # length is no power of two: 600 rows, a partial tile everywhere.
        dict(name="train_decoder_ln_r64", kind="train", model="decoder", norm="layer", mlp="gelu",
             vocab=2000, dim=1024, layers=1, heads=8, ffn=4096, seq=200, seqs=3, rank=64,
             targets=""),
        # Validation of the small decoder (width 512, 2 layers, MLP 1376).
        dict(name="eval_decoder_d512", kind="eval", model="decoder", norm="rms", mlp="swiglu",
             vocab=8192, dim=512, layers=2, heads=8, ffn=1376, seq=256, seqs=8, rank=8,
             targets="wq wv"),
        # The up projection of the d_model-2048 decoder at its own batch.
        dict(name="linear_8192x2048x5504", kind="linear", rows=8192, d_in=2048, d_out=5504,
             act="none"),
        # A layer whose sizes divide by nothing: 1000 rows, 770 -> 1531.
        dict(name="linear_1000x770x1531", kind="linear", rows=1000, d_in=770, d_out=1531,
             act="gelu"),
        # The same decoder's square projection with int8 frozen weights.
        dict(name="linear_q8_2048x2048x2048", kind="linear_q8", rows=2048, d_in=2048, d_out=2048,
             act="silu"),
        # A rank-16 adapter on a d_model-2048 projection.
        dict(name="adapter_8192x2048_r16", kind="adapter", rows=8192, d_in=2048, d_out=2048,
             rank=16),
        # Attention of the d_model-2048 decoder, 4 sequences.
        dict(name="attention_s1024_d128", kind="attention", seqs=4, seq=1024, heads=16, width=128),
        # A head width between the tuned ones and an odd length.
        dict(name="attention_s333_d80", kind="attention", seqs=3, seq=333, heads=8, width=80),
        # The loss over a 32000-class head.
        dict(name="loss_xent_2048x32000", kind="loss", loss="xent", rows=2048, classes=32000),
        # Norm, SwiGLU and residual of the d_model-2048 decoder's block.
        dict(name="norm_act_4096x2048x5504", kind="norm_act", rows=4096, dim=2048, ffn=5504,
             norm="rms", act="silu"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: a multiple of 64, of 8 or any whole number."""
    m = rng.choice([64, 64, 8, 1])
    return max(m, int(round(_log(rng, lo, hi) / m)) * m)


def draw(rng):
    kind = rng.choice(["train", "eval", "linear", "linear_q8", "adapter", "attention", "loss",
                       "norm_act"])
    if kind == "train" and rng.random() < 0.25:
        return dict(kind="train", model="mlp", batch=_log(rng, 16, 512), d_in=_width(rng, 64, 512),
                    hidden=_width(rng, 64, 1024), d_out=_width(rng, 16, 512),
                    rank=rng.choice([4, 8, 16]))
    if kind in ("train", "eval"):
        norm, mlp = rng.choice([("rms", "swiglu"), ("rms", "swiglu"), ("layer", "gelu")])
        dim, width = rng.choice([(256, 64), (512, 64), (512, 128), (768, 64), (1024, 128),
                                 (1024, 64), (1536, 128), (640, 80)])
        seq = _log(rng, 32, 512)
        return dict(kind=kind, model="decoder", norm=norm, mlp=mlp, vocab=_log(rng, 500, 8192),
                    dim=dim, layers=rng.choice([1, 2]), heads=dim // width,
                    ffn=int(dim * rng.choice([2, 2.6875, 4])), seq=seq,
                    seqs=rng.randint(1, max(1, 2048 // seq)), rank=rng.choice([8, 16, 64]),
                    targets=rng.choice(["wq wv", "wq wk wv wo"]))
    if kind in ("linear", "linear_q8"):
        return dict(kind=kind, rows=_log(rng, 64, 8192), d_in=_width(rng, 128, 4096),
                    d_out=_width(rng, 128, 5504),
                    act=rng.choice(["none", "relu", "gelu", "silu"]))
    if kind == "adapter":
        return dict(kind=kind, rows=_log(rng, 64, 8192), d_in=_width(rng, 256, 4096),
                    d_out=_width(rng, 256, 4096), rank=rng.choice([8, 16, 16, 32, 64]))
    if kind == "attention":
        seq = _log(rng, 32, 1024)
        return dict(kind=kind, seqs=rng.randint(1, max(1, min(8, 4096 // seq))), seq=seq,
                    heads=rng.choice([2, 4, 8, 16]), width=rng.choice([32, 64, 64, 80, 128, 128]))
    if kind == "loss":
        classes = rng.choice([256, 1000, 2048, 8192, 32000, _log(rng, 100, 32000)])
        return dict(kind=kind, loss=rng.choice(["xent", "xent", "kl"]),
                    rows=_log(rng, 32, max(64, min(8192, (1 << 26) // classes))), classes=classes)
    dim = _width(rng, 128, 4096)
    return dict(kind=kind, rows=_log(rng, 64, 4096), dim=dim,
                ffn=min(5504, int(dim * rng.choice([2, 2.6875, 4]))),
                norm=rng.choice(["rms", "layer"]), act=rng.choice(["silu", "gelu", "relu"]))


# ------------------------------------------------------------------- inputs

def _rng(case, seed):
    """A generator of the seed alone (the case sets only the shapes)."""
    g = torch.Generator(device=_DEV)
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=_DEV, dtype=torch.float32).mul_(std)


class _View:
    """A float32 range of device memory, for torch.as_tensor (no copy)."""

    def __init__(self, ptr, count, owner):
        self.__cuda_array_interface__ = dict(shape=(count,), typestr="<f4", data=(ptr, False),
                                             version=2, strides=None)
        self.owner = owner


_PLANS = {}  # the frozen model a user's program loads once: plan bytes by case


def _workload(case):
    if case["model"] == "mlp":
        model = configs.mlp_model(case["d_in"], case["hidden"], case["d_out"])
        cfg = planner.UpdateConfig(batch=case["batch"], loss="xent", lr=1e-3, weight_decay=0.01,
                                   lora=planner.LoraSpec(rank=case["rank"], alpha=16.0, seed=7))
        return model, cfg
    model = configs.decoder_model(case["vocab"], case["dim"], case["layers"], case["heads"],
                                  case["ffn"], case["seq"], norm=case["norm"], mlp=case["mlp"])
    cfg = planner.UpdateConfig(batch=case["seqs"] * case["seq"], loss="xent", lr=1e-3,
                               token_input=True,
                               lora=planner.LoraSpec(rank=case["rank"], alpha=16.0, seed=7,
                                                     targets=tuple(case["targets"].split())))
    return model, cfg


def _plan(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "kind")))
    if key not in _PLANS:
        while len(_PLANS) >= 2:
            _PLANS.pop(next(iter(_PLANS)))
        model, cfg = _workload(case)
        _PLANS[key] = (model, cfg, planner.compile_update(model, cfg))
    return _PLANS[key]


_STEP = 50  # a step in the middle of a run: the moments are warm


def _slots(plan):
    """The persistent segment's tensors: id -> (byte offset of p, of m, of v, count)."""
    out = {}
    for w in plan.train:
        if w["opcode"] == planner.OP["AdamWStep"]:
            p, _, m, v = w["inp"]
            out[p] = (p, m, v, w["out"][0])
    return {pid: out[ref] for pid, ref, _, _ in plan.params}


def _state_values(case, plan, seed):
    """Adapter and moment values in mid-training, by the seed: A as initialised
    (1/sqrt(fan_in)), B grown to 0.02, moments of 1e-4-sized gradients."""
    r = np.random.default_rng([int(seed), 11])
    image = np.zeros(plan.header["persistent_size"] // 4, np.float32)
    for pid, (p, m, v, n) in sorted(_slots(plan).items()):
        std = 1.0 / math.sqrt(n // case["rank"]) if pid.endswith("lora_A") else 0.02
        image[p // 4:p // 4 + n] = r.standard_normal(n, dtype=np.float32) * np.float32(std)
        image[m // 4:m // 4 + n] = r.standard_normal(n, dtype=np.float32) * np.float32(1e-4)
        image[v // 4:v // 4 + n] = (0.5 + r.random(n, dtype=np.float32)) * np.float32(1e-8)
    return image


def _batch(case, cfg, seed):
    r = np.random.default_rng([int(seed), 12])
    if case["model"] == "mlp":
        return (r.standard_normal((case["batch"], case["d_in"]), dtype=np.float32),
                r.integers(0, case["d_out"], case["batch"]).astype(np.int32))
    recs = configs.zipf_tokens(r, case["vocab"], case["seqs"] * (case["seq"] + 1))
    recs = recs.reshape(case["seqs"], case["seq"] + 1)
    return (np.ascontiguousarray(recs[:, :-1]).reshape(-1),
            np.ascontiguousarray(recs[:, 1:]).reshape(-1))


def _prepare_engine(case, seed):
    _, cfg, plan = _plan(case)
    e = DeviceUpdateEngine(plan.blob)
    e.write(0, _state_values(case, plan, seed))
    e.set_step(_STEP)
    x, y = _batch(case, cfg, seed)
    s = dict(kind=case["kind"], engine=e, x=torch.from_numpy(x).to(_DEV),
             y=torch.from_numpy(y).to(_DEV), views={})

    def view(off, n):
        return torch.as_tensor(_View(e.arena_ptr + off, n, e), device=_DEV)

    if case["kind"] == "train":
        e.build()
        for pid, (p, m, v, n) in sorted(_slots(plan).items()):
            s["views"][pid] = dict(p=view(p, n), m=view(m, n), v=view(v, n))
    else:
        e.build(PROGRAM_EVAL)
        xent = [w for w in plan.eval if w["opcode"] == planner.OP["SoftmaxXEntFwd"]][-1]
        s["views"]["probs"] = view(xent["inp"][3], cfg.batch * case["vocab"])
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "eval"):
        return _prepare_engine(case, seed)
    g = _rng(case, seed)
    s = dict(kind=kind, case=case)
    empty = lambda *shape: torch.empty(*shape, device=_DEV, dtype=torch.float32)  # noqa: E731
    if kind in ("linear", "linear_q8"):
        M, K, N = case["rows"], case["d_in"], case["d_out"]
        s.update(x=_randn(g, M, K), dy=_randn(g, M, N, std=1e-3), y=empty(M, N), dx=empty(M, K))
        if kind == "linear":
            s.update(w=_randn(g, K, N, std=1.0 / math.sqrt(K)), b=_randn(g, N, std=0.02),
                     dw=empty(K, N))
        else:
            s.update(w=torch.randint(-127, 128, (K, N), generator=g, device=_DEV, dtype=torch.int8),
                     scale=float(np.float32(1.0 / (74.0 * math.sqrt(K)))))
    elif kind == "adapter":
        T, K, N, r = case["rows"], case["d_in"], case["d_out"], case["rank"]
        s.update(x=_randn(g, T, K), a=_randn(g, K, r, std=1.0 / math.sqrt(K)),
                 b=_randn(g, r, N, std=0.02), y=_randn(g, T, N), dy=_randn(g, T, N, std=1e-3),
                 t=empty(T, r), u=empty(T, N), s=empty(T, N), out=empty(T, N), du=empty(T, N),
                 dt=empty(T, r), da=empty(K, r), db=empty(r, N), dx=empty(T, K))
    elif kind == "attention":
        B, S, H, d = case["seqs"], case["seq"], case["heads"], case["width"]
        T, D = B * S, H * d
        for k in ("q", "k", "v"):
            s[k] = _randn(g, T, D)
        s["do"] = _randn(g, T, D, std=1e-2)
        for k in ("qr", "kr", "o", "dv", "dqr", "dkr", "dq", "dk"):
            s[k] = empty(T, D)
        for k in ("p", "dp", "ds"):
            s[k] = empty(B * H * S, S)
    elif kind == "loss":
        N, C = case["rows"], case["classes"]
        s.update(logits=_randn(g, N, C, std=2.0), loss=empty(1), dl=empty(N, C),
                 seed=torch.ones(1, device=_DEV), probs=empty(N, C))
        if case["loss"] == "kl":
            s.update(teacher=_randn(g, N, C, std=2.0), probs_t=empty(N, C))
        else:
            s["labels"] = torch.randint(0, C, (N,), generator=g, device=_DEV, dtype=torch.int32)
    else:
        T, D, F = case["rows"], case["dim"], case["ffn"]
        s.update(x=_randn(g, T, D), gamma=1.0 + _randn(g, D, std=0.1), beta=_randn(g, D, std=0.1),
                 gate=_randn(g, T, F), up=_randn(g, T, F), dh=_randn(g, T, F, std=1e-2),
                 dn=_randn(g, T, D, std=1e-2), res=_randn(g, T, D, std=1e-2),
                 n=empty(T, D), mean=empty(T), rstd=empty(T), act=empty(T, F), h=empty(T, F),
                 dact=empty(T, F), dup=empty(T, F), dgate=empty(T, F), dx=empty(T, D),
                 dsum=empty(T, D))
    return s


# ---------------------------------------------------------------- one pass

def _call(name, *args):
    rc = getattr(lib(), "seeml_hip_" + name)(
        *[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args],
        torch.cuda.current_stream().cuda_stream)
    if rc != 0:
        raise RuntimeError("%s: %s" % (name, lib().seeml_hip_kernel_error().decode()))


def run(s):
    kind = s["kind"]
    if kind == "train":
        loss = s["engine"].train_step(s["x"], s["y"])
        return dict(loss=loss, state=s["views"])
    if kind == "eval":
        s["engine"].stage(s["x"], s["y"])
        s["engine"].run(PROGRAM_EVAL)
        return dict(loss=s["engine"].loss(), probs=s["views"]["probs"])
    c = s["case"]
    if kind == "linear":
        M, K, N = c["rows"], c["d_in"], c["d_out"]
        _call("gemm_nn", s["x"], s["w"], s["y"], M, N, K, s["b"], _ACTS[c["act"]])
        _call("gemm_nt", s["dy"], s["w"], s["dx"], M, K, N)
        _call("gemm_tn", s["x"], s["dy"], s["dw"], K, N, M)
        return dict(y=s["y"], dx=s["dx"], dw=s["dw"])
    if kind == "linear_q8":
        M, K, N = c["rows"], c["d_in"], c["d_out"]
        _call("gemm_nn_q8", s["x"], s["w"], s["y"], M, N, K, s["scale"], _ACTS[c["act"]])
        _call("gemm_nt_q8", s["dy"], s["w"], s["dx"], M, K, N, s["scale"])
        return dict(y=s["y"], dx=s["dx"])
    if kind == "adapter":
        T, K, N, r = c["rows"], c["d_in"], c["d_out"], c["rank"]
        alpha = 16.0 / r
        _call("gemm_nn", s["x"], s["a"], s["t"], T, r, K, None, 0)
        _call("gemm_nn", s["t"], s["b"], s["u"], T, N, r, None, 0)
        _call("scale", s["u"], s["s"], alpha, T * N)
        _call("add_ew", s["y"], s["s"], s["out"], T * N)
        _call("scale", s["dy"], s["du"], alpha, T * N)
        _call("gemm_nt", s["du"], s["b"], s["dt"], T, r, N)
        _call("gemm_tn", s["t"], s["du"], s["db"], r, N, T)
        _call("gemm_tn", s["x"], s["dt"], s["da"], K, r, T)
        _call("gemm_nt", s["dt"], s["a"], s["dx"], T, K, r)
        return {k: s[k] for k in ("t", "out", "dt", "da", "db", "dx")}
    if kind == "attention":
        g = (c["seqs"], c["seq"], c["heads"], c["width"])
        _call("rope_fwd", s["q"], s["qr"], *g, 10000.0)
        _call("rope_fwd", s["k"], s["kr"], *g, 10000.0)
        _call("attn_fwd", s["qr"], s["kr"], s["v"], s["o"], s["p"], *g)
        _call("attn_dp", s["do"], s["v"], s["dp"], *g)
        _call("attn_dv", s["p"], s["do"], s["dv"], *g)
        _call("softmax_rows_bwd", s["p"], s["dp"], s["ds"], g[0] * g[1] * g[2], g[1])
        _call("attn_dq", s["ds"], s["kr"], s["dqr"], *g)
        _call("attn_dk", s["ds"], s["qr"], s["dkr"], *g)
        _call("rope_bwd", s["dqr"], s["dq"], *g, 10000.0)
        _call("rope_bwd", s["dkr"], s["dk"], *g, 10000.0)
        return {k: s[k] for k in ("o", "p", "ds", "dq", "dk", "dv")}
    if kind == "loss":
        N, C = c["rows"], c["classes"]
        if c["loss"] == "kl":
            _call("kl_distill_fwd", s["logits"], s["teacher"], s["loss"], s["probs"], s["probs_t"],
                  N, C, 2.0)
            _call("kl_distill_bwd", s["probs"], s["probs_t"], s["seed"], s["dl"], N, C, 2.0)
            return {k: s[k] for k in ("loss", "probs", "probs_t", "dl")}
        _call("softmax_xent_fwd", s["logits"], s["labels"], s["loss"], s["probs"], N, C)
        _call("softmax_xent_bwd", s["probs"], s["labels"], s["seed"], s["dl"], N, C)
        return {k: s[k] for k in ("loss", "probs", "dl")}
    T, D, F = c["rows"], c["dim"], c["ffn"]
    act = c["act"]
    if c["norm"] == "rms":
        _call("rms_norm_fwd", s["x"], s["gamma"], s["n"], s["rstd"], T, D)
    else:
        _call("layer_norm_fwd", s["x"], s["gamma"], s["beta"], s["n"], s["mean"], s["rstd"], T, D)
    _call(act + "_fwd", s["gate"], s["act"], T * F)
    _call("mul_ew", s["act"], s["up"], s["h"], T * F)
    _call("mul_ew", s["dh"], s["act"], s["dup"], T * F)
    _call("mul_ew", s["dh"], s["up"], s["dact"], T * F)
    _call(act + "_bwd", s["dact"], s["gate"], s["dgate"], T * F)
    if c["norm"] == "rms":
        _call("rms_norm_bwd", s["dn"], s["x"], s["gamma"], s["rstd"], s["dx"], T, D)
    else:
        _call("layer_norm_bwd", s["dn"], s["x"], s["gamma"], s["mean"], s["rstd"], s["dx"], T, D)
    _call("add_ew", s["res"], s["dx"], s["dsum"], T * D)
    return {k: s[k] for k in ("n", "h", "dup", "dgate", "dsum")}


# ------------------------------------------------- the work of one pass

def work(case):
    """What a pass cannot do without: each input read once, each output
    written once; multiply-adds as two operations, causal halves counted once."""
    kind = case["kind"]
    if kind in ("linear", "linear_q8"):
        M, K, N = case["rows"], case["d_in"], case["d_out"]
        if kind == "linear":  # x, w, b, dy in; y, dx, dw out
            return dict(flops=6.0 * M * K * N, bytes=4.0 * (2 * M * K + 2 * M * N + 2 * K * N + N))
        return dict(flops=4.0 * M * K * N, bytes=4.0 * (2 * M * K + 2 * M * N) + K * N)
    if kind == "adapter":
        T, K, N, r = case["rows"], case["d_in"], case["d_out"], case["rank"]
        # x, y, dy, a, b in; out, dx, t, dt, da, db out
        return dict(flops=6.0 * T * r * (K + N), bytes=4.0 * (2 * T * K + 3 * T * N
                                                              + 2 * r * (K + N) + 2 * T * r))
    if kind == "attention":
        B, S, H, d = case["seqs"], case["seq"], case["heads"], case["width"]
        half = B * H * S * (S + 1) / 2.0
        # q, k, v, do in; o, dq, dk, dv and the P, dS rows out
        return dict(flops=6 * 2.0 * half * d, bytes=4.0 * (8 * B * S * H * d + 2 * B * H * S * S))
    if kind == "loss":
        n = case["rows"] * case["classes"]
        return dict(flops=0.0, bytes=4.0 * n * (5 if case["loss"] == "kl" else 3))
    if kind == "norm_act":
        # x, dn, res in, n, dsum out; gate, up, dh in, h, dup, dgate out
        return dict(flops=0.0, bytes=4.0 * case["rows"] * (5 * case["dim"] + 6 * case["ffn"]))
    train = case["kind"] == "train"
    if case["model"] == "mlp":
        T, r = case["batch"], case["rank"]
        i, h, o = case["d_in"], case["hidden"], case["d_out"]
        base = 2.0 * T * (i * h + h * o) + (2.0 * T * h * o if train else 0.0)
        lora = 2.0 * T * r * (i + 2 * h + o) * (3 if train else 1)
        params = r * (i + 2 * h + o)
        weights = i * h + h * o + h + o
        return dict(flops=base + lora, bytes=4.0 * (weights + T * i + T + (6 if train else 1) * params))
    T, D, F, V, L = (case["seqs"] * case["seq"], case["dim"], case["ffn"], case["vocab"],
                     case["layers"])
    S, r = case["seq"], case["rank"]
    ups = 2 if case["mlp"] == "swiglu" else 1
    shapes = {"wq": (D, D), "wk": (D, D), "wv": (D, D), "wo": (D, D), "wu": (D, F), "wd": (F, D)}
    if ups == 2:
        shapes["wg"] = (D, F)
    targets = case["targets"].split()
    layer = sum(a * b for a, b in shapes.values())
    adapted = [s for n, s in shapes.items() if not targets or n in targets] * L
    if not targets:
        adapted.append((D, V))
    params = sum(r * (a + b) for a, b in adapted)
    weights = L * layer + D * V
    attn = L * 2 * 2.0 * case["seqs"] * S * (S + 1) / 2.0 * D
    flops = 2.0 * T * weights + attn + 2.0 * T * params
    if train:  # input gradients (not below the first layer's inputs), dA, dB
        flops += 2.0 * T * (weights - 3 * D * D) + 2.0 * attn + 4.0 * T * params
    nbytes = 4.0 * (weights + 2 * T + T * D + (6 if train else 1) * params)
    if not train:
        nbytes += 4.0 * T * V
    return dict(flops=flops, bytes=nbytes)


# ------------------------------------------------------------- tolerances

def tolerance(case):
    """Everything is computed in 32 bits. `rel` is about four times what the
    outputs were seen to differ by from the same sums in 64 bits."""
    return dict(rel=_TOL[case["kind"]])


_TOL = {
    "train": 2e-5,
    "eval": 4e-6,
    "linear": 8e-6,
    "linear_q8": 8e-6,
    "adapter": 4e-6,
    "attention": 4e-6,
    "loss": 2e-6,
    "norm_act": 1e-6,
}


# -------------------------------------------------- the same in 64 bits

def _act64(name, x):
    if name == "relu":
        return torch.relu(x)
    if name == "gelu":
        return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x * x * x)))
    if name == "silu":
        return x * torch.sigmoid(x)
    return x


def _norm64(kind, x, gamma, beta):
    if kind == "rms":
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * gamma
    mu = x.mean(-1, keepdim=True)
    xc = x - mu
    return xc * torch.rsqrt((xc * xc).mean(-1, keepdim=True) + 1e-5) * gamma + beta


def _rope64(x, B, S, H, d):
    """Interleaved pairs (2c, 2c+1) rotated by s * f_c. The plan format defines
    f_c by repeated float32 products (f_0 = 1, f_c+1 = f_c * 10000^(-2/d)) and
    the angle as the float32 product s * f_c; from there on, 64 bits."""
    f = np.ones(d // 2, np.float32)
    for c in range(1, d // 2):
        f[c] = f[c - 1] * np.float32(10000.0 ** float(np.float32(-2.0) / np.float32(d)))
    ang = np.arange(S, dtype=np.float32)[:, None] * f[None, :]
    ang = torch.from_numpy(ang).to(x.device).double()
    cs, sn = ang.cos()[None, :, None, :], ang.sin()[None, :, None, :]
    v = x.reshape(B, S, H, d // 2, 2)
    a, b = v[..., 0], v[..., 1]
    return torch.stack((a * cs - b * sn, a * sn + b * cs), -1).reshape(B * S, H * d)


def _heads64(x, B, S, H, d):
    return x.reshape(B, S, H, d).permute(0, 2, 1, 3).contiguous()


def _rows64(x):
    B, H, S, d = x.shape
    return x.permute(0, 2, 1, 3).reshape(B * S, H * d)


def _causal64(S):
    return torch.ones(S, S, device=_DEV, dtype=torch.bool).triu(1)


def _probs64(q, k, d):
    s = torch.matmul(q, k.transpose(-1, -2)) / math.sqrt(d)
    return torch.softmax(s.masked_fill(_causal64(s.shape[-1]), -math.inf), -1)


def _forward64(case, w, lora, x):
    """The model of a train / eval case over weights `w` and adapters `lora`."""
    scale = 16.0 / case["rank"]

    def mm(a, name):
        y = a @ w[name]
        if name + ".lora_A" in lora:
            y = y + scale * ((a @ lora[name + ".lora_A"]) @ lora[name + ".lora_B"])
        return y

    if case["model"] == "mlp":
        return mm(torch.relu(mm(x, "w1") + w["b1"]), "w2") + w["b2"]
    B, S, H = case["seqs"], case["seq"], case["heads"]
    d = case["dim"] // H
    e = w["emb"][x.long()]
    for i in range(case["layers"]):
        p = "l%d." % i
        n = _norm64(case["norm"], e, w[p + "g1"], w.get(p + "g1b"))
        q = _heads64(_rope64(mm(n, p + "wq"), B, S, H, d), B, S, H, d)
        k = _heads64(_rope64(mm(n, p + "wk"), B, S, H, d), B, S, H, d)
        v = _heads64(mm(n, p + "wv"), B, S, H, d)
        e = e + mm(_rows64(torch.matmul(_probs64(q, k, d), v)), p + "wo")
        n = _norm64(case["norm"], e, w[p + "g2"], w.get(p + "g2b"))
        if case["mlp"] == "swiglu":
            e = e + mm(_act64("silu", mm(n, p + "wg")) * mm(n, p + "wu"), p + "wd")
        else:
            e = e + mm(_act64("gelu", mm(n, p + "wu") + w[p + "bu"]), p + "wd") + w[p + "bd"]
    return mm(_norm64(case["norm"], e, w["gf"], w.get("gfb")), "wh")


def _exact_engine(case, seed):
    model, cfg, plan = _plan(case)
    h = plan.header
    blob = np.frombuffer(plan.blob, np.uint8)
    f64 = lambda a: torch.from_numpy(np.array(a, np.float32)).to(_DEV).double()  # noqa: E731
    w = {}
    for t in model.tensors:
        if t.const:
            n = int(np.prod(t.dims))
            off = h["rodata_offset"] + plan.weights[t.name]
            w[t.name] = f64(blob[off:off + 4 * n].view(np.float32)).reshape(t.dims)
    image = _state_values(case, plan, seed)
    slots = _slots(plan)
    lora = {}
    for pid, (p, _, _, n) in slots.items():
        lora[pid] = f64(image[p // 4:p // 4 + n])
        lora[pid] = lora[pid].reshape((n // case["rank"], case["rank"]) if pid.endswith("lora_A")
                                      else (case["rank"], n // case["rank"]))
    x, y = _batch(case, cfg, seed)
    x = torch.from_numpy(x).to(_DEV)
    x = x.double() if case["model"] == "mlp" else x
    labels = torch.from_numpy(y).to(_DEV).long()
    train = case["kind"] == "train"
    if train:
        for t in lora.values():
            t.requires_grad_(True)
    logits = _forward64(case, w, lora, x)
    loss = torch.nn.functional.cross_entropy(logits, labels)
    if not train:
        return dict(loss=float(loss), probs=torch.softmax(logits, -1).reshape(-1))
    loss.backward()
    state = {}
    b1, b2, lr, wd, eps = (float(np.float32(v)) for v in (cfg.beta1, cfg.beta2, cfg.lr,
                                                          cfg.weight_decay, cfg.eps))
    for pid, (p, m, v, n) in slots.items():
        g = lora[pid].grad.reshape(-1)
        m1 = b1 * f64(image[m // 4:m // 4 + n]) + (1.0 - b1) * g
        v1 = b2 * f64(image[v // 4:v // 4 + n]) + (1.0 - b2) * g * g
        p0 = lora[pid].detach().reshape(-1)
        mh, vh = m1 / (1.0 - b1 ** (_STEP + 1)), v1 / (1.0 - b2 ** (_STEP + 1))
        state[pid] = dict(p=p0 - lr * (mh / (vh.sqrt() + eps) + wd * p0), m=m1, v=v1)
    return dict(loss=float(loss.detach()), state=state)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("train", "eval"):
        return _exact_engine(case, seed)
    s = prepare(case, seed)
    D = {k: v.double() for k, v in s.items()
         if isinstance(v, torch.Tensor) and v.dtype in (torch.float32, torch.int8)}
    c = case
    if kind == "linear":
        return dict(y=_act64(c["act"], D["x"] @ D["w"] + D["b"]), dx=D["dy"] @ D["w"].t(),
                    dw=D["x"].t() @ D["dy"])
    if kind == "linear_q8":
        return dict(y=_act64(c["act"], s["scale"] * (D["x"] @ D["w"])),
                    dx=s["scale"] * (D["dy"] @ D["w"].t()))
    if kind == "adapter":
        alpha = 16.0 / c["rank"]
        t = D["x"] @ D["a"]
        du = alpha * D["dy"]
        dt = du @ D["b"].t()
        return dict(t=t, out=D["y"] + alpha * (t @ D["b"]), dt=dt, da=D["x"].t() @ dt,
                    db=t.t() @ du, dx=dt @ D["a"].t())
    if kind == "attention":
        g = (c["seqs"], c["seq"], c["heads"], c["width"])
        d = g[3]
        q, k = (_heads64(_rope64(D[n], *g), *g) for n in ("q", "k"))
        v, do = _heads64(D["v"], *g), _heads64(D["do"], *g)
        p = _probs64(q, k, d)
        dp = torch.matmul(do, v.transpose(-1, -2)).masked_fill(_causal64(g[1]), 0.0)
        ds = p * (dp - (p * dp).sum(-1, keepdim=True))
        dq = _rows64(torch.matmul(ds, k) / math.sqrt(d))
        dk = _rows64(torch.matmul(ds.transpose(-1, -2), q) / math.sqrt(d))
        flip = torch.tensor([1.0, -1.0], device=_DEV, dtype=torch.float64).repeat(g[2] * d // 2)
        back = lambda z: _rope64(z * flip, *g) * flip  # the rotation by -t  # noqa: E731
        return dict(o=_rows64(torch.matmul(p, v)), p=p.reshape(-1, g[1]), ds=ds.reshape(-1, g[1]),
                    dq=back(dq), dk=back(dk),
                    dv=_rows64(torch.matmul(p.transpose(-1, -2), do)))
    if kind == "loss":
        N = c["rows"]
        if c["loss"] == "kl":
            T = 2.0
            ps, pt = torch.softmax(D["logits"] / T, -1), torch.softmax(D["teacher"] / T, -1)
            loss = (pt * (pt.log() - ps.log())).sum() / N
            return dict(loss=loss.reshape(1), probs=ps, probs_t=pt, dl=(ps - pt) / (N * T))
        p = torch.softmax(D["logits"], -1)
        lab = s["labels"].long()
        dl = p / N
        dl[torch.arange(N, device=_DEV), lab] -= 1.0 / N
        loss = torch.nn.functional.cross_entropy(D["logits"], lab)
        return dict(loss=loss.reshape(1), probs=p, dl=dl)
    x = D["x"].clone().requires_grad_(True)
    gate = D["gate"].clone().requires_grad_(True)
    n = _norm64(c["norm"], x, D["gamma"], D["beta"])
    a = _act64(c["act"], gate)
    n.backward(D["dn"])
    a.backward(D["dh"] * D["up"])
    return dict(n=n.detach(), h=(a * D["up"]).detach(), dup=(D["dh"] * a).detach(),
                dgate=gate.grad, dsum=D["res"] + x.grad)
