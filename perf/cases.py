"""The work that users of this framework have it do, as cases that can be timed and compared.

Every case goes through a public entry point: the engine (EvalLogits, EvalLoss, Step / TrainBatch), the KV-cache
decoder (Prefill, Generate, Step), the mixture-of-experts layer, the classifier-head loss on device buffers, and the
per-object layer seam.  `exact` gives the same results in 64-bit plain torch, without this framework's code.

Weights are N(0, 0.02) (the initialisation that every configuration here uses) with norm gains around 1; the decoder's
embedding is wider, see `_serve_params`.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "autoresearch-go-ane_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ane  # noqa: E402
from ane import _lib, objects  # noqa: E402
from ane.moe import MoeConfig, MoeLayer, moe_param_count  # noqa: E402

EPS = 1e-5

# The optimizer settings in use here: the llama2 training benchmark's, and the reference experiment's for nanochat.
TRAIN_OPTIONS = {
    "llama2": dict(LR=3e-4, AdamBeta1=0.9, AdamBeta2=0.95, AdamEps=1e-8, WeightDecay=0.1, Seed=42),
    "nanochat": dict(LR=3e-4, Seed=42, AdamBeta1=0.8, AdamBeta2=0.95, AdamEps=1e-10, WeightDecay=0.0, GradClip=1.0,
                     LossScale=256.0, EmbedLRMult=1.0, ScalarLRMult=1.0, LambdaLRMult=0.01, LambdaBeta1=0.96,
                     LambdaBeta2=0.95),
}


def _model(arch="llama2", dim=768, hidden=2048, heads=12, layers=12, vocab=32000, seq=256, **kw):
    return dict(arch=arch, dim=dim, hidden=hidden, heads=heads, layers=layers, vocab=vocab, seq=seq, **kw)


def listed():
    return [
        # One window of the small model of the tests: what the shortest call costs (latency, launches).
        dict(name="logits_tiny", kind="logits", **_model(dim=128, hidden=256, heads=2, layers=2, vocab=512, seq=64)),
        # The reference's BenchmarkEvalLogits: one 256-token window of its own model, logits copied out.
        dict(name="logits_window", kind="logits", **_model("nanochat")),
        # The headline: forward and loss of 32 windows of stories110M.
        dict(name="loss_b32", kind="loss", batch=32, **_model()),
        # The harness's validation loss of the reference's model: 39 windows (10,000 tokens).
        dict(name="loss_b39_nanochat", kind="loss", batch=39, **_model("nanochat")),
        # Scoring a few longer texts: a ragged number of tokens, sequences beyond the training length.
        dict(name="loss_b5_seq448", kind="loss", batch=5, **_model(seq=448)),
        # Training at batch 16: eight optimizer steps, then the weights read back as a checkpoint does.
        dict(name="train_b16", kind="train", batch=16, steps=8, accum=16, **_model()),
        # The reference's BenchmarkStep: one window a step, an update every eight, and the weights read back.
        dict(name="step_b1_nanochat", kind="train", batch=1, steps=32, accum=8, **_model("nanochat")),
        # Serving a full batch: prefill of 64 prompts of 1024 tokens, greedy generation, then logits for sampling.
        dict(name="serve_b64", kind="serve", batch=64, prefix=1024, steps=64, kv_heads=4, **_model(seq=1024)),
        # Serving a few users: three short prompts, where every step is latency.
        dict(name="serve_b3", kind="serve", batch=3, prefix=192, steps=64, kv_heads=4, **_model(seq=1024)),
        # The mixture-of-experts layer over a batch of activations from the host.
        dict(name="moe_8192", kind="moe", tokens=8192, dim=768, hidden=2048, experts=8),
        # The classifier head's loss on the caller's own device buffers, as a part of another program's forward.
        dict(name="head_8192", kind="head", tokens=8192, seq=256, dim=768, vocab=32000, softcap=0, noalloc=1),
        # One layer through the per-object seam, as the reference's engine drives it in training: forward with the
        # activations kept, attention backward, FFN backward, all on host slices.
        dict(name="layer_seam", kind="layer", dim=768, hidden=2048, heads=12, seq=256),
    ]


def _log(rng, lo, hi, step=1):
    """A size between lo and hi, spread over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def _drawn_model(rng, arch=None, top_seq=512):
    heads = rng.choice([2, 3, 4, 6, 8, 10, 12])
    return _model(arch or rng.choice(["llama2", "llama2", "nanochat"]), dim=64 * heads,
                  hidden=64 * rng.randint(2 * heads, 32) if heads < 16 else 2048, heads=heads,
                  layers=rng.randint(2, 12), vocab=_log(rng, 512, 32000, 64), seq=64 * rng.randint(1, top_seq // 64))


def draw(rng):
    kind = rng.choice(["logits", "loss", "loss", "train", "train", "serve", "serve", "moe", "head", "layer"])
    if kind == "logits":
        return dict(kind=kind, **_drawn_model(rng))
    if kind == "loss":
        # half of them on the full-size model, over the batch; seq * batch stays within the listed ones
        m = _model(rng.choice(["llama2", "nanochat"]), seq=64 * rng.randint(1, 8)) if rng.random() < 0.5 else _drawn_model(rng)
        return dict(kind=kind, batch=_log(rng, 1, min(40, 9984 // m["seq"])), **m)
    if kind == "train":
        m = _model(rng.choice(["llama2", "nanochat"]), seq=64 * rng.randint(1, 4)) if rng.random() < 0.5 else _drawn_model(rng, top_seq=256)
        batch = _log(rng, 1, 16)
        calls = rng.choice([1, 1, 2, 4])  # calls that one update gathers
        return dict(kind=kind, batch=batch, steps=8, accum=batch * calls, **m)
    if kind == "serve":
        heads, kv = rng.choice([(12, 4), (12, 4), (12, 12), (8, 4), (8, 2), (4, 2), (6, 3)])
        m = _model(dim=64 * heads, heads=heads, hidden=2048 if heads == 12 else 64 * rng.randint(heads, 32),
                   layers=rng.randint(2, 12), vocab=_log(rng, 1024, 32000, 64), seq=1024)
        return dict(kind=kind, batch=_log(rng, 1, 64), prefix=64 * rng.randint(1, 16), steps=rng.randint(8, 64),
                    kv_heads=kv, **m)
    if kind == "moe":
        return dict(kind=kind, tokens=_log(rng, 1, 8192), dim=64 * rng.choice([4, 6, 8, 12]),
                    hidden=64 * rng.randint(8, 32), experts=rng.choice([4, 8, 8, 16]))
    if kind == "head":
        seq = 64 * rng.randint(1, 8)
        return dict(kind=kind, tokens=seq * max(1, _log(rng, 64, 8192) // seq), seq=seq, dim=64 * rng.randint(4, 12),
                    vocab=_log(rng, 1024, 32000, 256), softcap=rng.choice([0, 1]), noalloc=rng.choice([0, 1]))
    heads = rng.choice([4, 6, 8, 12])
    return dict(kind=kind, dim=64 * heads, hidden=64 * rng.randint(2 * heads, 32), heads=heads, seq=64 * rng.randint(1, 4))


# ---- inputs ------------------------------------------------------------------------------------------------------------


def _gen(seed, stream):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 16 + stream)


def _cfg(case):
    return ane.Config(**{k: case[k] for k in ("arch", "dim", "hidden", "heads", "layers", "vocab", "seq")},
                      kv_heads=case.get("kv_heads", 0))


def _params(cfg, seed):
    """N(0, 0.02) matrices, norm gains 1 + N(0, 0.1), nanochat's scalars as they are initialised; on the host."""
    flat = torch.randn(ane.param_count(cfg), generator=_gen(seed, 0), device="cuda").mul_(0.02)
    start = {"resid_lambdas": 1.0, "x0_lambdas": 0.1, "smear_lambda": 0.01, "backout_lambda": 0.01}
    for name, off, shape in ane.param_layout(cfg):
        part = flat[off:off + math.prod(shape)]
        if name.split(".")[-1] in ("g_att", "g_ffn", "g_final"):
            part.mul_(5.0).add_(1.0)
        elif name in start:
            part.fill_(start[name])
    return flat.cpu().numpy()


def _serve_params(cfg, seed):
    """As `_params`, with an embedding of N(0, 0.2): beside it each position's own token stands out of the random
    layers, so the greedy choice has the clear margin that trained weights give it.  With 0.02 throughout, about one
    token in a hundred lies within a rounding of the runner-up, and what follows it is another text."""
    flat = _params(cfg, seed)
    for name, off, shape in ane.param_layout(cfg):
        if name == "embed":
            flat[off:off + math.prod(shape)] *= np.float32(10.0)
    return flat


def _tokens(case, seed, rows, cols):
    return torch.randint(0, case["vocab"], (rows, cols), generator=_gen(seed, 1), device="cuda").cpu().numpy().astype(np.uint16)


def _normal(seed, stream, *shape, std=1.0):
    return torch.randn(shape, generator=_gen(seed, stream), device="cuda").mul_(std)


def _layer_weights(case, seed):
    d, h = case["dim"], case["hidden"]
    shapes = dict(wq=(d, d), wk=(d, d), wv=(d, d), wo=(d, d), w1=(h, d), w2=(d, h))
    return {n: _normal(seed, i, *s, std=s[1] ** -0.5) for i, (n, s) in enumerate(shapes.items())}


def _layer_inputs(case, seed):
    """Channel-first [C, seq] activations and gradients of one layer."""
    d, h, s = case["dim"], case["hidden"], case["seq"]
    return {n: _normal(seed, 6 + i, c, s) for i, (n, c) in enumerate(
        [("x", d), ("q", d), ("k", d), ("v", d), ("dx2", d), ("dffn", d), ("h1", h)])}


def _moe_inputs(case, seed):
    cfg = MoeConfig(dim=case["dim"], hidden=case["hidden"], experts=case["experts"])
    return cfg, _normal(seed, 0, moe_param_count(cfg), std=0.02), _normal(seed, 1, case["tokens"], case["dim"])


def _head_inputs(case, seed):
    xn = _normal(seed, 0, case["tokens"], case["dim"]).half()
    embed = _normal(seed, 1, case["vocab"], case["dim"], std=0.3 if case["softcap"] else 0.05).half()
    return xn, embed, torch.from_numpy(_tokens(case, seed, 1, case["tokens"])[0].view(np.int16)).cuda()


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("logits", "loss", "train"):
        cfg, params = _cfg(case), _params(_cfg(case), seed)
        if kind == "train":
            s["eng"] = ane.Open(ane.Options(Config=cfg, Params=params, MaxBatch=case["batch"], AccumSteps=case["accum"],
                                            Tokens=_tokens(case, seed, 1, 64 * (cfg.seq + 1))[0],
                                            **TRAIN_OPTIONS[cfg.arch]))
        else:
            rows = case.get("batch", 1)
            ids = _tokens(case, seed, rows, cfg.seq + 1)
            s["tok"], s["tgt"] = np.ascontiguousarray(ids[:, :-1]), np.ascontiguousarray(ids[:, 1:])
            s["eng"] = ane.Open(ane.Options(Config=cfg, Params=params, MaxBatch=rows))
    elif kind == "serve":
        cfg = _cfg(case)
        s["dec"] = ane.Decoder(cfg, _serve_params(cfg, seed), max_batch=case["batch"],
                               max_ctx=case["prefix"] + case["steps"] + 1)
        s["prefix"] = _tokens(case, seed, case["batch"], case["prefix"])
    elif kind == "moe":
        cfg, params, x = _moe_inputs(case, seed)
        s["layer"], s["x"] = MoeLayer(cfg, params.cpu().numpy(), max_tokens=case["tokens"]), x.cpu().numpy()
    elif kind == "head":
        s["xn"], s["embed"], s["tgt"] = _head_inputs(case, seed)
        s["loss"] = torch.zeros(case["tokens"] // case["seq"], device="cuda")
        s["lse"] = torch.zeros(case["tokens"], device="cuda")
    else:
        w = {n: t.cpu().numpy() for n, t in _layer_weights(case, seed).items()}
        s["fwd"] = objects.compile_stories_layer_forward(w, case["seq"], heads=case["heads"])
        s["bwd"] = objects.compile_stories_layer_backward(w, case["seq"], heads=case["heads"])
        s["in"] = {n: t.cpu().numpy().ravel() for n, t in _layer_inputs(case, seed).items()}
        s["cache"] = objects.LayerCache(case["dim"], case["hidden"], case["seq"])
        n, nh = case["dim"] * case["seq"], case["hidden"] * case["seq"]
        s["out"] = {k: np.zeros(nh if k == "dh1" else n, np.float32) for k in ("out", "dxa", "dq", "dk", "dv", "dxf", "dh1")}
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "logits":
        return s["eng"].EvalLogits(s["tok"][0])
    if kind == "loss":
        mean, per = s["eng"].EvalLoss(s["tok"], s["tgt"])
        return {"mean": mean, "per_sequence": per}
    if kind == "train":
        eng, n = s["eng"], case["batch"]
        losses = [(eng.Step() if n == 1 else eng.TrainBatch(n)).loss for _ in range(case["steps"])]
        return {"losses": np.array(losses, np.float32), "params": eng.Params()}
    if kind == "serve":
        dec = s["dec"]
        first, _ = dec.Prefill(s["prefix"])
        more = dec.Generate(case["steps"])
        _, logits = dec.Step(want_logits=True)
        return {"first": first.astype(np.int32), "tokens": more.astype(np.int32), "logits": logits}
    if kind == "moe":
        out, experts, weights = s["layer"].Forward(s["x"])
        return {"out": out, "experts": experts, "weights": weights}
    if kind == "head":
        lib = _lib.load()
        call = lib.ane_head_loss_noalloc if case["noalloc"] else lib.ane_head_loss
        p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
        rc = call(p(s["xn"]), p(s["embed"]), p(s["tgt"]), case["tokens"], case["dim"], case["vocab"], case["seq"],
                  case["softcap"], p(s["loss"]), p(s["lse"]), C.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc != _lib.ANE_OK:
            raise RuntimeError(lib.ane_op_last_error().decode())
        return {"loss": s["loss"], "lse": s["lse"]}
    i, o, cache = s["in"], s["out"], s["cache"]
    s["fwd"].run_with_taps(o["out"], i["x"], cache)
    s["bwd"].run_attention(o["dxa"], o["dq"], o["dk"], o["dv"], i["q"], i["k"], i["v"], i["dx2"])
    s["bwd"].run_ffn(o["dxf"], o["dh1"], i["dffn"], i["h1"])
    return {**o, **{n: getattr(cache, n) for n in _lib.LAYER_TAPS}}


# ---- what a pass cannot do without -------------------------------------------------------------------------------------


def _forward_flops(case, seqs, seq):
    """Matrix products of the layers (causal attention: the lower triangle), without the classifier."""
    d, h, kv = case["dim"], case["hidden"], case.get("kv_heads", 0) or case["heads"]
    up = 2 if case["arch"] == "llama2" else 1
    proj = d * (d + 128 * kv) + d * d + (up + 1) * d * h
    return 2.0 * seqs * seq * (case["layers"] * proj + (d * d if up == 1 else 0)) + \
        case["layers"] * 4.0 * d * seqs * seq * (seq + 1) / 2


def _weights(case):
    """Elements of all matrices, the embedding among them (value-embedding tables are looked up, not read)."""
    d, h, kv = case["dim"], case["hidden"], case.get("kv_heads", 0) or case["heads"]
    up = 2 if case["arch"] == "llama2" else 1
    return case["layers"] * (d * (d + 128 * kv) + d * d + (up + 1) * d * h) + case["vocab"] * d + (d * d if up == 1 else 0)


def work(case):
    kind = case["kind"]
    if kind == "layer":
        d, h, s = case["dim"], case["hidden"], case["seq"]
        flops = 2.0 * s * (4 * d * d + 2 * d * h) * 2 + 4.0 * d * s * (s + 1) / 2 * 3.5
        return {"bytes": 4.0 * s * (18 * d + 4 * h) + 2.0 * (4 * d * d + 2 * d * h) * 2, "flops": flops}
    if kind == "head":
        t, d, v = case["tokens"], case["dim"], case["vocab"]
        return {"bytes": 2.0 * d * (t + v) + 6.0 * t, "flops": 2.0 * t * d * v}
    if kind == "moe":
        t, d, h, e = case["tokens"], case["dim"], case["hidden"], case["experts"]
        return {"bytes": 8.0 * t * d + 16.0 * t + 6.0 * min(e, 2 * t) * d * h, "flops": 12.0 * t * d * h + 2.0 * t * d * e}
    cfg = _cfg(case)
    d, v, s = case["dim"], case["vocab"], case["seq"]
    if kind == "serve":
        b, p, n = case["batch"], case["prefix"], case["steps"]
        row = case["layers"] * 256 * case["kv_heads"]  # K and V of one position, fp16
        flops = _forward_flops(case, b, p) + 2.0 * b * d * v
        nbytes = 2.0 * _weights(case) + b * p * row
        for k in range(n + 1):
            nbytes += 2.0 * _weights(case) + b * row * (p + k + 1)
            flops += 2.0 * b * _weights(case) + case["layers"] * 4.0 * d * b * (p + k + 1)
        return {"bytes": nbytes + 4.0 * b * v, "flops": flops}
    rows = case.get("batch", 1)
    flops = _forward_flops(case, rows, s) + 2.0 * rows * s * d * v
    if kind == "train":
        total, updates = ane.param_count(cfg), case["steps"] * case["batch"] // case["accum"]
        # per call the fp16 weights forward and backward and the gradient written; per update 30 bytes a parameter
        return {"bytes": case["steps"] * 8.0 * _weights(case) + updates * 30.0 * total + 4.0 * total,
                "flops": 3.0 * case["steps"] * flops}
    return {"bytes": 2.0 * _weights(case) + (4.0 * v * s if kind == "logits" else 0) + 4.0 * rows * s, "flops": flops}


# Each about four times the largest error against the 64-bit result that the path showed (logits 5.7e-4, loss 4e-6,
# trained weights 2.1e-3 after eight updates, decoder logits 1e-3, experts 5.1e-4, head 4.4e-8, layer 6.6e-4).  `max` of
# the trained weights: a gradient within rounding of zero changes sign, and AdamW moves such a weight the other way.
TOLERANCE = {
    "logits": {"rel": 2.5e-3},
    "loss": {"rel": 2e-5},
    "train": {"rel": 8e-3, "max": 0.5},
    "serve": {"rel": 4e-3, "differ": 0.005},
    "moe": {"rel": 2e-3, "differ": 0.0005},
    "head": {"rel": 2e-6},
    "layer": {"rel": 2.5e-3},
}


def tolerance(case):
    return TOLERANCE[case["kind"]]


# ---- the same results in 64 bits ---------------------------------------------------------------------------------------


def _rms(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)


def _rope(x, theta, at=0):
    """x [..., S, heads, 64]: channels (2i, 2i + 1) of each head turned by position * theta^(-2i/64)."""
    n, half = x.shape[-3], x.shape[-1] // 2
    pos = torch.arange(at, at + n, dtype=torch.float64, device=x.device)[:, None]
    ang = pos * theta ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    c, s = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([e * c - o * s, o * c + e * s], -1).flatten(-2)


def _attend(q, k, v, scale, at=0):
    """q [B, S, H, 64], k and v [B, K, G, 64] -> [B, S, H * 64]; query row i sees keys up to at + i."""
    rep = q.shape[2] // k.shape[2]
    q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
    if rep > 1:
        k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    w = (q @ k.transpose(2, 3).contiguous()) * scale
    seen = torch.arange(k.shape[2], device=q.device)[None, :] <= at + torch.arange(q.shape[2], device=q.device)[:, None]
    w = torch.softmax(w.masked_fill(~seen, float("-inf")), -1)
    return (w @ v).transpose(1, 2).flatten(2)


def _qknorm(x, quirks):
    r = torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
    if not quirks:
        return 1.2 * x * r
    return 1.2 * x * r.detach() + 1.44 * (x.detach() * r - x.detach() * r.detach())


def _views(cfg, flat):
    return {name: flat[off:off + math.prod(shape)].view(shape) for name, off, shape in ane.param_layout(cfg)}


def _logits(cfg, P, tok, quirks=False):
    """Logits [B, S, V] of whole windows.  quirks: the gradient is that of the reference's own backward, which takes the
    attention probabilities at scale 1, leaves out the rotation, weights the QK-norm's projection term by 1.44 and lets
    the first residual's gradient join before the smear."""
    nano, (B, S), NH = cfg.arch == "nanochat", tok.shape, cfg.heads
    heads = lambda t: t.view(B, S, -1, 64)  # noqa: E731
    x = P["embed"][tok]
    x0 = mid = None
    if nano:
        x = base = _rms(x)
        gate = torch.sigmoid(x @ P["smear_gate"].T)
        x = x + P["smear_lambda"] * gate * F.pad(x, (0, 0, 1, 0))[:, :-1]
        x0 = x + (base - x).detach() if quirks else base
    for l in range(cfg.layers):
        p = lambda n: P["layers.%d.%s" % (l, n)]  # noqa: E731
        xn = _rms(x) if nano else _rms(x) * p("g_att")
        q, k, v = heads(xn @ p("wq").T), heads(xn @ p("wk").T), heads(xn @ p("wv").T)
        qr, kr = _rope(q, cfg.rope_theta), _rope(k, cfg.rope_theta)
        if quirks:
            qr, kr = q + (qr - q).detach(), k + (kr - k).detach()
        if nano:
            qr, kr = _qknorm(qr, quirks), _qknorm(kr, quirks)
        if "layers.%d.ve_embed" % l in P:
            g = torch.sigmoid(x[..., :12] @ p("ve_gate").view(NH, 12).T)
            v = v + 3.0 * g[..., None] * heads(p("ve_embed")[tok])
        att = _attend(qr, kr, v, 0.125)
        if quirks:
            one = _attend(qr, kr, v, 1.0)
            att = one + (att - one).detach()
        if nano:
            rl, xl = P["resid_lambdas"][l], P["x0_lambdas"][l]
            x2 = rl * x + att @ p("wo").T + xl * x0
            x = rl * x2 + torch.relu(_rms(x2) @ p("w1").T) ** 2 @ p("w2").T + xl * x0
            mid = x if l == cfg.layers // 2 - 1 else mid
        else:
            x = x + att @ p("wo").T
            xn = _rms(x) * p("g_ffn")
            x = x + (F.silu(xn @ p("w1").T) * (xn @ p("w3").T)) @ p("w2").T
    if nano:
        x = _rms(x - P["backout_lambda"] * mid)
        return 15.0 * torch.tanh(x @ P["embed"].T / 15.0)
    return (_rms(x) * P["g_final"]) @ P["embed"].T


def _per_sequence(logits, tgt):
    return F.cross_entropy(logits.flatten(0, 1), tgt.flatten(), reduction="none").view(tgt.shape).mean(1)


def _cuda64(a):
    return torch.as_tensor(a, device="cuda").to(torch.float64)


def _ids(a):
    return torch.from_numpy(a.astype(np.int64)).cuda()


def _exact_train(case, cfg, seed):
    """The windows of the drand48 sampler, the gradient of their mean loss, global-norm clip and AdamW."""
    o = TRAIN_OPTIONS[cfg.arch]
    nano, D = cfg.arch == "nanochat", cfg.dim
    flat = _cuda64(_params(cfg, seed)).requires_grad_(True)
    stream = _ids(_tokens(case, seed, 1, 64 * (cfg.seq + 1))[0])
    state, limit = (o["Seed"] << 16) | 0x330E, stream.numel() - cfg.seq - 1
    lr, wd = torch.full_like(flat, o["LR"], requires_grad=False), torch.zeros_like(flat, requires_grad=False)
    b1, b2 = torch.full_like(wd, o["AdamBeta1"]), torch.full_like(wd, o["AdamBeta2"])
    clipped = torch.ones_like(wd, dtype=torch.bool)
    for name, off, shape in ane.param_layout(cfg):
        at, leaf = slice(off, off + math.prod(shape)), name.split(".")[-1]
        if leaf in ("wq", "wk", "wv", "wo", "w1", "w2", "w3", "smear_gate"):
            wd[at] = o["WeightDecay"]
        if leaf in ("resid_lambdas", "x0_lambdas"):
            lr[at], b1[at], b2[at] = o["LR"] * o["LambdaLRMult"], o["LambdaBeta1"], o["LambdaBeta2"]
        if leaf in ("g_final", "smear_gate", "smear_lambda", "backout_lambda", "resid_lambdas", "x0_lambdas"):
            clipped[at] = False
    m, v, losses, pending, t = torch.zeros_like(wd), torch.zeros_like(wd), [], 0, 0
    for _ in range(case["steps"]):
        rows = []
        for _ in range(case["batch"]):
            state = (0x5DEECE66D * state + 0xB) & ((1 << 48) - 1)
            at = min(int(state / 2.0 ** 48 * limit), limit - 1)
            rows.append(stream[at:at + cfg.seq + 1])
        ids = torch.stack(rows)
        per = _per_sequence(_logits(cfg, _views(cfg, flat), ids[:, :-1], nano), ids[:, 1:])
        per.sum().backward()
        losses.append(float(per.detach().mean()))
        pending += case["batch"]
        if pending >= case["accum"]:
            t += 1
            with torch.no_grad():
                g = flat.grad / pending
                norm = float(g[clipped].norm())
                if o.get("GradClip", 0) > 0 and norm > o["GradClip"]:
                    g[clipped] *= o["GradClip"] / norm
                m = b1 * m + (1 - b1) * g
                v = b2 * v + (1 - b2) * g * g
                upd = m / (1 - b1 ** t) / (torch.sqrt(v / (1 - b2 ** t)) + o["AdamEps"]) + wd * flat
                flat -= lr * upd
            flat.grad, pending = None, 0
    return {"losses": np.array(losses), "params": flat.detach()}


def _exact_serve(case, cfg, seed):
    """Greedy decoding with every key and value kept in 64 bits; a few sequences at a time."""
    P = _views(cfg, _cuda64(_serve_params(cfg, seed)))
    prefix = _ids(_tokens(case, seed, case["batch"], case["prefix"]))
    first, tokens, last = [], [], []
    for rows in prefix.split(4):
        keys, vals = [None] * cfg.layers, [None] * cfg.layers

        def feed(tok, at):
            x = P["embed"][tok]
            for l in range(cfg.layers):
                p = lambda n: P["layers.%d.%s" % (l, n)]  # noqa: E731
                heads = lambda t: t.view(*tok.shape, -1, 64)  # noqa: E731
                xn = _rms(x) * p("g_att")
                q, k, v = (heads(xn @ p(n).T) for n in ("wq", "wk", "wv"))
                k = _rope(k, cfg.rope_theta, at)
                keys[l] = k if keys[l] is None else torch.cat([keys[l], k], 1)
                vals[l] = v if vals[l] is None else torch.cat([vals[l], v], 1)
                x = x + _attend(_rope(q, cfg.rope_theta, at), keys[l], vals[l], 0.125, at) @ p("wo").T
                xn = _rms(x) * p("g_ffn")
                x = x + (F.silu(xn @ p("w1").T) * (xn @ p("w3").T)) @ p("w2").T
            return (_rms(x[:, -1]) * P["g_final"]) @ P["embed"].T

        at = case["prefix"]
        nxt = feed(rows, 0).argmax(-1)
        got = [nxt]
        for _ in range(case["steps"]):
            nxt = feed(nxt[:, None], at).argmax(-1)
            got.append(nxt)
            at += 1
        last.append(feed(nxt[:, None], at))
        first.append(got[0])
        tokens.append(torch.stack(got[1:], 1))
    return {"first": torch.cat(first).int(), "tokens": torch.cat(tokens).int(), "logits": torch.cat(last)}


def _exact_moe(case, seed):
    cfg, params, x = _moe_inputs(case, seed)
    params, x = params.double(), x.double()
    E, D, H = cfg.experts, cfg.dim, cfg.hidden
    top, which = (x @ params[:E * D].view(E, D).T).topk(2, dim=1)
    weights = torch.softmax(top, 1)
    out = torch.zeros_like(x)
    for e in range(E):
        at = E * D + e * 3 * H * D
        w1, w3, w2 = params[at:at + H * D].view(H, D), params[at + H * D:at + 2 * H * D].view(H, D), params[at + 2 * H * D:at + 3 * H * D].view(D, H)
        t, slot = (which == e).nonzero(as_tuple=True)
        if t.numel():
            y = (F.silu(x[t] @ w1.T) * (x[t] @ w3.T)) @ w2.T
            out.index_add_(0, t, y * weights[t, slot, None])
    return {"out": out, "experts": None, "weights": weights}


def _exact_head(case, seed):
    xn, embed, tgt = _head_inputs(case, seed)
    tgt = tgt.long() & 0xFFFF
    lse, picked = [], []
    for rows, t in zip(xn.split(2048), tgt.split(2048)):
        lg = rows.double() @ embed.double().T
        if case["softcap"]:
            lg = 15.0 * torch.tanh(lg / 15.0)
        lse.append(torch.logsumexp(lg, 1))
        picked.append(lg.gather(1, t[:, None])[:, 0])
    lse, picked = torch.cat(lse), torch.cat(picked)
    nll = torch.clamp(lse - picked, max=-math.log(1e-10))
    return {"loss": nll.view(-1, case["seq"]).mean(1), "lse": lse}


def _exact_layer(case, seed):
    w = {n: t.double() for n, t in _layer_weights(case, seed).items()}
    i = {n: t.double().T.contiguous() for n, t in _layer_inputs(case, seed).items()}  # token-major
    heads = lambda t: t.view(1, case["seq"], -1, 64)  # noqa: E731
    r = {}
    r["x_norm"] = _rms(i["x"])
    q, k, v = (heads(r["x_norm"] @ w[n].T) for n in ("wq", "wk", "wv"))
    q, k = _rope(q, 1e5), _rope(k, 1e5)
    r["q"], r["k"], r["v"] = (t.flatten(2)[0] for t in (q, k, v))
    r["att_out"] = _attend(q, k, v, 0.125)[0]
    r["x2"] = i["x"] + r["att_out"] @ w["wo"].T
    r["x2_norm"] = _rms(r["x2"])
    r["h1"] = r["x2_norm"] @ w["w1"].T
    r["gate"] = torch.relu(r["h1"]) ** 2
    r["out"] = r["x2"] + r["gate"] @ w["w2"].T
    q, k, v = (heads(i[n]).requires_grad_(True) for n in "qkv")
    dq, dk, dv = torch.autograd.grad(_attend(q, k, v, 0.125), (q, k, v), (i["dx2"] @ w["wo"])[None])
    r["dq"], r["dk"], r["dv"] = (t.flatten(2)[0] for t in (dq, dk, dv))
    r["dxa"] = r["dq"] @ w["wq"] + r["dk"] @ w["wk"] + r["dv"] @ w["wv"]
    r["dh1"] = (i["dffn"] @ w["w2"]) * 2.0 * torch.relu(i["h1"])
    r["dxf"] = r["dh1"] @ w["w1"]
    return {n: t.T.contiguous().view(-1) for n, t in r.items()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "moe":
        return _exact_moe(case, seed)
    if kind == "head":
        return _exact_head(case, seed)
    if kind == "layer":
        return _exact_layer(case, seed)
    cfg = _cfg(case)
    if kind == "train":
        return _exact_train(case, cfg, seed)
    with torch.no_grad():
        if kind == "serve":
            return _exact_serve(case, cfg, seed)
        P = _views(cfg, _cuda64(_params(cfg, seed)))
        ids = _ids(_tokens(case, seed, case.get("batch", 1), cfg.seq + 1))
        if kind == "logits":
            return _logits(cfg, P, ids[:, :-1])[0].T.contiguous().view(-1)
        per = torch.cat([_per_sequence(_logits(cfg, P, b[:, :-1]), b[:, 1:]) for b in ids.split(4)])
        return {"mean": float(per.mean()), "per_sequence": per}
