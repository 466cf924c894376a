"""The work whose speed is followed: one pass each of what a GRPO actor-learner does with this package.

Learner and sampler, at the vocabulary of Qwen2.5 (151,936):
  sample     one decode step's sampling over [rows, vocab] logits, plain (T = 1) or with top-p
  policy     a mini-batch's training passes over resident logits: plan with GRPO, one fused forward and backward per
             micro-batch, fold; returns the logits' gradients
  reference  old / reference log-probs and entropies of packed tokens from hidden states, lm_head inside
Rollout engine, bf16, two of the hybrid decoders with four layer runs in the proportions of `bench.py --hybrid`
(Dovidra: latent attention and gated delta rule, a loop run twice; Tativik: latent attention with low-rank queries
and sinks, generalized delta rule, routed experts), through the engine's runner, logits instead of samples:
  prompts    prompts from position 0, several at once or a long one
  decode     a decode step of `rows` sequences with about `context` tokens behind them
  mixed      a step that continues prompts while other sequences decode

Sizes: the batch shapes of bench.py and bench_hybrid.py, widths 1536 to 4096, odd counts and lengths in `draw`."""

import math
import random

import numpy as np
import torch
import torch.nn.functional as F

from skyrl_amd import ops
from skyrl_amd.inference_engines.engine import BLOCK_SIZE, ModelRunner, Request, RequestParams, ScheduledBatch
from skyrl_amd.inference_engines.hybrid import HybridDecoder

DEV = "cuda:0"
VOCAB = 151936         # Qwen2.5's
ENGINE_VOCAB = 32768   # bench_hybrid.py's
RUNS = 4               # layer runs of the engine's models
WINDOW = 1024
EPS = 1e-6


def listed():
    return [
        # the smallest call: one interactive sequence's next token
        {"name": "sample_one_row", "kind": "sample", "rows": 1, "vocab": VOCAB, "temperature": 1.0, "top_p": 1.0},
        # a rollout batch with the usual evaluation filter
        {"name": "sample_512_top_p", "kind": "sample", "rows": 512, "vocab": VOCAB, "temperature": 0.6, "top_p": 0.95},
        # a learner's mini-batch of two micro-batches, responses of up to 512 tokens
        {"name": "policy_16x512", "kind": "policy", "rows": 16, "micro": 8, "length": 512, "group": 8, "vocab": VOCAB},
        # the reference model's pass over a packed micro-batch
        {"name": "reference_8192", "kind": "reference", "tokens": 8192, "width": 1536, "vocab": VOCAB},
        # a long document
        {"name": "dovidra_prompt_8192", "kind": "prompts", "model": "dovidra", "width": 2048, "rows": 1, "longest": 8192},
        # interactive decoding
        {"name": "dovidra_decode_1", "kind": "decode", "model": "dovidra", "width": 2048, "rows": 1, "context": 2048},
        # rollout decoding
        {"name": "dovidra_decode_64", "kind": "decode", "model": "dovidra", "width": 2048, "rows": 64, "context": 2048},
        # the start of a rollout batch: ragged prompts
        {"name": "tativik_prompts_8", "kind": "prompts", "model": "tativik", "width": 2048, "rows": 8, "longest": 1024},
        # continuous batching: three prompts admitted (one of them continued) while 48 sequences decode
        {"name": "tativik_mixed", "kind": "mixed", "model": "tativik", "width": 2048, "rows": 48, "context": 1536,
         "prompts": 3, "longest": 700},
        {"name": "tativik_decode_1", "kind": "decode", "model": "tativik", "width": 2048, "rows": 1, "context": 2048},
        {"name": "tativik_decode_64", "kind": "decode", "model": "tativik", "width": 2048, "rows": 64, "context": 2048},
        # a full rollout batch
        {"name": "tativik_decode_256", "kind": "decode", "model": "tativik", "width": 2048, "rows": 256, "context": 1024},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("sample", "policy", "reference", "prompts", "prompts", "decode", "decode", "decode", "mixed"))
    if kind == "sample":
        top_p = rng.choice((1.0, 0.95, 0.9))
        return {"kind": kind, "rows": _log(rng, 1, 512), "vocab": rng.choice((VOCAB, 50257, 32768)),
                "temperature": 1.0 if top_p == 1.0 else rng.choice((0.6, 1.0)), "top_p": top_p}
    if kind == "policy":
        group = rng.choice((4, 8))
        rows = group * rng.randint(1, 16 // group)
        return {"kind": kind, "rows": rows, "micro": rng.choice((3, 4, 8)), "length": _log(rng, 9, 511), "group": group,
                "vocab": VOCAB}
    if kind == "reference":
        return {"kind": kind, "tokens": _log(rng, 200, 8191), "width": rng.choice((1536, 2048)), "vocab": VOCAB}
    model, width = rng.choice(("dovidra", "tativik")), rng.choice((1536, 2048, 2048, 4096))
    if kind == "prompts":
        rows = _log(rng, 1, 8)
        return {"kind": kind, "model": model, "width": width, "rows": rows,
                "longest": _log(rng, 40, (8000 if width < 4096 else 2000) // rows)}
    if kind == "decode":
        return {"kind": kind, "model": model, "width": width, "rows": _log(rng, 1, 256 if width < 4096 else 64),
                "context": _log(rng, 64, 3000)}
    return {"kind": kind, "model": model, "width": width, "rows": _log(rng, 1, 96), "context": _log(rng, 64, 3000),
            "prompts": rng.randint(1, 4), "longest": _log(rng, 40, 900)}


# ---------------------------------------------------------------- the engine's models
def _config(model, width):
    heads, ff = width // 128, 3 * width
    latent = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
              "mask": {"size": WINDOW}, "rot": {"base": 10000.0, "dims": 64}}
    cfg = {"norm": {"eps": EPS}, "vocab": ENGINE_VOCAB, "width": width}
    if model == "dovidra":
        latent["rot"]["scaling"] = {"factor": 16.0, "original": 4096, "fast": 32.0, "slow": 1.0}
        mlp = {"kind": "dense", "ff": ff}
        layers = [{"type": "latent_attention", "mlp": mlp, "mixer": latent},
                  {"type": "delta", "mlp": mlp, "mixer": {"heads": 2 * heads, "kv_heads": heads, "dim": 128, "vdim": 128,
                                                          "conv": 4}}]
        return dict(cfg, architecture="Dovidra", layers=layers, loop={"start": 0, "stop": 2, "times": RUNS // 2},
                    logit_softcap=30.0)
    mlp = {"kind": "moe", "expert": {"ff": ff // 8}, "router": {"experts": 64, "top": 8, "groups": {"count": 8, "keep": 4}}}
    latent["q_rank"] = width * 3 // 8
    layers = [{"type": "general_delta", "mlp": mlp, "mixer": {"heads": width // 64, "dim": 64, "decay_rank": 64}} if i % 2
              else {"type": "latent_attention", "mlp": mlp, "mixer": latent} for i in range(RUNS)]
    return dict(cfg, architecture="Tativik", layers=layers, norm={"eps": EPS, "groups": 4}, residual_mult=0.5)


def _model(case, seed, max_len):
    """Random weights; gates, decays and norms spread as a trained model's are."""
    model = HybridDecoder(_config(case["model"], case["width"]), DEV, dtype=torch.bfloat16, seed=seed, max_model_len=max_len)
    g = torch.Generator(device=DEV).manual_seed(seed + 1)
    for name, t in model.hf_named_tensors():
        last = name.rsplit(".", 1)[-1]
        if last == "A_log":    # rates of 1 to 16
            t.uniform_(1.0, 16.0, generator=g).log_()
        elif last == "dt_bias":  # time steps of 0.001 to 0.1
            t.uniform_(math.log(0.001), math.log(0.1), generator=g).exp_().expm1_().log_()
        elif last == "conv":
            t.normal_(0.0, 0.5, generator=g)
        elif last in ("w0", "sink"):
            t.normal_(-1.0, 1.0, generator=g)
        elif name.endswith("a.b"):
            t.normal_(0.0, 1.0, generator=g)
        elif last == "correction":
            t.normal_(0.0, 0.05, generator=g)
        elif "norm" in last:
            t.normal_(1.0, 0.1, generator=g)
    if case["model"] == "tativik":  # a trained router is decided: tokens lean to two experts in each of four groups
        lean = torch.rand(ENGINE_VOCAB, 8, device=DEV, generator=g).topk(4, -1).indices
        two = torch.rand(ENGINE_VOCAB, 4, 8, device=DEV, generator=g).topk(2, -1).indices
        ways = torch.randn(64, case["width"], device=DEV, generator=g) * case["width"] ** -0.5
        model.embed.add_(0.2 * torch.zeros(ENGINE_VOCAB, 64, device=DEV).scatter_(1, (lean[..., None] * 8 + two).flatten(1), 1.0) @ ways)
        for name, t in model.hf_named_tensors():
            if name.endswith("mlp.router"):
                t.copy_(0.5 * ways)
    model.load_weights(())
    return model


def _sequences(case, rng):
    """[(tokens behind, tokens of the step)] of the engine's cases."""
    kind = case["kind"]
    new = lambda n: [(0, case["longest"] if i == 0 else rng.randint(max(1, case["longest"] // 3), case["longest"]))  # noqa: E731
                     for i in range(n)]
    if kind == "prompts":
        return new(case["rows"])
    c = case["context"]
    old = [(rng.randint(max(1, c * 3 // 4), c + c // 4), 1) for _ in range(case["rows"])]
    if kind == "decode":
        return old
    fresh = new(case["prompts"])
    return old + [(BLOCK_SIZE * 20 + 5, fresh[0][1])] + fresh[1:]  # the first one has had a portion before


def _engine(case, seed):
    rng = random.Random(seed)
    seqs = _sequences(case, random.Random(7))  # a step's shape belongs to the case
    max_len = -(-max(2048, *(s + n for s, n in seqs)) // BLOCK_SIZE) * BLOCK_SIZE
    need = [-(-(s + n) // BLOCK_SIZE) for s, n in seqs]
    order = list(range(sum(need)))
    rng.shuffle(order)
    rows = next((b for b in ModelRunner.BUCKETS if b >= len(seqs)), len(seqs))
    ids = np.random.default_rng(seed).integers(0, ENGINE_VOCAB, (len(seqs), max(s + n for s, n in seqs)))
    reqs = []
    for i, (s, n) in enumerate(seqs):
        reqs.append(Request(rid=i, prompt=ids[i, :s + n].tolist(), params=RequestParams(), key=i, row=i, num_computed=s,
                            blocks=[order.pop() for _ in range(need[i])]))
    with torch.no_grad():
        runner = ModelRunner(_model(case, seed, max_len), sum(need), rows)
        batch = ScheduledBatch("decode" if case["kind"] == "decode" else "portions", reqs,
                               np.zeros(len(reqs), dtype=np.int64), [()] * len(reqs), [n for _, n in seqs])
        state = {"kind": "engine", "runner": runner, "batch": batch, "want": [(i, n - 1) for i, (_, n) in enumerate(seqs)],
                 "case": case}
        if case["kind"] == "decode":  # the runner's captured step of this size, as an engine that is running has it
            run(state)
        g = torch.Generator(device=DEV).manual_seed(seed + 2)
        for t in _caches(runner):  # what earlier tokens left: normed latents, states, convolution inputs
            t.normal_(0.0, 0.3 if t.dtype == torch.float32 else 1.0, generator=g)
    return state


def _caches(runner):
    return [t for run_ in runner.cache.runs for t in (run_ if isinstance(run_, tuple) else (run_,))]


# ---------------------------------------------------------------- the interface
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("prompts", "decode", "mixed"):
        return _engine(case, seed)
    g = torch.Generator(device=DEV).manual_seed(seed)
    if kind == "sample":
        logits = _logits((case["rows"], case["vocab"]), g)
        return {"kind": kind, "logits": logits, "ids": torch.randperm(1 << 16, device=DEV, generator=g)[:case["rows"]],
                "args": {"temperature": case["temperature"], "top_p": case["top_p"], "seed": seed, "step": seed % 1000}}
    if kind == "policy":
        n, R, V = case["rows"], case["length"], case["vocab"]
        z = _logits((n * R, V), g).view(n, R, V)
        labels = torch.randint(0, V, (n, R), device=DEV, generator=g)
        lp = torch.empty(n, R, device=DEV)
        for i in range(n):  # tokens a policy samples are likely ones
            labels[i] = torch.where(torch.rand(R, device=DEV, generator=g) < 0.8, z[i].argmax(-1), labels[i])
            lp[i] = torch.log_softmax(z[i].double(), -1).gather(1, labels[i][:, None])[:, 0]
        near = lambda: lp + 0.05 * torch.randn(n, R, device=DEV, generator=g)  # noqa: E731
        lens = torch.randint(max(1, R // 4), R + 1, (n,), device=DEV, generator=g)
        mask = (torch.arange(R, device=DEV)[None] < lens[:, None])
        return {"kind": kind, "z": z.requires_grad_(True), "labels": labels, "old": near(), "ref": near(), "case": case,
                "mask": mask.float(), "rmask": mask.to(torch.int64), "rows": mask.float().sum(1),
                "scores": (torch.rand(n, device=DEV, generator=g) < 0.4).float() + 0.1 * torch.rand(n, device=DEV, generator=g),
                "adv": torch.empty(n, R, device=DEV),
                "params": ops.make_ppo_params(use_kl_loss=True, kl_loss_coef=0.001, has_entropy=True)}
    T, W = case["tokens"], case["width"]
    hidden = torch.randn((T, W), device=DEV, generator=g).to(torch.bfloat16)
    weight = torch.empty((case["vocab"], W), device=DEV, dtype=torch.bfloat16).normal_(0.0, 0.05, generator=g)
    return {"kind": kind, "hidden": hidden, "weight": weight,
            "labels": torch.randint(0, case["vocab"], (T,), device=DEV, generator=g)}


def _logits(shape, g):
    """A language model's: a wide body and some likely tokens in every row."""
    z = torch.empty(shape, device=DEV, dtype=torch.bfloat16).normal_(0.0, 2.5, generator=g)
    step = shape[1] // 24
    at = torch.arange(24, device=DEV) * step + torch.randint(0, step, (shape[0], 24), device=DEV, generator=g)
    return z.scatter_(1, at, torch.empty(at.shape, device=DEV, dtype=torch.bfloat16).normal_(13.0, 2.5, generator=g))


def run(state):
    kind = state["kind"]
    if kind == "engine":
        with torch.no_grad():
            logits = state["runner"].portion_logits(state["batch"], state["want"])
        return {"logits": logits, "caches": _caches(state["runner"])}
    if kind == "sample":
        return ops.sample(state["logits"], seq_ids=state["ids"], **state["args"])
    if kind == "policy":
        c = state["case"]
        step = ops.PolicyTrainStep(state["old"], state["adv"], state["mask"], state["params"], c["micro"],
                                   ref_log_probs=state["ref"],
                                   grpo={"scores": state["scores"], "response_mask": state["rmask"],
                                         "group_size": c["group"], "loss_mask_row_sum": state["rows"]})
        grads = []
        for k in range(step.n_micro):
            i, j = step.rows(k)
            z = state["z"][i:j].detach().requires_grad_(True)
            grads += torch.autograd.grad(step.micro(k, z, state["labels"][i:j]), z)
        loss, metrics = step.fold()
        return {"grads": grads, "loss": loss, "final_loss": metrics[:, 0], "logp": step.logp, "entropy": step.entropy,
                "adv": state["adv"]}
    return ops.lmhead_logprob_fwd(state["hidden"], state["weight"], state["labels"])


def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": 2 * case["rows"] * case["vocab"], "flops": 0}
    if kind == "policy":
        return {"bytes": 4 * case["rows"] * case["length"] * case["vocab"], "flops": 0}
    if kind == "reference":
        T, W, V = case["tokens"], case["width"], case["vocab"]
        return {"bytes": 2 * W * (T + V), "flops": 2 * T * W * V}
    W, seqs = case["width"], _sequences(case, random.Random(7))
    T, H = sum(n for _, n in seqs), W // 128
    kept = lambda s, n: sum(min(WINDOW, s + j + 1) for j in range(n))  # noqa: E731
    pairs = sum(kept(s, n) for s, n in seqs)
    seen = sum(min(s + n, WINDOW + n - 1) for s, n in seqs)
    rank, row, ff = 512, 576, 3 * W
    if case["model"] == "dovidra":
        attn = W * H * 192 + W * row + 2 * 512 * H * 128 + H * 128 * W
        state, rule = 2 * H * 128 * 128, W * (2 * H * 128 + 4 * H * 128 + 4 * H) + 2 * H * 128 * W
        ff_w, ff_run = 3 * ff * W, 3 * ff * W
        layers = RUNS // 2
    else:
        q = W * 3 // 8
        attn = W * q + q * H * 192 + W * (row + H) + 2 * rank * H * 128 + H * 128 * W + W * W
        state, rule = W * 64, W * (5 * W + 64) + 64 * W + W * W + W * W
        ff_run = 3 * ff * W + 64 * W + W * W
        ff_w = 3 * (ff // 8) * W * min(64, 64 * (1 - (1 - 1 / 8) ** T)) + 64 * W + W * W
        layers = RUNS
    half = RUNS // 2
    weights = layers / 2 * (attn + rule + 2 * ff_w) + len(seqs) * W + ENGINE_VOCAB * W
    flops = 2 * T * half * (attn + rule + 2 * ff_run) + half * (pairs * H * 2 * 320 + T * state * 6)
    flops += 2 * len(seqs) * ENGINE_VOCAB * W
    moved = half * (seen * row * 2 + T * row * 2 + len(seqs) * state * 8)
    return {"bytes": 2 * weights + moved + 4 * len(seqs) * ENGINE_VOCAB, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":   # 32-bit sums; a token may move where two scores are within them
        return {"rel": 1e-5, "differ": 0.0}
    if kind == "policy":   # gradients are bf16, what they come from 32-bit
        return {"rel": 2e-3, "max": 0.02}
    if kind == "reference":  # logits in bf16, sums of them in 32 bits
        return {"rel": 1e-3, "max": 0.05}
    return {"rel": 0.03, "max": 0.99}  # bf16 through four layers; experts that are nearly tied change places


# ---------------------------------------------------------------- 64 bits
def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind == "sample":
            return None  # the tokens belong to the package's noise, the log-probs to the tokens
        if kind == "policy":
            return _policy64(state, case)
        if kind == "reference":
            out = []
            w = state["weight"].double()
            for h, l in zip(state["hidden"].split(1024), state["labels"].split(1024)):
                p = torch.log_softmax(h.double() @ w.T, -1)
                out.append((p.gather(1, l[:, None])[:, 0], -(p.exp() * p).sum(-1)))
            return tuple(torch.cat(t) for t in zip(*out))
        return _engine64(state, case)


def _policy64(s, c):
    n, R, G = c["rows"], c["length"], c["group"]
    sc, mask = s["scores"].double().view(-1, G), s["mask"].double()
    adv = ((sc - sc.mean(1, True)) / (sc.std(1, keepdim=True) + 1e-6)).view(-1, 1) * mask
    grads, losses, lps, ents = [], [], [], []
    for i in range(0, n, c["micro"]):
        j = min(n, i + c["micro"])
        glp, m = torch.zeros(j - i, R, device=DEV, dtype=torch.float64), mask[i:j]
        grad = torch.empty(j - i, R, c["vocab"], device=DEV, dtype=torch.float64)
        for k in range(j - i):
            p = torch.log_softmax(s["z"][i + k].double(), -1)
            lps.append(p.gather(1, s["labels"][i + k][:, None])[:, 0])
            ents.append(-(p.exp() * p).sum(-1))
            grad[k] = -p.exp_()
            grad[k].scatter_add_(1, s["labels"][i + k][:, None], torch.ones(R, 1, device=DEV, dtype=torch.float64))
        lp = torch.stack(lps[-(j - i):])
        with torch.enable_grad():
            x = lp.clone().requires_grad_(True)
            ratio = torch.exp((x - s["old"][i:j].double()).clamp(-20, 20))
            loss = -torch.min(ratio * adv[i:j], ratio.clamp(0.8, 1.2) * adv[i:j])
            pg = (loss * m).sum() / m.sum()
            (glp,) = torch.autograd.grad(pg, x)
        d = (s["ref"][i:j].double() - lp).clamp(-20, 20)
        kl = ((torch.exp(d) - d - 1).clamp(-10, 10) * m).sum(1) / m.sum(1)
        grads.append(grad.mul_(glp[..., None]))
        losses.append(pg.detach() + 0.001 * kl.mean())
    return {"grads": grads, "loss": torch.stack(losses), "final_loss": torch.stack(losses), "logp": torch.stack(lps),
            "entropy": torch.stack(ents), "adv": adv}


def _rms(x, groups=1):
    x = x.unflatten(-1, (groups, -1))
    return (x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)).flatten(-2)


def _layer_norm(x, w):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + EPS) * w


def _rotate(x, pos, rot, halves):
    D, base = rot["dims"], rot["base"]
    f, amp = base ** (-2.0 * torch.arange(D // 2, device=DEV, dtype=torch.float64) / D), 1.0
    sc = rot.get("scaling")
    if sc:  # YaRN
        dim = lambda turns: D * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(dim(sc["fast"])), 0), min(math.ceil(dim(sc["slow"])), D - 1)
        ramp = ((torch.arange(D // 2, device=DEV, dtype=torch.float64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f, amp = f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
    a = pos.double()[:, None] * f
    a = a.view(a.shape[:1] + (1,) * (x.dim() - 2) + a.shape[1:])
    c, s = a.cos() * amp, a.sin() * amp
    u, v = (x[..., :D // 2], x[..., D // 2:]) if halves else (x[..., 0::2], x[..., 1::2])
    u, v = u * c - v * s, v * c + u * s
    return torch.cat([u, v], -1) if halves else torch.stack([u, v], -1).flatten(-2)


class _Step:
    """The step's tokens: seqs = (first token, tokens, tokens behind, row, blocks)."""

    def __init__(self, state):
        at, self.seqs, ids, pos = 0, [], [], []
        for r, n in zip(state["batch"].requests, state["batch"].counts):
            s = r.num_computed
            self.seqs.append((at, n, s, r.row, torch.tensor(r.blocks, device=DEV)))
            ids += r.prompt[s:s + n]
            pos += range(s, s + n)
            at += n
        self.ids, self.pos = torch.tensor(ids, device=DEV), torch.tensor(pos, device=DEV)


def _latent64(h, w, p, m, step, cache, tativik):
    H, D, R, V, C = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
    T = h.shape[0]
    q = (_rms(h @ w(p + "dq").T) * w(p + "dq.norm")) @ w(p + "uq").T if tativik else h @ w(p + "q").T
    q = q.view(T, H, D + R)
    q = torch.cat([q[..., :D], _rotate(q[..., D:], step.pos, m["rot"], tativik)], -1)
    down = h @ w(p + "dkv").T
    rows = torch.cat([_rms(down[:, :C]) * w(p + "dkv.norm"), _rotate(down[:, C:], step.pos, m["rot"], tativik)], -1)
    uk, uv = w(p + "uk").view(H, D, C), w(p + "uv").view(H, V, C)
    flat, out = cache.view(-1, cache.shape[-1]), torch.empty(T, H, V, device=DEV, dtype=torch.float64)
    for at, n, s, _, blocks in step.seqs:
        slot = lambda a, b: (lambda x: blocks[x // BLOCK_SIZE] * BLOCK_SIZE + x % BLOCK_SIZE)(torch.arange(a, b, device=DEV))  # noqa: E731
        flat[slot(s, s + n)] = rows[at:at + n]
        for a in range(0, n, 512):
            b = min(n, a + 512)
            lo = max(0, s + a - WINDOW + 1)
            kv = flat[slot(lo, s + b)]
            qa = torch.einsum("thd,hdc->thc", q[at + a:at + b, :, :D], uk)
            x = (torch.einsum("thc,jc->htj", qa, kv[:, :C]) + torch.einsum("thr,jr->htj", q[at + a:at + b, :, D:], kv[:, C:])) * m["scale"]
            d = torch.arange(s + a, s + b, device=DEV)[:, None] - torch.arange(lo, s + b, device=DEV)[None]
            x = x.masked_fill((d < 0) | (d >= WINDOW), float("-inf"))
            if tativik:
                x = torch.cat([x, w(p + "sink").view(H, 1, 1).expand(H, b - a, 1)], -1)
            x = torch.softmax(x, -1)[..., :kv.shape[0]]
            out[at + a:at + b] = torch.einsum("htc,hvc->thv", x @ kv[:, :C], uv)
    if tativik:
        out *= torch.sigmoid(h @ w(p + "g").T)[:, :, None]
    return out.view(T, H * V) @ w(p + "o").T


def _unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _delta64(h, w, p, m, step, S_all, ring):
    H, K, D, V, taps = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"]
    T = h.shape[0]
    u = torch.cat([h @ w(p + n).T for n in "qkv"], 1)
    filt = torch.cat([w(p + n + ".conv") for n in "qkv"])
    y = torch.empty_like(u)
    for at, n, s, row, _ in step.seqs:
        back = torch.stack([ring[row, (s - j) % taps] if s - j >= 0 else torch.zeros_like(u[0]) for j in range(taps - 1, 0, -1)])
        x = torch.cat([back, u[at:at + n]])
        y[at:at + n] = sum(x[j:j + n] * filt[:, j] for j in range(taps))
        for j in range(max(0, n - taps), n):
            ring[row, (s + j) % taps] = u[at + j]
    q, k, v = F.silu(y).split([K * D, K * D, H * V], 1)
    q, k = ((_unit(t.view(T, K, D)) * f).repeat_interleave(H // K, 1) for t, f in ((q, D ** -0.5), (k, 1.0)))
    v, beta = v.view(T, H, V), torch.sigmoid(h @ w(p + "b").T)
    g = torch.exp(-torch.exp(w(p + "A_log")) * F.softplus(h @ w(p + "a").T + w(p + "dt_bias"), threshold=50.0))
    o = torch.empty(T, H, V, device=DEV, dtype=torch.float64)
    for at, n, s, row, _ in step.seqs:
        S = S_all[row] if s else torch.zeros_like(S_all[row])
        for t in range(at, at + n):
            S = S * g[t][:, None, None]
            S = S + k[t][..., None] * (beta[t][:, None] * (v[t] - (k[t][:, None] @ S)[:, 0]))[:, None]
            o[t] = (q[t][:, None] @ S)[:, 0]
        S_all[row] = S
    o = _rms(o) * w(p + "norm") * F.silu(h @ w(p + "g").T).view(T, H, V)
    return o.view(T, H * V) @ w(p + "o").T


def _general64(h, w, p, m, step, S_all):
    H, D, T = m["heads"], m["dim"], h.shape[0]
    r, k, v = ((h @ w(p + n).T).view(T, H, D) for n in "rkv")
    z = torch.tanh(h @ w(p + "w1").T) @ w(p + "w2").T + w(p + "w0")
    decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(z)).view(T, H, D)
    u = _unit(k)
    au = torch.sigmoid(h @ w(p + "a").T + w(p + "a.b")).view(T, H, D) * u
    o = torch.empty(T, H, D, device=DEV, dtype=torch.float64)
    for at, n, s, row, _ in step.seqs:
        S = S_all[row] if s else torch.zeros_like(S_all[row])
        for t in range(at, at + n):
            S = decay[t][..., None] * S - au[t][..., None] * (u[t][:, None] @ S) + k[t][..., None] * v[t][:, None]
            o[t] = (r[t][:, None] @ S)[:, 0]
        S_all[row] = S
    o = _rms(o).view(T, H * D) * w(p + "norm") * torch.sigmoid(h @ w(p + "g").T)
    return o @ w(p + "o").T


def _experts64(h, w, p, m):
    ro, T = m["router"], h.shape[0]
    score = torch.sigmoid(h @ w(p + "router").T)
    choice = score + w(p + "correction")
    n, keep = ro["groups"]["count"], ro["groups"]["keep"]
    best = choice.view(T, n, -1).topk(2, -1).values.sum(-1)
    kept = torch.zeros_like(best, dtype=torch.bool).scatter_(1, best.topk(keep, -1).indices, True)
    idx = choice.masked_fill(~kept.repeat_interleave(ro["experts"] // n, 1), float("-inf")).topk(ro["top"], -1).indices
    out = torch.zeros_like(h)
    for e in range(ro["experts"]):
        t = (idx == e).any(1).nonzero()[:, 0]
        if t.numel():
            x, q = h[t], f"{p}e{e}."
            out[t] += score[t, e, None] * ((F.silu(x @ w(q + "gate").T) * (x @ w(q + "up").T)) @ w(q + "down").T)
    return out


def _engine64(state, case):
    runner, step = state["runner"], _Step(state)
    cfg, tativik = _config(case["model"], case["width"]), case["model"] == "tativik"
    names = dict(runner.model.hf_named_tensors())
    w = lambda name: names[name].double()  # noqa: E731
    caches = [t.double() for t in _caches(runner)]
    left = iter(caches)
    group = lambda x, name: _rms(x, 4) * w(name)  # noqa: E731
    x = names["embed"][step.ids].double()
    x = group(x, "embed.norm") if tativik else x
    runs = range(RUNS) if tativik else [0, 1] * (RUNS // 2)
    for k, i in enumerate(runs):
        p, e = f"l{i}.", cfg["layers"][i]
        if not tativik and i == 0:
            x = x + w("loop.step")[k // 2]
        h = group(x, p + "norm1") if tativik else _layer_norm(x, w(p + "norm1"))
        if e["type"] == "latent_attention":
            y = _latent64(h, w, p + "mix.", e["mixer"], step, next(left), tativik)
        elif e["type"] == "delta":
            y = _delta64(h, w, p + "mix.", e["mixer"], step, next(left), next(left))
        else:
            y = _general64(h, w, p + "mix.", e["mixer"], step, next(left))
        if tativik:
            x = x + 0.5 * group(y * torch.sigmoid(h @ w(p + "rg1").T + w(p + "rg1.b")), p + "norm1b")
            h = group(x, p + "norm2")
            y = _experts64(h, w, p + "mlp.", e["mlp"]) * torch.sigmoid(h @ w(p + "rg2").T + w(p + "rg2.b"))
            x = x + 0.5 * group(y, p + "norm2b")
        else:
            x = x + y
            h = _layer_norm(x, w(p + "norm2"))
            y = F.gelu(h @ w(p + "mlp.gate").T, approximate="tanh") * (h @ w(p + "mlp.up").T)
            x = x + y @ w(p + "mlp.down").T
    x = x[torch.tensor([at + n - 1 for at, n, *_ in step.seqs], device=DEV)]
    x = group(x, "final.norm") if tativik else _layer_norm(x, w("final.norm"))
    logits = x @ w("head").T
    return {"logits": logits if tativik else 30.0 * torch.tanh(logits / 30.0), "caches": caches}
