"""What is measured of this framework's inference path: whole requests through its public entry points.

A state is what a serving program has in hand before a request: a device context with the weights of one of the
repository's configurations (kept for as long as the process lives, shared by the requests of that configuration, as
such a program shares it) and the token ids of the request, made from the seed alone.  A pass is the whole request:
every sequence starts empty, its prompt is processed, tokens are produced.

  generate  one prompt, greedy tokens after it, on one sequence: the reference's token loop (Device.generate).  The
            answer is the token ids.
  serve     several sequences at once: ragged prompts in one prefill call, then greedy steps for all of them
            (prefill_batch, greedy_token, decode_loop).  The answer is the token ids.
  stream    several sequences, one call per step, each fed a token that the caller chose (decode_step: a caller that
            streams, samples on the host or scores a continuation).  The answer is the last logits.
  prefill   prompts only: the time to the first token (prefill_batch, then the logits a caller picks from).
  score     logits and probabilities of every position of a text, and its loss (forward_full).

Models: the five benchmark configurations and the reference's compiled-in shape ("ref"), at full size; weights
N(0, 0.02), gains 1, gate biases N(0, 1); uniform random token ids.  `draw` spreads lengths, sequence counts and steps
over what those contexts hold.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

NAME = "mini_llm_cuda_amd"


def _package():
    if NAME not in sys.modules:
        pkg = os.path.join(os.getcwd(), "mini-llm-cuda_amd")
        spec = importlib.util.spec_from_file_location(NAME, os.path.join(pkg, "__init__.py"), submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[NAME] = mod
        try:
            spec.loader.exec_module(mod)
        except Exception:
            del sys.modules[NAME]
            raise
    return sys.modules[NAME]


def listed():
    return [
        # the smallest request: a few tokens of the tiny model, nothing but latency and host work
        {"name": "tiny-short", "task": "generate", "model": "1", "prompt": 5, "new": 12},
        # batch-1 generation at the sizes the configurations state: attention-only, hybrid, the reference's own shape
        {"name": "attn-generate", "task": "generate", "model": "2", "prompt": 64, "new": 512},
        {"name": "hybrid-generate", "task": "generate", "model": "3", "prompt": 128, "new": 384},
        {"name": "ref-generate", "task": "generate", "model": "ref", "prompt": 256, "new": 192},
        # a handful, a middling odd number and a full house of concurrent fp32 sequences, ragged prompts
        {"name": "hybrid-serve5", "task": "serve", "model": "4", "seqs": 5, "shortest": 20, "longest": 205, "steps": 48},
        {"name": "hybrid-serve19", "task": "serve", "model": "4", "seqs": 19, "shortest": 32, "longest": 333, "steps": 48},
        {"name": "hybrid-serve64", "task": "serve", "model": "4", "seqs": 64, "shortest": 32, "longest": 512, "steps": 64},
        # the large bf16 model: one stream, all eight, a single odd prompt, the whole prefill batch
        {"name": "large-stream1", "task": "stream", "model": "5", "seqs": 1, "shortest": 300, "longest": 300, "steps": 32},
        {"name": "large-stream8", "task": "stream", "model": "5", "seqs": 8, "shortest": 100, "longest": 900, "steps": 24},
        {"name": "large-prefill1", "task": "prefill", "model": "5", "seqs": 1, "shortest": 777, "longest": 777},
        {"name": "large-prefill8", "task": "prefill", "model": "5", "seqs": 8, "shortest": 2048, "longest": 2048},
        # scoring a text of the reference's own shape at every position
        {"name": "ref-score", "task": "score", "model": "ref", "tokens": 517},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    task = rng.choice(["generate", "generate", "serve", "serve", "stream", "prefill", "score"])
    if task == "generate":
        model = rng.choice(["1", "2", "3", "ref"])
        most, new = {"1": (144, 128), "2": (576, 512), "3": (768, 512), "ref": (640, 240)}[model]
        prompt = _log(rng, 2, most // 2)
        return {"task": task, "model": model, "prompt": prompt, "new": _log(rng, 8, min(new, most - prompt))}
    if task == "serve":
        longest = _log(rng, 24, 512)
        return {"task": task, "model": "4", "seqs": _log(rng, 2, 64), "shortest": _log(rng, 8, longest), "longest": longest,
                "steps": _log(rng, 12, 64)}
    if task == "stream":
        longest = _log(rng, 24, 1200)
        return {"task": task, "model": "5", "seqs": rng.randint(1, 8), "shortest": _log(rng, 8, longest), "longest": longest,
                "steps": _log(rng, 12, 32)}
    if task == "prefill":
        model = rng.choice(["4", "5", "5"])
        longest = _log(rng, 48, 512 if model == "4" else 2048)
        return {"task": task, "model": model, "seqs": _log(rng, 1, 64) if model == "4" else rng.randint(1, 8),
                "shortest": _log(rng, 17, longest), "longest": longest}
    return {"task": task, "model": rng.choice(["2", "ref"]), "tokens": _log(rng, 24, 570)}


# --------------------------------------------------------------------------------------------------------------------
# contexts
# --------------------------------------------------------------------------------------------------------------------
_contexts = {}


def _hparams(model):
    m = _package()
    return m.reference_defaults() if model == "ref" else m.config(int(model))


def _tensors(m, hp):
    """(layer, tensor id, shape, kind) of every tensor a context of these hyper-parameters needs."""
    d, F, V, p = hp.dim, hp.ffnDim, hp.vocabSize, hp.pleDim
    out = [(0, m.T_TOKEN_EMBEDDINGS, (V, d), "w"), (0, m.T_FINAL_RMS_GAMMA, (d,), "1")]
    for layer in range(hp.transformers):
        attn = hp.layerKinds[layer] == m.KIND_ATTENTION
        qk, vv = (d, d) if attn else (hp.gdnHeads * hp.gdnDk, hp.gdnHeads * hp.gdnDv)
        out += [(layer, m.T_RMS_GAMMA, (d,), "1"), (layer, m.T_QUERY, (qk, d), "w"), (layer, m.T_KEY, (qk, d), "w"),
                (layer, m.T_VALUE, (vv, d), "w"), (layer, m.T_OUTPUT_PROJ, (d, vv), "w"), (layer, m.T_RMS_GAMMA2, (d,), "1"),
                (layer, m.T_FFN_1A, (F, d), "w"), (layer, m.T_FFN_1B, (F, d), "w"), (layer, m.T_FFN_2, (d, F), "w")]
        if attn and hp.qkRmsNorm:
            out += [(layer, m.T_QUERY_RMS_GAMMA, (d,), "1"), (layer, m.T_KEY_RMS_GAMMA, (d,), "1")]
        if attn and hp.queryGating:
            out += [(layer, m.T_GATED_QUERY, (d, d), "w")]
        if not attn:
            out += [(layer, m.T_GDN_ALPHA_W, (hp.gdnHeads, d), "w"), (layer, m.T_GDN_ALPHA_B, (hp.gdnHeads,), "n"),
                    (layer, m.T_GDN_BETA_W, (hp.gdnHeads, d), "w"), (layer, m.T_GDN_BETA_B, (hp.gdnHeads,), "n")]
        if p:
            out += [(layer, m.T_PLE_TABLE, (V, p), "w"), (layer, m.T_PLE_GATE, (p, d), "w"), (layer, m.T_PLE_UP, (d, p), "w")]
    return out


def _context(model):
    if model not in _contexts:
        m, hp = _package(), _hparams(model)
        dev = m.Device(hp, 0)
        gen = torch.Generator(device="cuda:0")
        gen.manual_seed(100 + len(model))
        for layer, tid, shape, kind in _tensors(m, hp):
            if kind == "1":
                t = torch.ones(shape)
            else:
                t = (torch.randn(shape, device="cuda:0", generator=gen) * (0.02 if kind == "w" else 1.0)).cpu()
            dev.upload_tensor(layer, tid, t.numpy())
        dev.upload_rope(m.rope_table(hp.maxL, hp.headDim, hp.ropeDenomBase))
        dev.finalize()
        torch.cuda.empty_cache()
        _contexts[model] = dev
    return _contexts[model]


# --------------------------------------------------------------------------------------------------------------------
# requests
# --------------------------------------------------------------------------------------------------------------------
def _lengths(case):
    """Prompt lengths of a case's sequences: from the shortest to the longest, dealt in a scattered order."""
    n, lo, hi = case["seqs"], case["shortest"], case["longest"]
    if n == 1:
        return [hi]
    return [lo + (hi - lo) * ((i * 7 + 3) % n) // (n - 1) for i in range(n)] if n % 7 else [lo + (hi - lo) * i // (n - 1) for i in range(n)]


def prepare(case, seed):
    dev = _context(case["model"])
    rng = np.random.default_rng([int(seed), 17])
    V = dev.hp.vocabSize

    def ids(*shape):
        return rng.integers(0, V, size=shape, dtype=np.int32)

    s = {"task": case["task"], "dev": dev}
    if case["task"] == "generate":
        s.update(prompt=ids(case["prompt"]), new=case["new"])
    elif case["task"] == "score":
        s.update(text=ids(case["tokens"]))
    else:
        s.update(seqs=list(range(case["seqs"])), prompts=[ids(n) for n in _lengths(case)])
        if case["task"] == "serve":
            s.update(steps=case["steps"])
        elif case["task"] == "stream":
            s.update(feed=ids(case["steps"], case["seqs"]))
    return s


def run(s):
    dev, task = s["dev"], s["task"]
    if task == "generate":
        return dev.generate(s["prompt"], s["new"])[0]
    dev.reset()
    if task == "score":
        logits, probs, nll = dev.forward_full(0, s["text"])
        return {"logits": logits, "probs": probs, "nll": nll}
    dev.prefill_batch(s["seqs"], s["prompts"])
    if task == "prefill":
        return np.stack([dev.logits(q) for q in s["seqs"]])
    if task == "serve":
        first = [dev.greedy_token(q) for q in s["seqs"]]
        return {"first": np.array(first, dtype=np.int32), "rest": dev.decode_loop(first, s["steps"])}
    for last in s["feed"]:
        dev.decode_step(last)
    return np.stack([dev.logits(q) for q in s["seqs"]])


# --------------------------------------------------------------------------------------------------------------------
# what a request cannot do without
# --------------------------------------------------------------------------------------------------------------------
def _matrices(m, hp):
    """Weight-matrix elements one token multiplies on its way through the stack (LM head and tables excluded)."""
    d, F, total = hp.dim, hp.ffnDim, 0
    for t in range(hp.transformers):
        if hp.layerKinds[t] == m.KIND_ATTENTION:
            total += 4 * d * d + 3 * d * F + (d * d if hp.queryGating else 0)
        else:
            total += 2 * hp.gdnHeads * hp.gdnDk * d + 2 * hp.gdnHeads * hp.gdnDv * d + 3 * d * F + 2 * hp.gdnHeads * d
        total += 2 * hp.pleDim * d
    return total


def work(case):
    m, hp = _package(), _hparams(case["model"])
    wb = 2 if hp.weightDtype == m.DTYPE_BF16 else 4
    d, V = hp.dim, hp.vocabSize
    n_attn = sum(1 for t in range(hp.transformers) if hp.layerKinds[t] == m.KIND_ATTENTION)
    n_gdn = hp.transformers - n_attn
    mats, head = _matrices(m, hp), V * d
    state = n_gdn * hp.gdnHeads * hp.gdnDk * hp.gdnDv
    if case["task"] == "generate":
        lens, steps = [case["prompt"]], case["new"] - 1
    elif case["task"] == "score":
        lens, steps = [case["tokens"]], 0
    else:
        lens, steps = _lengths(case), case.get("steps", 0)
    rows, nseq = sum(lens), len(lens)
    heads = rows if case["task"] == "score" else nseq  # positions of the prompts whose logits are wanted
    # prompts: weights once, K and V rows and GDN states written; causal attention over the prompt
    nbytes = wb * (mats + head) + 2 * 4 * d * n_attn * rows + 4 * state * nseq + (4 * V * nseq if steps == 0 else 0)
    flops = 2.0 * mats * rows + 2.0 * head * heads + sum(2.0 * n_attn * d * n * n for n in lens) + 6.0 * state * rows
    if case["task"] == "score":
        nbytes += 2 * 4 * V * rows  # logits and probabilities of every position (the one row above is among them)
    # steps: weights once each, every sequence's K and V rows read and one row written, states read and written
    for i in range(steps):
        kv = sum(n + i + 1 for n in lens)
        nbytes += wb * (mats + head) + 2 * 4 * d * n_attn * (kv + nseq) + 2 * 4 * state * nseq
        flops += 2.0 * (mats + head) * nseq + 4.0 * n_attn * d * kv + 6.0 * state * nseq
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    if case["task"] in ("generate", "serve"):
        return {"differ": 0.01}  # token ids; two correct fp32 sums part only where two logits all but tie
    if case["model"] == "5":
        return {"rel": 1e-2}  # bf16 weights, half activations
    return {"rel": 2e-5}  # logits of 12 to 16 fp32 layers
