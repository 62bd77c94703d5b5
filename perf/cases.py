"""The work this framework is timed on: its public calls, as a program that serves, scores or exports a model makes them.

Two model families go through it. The int8 step (``Yggdrasil`` on a YGG1 file) reads, scores and generates token
streams; the float step (``FloatYggdrasil`` on a checkpoint) serves an unquantised model in f32 and, in f64, gives the
calibration maxima of the int8 export. The shapes are the reference's trained ones (5 layers, block 16, router depth 10:
small, medium and large by state width, readout rank and layer-input rank), the batch-4096 configuration ("c4", 3.6 GB)
and the five-symbol DNA configuration ("c3", state width 96).

A case's "kind" is the call:

  step         ``Yggdrasil.step``: one token for each of ``streams`` streams, states carried (interactive serving)
  read         ``Yggdrasil.run`` of one known stream and ``softmax`` of its logits (the reference's time mode)
  run          ``Yggdrasil.run``: ``tokens`` tokens of each stream, all logits (prompts, batch evaluation)
  score        ``Yggdrasil.score``: bits of host windows, end to end
  generate     ``Yggdrasil.generate``: host prompts, ``tokens`` sampled tokens each, with their logits
  float_step   ``FloatYggdrasil.step`` in f32
  float_run    ``FloatYggdrasil.run`` in f32
  float_score  ``FloatYggdrasil.score`` in f32 of host windows, end to end
  calibrate    ``FloatYggdrasil.run`` in f64 with the calibration maxima (the export's pass over its windows)

A program loads its model once, so the loaded models are kept here between calls (the two used last); what a seed
changes is the tokens, the states and the sampling.
"""
import functools
import math
import os
import tempfile

import numpy as np
import torch

from yggdrasil_amd import float_model, synth
from yggdrasil_amd.inference import Yggdrasil

# state width, readout rank, layer-input rank, input rank of the trained shapes
SHAPES = {"small": (64, 8, 16, 32), "medium": (128, 16, 32, 32), "large": (256, 32, 64, 64)}
DEPTH, LAYERS, VOCAB, TOKEN_DIM, BLOCK = 10, 5, 256, 16, 16
FLOAT_KINDS = ("float_step", "float_run", "float_score", "calibrate")


def listed():
    return [
        # one interactive stream, the smallest call: a launch and its host path
        dict(name="step_small_b1", kind="step", shape="small", scales="tensor", streams=1, tokens=1),
        # a server's step over the requests in flight
        dict(name="step_medium_b48", kind="step", shape="medium", scales="tensor", streams=48, tokens=1),
        # reading one document on the published model's shape, with the time mode's softmax; an odd length
        dict(name="read_large_t1001", kind="read", shape="large", scales="tensor", streams=1, tokens=1001),
        # prompts of a batch on a model exported with factored storage (the small file)
        dict(name="run_factored_b60_t250", kind="run", shape="medium", scales="tensor", storage="factored", streams=60,
             tokens=250),
        # evaluation windows of DNA, host tokens to bits
        dict(name="score_c3_b700_t513", kind="score", shape="c3", scales="tensor", streams=700, tokens=513),
        # the headline batch: 4096 streams of 1024 tokens, the largest
        dict(name="run_c4_b4096_t1024", kind="run", shape="c4", scales="tensor", storage="table", streams=4096,
             tokens=1024),
        # one user's completion
        dict(name="generate_medium_b1", kind="generate", shape="medium", scales="tensor", streams=1, prompt=48,
             tokens=200, temperature=0.8, top_k=20),
        # completions of a batch of users, on a model exported with group scales; greedy
        dict(name="generate_group_b96", kind="generate", shape="small", scales="group", streams=96, prompt=33,
             tokens=100, temperature=0.0, top_k=0),
        # one interactive stream of an unquantised checkpoint
        dict(name="float_step_large_b1", kind="float_step", shape="large", streams=1, tokens=1),
        # prompts of a batch on a checkpoint
        dict(name="float_run_medium_b9", kind="float_run", shape="medium", streams=9, tokens=100),
        # validation bits of a checkpoint after training
        dict(name="float_score_large_b256", kind="float_score", shape="large", streams=256, tokens=129),
        # the export's calibration over its windows
        dict(name="calibrate_medium_b500", kind="calibrate", shape="medium", streams=500, tokens=200),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of one of the kinds, its sizes spread over the logarithm of the kind's range."""
    kind = rng.choice(["step", "step", "read", "run", "run", "score", "generate", "generate", *FLOAT_KINDS])
    c = dict(kind=kind, shape=rng.choice(list(SHAPES)))
    if kind not in FLOAT_KINDS:
        c["scales"] = rng.choice(["tensor", "tensor", "group"])
    if kind in ("step", "float_step"):
        c.update(streams=_log_int(rng, 1, 2048 if kind == "step" else 512), tokens=1)
    elif kind == "read":
        c.update(streams=1, tokens=_log_int(rng, 100, 2000))
    elif kind == "run":
        c.update(storage=rng.choice(["table", "factored"]), streams=_log_int(rng, 8, 1000),
                 tokens=_log_int(rng, 50, 500))
    elif kind == "score":
        if rng.random() < 0.5:
            c.update(shape="c3", scales="tensor")
        c.update(streams=_log_int(rng, 20, 1000), tokens=_log_int(rng, 100, 700))
    elif kind == "generate":
        c.update(streams=rng.choice([1, _log_int(rng, 2, 256)]), prompt=_log_int(rng, 4, 200),
                 tokens=_log_int(rng, 20, 200), temperature=rng.choice([0.0, 0.8, 1.0]), top_k=rng.choice([0, 20]))
    elif kind == "float_run":
        # (at most about 1000 stream steps, see tolerance)
        c.update(streams=_log_int(rng, 1, 32))
        c.update(tokens=_log_int(rng, 16, min(200, 1024 // c["streams"])))
    elif kind == "float_score":
        c.update(streams=_log_int(rng, 16, 256), tokens=_log_int(rng, 32, 129))
    else:
        c.update(streams=_log_int(rng, 64, 500), tokens=_log_int(rng, 64, 200))
    return c


# ------------------------------------------------------------------------------------------------------ models
def _int8_spec(shape, scales, storage):
    if shape == "c4":
        return synth.C4, 3
    if shape == "c3":
        return synth.C3, 2
    n, R, R2, K = SHAPES[shape]
    return synth.ModelSpec(n, BLOCK, DEPTH, VOCAB, LAYERS, R, R2, input_rank=K if storage == "factored" else 0,
                           group=scales == "group", router="gauss"), 5


@functools.lru_cache(maxsize=2)
def _int8_model(shape, scales, storage):
    spec, seed = _int8_spec(shape, scales, storage)
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "model.bin")
        synth.write_model(spec, seed, path)
        return Yggdrasil.load(path)


@functools.lru_cache(maxsize=2)
def _checkpoint(shape):
    """A random checkpoint's arrays by their flat keys: decays in [0.6, 1), small rotation generators, as the
    framework's own random checkpoints are distributed."""
    n, R, R2, K = SHAPES[shape]
    rng = np.random.default_rng(5)
    out = {}
    for l in range(LAYERS):
        E = 2 ** DEPTH if l else VOCAB
        pre = f"routed_layers/{l - 1}/" if l else "token_layer/"
        p = {"token_embed": rng.normal(0, 1.0, (VOCAB, K)), "input_proj": rng.normal(0, 0.3 / math.sqrt(K), (E, n, K)),
             "bias": rng.normal(0, 0.1, (E, n)), "readout": rng.normal(0, 1 / math.sqrt(n), (E, R, n)),
             "unembed": rng.normal(0, 1 / math.sqrt(R), (VOCAB, R)),
             "rotation": rng.normal(0, 0.3, (E, n // BLOCK, BLOCK, BLOCK)), "decay": rng.uniform(0.6, 1.0, (E, n))}
        if l:
            p["router_embed"] = rng.normal(0, 1.0, (VOCAB, TOKEN_DIM))
            p["router_weight"] = rng.normal(0, 1 / math.sqrt(TOKEN_DIM + n), (E - 1, TOKEN_DIM + n))
            p["router_bias"] = rng.normal(0, 0.1, E - 1)
            p["layer_input_down"] = rng.normal(0, 1 / math.sqrt(n), (R2, n))
            p["layer_input_proj"] = rng.normal(0, 0.3 / math.sqrt(R2), (E, n, R2))
        out.update({pre + k: v.astype(np.float32) for k, v in p.items()})
    out["output_bias"] = rng.normal(0, 0.1, VOCAB).astype(np.float32)
    return out


@functools.lru_cache(maxsize=2)
def _float_model(shape, precision):
    raw, bias = float_model.from_params(_checkpoint(shape))
    return float_model.FloatYggdrasil(float_model.float_layers(raw, blas=True), bias, precision=precision)


# ------------------------------------------------------------------------------------------------------ inputs
def _generator(seed):
    return torch.Generator("cuda").manual_seed(1000003 * (seed + 1) % (1 << 31))


def _tokens(case, seed, width):
    """(streams, width) int32 on the GPU: Zipf(1.1) bytes, or the DNA configuration's four even symbols and a rare
    fifth."""
    if case["shape"] == "c3":
        p = torch.tensor([0.24975] * 4 + [0.001], dtype=torch.float64, device="cuda")
    else:
        p = torch.arange(1, VOCAB + 1, dtype=torch.float64, device="cuda") ** -1.1
    cum = torch.cumsum(p / p.sum(), 0)
    u = torch.rand(case["streams"], width, dtype=torch.float64, device="cuda", generator=_generator(seed))
    return torch.searchsorted(cum, u).clamp_(max=len(p) - 1).to(torch.int32)


def _float_state(case, seed):
    """A carried float state: the spread the recurrence settles at (about 0.6 per coordinate)."""
    n = SHAPES[case["shape"]][0]
    g = _generator(seed + 7)
    return 0.6 * torch.randn(case["streams"], LAYERS, n, dtype=torch.float32, device="cuda", generator=g)


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind in FLOAT_KINDS:
        s["model"] = _float_model(case["shape"], 64 if kind == "calibrate" else 32)
        x = _tokens(case, seed, case["tokens"])
        if kind == "float_step":
            s["tokens"], s["state"] = x[:, 0].contiguous(), _float_state(case, seed)
        else:
            s["tokens"] = x if kind == "float_run" else x.cpu().numpy()
        return s
    s["model"] = m = _int8_model(case["shape"], case["scales"], case.get("storage", "table"))
    if kind == "step":
        x = _tokens(case, seed, 17)
        s["state"], s["tokens"] = m.run(x[:, :16].contiguous(), logits=False)["state"], x[:, 16].contiguous()
    elif kind in ("read", "run"):
        s["tokens"] = _tokens(case, seed, case["tokens"])
    elif kind == "score":
        s["tokens"] = _tokens(case, seed, case["tokens"]).cpu().numpy()
    else:
        s["tokens"], s["seed"] = _tokens(case, seed, case["prompt"]).cpu().numpy(), seed
    return s


def run(state):
    case, m, x = state["case"], state["model"], state["tokens"]
    kind = case["kind"]
    if kind in ("step", "float_step"):
        logits, new = m.step(x, state["state"])
        return {"logits": logits, "state": new}
    if kind == "read":
        r = m.run(x)
        p, lse = m.softmax(r["logits"])
        return {"logits": r["logits"], "state": r["state"], "probs": p, "lse": lse}
    if kind in ("run", "float_run"):
        r = m.run(x)
        return {"logits": r["logits"], "state": r["state"]}
    if kind in ("score", "float_score"):
        return {"bits": m.score(x)}
    if kind == "generate":
        text, logits = m.generate(x, case["tokens"], temperature=case["temperature"], top_k=case["top_k"],
                                  seed=state["seed"], return_logits=True)
        return {"text": text, "logits": logits}
    r = m.run(x, logits=False, stats=True)
    return {"state": r["state"], "stats": r["stats"]}


# ------------------------------------------------------------------------------------------------------ measures
def _shape_of(case):
    """(n, R, R2, K, depth, layers, vocab)."""
    if case["shape"] in SHAPES:
        return (*SHAPES[case["shape"]], DEPTH, LAYERS, VOCAB)
    sp = synth.C4 if case["shape"] == "c4" else synth.C3
    return sp.d_state, sp.readout_rank, sp.layer_input_rank, 0, sp.router_depth, sp.n_layers, sp.vocab


def _distinct(total, draws):
    """Expected number of distinct items among uniform draws."""
    return total * -math.expm1(draws * math.log1p(-1 / total)) if total > 1 else 1.0


def work(case):
    """Bytes: each distinct weight that the tokens' routes touch read once, tokens and states read, results written.
    Operations: two per product term of the step."""
    n, R, R2, K, D, L, V = _shape_of(case)
    kind, B = case["kind"], case["streams"]
    per = case["tokens"] + case.get("prompt", 1) - 1
    if kind in ("score", "float_score"):
        per = case["tokens"] - 1
    N, E = B * per, 2 ** D
    wide = {"calibrate": 8}.get(kind, 4) if kind in FLOAT_KINDS else 1
    entry = wide if kind in FLOAT_KINDS else 2            # transition and table entries
    F = TOKEN_DIM if kind in FLOAT_KINDS else 0
    weights = V * R * wide * L + _distinct(V, N) * (n * BLOCK * entry + n * entry + R * n * wide)
    leaf = n * BLOCK * entry + (n * R2 + R * n) * wide
    leaves = _distinct(E, N)
    if case.get("storage") == "factored":
        rows = leaves * n * (K + 2) + V * K
    else:
        rows = _distinct(E * V, N) * n * entry
    nodes = sum(_distinct(2 ** d, N) for d in range(D))
    node = (F + n) * wide + (wide if F else 0)
    thresholds = 0 if F else 4 * sum(_distinct(2 ** d * V, N) for d in range(D))
    weights += (L - 1) * (leaves * leaf + rows + nodes * node + thresholds + R2 * n * wide + V * F * wide)
    state = B * L * n * wide
    out = state
    if kind in ("step", "read", "run", "float_step", "float_run"):
        out += N * V * 4
    if kind == "read":
        out += N * (V + 1) * 4
    if kind == "generate":
        out += B * case["tokens"] * (V + 1) * 4
    if kind in ("score", "float_score"):
        out = B * 8
    given = N * (8 if kind in ("score", "float_score") else 4) + (state if kind in ("step", "float_step") else 0)
    macs = L * (n * BLOCK + R * n + V * R) + (L - 1) * (D * (n + F) + 2 * n * R2)
    if case.get("storage") == "factored":
        macs += (L - 1) * n * K
    return {"bytes": weights + given + out, "flops": 2 * N * macs}


def tolerance(case):
    # int8: integer sums and f32 operations in a fixed order, equal to the reference's to the bit
    kind = case["kind"]
    if kind not in FLOAT_KINDS:
        return "exact"
    # f64 sums of up to 272 terms over the recurrence: 1.8e-15 and 1.6e-14 from exact()
    if kind == "calibrate":
        return {"rel": 1e-14, "max": 1e-13}
    # A router score within f32 rounding of 0 turns the other way in another summation order, in about one of 2e5
    # stream steps, and the stream's next logits are another leaf's. One such turn moved a row of bits by 0.014 of its
    # value at most, and all rows by 9e-4 (12 runs of 33k stream steps, 3 with a turn); without one 7e-9 and 2e-8.
    if kind == "float_score":
        return {"rel": 4e-3, "max": 0.06}
    # f32 sums of up to 272 terms through five layers and the recurrence: 2.9e-7 and 1.9e-6 from exact(); these cases
    # are at most about 1000 stream steps, so that hardly any meets a turn, which no bound on logits would hold
    return {"rel": 1.2e-6, "max": 8e-6}


def exact(case, seed):
    """The float step in 64 bits. The int8 results have no such value: they are whole numbers rounded at f32 steps that
    the file format fixes, and are compared bit for bit. Nor have the bits of tens of thousands of f32 stream steps,
    some of which turn otherwise at a router score near 0 (tolerance)."""
    kind = case["kind"]
    if kind not in FLOAT_KINDS or kind == "float_score":
        return None
    s = prepare(case, seed)
    x = torch.as_tensor(s["tokens"], device="cuda").long().reshape(case["streams"], -1)
    p = {k: torch.as_tensor(v, device="cuda").double() for k, v in _checkpoint(case["shape"]).items()}
    n, R, R2, K = SHAPES[case["shape"]]
    B, T = x.shape
    layers = []
    for l in range(LAYERS):
        y = {k.rsplit("/", 1)[1]: v for k, v in p.items() if k.startswith(f"routed_layers/{l - 1}/" if l else
                                                                           "token_layer/")}
        g = y["rotation"]
        y["A"] = y["decay"].reshape(*g.shape[:3], 1) * torch.linalg.matrix_exp(0.5 * (g - g.transpose(-1, -2)))
        layers.append(y)
    h = s["state"].double().clone() if "state" in s else torch.zeros(B, LAYERS, n, dtype=torch.float64, device="cuda")
    stats = torch.zeros(LAYERS, 3 + n // 16 + R, dtype=torch.float64, device="cuda")
    logits = []

    def times(m, v):                                      # (B, i, j) (B, j) -> (B, i)
        return (m * v[:, None, :]).sum(-1)

    for t in range(T):
        xt, below = x[:, t], None
        lg = p["output_bias"].expand(B, VOCAB).clone()
        for l, y in enumerate(layers):
            r = xt
            if l:
                f = torch.cat([y["router_embed"][xt], below], -1)
                node = torch.zeros_like(xt)
                for _ in range(DEPTH):
                    node = 2 * node + 1 + ((f * y["router_weight"][node]).sum(-1) + y["router_bias"][node] > 0)
                r = node - (2 ** DEPTH - 1)
            new = times(y["input_proj"][r], y["token_embed"][xt]) + y["bias"][r]
            if l:
                zl = below @ y["layer_input_down"].T
                new = new + times(y["layer_input_proj"][r], zl)
                stats[l, 1] = torch.maximum(stats[l, 1], zl.abs().max())
            old = h[:, l].reshape(B * n // BLOCK, BLOCK)
            new = new + times(y["A"][r].reshape(-1, BLOCK, BLOCK), old).reshape(B, n)
            z = times(y["readout"][r], new)
            h[:, l] = new
            below = new / torch.sqrt((new * new).mean(-1, keepdim=True) + 1e-6)
            lg = lg + z @ y["unembed"].T
            if kind == "calibrate":
                a, az = new.abs(), z.abs()
                stats[l] = torch.maximum(stats[l], torch.cat([
                    a.max().reshape(1), stats[l, 1:2], az.max().reshape(1),
                    a.reshape(B, n // 16, 16).amax((0, 2)), az.amax(0)]))
        if kind != "calibrate":
            logits.append(lg)
    if kind == "calibrate":
        return {"state": h, "stats": stats}
    return {"logits": logits[0] if kind == "float_step" else torch.stack(logits, 1), "state": h}
