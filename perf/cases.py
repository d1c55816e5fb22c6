"""The work a program built on this package has it do, as cases that can be timed
and compared: the Hyena mixers at decode, speculative verify and prefill, the fp8
projections, the attention layers, and a four-layer model (one layer of each
kind) at decode and prefill.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a program has in hand before the call, on the GPU
  run(state)           one pass through the public entry points, its outputs
  work(case)           bytes and flops that a pass cannot do without
  tolerance(case)      how far another correct implementation may be off
  exact(case, seed)    what run() returns, in 64 bits and plain torch

Decode and verify steps have fixed shapes and run as one HIP graph replay, as a
serving program runs them; prefill steps and single projections are eager calls.
A mixer case runs one layer of each kind (hcs, hcm, hcl), the three in equal
number in the released layer maps, each on its own hidden rows.
"""

import itertools
import math

import torch

from evo2_flash_amd.attention import PAGE
from evo2_flash_amd.config import HyenaConfig
from evo2_flash_amd.fp8 import Fp8StaticLinear
from evo2_flash_amd.fp8_emul import static_fp8_linear_emulated
from evo2_flash_amd.metadata import HyenaMamba2Metadata, build_metadata
from evo2_flash_amd.mixers import load_mixer_params, make_mixer, set_forward_context
from evo2_flash_amd.model import Evo2Attention, Evo2DecodeModel
from evo2_flash_amd.state import HyenaStatePool
from evo2_flash_amd.synthetic import mixer_params, quantize_weight_e4m3

DEV = "cuda"
BF16 = torch.bfloat16
KINDS = ("hcs", "hcm", "hcl")
ROPE_THETA, ROPE_FACTOR = 10000.0, 128.0
EPS = 1e-6
VOCAB = 512
# hidden size -> MLP width of the 1B, 7B and 40B configurations
INTERMEDIATE = {1920: 5120, 4096: 11264, 8192: 22528}
_names = itertools.count()


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one sequence generating, 7B shape: the smallest step, launches and latency
        {"name": "mixers_decode_1", "path": "mixers_decode", "hidden": 4096, "batch": 1},
        # the benchmark's decode batch
        {"name": "mixers_decode_64", "path": "mixers_decode", "hidden": 4096, "batch": 64},
        # speculative verify: 64 requests of up to 3 drafts and their anchor token
        {"name": "mixers_verify_64", "path": "mixers_verify", "hidden": 4096, "requests": 64,
         "drafts": 3},
        # one odd-length prompt through 1B-shaped mixers
        {"name": "mixers_prefill_1b_2047", "path": "mixers_prefill", "hidden": 1920,
         "tokens": 2047, "segments": 1, "resumed": 0},
        # a scheduler step of several ragged prompts, two of them continued
        {"name": "mixers_prefill_ragged", "path": "mixers_prefill", "hidden": 4096,
         "tokens": 6001, "segments": 7, "resumed": 2},
        # the benchmark's long prompt, 7B shape: the largest
        {"name": "mixers_prefill_32k", "path": "mixers_prefill", "hidden": 4096,
         "tokens": 32768, "segments": 1, "resumed": 0},
        # one fp8 projection over a chunk of prompt, 7B in_proj
        {"name": "fp8_linear_777", "path": "fp8_linear", "tokens": 777, "inputs": 4096,
         "outputs": 12288},
        # an FP8-surgery layer's projection (Hopper accumulation, bit for bit)
        {"name": "fp8_emulated_300", "path": "fp8_emulated", "tokens": 300, "inputs": 4096,
         "outputs": 12288},
        # an attention layer over a long prompt, 7B shape
        {"name": "attention_prefill_16k", "path": "attention_prefill", "hidden": 4096,
         "sequences": 1, "tokens": 16384},
        # an attention layer at decode, batch 8 at ragged positions up to 8k
        {"name": "attention_decode_8", "path": "attention_decode", "hidden": 4096, "batch": 8,
         "context": 8192, "shared": 0},
        # a whole small model's decode step at the batch of the published step time
        {"name": "model_decode_8", "path": "model_decode", "hidden": 4096, "batch": 8,
         "context": 4096},
        # a whole small model over a prompt of odd length
        {"name": "model_prefill_3001", "path": "model_prefill", "hidden": 4096, "sequences": 1,
         "tokens": 3001},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(("mixers_decode", "mixers_verify", "mixers_prefill", "mixers_prefill",
                       "fp8_linear", "fp8_emulated", "attention_prefill", "attention_decode",
                       "model_decode", "model_prefill"))
    hidden = rng.choice((1920, 4096, 4096, 8192))
    if path == "mixers_decode":
        return {"path": path, "hidden": hidden, "batch": _log(rng, 1, 128)}
    if path == "mixers_verify":
        drafts = rng.randint(1, 7)
        return {"path": path, "hidden": min(hidden, 4096), "requests": _log(rng, 1, 256 // (drafts + 1)),
                "drafts": drafts}
    if path == "mixers_prefill":
        tokens = _log(rng, 40, {1920: 32768, 4096: 32768, 8192: 8192}[hidden])
        segments = rng.randint(1, min(8, tokens // 8))
        return {"path": path, "hidden": hidden, "tokens": tokens, "segments": segments,
                "resumed": rng.randint(0, segments)}
    if path in ("fp8_linear", "fp8_emulated"):
        outputs = rng.choice((hidden, 3 * hidden, 3 * hidden))
        most = 8192 if path == "fp8_linear" else max(2, 400 * 4096 * 12288 // (hidden * outputs))
        return {"path": path, "tokens": _log(rng, 1, min(most, 8192)), "inputs": hidden,
                "outputs": outputs}
    if path == "attention_prefill":
        sequences = rng.randint(1, 4)
        return {"path": path, "hidden": hidden, "sequences": sequences,
                "tokens": _log(rng, 50, int(16384 / sequences ** 0.5 / max(1, hidden // 4096)))}
    if path == "attention_decode":
        batch = _log(rng, 1, 64)
        context = _log(rng, 60, min(16384, 8 * 16384 * 4096 // (batch * hidden)))
        shared = rng.choice((0, 0, 1)) * (context // 2 // PAGE) * PAGE
        return {"path": path, "hidden": hidden, "batch": batch, "context": context,
                "shared": shared if batch > 1 else 0}
    hidden = min(hidden, 4096)
    if path == "model_decode":
        batch = _log(rng, 1, 64)
        return {"path": path, "hidden": hidden, "batch": batch,
                "context": _log(rng, 60, min(8192, 8 * 16384 // batch))}
    sequences = rng.randint(1, 3)
    return {"path": path, "hidden": hidden, "sequences": sequences,
            "tokens": _log(rng, 50, 3000 // sequences)}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) % (1 << 40))


def _ints(seed):
    return torch.Generator().manual_seed(int(seed) % (1 << 40) + 7)


def _config(hidden, layers=3):
    return HyenaConfig(hidden_size=hidden, num_hidden_layers=layers,
                       num_attention_heads=hidden // 128, intermediate_size=INTERMEDIATE[hidden],
                       vocab_size=VOCAB, hcs_layer_idxs=[0], hcm_layer_idxs=[1],
                       hcl_layer_idxs=[2], attn_layer_idxs=[3] if layers > 3 else [],
                       rms_norm_eps=EPS, use_fp8_input_projections=True)


def _rows(n, hidden, g):
    """RMS-normalised activations, what a pre-norm hands to a layer."""
    return torch.randn(n, hidden, generator=g, device=DEV).to(BF16)


def _fill_pool(pool, g):
    """States a prefill leaves: bf16-valued windows, fp32 recurrence states."""
    conv, inner, ssm = pool.kv_cache
    conv.copy_(torch.randn(conv.shape, generator=g, device=DEV))
    inner.copy_((torch.randn(inner.shape, generator=g, device=DEV) * 0.5).to(BF16))
    ssm.copy_(torch.randn(ssm.shape, generator=g, device=DEV))


def _segments(case, seed):
    """Ragged segment lengths that add up to the case's tokens."""
    n, total = case["segments"], case["tokens"]
    share = torch.rand(n, generator=_ints(seed)).add_(0.15)
    lens = (share / share.sum() * (total - n)).long().add_(1)
    lens[0] += total - int(lens.sum())
    return lens.tolist()


def _positions(batch, context, shared, seed):
    """Where each sequence stands: the second half of the context, one at its end."""
    lo = max(shared, context // 2)
    pos = torch.randint(lo, context, (batch,), generator=_ints(seed)) if lo < context - 1 else \
        torch.full((batch,), context - 1)
    pos[0] = context - 1
    return pos.to(torch.int64)


def _mixer_inputs(case, seed):
    """The three mixers with their states and each one's hidden rows."""
    path, hidden = case["path"], case["hidden"]
    g = _gen(seed)
    spec = case["drafts"] if path == "mixers_verify" else 0
    cfg = _config(hidden)
    s = {"mixers": [], "pools": [], "hidden": []}
    if path == "mixers_decode":
        n = rows = case["batch"]
        s["slots"] = (torch.randperm(n, generator=_ints(seed)) + 1).tolist()
    elif path == "mixers_prefill":
        s["lens"] = _segments(case, seed)
        n, rows = case["segments"], case["tokens"]
        s["slots"] = (torch.randperm(n, generator=_ints(seed)) + 1).tolist()
        s["resumed"] = [1 if j >= n - case["resumed"] else 0 for j in range(n)]
    else:
        q = spec + 1
        nreq = case["requests"]
        n = nreq * q
        lens = torch.randint(1, q + 1, (nreq,), generator=_ints(nreq))  # by the case alone
        lens[0] = q
        s["rows"] = [0] + torch.cumsum(lens, 0).tolist()
        rows = s["rows"][-1]
        s["slots"] = (torch.randperm(n, generator=_ints(seed + 1)) + 1).view(nreq, q)
        # tokens computed before, and how many of the last step's rows are
        # accepted: the step advances by that before it verifies the next drafts
        s["computed"] = torch.randint(1000, 9000, (nreq,), generator=_ints(seed + 2))
        s["accepted"] = torch.randint(1, q + 1, (nreq,), generator=_ints(seed + 3))
    for layer, kind in enumerate(KINDS):
        mixer = make_mixer(cfg, layer, prefix=f"perf.{next(_names)}.{kind}", device=DEV,
                           num_spec=spec)
        load_mixer_params(mixer, mixer_params(kind, hidden, seed * 8 + layer, device=DEV))
        pool = HyenaStatePool(n + 1, hidden, DEV, num_spec=spec)
        _fill_pool(pool, g)
        if spec:
            col = torch.arange(spec + 1)[None, :]
            stamp = (s["computed"][:, None] + col + 1).float().to(DEV)
            pool.stamps()[s["slots"].to(DEV)] = stamp
        mixer.kv_cache = pool.kv_cache
        s["mixers"].append(mixer)
        s["pools"].append(pool)
        s["hidden"].append(_rows(rows, hidden, g))
    return s


def _linear_inputs(case, seed):
    g = _gen(seed)
    k, n = case["inputs"], case["outputs"]
    w8, scale = quantize_weight_e4m3(torch.randn(n, k, generator=g, device=DEV) * 0.02)
    return {"x": _rows(case["tokens"], k, g), "w8": w8, "weight_scale": scale,
            "input_scale": torch.full((1,), 6.0 / 448.0, device=DEV)}


def _attention_inputs(case, seed):
    """One attention layer, its pages named by a random block table."""
    g = _gen(seed)
    hidden = case["hidden"]
    decode = case["path"] == "attention_decode"
    batch = case["batch"] if decode else case["sequences"]
    tokens = case["context"] if decode else case["tokens"]
    shared = case["shared"] // PAGE if decode else 0
    per = -(-tokens // PAGE)
    num_pages = shared + batch * (per - shared) + 1
    perm = torch.randperm(num_pages - 1, generator=_ints(seed)) + 1
    table = torch.empty(batch, per, dtype=torch.int32)
    table[:, :shared] = perm[:shared].int()
    table[:, shared:] = perm[shared:].int().view(batch, per - shared)
    layer = Evo2Attention(_config(hidden), num_pages, per, batch, ROPE_THETA, ROPE_FACTOR, DEV)
    layer.shared_pages = shared
    for lin in (layer.qkv_proj, layer.o_proj):
        lin.weight.data.copy_(torch.randn(lin.weight.shape, generator=g, device=DEV) * 0.02)
    layer.o_proj.bias.data.copy_(torch.randn(hidden, generator=g, device=DEV) * 0.02)
    s = {"layer": layer, "table": table.to(DEV)}
    if decode:
        for pages in (layer.cache.k, layer.cache.v):
            pages.copy_(torch.randn(pages.shape, generator=g, device=DEV, dtype=BF16))
        s["positions"] = _positions(batch, tokens, case["shared"], seed).to(DEV)
        s["x"] = _rows(batch, hidden, g)
    else:
        s["x"] = _rows(batch * tokens, hidden, g)
    return s


def _model_inputs(case, seed):
    """The four-layer model with random weights, states and pages, and tokens."""
    decode = case["path"] == "model_decode"
    batch = case["batch"] if decode else case["sequences"]
    context = case["context"] if decode else case["tokens"]
    model = Evo2DecodeModel(_config(case["hidden"], 4), max_batch=batch, max_ctx=context,
                            device=DEV, rope_theta=ROPE_THETA, rope_factor=ROPE_FACTOR,
                            name=f"perf.{next(_names)}", page_seed=seed % 1000003)
    model.init_random(seed, state_scale=0.5 if decode else 0.0, kv_scale=0.5 if decode else 0.0)
    ids = torch.tensor([65, 67, 71, 84])  # A, C, G, T
    shape = (batch,) if decode else (batch, context)
    tokens = ids[torch.randint(0, 4, shape, generator=_ints(seed))].to(DEV)
    s = {"model": model, "tokens": tokens}
    if decode:
        s["positions"] = _positions(batch, context, 0, seed).to(DEV)
    return s


def _inputs(case, seed):
    path = case["path"]
    if path.startswith("mixers"):
        return _mixer_inputs(case, seed)
    if path.startswith("fp8"):
        return _linear_inputs(case, seed)
    if path.startswith("attention"):
        return _attention_inputs(case, seed)
    return _model_inputs(case, seed)


def _captured(step, keep):
    """A HIP graph of one step; the tensors of `keep`, which the warm-up
    changes, hold afterwards what they held before."""
    kept = [t.clone() for t in keep]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = step()
    torch.cuda.current_stream().wait_stream(side)
    for t, old in zip(keep, kept):
        t.copy_(old)
    return graph, out


def prepare(case, seed):
    path = case["path"]
    s = _inputs(case, seed)
    s["path"] = path
    if path == "mixers_decode":
        m = build_metadata(decode_slots=s["slots"], device=DEV)
        s["graph"], s["out"] = _captured(lambda: _step(s, m), [p.raw for p in s["pools"]])
    elif path == "mixers_verify":
        n, rows = case["requests"], s["rows"]
        m = HyenaMamba2Metadata(num_decodes=n, num_decode_tokens=rows[-1])
        m.state_indices_tensor_d = s["slots"].to(DEV, torch.int32)
        m.query_start_loc_d = torch.tensor(rows, dtype=torch.int32, device=DEV)
        m.num_computed_tokens_d = s["computed"].to(DEV, torch.int32)
        accepted = s["accepted"].to(DEV, torch.int32)

        def step():
            m.num_computed_tokens_d.add_(accepted)  # the scheduler's counts of this step
            return _step(s, m)

        s["graph"], s["out"] = _captured(
            step, [m.num_computed_tokens_d] + [p.raw for p in s["pools"]])
    elif path == "mixers_prefill":
        s["meta"] = build_metadata(prefill_lens=s["lens"], prefill_slots=s["slots"],
                                   has_init=s["resumed"], device=DEV)
    elif path == "fp8_linear":
        lin = Fp8StaticLinear(case["inputs"], case["outputs"], device=DEV)
        lin.input_scale.data.copy_(s["input_scale"])
        lin.weight_scale.data.copy_(s["weight_scale"])
        lin.weight.weight_loader(lin.weight, s["w8"])
        lin.process_weights_after_loading()
        s["linear"] = lin
    elif path == "fp8_emulated":
        s["w_t"] = s["w8"].to(BF16).t().contiguous()
    elif path == "attention_decode":
        layer = s["layer"]
        s["graph"], s["out"] = _captured(
            lambda: layer.forward_decode(s["x"], s["positions"], s["table"]), [])
    elif path == "model_decode":
        model = s["model"]
        s["graph"], s["out"] = _captured(
            lambda: model.decode_step(s["tokens"], s["positions"]),
            [p.raw for p in model.pools.values()])
    return s


# ---------------------------------------------------------------- one pass
def _step(s, meta):
    with set_forward_context(meta):
        return [mixer(x) for mixer, x in zip(s["mixers"], s["hidden"])]


def _states(pools):
    """The states a step writes: each kind's short window and its own slice."""
    return [list(p.kv_cache) for p in pools]


def run(state):
    s, path = state, state["path"]
    if path in ("mixers_decode", "mixers_verify"):
        s["graph"].replay()
        return {"out": s["out"], "states": _states(s["pools"])}
    if path == "mixers_prefill":
        out = _step(s, s["meta"])
        return {"out": out, "states": _states(s["pools"])}
    if path == "fp8_linear":
        return s["linear"](s["x"])[0]
    if path == "fp8_emulated":
        return static_fp8_linear_emulated(s["x"], s["w_t"], s["input_scale"], s["weight_scale"])
    if path == "attention_prefill":
        layer, x = s["layer"], s["x"]
        n = s["table"].shape[0]
        out = layer.forward_prefill(x, n, x.shape[0] // n, s["table"])
        return {"out": out, "k": layer.cache.k, "v": layer.cache.v}
    if path == "attention_decode":
        s["graph"].replay()
        return {"out": s["out"], "k": s["layer"].cache.k, "v": s["layer"].cache.v}
    model = s["model"]
    cache = model.layers[3].mixer.cache
    if path == "model_decode":
        s["graph"].replay()
        out = s["out"]
    else:
        out = model.prefill(s["tokens"])
    return {"logits": out, "states": _states(model.pools.values()), "k": cache.k, "v": cache.v}


# ---------------------------------------------------------------- what a pass costs
def _window_bytes(kind, hidden):
    return {"hcs": 6, "hcm": 127, "hcl": 16}[kind] * hidden * 4


def _mixer_work(hidden, rows, state_bytes):
    """One layer of each kind over `rows` rows: in_proj (e4m3) and out_proj
    (bf16) weights, the hidden rows in and out, the states' bytes."""
    h = hidden
    by = 3 * (3 * h * h + 2 * h * h + 4 * rows * h) + state_bytes
    inner = sum(2 * k for k in (7, 128)) + 4 * 16  # multiply-adds of FIR taps and poles
    return by, rows * (3 * 8 * h * h + inner * h)


def work(case):
    path = case["path"]
    if path.startswith("fp8"):
        t, k, n = case["tokens"], case["inputs"], case["outputs"]
        wb = n * k * (1 if path == "fp8_linear" else 2)
        return {"bytes": wb + 2 * t * (k + n), "flops": 2 * t * k * n}
    h = case["hidden"]
    windows = [_window_bytes(k, h) for k in KINDS]
    short = 3 * (2 * 3 * h * 2)
    if path == "mixers_decode":
        by, fl = _mixer_work(h, case["batch"], case["batch"] * 2 * (sum(windows) + short))
        return {"bytes": by, "flops": fl}
    if path == "mixers_verify":
        rows = case["requests"] * (case["drafts"] + 2) / 2  # ragged: half the drafts on average
        by, fl = _mixer_work(h, rows, (case["requests"] + rows) * sum(windows)
                             + case["requests"] * 2 * short)
        return {"bytes": by, "flops": fl}
    if path == "mixers_prefill":
        by, fl = _mixer_work(h, case["tokens"], case["segments"] * (sum(windows) + short))
        return {"bytes": by, "flops": fl}
    if path == "attention_prefill":
        n, t = case["sequences"], case["tokens"]
        return {"bytes": 8 * h * h + n * t * h * 8,
                "flops": n * t * 8 * h * h + n * 2 * h * t * t}
    if path == "attention_decode":
        kv = case["shared"] + case["batch"] * (0.75 * case["context"] - case["shared"]) \
            if case["shared"] else case["batch"] * 0.75 * case["context"]
        return {"bytes": 8 * h * h + max(kv, case["context"]) * h * 4 + 4 * case["batch"] * h,
                "flops": case["batch"] * (8 * h * h + 3 * h * case["context"])}
    f = INTERMEDIATE[h]
    mlp = 4 * 3 * h * f * 2
    if path == "model_decode":
        b, c = case["batch"], case["context"]
        by, fl = _mixer_work(h, b, b * 2 * (sum(windows) + short))
        return {"bytes": by + mlp + 8 * h * h + b * 0.75 * c * h * 4 + VOCAB * h * 2,
                "flops": fl + b * (mlp + 8 * h * h + 3 * h * c + 2 * VOCAB * h)}
    n, t = case["sequences"], case["tokens"]
    by, fl = _mixer_work(h, n * t, n * (sum(windows) + short))
    return {"bytes": by + mlp + 8 * h * h + n * t * h * 4,
            "flops": fl + n * t * (mlp + 8 * h * h) + n * 2 * h * t * t + n * 2 * VOCAB * h}


def tolerance(case):
    return {
        # the emulated accumulator is defined bit for bit
        "fp8_emulated": "exact",
        # one bf16 rounding of an fp32 sum: 1.7e-3 from the 64-bit value
        "fp8_linear": {"rel": 7e-3},
        # bf16 at z, u, y, the gate and the projection's output: 4e-3 to 5.5e-3
        "mixers_decode": {"rel": 2e-2}, "mixers_verify": {"rel": 2e-2},
        "mixers_prefill": {"rel": 2e-2},
        # bf16 q, k, v, softmax weights (prefill) and outputs: 5.5e-3 and 3.5e-3
        "attention_prefill": {"rel": 2e-2}, "attention_decode": {"rel": 1.5e-2},
        # four layers one after the other: 0.9e-2 to 2e-2
        "model_decode": {"rel": 3e-2}, "model_prefill": {"rel": 3e-2},
    }[case["path"]]


# ---------------------------------------------------------------- 64-bit values
def _d(t):
    return t.detach().to(torch.float64)


def _e4m3(x, scale):
    """The static quantisation, which the projection is defined on."""
    q = (x.detach().float() / scale.float()).clamp(-448.0, 448.0)
    return q.to(torch.float8_e4m3fn).double()


def _fp8_linear(x, w8, input_scale, weight_scale):
    y = _e4m3(x, input_scale) @ w8.float().double().t()
    return y * _d(input_scale) * _d(weight_scale)


def _short(z, w, left):
    """The K=3 filter over rows z (n, 3H) after the two rows `left`; (x2, x1 v)."""
    w = _d(w).reshape(-1, 3)
    p = torch.cat([left, z])
    n = z.shape[0]
    zf = p[:n] * w[:, 0] + p[1:n + 1] * w[:, 1] + p[2:] * w[:, 2]
    return zf[:, 0::3], zf[:, 1::3] * zf[:, 2::3]


def _inner(kind, mixer, u, left):
    """The inner operator over rows u (n, H): its outputs, and the states
    after each row (hcl) or the rows with their history in front (FIRs)."""
    if kind == "hcl":
        p, r = _d(mixer.log_poles)[..., 0].exp(), _d(mixer.residues)
        st, y = left.clone(), torch.empty_like(u)
        states = []
        for i in range(u.shape[0]):
            st = torch.addcmul(u[i][:, None].expand_as(st), st, p)
            torch.sum(r * st, -1, out=y[i])
            states = (states + [st])[-8:]
        return y, states
    w = _d(mixer.conv).reshape(u.shape[1], -1)
    k = w.shape[1]
    p = torch.cat([left, u])
    y = torch.zeros_like(u)
    for i in range(k):
        y.addcmul_(p[i:i + u.shape[0]], w[:, i])
    return y, p


def _mixer_rows(kind, mixer, z, conv_left, inner_left):
    """(out_proj output before nothing else, u, inner states) of one segment."""
    x2, u = _short(z, mixer.short_filter, conv_left)
    y, states = _inner(kind, mixer, u, inner_left)
    if mixer.D is not None:
        y = y + _d(mixer.D) * u
    return x2 * y, states


def _out_proj(mixer, g):
    return g @ _d(mixer.out_proj.weight).t() + _d(mixer.out_proj.bias)


def _project(mixer, x):
    p = mixer.in_proj
    return _fp8_linear(x, p.weight, p.input_scale, p.weight_scale)


def _sequence(kind, mixer, z, pool_d, slot, resumed):
    """One segment from its block's state; writes the block's final state."""
    conv, inner, ssm = pool_d
    k = {"hcs": 7, "hcm": 128, "hcl": 0}[kind]
    left = conv[slot, :2] if resumed else torch.zeros_like(conv[slot, :2])
    if kind == "hcl":
        il = ssm[slot] if resumed else torch.zeros_like(ssm[slot])
    else:
        il = inner[slot, :k - 1] if resumed else torch.zeros_like(inner[slot, :k - 1])
    g, states = _mixer_rows(kind, mixer, z, left, il)
    conv[slot, :2] = torch.cat([left, z])[-2:]
    if kind == "hcl":
        ssm[slot] = states[-1]
    else:
        inner[slot, :k - 1] = states[-(k - 1):]
    return g


def _exact_mixer(kind, mixer, x, pool, lens, slots, resumed):
    """One mixer over packed segments: its output and states."""
    pool_d = [_d(t).clone() for t in pool.kv_cache]
    z = _project(mixer, x)
    parts, a = [], 0
    for n, slot, res in zip(lens, slots, resumed):
        parts.append(_sequence(kind, mixer, z[a:a + n], pool_d, slot, res))
        a += n
    return _out_proj(mixer, torch.cat(parts)), pool_d


def _exact_decode(kind, mixer, x, pool, slots):
    """One token of every sequence at once: rows are independent."""
    conv, inner, ssm = pool_d = [_d(t).clone() for t in pool.kv_cache]
    slots = torch.as_tensor(slots, device=x.device).long()
    z = _project(mixer, x)
    w = _d(mixer.short_filter).reshape(-1, 3)
    old = conv[slots]
    zf = old[:, 0] * w[:, 0] + old[:, 1] * w[:, 1] + z * w[:, 2]
    conv[slots] = torch.stack([old[:, 1], z], 1)
    x2, u = zf[:, 0::3], zf[:, 1::3] * zf[:, 2::3]
    if kind == "hcl":
        st = ssm[slots] * _d(mixer.log_poles)[..., 0].exp() + u[:, :, None]
        ssm[slots] = st
        y = (st * _d(mixer.residues)).sum(-1)
    else:
        taps = _d(mixer.conv).reshape(u.shape[1], -1).t()
        k = taps.shape[0]
        win = torch.cat([inner[slots][:, :k - 1], u[:, None]], 1)
        inner[slots, :k - 1] = win[:, 1:]
        y = (win * taps).sum(1)
    if mixer.D is not None:
        y = y + _d(mixer.D) * u
    return _out_proj(mixer, x2 * y), pool_d


def _exact_verify(kind, mixer, x, pool, s):
    """Each request from its live snapshot, one snapshot a row written."""
    conv, inner, ssm = [_d(t).clone() for t in pool.kv_cache]
    conv0, inner0, ssm0 = conv.clone(), inner.clone(), ssm.clone()
    z = _project(mixer, x)
    q = s["slots"].shape[1]
    k = {"hcs": 7, "hcm": 128, "hcl": 0}[kind]
    parts = []
    for r, row in enumerate(s["slots"].tolist()):
        acc = int(s["accepted"][r])
        a, b = s["rows"][r], s["rows"][r + 1]
        left = conv0[row[0], acc - 1:acc + 1]
        live = ssm0[row[acc - 1], :, :16] if kind == "hcl" else inner0[row[acc - 1], :k - 1]
        g, states = _mixer_rows(kind, mixer, z[a:b], left, live)
        parts.append(g)
        conv[row[0], 0] = left[1]
        conv[row[0], 1:1 + b - a] = z[a:b]
        done = int(s["computed"][r]) + acc
        for p in range(b - a):
            if kind == "hcl":
                ssm[row[p], :, :16] = states[p - (b - a)]
            else:
                inner[row[p], :k - 1] = states[p + 1:p + k]
            ssm[row[p], 0, 16] = done + p + 1
        assert q >= b - a
    return _out_proj(mixer, torch.cat(parts)), [conv, inner, ssm]


def _rotary(x, positions):
    """Neox rotary on (n, heads, head_dim) with linear position scaling."""
    half = x.shape[-1] // 2
    inv = ROPE_THETA ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    ang = (positions.double() / ROPE_FACTOR)[:, None] * inv
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _qkv(layer, x, positions):
    n, heads = x.shape[0], layer.heads
    qkv = (_d(x) @ _d(layer.qkv_proj.weight).t()).view(n, 3, heads, 128)
    return _rotary(qkv[:, 0], positions), _rotary(qkv[:, 1], positions), qkv[:, 2]


def _o_proj(layer, o):
    return o.reshape(o.shape[0], -1) @ _d(layer.o_proj.weight).t() + _d(layer.o_proj.bias)


def _exact_attention_decode(layer, x, positions, table):
    q, k, v = _qkv(layer, x, positions)
    kc, vc = layer.cache.k.clone(), layer.cache.v.clone()
    page = table.gather(1, (positions // PAGE)[:, None])[:, 0].long()
    kc[page, :, :, positions % PAGE] = k.to(kc.dtype)
    vc[page, :, positions % PAGE] = v.to(vc.dtype)
    out = torch.empty_like(q)
    for b in range(x.shape[0]):
        n = int(positions[b]) + 1
        pages = table[b, :-(-n // PAGE)].long()
        kd = _d(kc[pages]).permute(1, 2, 0, 3).reshape(layer.heads, 128, -1)[..., :n]
        vd = _d(vc[pages]).permute(1, 0, 2, 3).reshape(layer.heads, -1, 128)[:, :n]
        kd[..., -1], vd[:, -1] = k[b], v[b]
        w = torch.softmax((q[b][:, :, None] * kd).sum(1) * 128 ** -0.5, -1)
        out[b] = (w[:, :, None] * vd).sum(1)
    return _o_proj(layer, out)


def _exact_attention_prefill(layer, x, n, table):
    length = x.shape[0] // n
    pos = torch.arange(length, device=x.device).repeat(n)
    q, k, v = _qkv(layer, x, pos)
    out = torch.empty_like(q)
    mask = torch.ones(length, length, dtype=torch.bool, device=x.device).triu_(1)
    for b in range(n):
        rows = slice(b * length, (b + 1) * length)
        for h in range(layer.heads):
            sc = q[rows, h].contiguous() @ k[rows, h].t().contiguous()
            sc = sc.mul_(128 ** -0.5).masked_fill_(mask, float("-inf"))
            out[rows, h] = torch.softmax(sc, -1) @ v[rows, h].contiguous()
    per = -(-length // PAGE)
    kc = torch.zeros(layer.cache.k.shape, dtype=torch.float64, device=x.device)
    vc = torch.zeros(layer.cache.v.shape, dtype=torch.float64, device=x.device)

    def paged(t):
        t = torch.nn.functional.pad(t.view(n, length, layer.heads, 128),
                                    (0, 0, 0, 0, 0, per * PAGE - length))
        return t.view(n * per, PAGE, layer.heads, 128)

    pages = table[:n, :per].reshape(-1).long()
    kc[pages] = paged(k).permute(0, 2, 3, 1)
    vc[pages] = paged(v).permute(0, 2, 1, 3)
    return _o_proj(layer, out), kc, vc


def _norm(x, w):
    n = x.square().sum(-1, keepdim=True).sqrt() * x.shape[-1] ** -0.5 + EPS
    return _d(w) * x / n


def _exact_model(case, s):
    model = s["model"]
    decode = case["path"] == "model_decode"
    x = _d(model.embed)[s["tokens"].reshape(-1)]
    slots = model.slots.tolist()
    for i, layer in enumerate(model.layers):
        pre = _norm(x, layer.pre_norm.weight)
        if layer.kind == "attn":
            if decode:
                m = _exact_attention_decode(layer.mixer, pre, s["positions"], model.block_table)
            else:
                m = _exact_attention_prefill(layer.mixer, pre, case["sequences"],
                                             model.block_table)[0]
        elif decode:
            m = _exact_decode(layer.kind, layer.mixer, pre.to(BF16), model.pools[i], slots)[0]
        else:
            n = case["sequences"]
            m = _exact_mixer(layer.kind, layer.mixer, pre.to(BF16), model.pools[i],
                             [case["tokens"]] * n, slots, [0] * n)[0]
        x = x + m
        post = _norm(x, layer.post_norm.weight)
        z1, z2 = (post @ _d(lin.weight).t() for lin in (layer.mlp.l1, layer.mlp.l2))
        if layer.mlp.use_act:
            z1 = torch.nn.functional.gelu(z1)
        x = x + (z1 * z2) @ _d(layer.mlp.l3.weight).t()
    if not decode:
        x = x.view(case["sequences"], case["tokens"], -1)[:, -1]
    return {"logits": _norm(x, model.norm.weight) @ _d(model.embed).t()}


def exact(case, seed):
    path = case["path"]
    with torch.no_grad():
        s = _inputs(case, seed)
        if path.startswith("fp8"):
            return _fp8_linear(s["x"], s["w8"], s["input_scale"], s["weight_scale"])
        if path == "attention_decode":
            return {"out": _exact_attention_decode(s["layer"], s["x"], s["positions"],
                                                   s["table"]), "k": None, "v": None}
        if path == "attention_prefill":
            out, k, v = _exact_attention_prefill(s["layer"], s["x"], case["sequences"],
                                                 s["table"])
            return {"out": out, "k": k, "v": v}
        if path.startswith("model"):
            return _exact_model(case, s)
        outs, states = [], []
        for kind, mixer, pool, x in zip(KINDS, s["mixers"], s["pools"], s["hidden"]):
            if path == "mixers_decode":
                o, st = _exact_decode(kind, mixer, x, pool, s["slots"])
            elif path == "mixers_verify":
                o, st = _exact_verify(kind, mixer, x, pool, s)
            else:
                o, st = _exact_mixer(kind, mixer, x, pool, s["lens"], s["slots"], s["resumed"])
            outs.append(o)
            states.append(st)
        return {"out": outs, "states": states}
