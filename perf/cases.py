"""The work this framework is timed on, through the calls a program makes: decode steps of a batch
over its paged cache, prefills, the LocDiT sampler, the local encoder and the whole patch step, each
through host arrays as `tgx` takes them.

Shapes are the repository's own: the 24-layer MiniCPM-4 backbone (hidden 1024, 16 heads over 2 KV
heads of 64 dimensions), VoxCPM2's wider LM (hidden 2048, heads of 128 dimensions; four of its
layers), the 8-layer residual LM without RoPE and the 4-layer local stacks. Weights are random, the
same for every state: a program loads them once and keeps its decoder, so `prepare` takes the handle
of the case's shape (made at its first use), hands the state cache slots of its own in it and fills
them with the state's prompts. `exact` restates each path in float64 with torch alone.
"""

import math
import random
import sys
import weakref
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "tgtts-v4_amd"))
import tgx  # noqa: E402
from tgx import patch as tgx_patch  # noqa: E402

EPS = 1e-5
THETA = 10000.0
FEAT, FRAMES, TIMESTEPS = 64, 4, 10
LATENT, LEVELS = 256, 9
PATCH_SLOTS = 16

STACKS = {
    "backbone": dict(hidden=1024, inner=4096, heads=16, kv_heads=2, head_dim=64, layers=24),
    "wide": dict(hidden=2048, inner=6144, heads=16, kv_heads=2, head_dim=128, layers=4),
    "residual": dict(hidden=1024, inner=4096, heads=16, kv_heads=2, head_dim=64, layers=8, rope=False),
    "dit": dict(hidden=1024, inner=4096, heads=16, kv_heads=2, head_dim=64, layers=4),
    "encoder": dict(hidden=1024, inner=4096, heads=16, kv_heads=2, head_dim=64, layers=4),
}
# The decoders the cases run on: rows a step, positions a slot holds.
CAPACITY = {("backbone", 1): 4096, ("backbone", 4): 16384, ("backbone", 16): 4096, ("backbone", 64): 2112, ("wide", 8): 2112}
STATES = 4  # states whose slots a decoder holds at once


def listed():
    return [
        # One request speaking alone, half a minute in: the latency a single user meets.
        dict(name="decode_1", kind="decode", stack="backbone", batch=1, rows=1, low=511, high=511, steps=4),
        # A server's decoder of 16 rows with 13 requests under way, at ragged positions.
        dict(name="decode_13_of_16", kind="decode", stack="backbone", batch=16, rows=13, low=64, high=1024, steps=4),
        # A full batch of 64 requests.
        dict(name="decode_64", kind="decode", stack="backbone", batch=64, rows=64, low=64, high=1024, steps=4),
        # Long-form reading: few requests, far into their caches.
        dict(name="decode_long", kind="decode", stack="backbone", batch=4, rows=2, low=5003, high=12007, steps=4),
        # VoxCPM2's own layer sizes, 128-dimension heads, a part-filled batch.
        dict(name="decode_wide", kind="decode", stack="wide", batch=8, rows=5, low=33, high=700, steps=4),
        # A short text prompt: the wait before a request's first step.
        dict(name="prefill_57", kind="prefill", stack="backbone", batch=16, runs=1, low=57, high=57, start=0),
        # Three requests' next pieces of their prompts, behind pieces already cached.
        dict(name="prefill_resumed", kind="prefill", stack="backbone", batch=16, runs=3, low=77, high=513, start=300),
        # Long prompts of a full batch, the largest call.
        dict(name="prefill_8x2048", kind="prefill", stack="backbone", batch=16, runs=8, low=2048, high=2048, start=0),
        # The LocDiT's ten Euler steps for one request and for a full patch batch.
        dict(name="sample_1", kind="sample", rows=1, guidance=2.0),
        dict(name="sample_16", kind="sample", rows=16, guidance=2.0),
        # One patch through the local encoder: the smallest call.
        dict(name="encode_1", kind="encode", rows=1),
        # The whole patch step of 16 requests: encoder, both LMs and their heads, sampler; twice, each
        # patch conditioning the next.
        dict(name="patch_16", kind="patch", rows=16, low=64, high=512, steps=2),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "sample", "encode", "patch"])
    if kind == "decode":
        if rng.random() < 0.25:
            stack, batch = "wide", 8
            rows = rng.randint(1, batch)
        else:
            stack, rows = "backbone", _log(rng, 1, 64)
            batch = next(b for b in (1, 4, 16, 64) if b >= rows)
        high = _log(rng, 8, CAPACITY[stack, batch] - 64)
        low = max(1, int(high * rng.uniform(0.05, 1.0)))
        return dict(kind=kind, stack=stack, batch=batch, rows=rows, low=low, high=high, steps=4)
    if kind == "prefill":
        wide = rng.random() < 0.25
        high = _log(rng, 1, 1024 if wide else 2048)
        return dict(kind=kind, stack="wide" if wide else "backbone", batch=8 if wide else 16, runs=_log(rng, 1, 8),
                    low=max(1, int(high * rng.uniform(0.05, 1.0))), high=high,
                    start=0 if rng.random() < 0.5 else _log(rng, 1, 1000))
    if kind == "patch":
        high = _log(rng, 8, 1500)
        return dict(kind=kind, rows=rng.randint(1, PATCH_SLOTS), low=max(1, int(high * rng.uniform(0.05, 1.0))), high=high, steps=2)
    if kind == "sample":
        return dict(kind=kind, rows=rng.randint(1, 16), guidance=round(rng.uniform(1.0, 3.0), 2))
    return dict(kind=kind, rows=rng.randint(2, 32))


def _spread(low, high, n):
    """n lengths over low .. high, the first the highest, the same for every seed."""
    return [int(round(high - (high - low) * ((i * 0.6180339887498949) % 1.0))) for i in range(n)]


# ---- weights: drawn once for each stack, kept as bf16 on the host and (for `exact`) on the GPU ----

_made = {}


def _once(key, make):
    if key not in _made:
        _made[key] = make()
    return _made[key]


def _shapes(stack):
    s = STACKS[stack]
    h, i = s["hidden"], s["inner"]
    qkv = (s["heads"] + 2 * s["kv_heads"]) * s["head_dim"]
    out = {}
    for l in range(s["layers"]):
        out[f"layers.{l}.input_layernorm"] = (h,)
        out[f"layers.{l}.qkv_proj"] = (qkv, h)
        out[f"layers.{l}.o_proj"] = (h, s["heads"] * s["head_dim"])
        out[f"layers.{l}.post_attention_layernorm"] = (h,)
        out[f"layers.{l}.gate_up_proj"] = (2 * i, h)
        out[f"layers.{l}.down_proj"] = (h, i)
    out["norm"] = (h,)
    if stack == "dit":
        out.update({"in_proj.weight": (h, FEAT), "cond_proj.weight": (h, FEAT), "out_proj.weight": (FEAT, h),
                    "in_proj.bias": (h,), "cond_proj.bias": (h,), "out_proj.bias": (FEAT,)})
        for m in ("time_mlp", "delta_time_mlp"):
            out.update({f"{m}.linear_1.weight": (h, h), f"{m}.linear_1.bias": (h,),
                        f"{m}.linear_2.weight": (h, h), f"{m}.linear_2.bias": (h,)})
    if stack == "encoder":
        out.update({"in_proj.weight": (h, FEAT), "in_proj.bias": (h,), "special_token": (h,)})
    return out


HEADS = {
    "enc_to_lm_proj.weight": (1024, 1024), "enc_to_lm_proj.bias": (1024,),
    "fsq_layer.in_proj.weight": (LATENT, 1024), "fsq_layer.in_proj.bias": (LATENT,),
    "fsq_layer.out_proj.weight": (1024, LATENT), "fsq_layer.out_proj.bias": (1024,),
    "fusion_concat_proj.weight": (1024, 2048), "fusion_concat_proj.bias": (1024,),
    "lm_to_dit_proj.weight": (1024, 1024), "lm_to_dit_proj.bias": (1024,),
    "res_to_dit_proj.weight": (1024, 1024), "res_to_dit_proj.bias": (1024,),
    "stop_proj.weight": (1024, 1024), "stop_proj.bias": (1024,),
    "stop_head.weight": (2, 1024),
}


def _weights(stack):
    """bf16 tensors on the GPU by name: projections N(0, 0.02), gains near 1."""

    def make():
        g = torch.Generator("cuda").manual_seed(1000 + sorted([*STACKS, "heads"]).index(stack))
        out = {}
        for name, shape in (HEADS if stack == "heads" else _shapes(stack)).items():
            v = torch.randn(shape, generator=g, device="cuda")
            v = 1 + 0.02 * v if name.endswith("norm") else v if name == "special_token" else 0.02 * v
            out[name] = v.to(torch.bfloat16)
        return out

    return _once(("weights", stack), make)


def _load(handle, stack, prefix=""):
    for name, v in _weights(stack).items():
        handle.load(prefix + name, v.view(torch.uint16).cpu().numpy())


# ---- handles a program keeps ----


def _context():
    return _once("context", lambda: tgx.Context(0))


def _shape(stack, capacity):
    return tgx.Shape(capacity=capacity, eps=EPS, rope_theta=THETA, **STACKS[stack])


class _Slots:
    """Cache slots of one decoder (or of an LM side's two), handed to states and taken back when a
    state is dropped."""

    def __init__(self, decoders, count):
        self.decoders, self.free = decoders, list(range(count))

    def take(self, state, n):
        got, self.free = self.free[:n], self.free[n:]
        if len(got) < n:
            raise RuntimeError("more states than the decoder holds slots for")
        weakref.finalize(state, self.give, got).atexit = False
        return got

    def give(self, slots):
        for s in slots:
            for d in self.decoders:
                d.release_slot(s)
        self.free = slots + self.free


def _decoder(stack, batch):
    def make():
        count = STATES * max(batch, 8)
        d = tgx.Decoder(_context(), _shape(stack, CAPACITY[stack, batch]), tgx.Batch(rows=batch, slots=count))
        _load(d, stack)
        return d, _Slots([d], count)

    return _once(("decoder", stack, batch), make)


def _sampler(rows, owner="alone"):
    def make():
        s = tgx_patch.Sampler(_context(), _shape("dit", 16), tgx_patch.PatchShape(FEAT, FRAMES, TIMESTEPS, rows))
        _load(s, "dit")
        return s

    return _once(("sampler", rows, owner), make)


def _encoder(rows, owner="alone"):
    def make():
        e = tgx_patch.Encoder(_context(), _shape("encoder", 16), tgx_patch.PatchShape(FEAT, FRAMES, TIMESTEPS, rows))
        _load(e, "encoder")
        return e

    return _once(("encoder", rows, owner), make)


def _patch_step():
    def make():
        count = STATES * PATCH_SLOTS
        side = tgx_patch.LmSide(_context(), _shape("backbone", 2048), _shape("residual", 2048),
                                tgx.Batch(rows=PATCH_SLOTS, slots=count), tgx_patch.HeadsShape(1024, 1024, LATENT, LEVELS))
        _load(side, "backbone", "base_lm.")
        _load(side, "residual", "residual_lm.")
        _load(side, "heads")
        step = tgx_patch.PatchStep(_encoder(PATCH_SLOTS, "patch"), side, _sampler(PATCH_SLOTS, "patch"))
        return step, side, _Slots([side.decoder(0), side.decoder(1)], count)

    return _once("patch", make)


# ---- inputs ----


class State:
    pass


def _normal(seed, what, *shape):
    g = torch.Generator("cuda").manual_seed(seed * 64 + what)
    return torch.randn(shape, generator=g, device="cuda")


def _inputs(case, seed):
    """The case's inputs as float32 tensors on the GPU: `prompts` (one a request) already in the
    caches, and what `run` passes."""
    kind = case["kind"]
    if kind == "decode":
        lens = _spread(case["low"], case["high"], case["rows"])
        h = STACKS[case["stack"]]["hidden"]
        return dict(lens=lens, prompt=_normal(seed, 0, sum(lens), h), x=_normal(seed, 1, case["steps"], case["batch"], h))
    if kind == "prefill":
        lens = _spread(case["low"], case["high"], case["runs"])
        starts = _spread(case["start"] // 2, case["start"], case["runs"])
        h = STACKS[case["stack"]]["hidden"]
        return dict(lens=lens, starts=starts, prompt=_normal(seed, 0, sum(starts), h), x=_normal(seed, 1, sum(lens), h))
    rows = case["rows"]
    if kind == "sample":
        return dict(mu=_normal(seed, 0, rows, 2, 1024) * 0.5, cond=_normal(seed, 1, rows, FEAT, FRAMES),
                    noise=_normal(seed, 2, rows, FEAT, FRAMES))
    if kind == "encode":
        return dict(patches=_normal(seed, 0, rows, FEAT, FRAMES))
    lens = _spread(case["low"], case["high"], rows)
    return dict(lens=lens, prompt=_normal(seed, 0, sum(lens), 1024), residual_prompt=_normal(seed, 1, sum(lens), 1024),
                cond=_normal(seed, 2, rows, FEAT, FRAMES), noise=_normal(seed, 3, case["steps"], rows, FEAT, FRAMES))


def _sampling(case):
    return np.array([[1.0, case.get("guidance", 2.0)]] * case["rows"], dtype=np.float32)  # temperature, guidance


def prepare(case, seed):
    got = {k: v.cpu().numpy() if isinstance(v, torch.Tensor) else v for k, v in _inputs(case, seed).items()}
    s = State()
    s.kind, s.case, s.inputs = case["kind"], case, got
    if s.kind == "decode":
        s.decoder, slots = _decoder(case["stack"], case["batch"])
        took = slots.take(s, case["rows"])
        s.decoder.prefill_runs([(k, 0, n) for k, n in zip(took, got["lens"])], got["prompt"])
        spare = [None] * (case["batch"] - case["rows"])
        s.rows = [[tgx.Row(n + t, k) for k, n in zip(took, got["lens"])] + spare for t in range(case["steps"])]
    elif s.kind == "prefill":
        s.decoder, slots = _decoder(case["stack"], case["batch"])
        took = slots.take(s, case["runs"])
        before = [(k, 0, n) for k, n in zip(took, got["starts"]) if n]
        if before:
            s.decoder.prefill_runs(before, got["prompt"])
        s.runs = list(zip(took, got["starts"], got["lens"]))
    elif s.kind == "sample":
        s.sampler = _sampler(case["rows"])
    elif s.kind == "encode":
        s.encoder = _encoder(case["rows"])
    else:
        s.step, side, slots = _patch_step()
        took = slots.take(s, case["rows"])
        for which, prompt in enumerate((got["prompt"], got["residual_prompt"])):
            side.decoder(which).prefill_runs([(k, 0, n) for k, n in zip(took, got["lens"])], prompt)
        s.rows = [[tgx.Row(n + t, k) for k, n in zip(took, got["lens"])] for t in range(case["steps"])]
    return s


def run(state):
    s, got = state, state.inputs
    if s.kind == "decode":
        n = s.case["rows"]
        return [s.decoder.step_rows(rows, x)[:n] for rows, x in zip(s.rows, got["x"])]
    if s.kind == "prefill":
        return s.decoder.prefill_runs(s.runs, got["x"])
    if s.kind == "sample":
        return s.sampler.sample(got["mu"], got["cond"], got["noise"], _sampling(s.case))
    if s.kind == "encode":
        return s.encoder.encode(got["patches"])
    cond, out = got["cond"], []
    for rows, noise in zip(s.rows, got["noise"]):
        cond, stop = s.step.run_rows(rows, cond, noise, _sampling(s.case))
        out += [cond, stop]
    return out


# ---- what a pass cannot do without ----


def _stack_work(stack, rows, attended, kv_read, kv_written):
    """A stack over `rows` positions that attend to `attended` positions in all."""
    s = STACKS[stack]
    h, d, L = s["hidden"], s["head_dim"], s["layers"]
    params = L * ((s["heads"] + 2 * s["kv_heads"]) * d * h + s["heads"] * d * h + 3 * h * s["inner"])
    position = L * 2 * s["kv_heads"] * d * 2
    return (2 * params + L * 2 * h * 2 + position * (kv_read + kv_written) + rows * h * 8,
            2 * params * rows + 4 * L * s["heads"] * d * attended)


def work(case):
    kind, total = case["kind"], [0, 0]

    def add(pair):
        total[0] += pair[0]
        total[1] += pair[1]

    if kind == "decode":
        lens = _spread(case["low"], case["high"], case["rows"])
        for t in range(case["steps"]):
            reach = sum(n + t + 1 for n in lens)
            add(_stack_work(case["stack"], case["rows"], reach, reach, case["rows"]))
    elif kind == "prefill":
        lens = _spread(case["low"], case["high"], case["runs"])
        starts = _spread(case["start"] // 2, case["start"], case["runs"])
        add(_stack_work(case["stack"], sum(lens), sum(n * s + n * (n + 1) // 2 for n, s in zip(lens, starts)), sum(starts), sum(lens)))
    elif kind == "sample":
        add(_dit_work(case["rows"]))
    elif kind == "encode":
        add(_encoder_work(case["rows"]))
    else:
        lens = _spread(case["low"], case["high"], case["rows"])
        heads = sum(math.prod(v) for v in HEADS.values())
        for t in range(case["steps"]):
            reach = sum(n + t + 1 for n in lens)
            for stack in ("backbone", "residual"):
                add(_stack_work(stack, case["rows"], reach, reach, case["rows"]))
            add((2 * heads, 2 * heads * case["rows"]))
            add(_encoder_work(case["rows"]))
            add(_dit_work(case["rows"]))
    return {"bytes": total[0], "flops": total[1]}


def _dit_work(rows):
    tokens, evaluations = rows * 2 * (3 + 2 * FRAMES), TIMESTEPS - 1
    b, f = _stack_work("dit", tokens, tokens * (3 + 2 * FRAMES), 0, 0)
    return b + rows * (2 * 1024 + 3 * FEAT * FRAMES) * 4, f * evaluations


def _encoder_work(rows):
    b, f = _stack_work("encoder", rows * (1 + FRAMES), rows * (1 + FRAMES) ** 2, 0, 0)
    return b + rows * (FEAT * FRAMES + 1024) * 4, f


def tolerance(case):
    # bf16 operands, float32 sums. Over the backbone's 24 layers an output is 0.0042 off `exact`, and
    # a position decoded is 0.0048 off the same position prefilled (the same sums in another order);
    # a sample or an embedding is 0.0025 off `exact`. The patch step's quantizer turns such
    # differences into whole levels here and there: 0.02 to 0.1 off `exact`.
    return {"rel": 3e-2 if case["kind"] == "patch" else 1e-2}


# ---- the same in float64, by torch alone ----


def _rms(x, gain):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gain.double()


def _rope(v, places):
    """Rotate-half RoPE of [T, heads, d]; the angles in float32, as the model's tables have them."""
    d = v.shape[-1]
    inv = np.float32(1) / np.power(np.float32(THETA), np.arange(0, d, 2, dtype=np.float32) / np.float32(d), dtype=np.float32)
    angle = torch.from_numpy(places.astype(np.float32)[:, None] * inv).to(v.device).double()[:, None, :]
    cos, sin = torch.cos(angle), torch.sin(angle)
    a, c = v[..., : d // 2], v[..., d // 2:]
    return torch.cat([a * cos - c * sin, c * cos + a * sin], -1)


def _attend(q, k, v, first):
    """q [T, heads, d] over k, v [P, kv_heads, d]: query t sees keys 0 .. first + t (all, if None)."""
    group = q.shape[1] // k.shape[1]
    k = k.repeat_interleave(group, 1).transpose(0, 1).contiguous()
    v = v.repeat_interleave(group, 1).transpose(0, 1).contiguous()
    out = []
    for t0 in range(0, q.shape[0], 1024):
        part = q[t0: t0 + 1024].transpose(0, 1)
        scores = torch.matmul(part, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
        if first is not None:
            at = torch.arange(t0, t0 + part.shape[1], device=q.device)[:, None] + first
            scores.masked_fill_(torch.arange(k.shape[1], device=q.device)[None, :] > at, -math.inf)
        out.append(torch.matmul(torch.softmax(scores, -1), v).transpose(0, 1))
    return torch.cat(out)


def _stack(stack, x, lens, causal=True):
    """The stack over sequences of `lens` positions laid one after another in x, float64."""
    s, w = STACKS[stack], _weights(stack)
    H, KV, d = s["heads"], s["kv_heads"], s["head_dim"]
    places = np.concatenate([np.arange(n) for n in lens])
    ends = np.cumsum(lens)
    W = lambda l, name: w[f"layers.{l}.{name}"].double().t()  # noqa: E731
    x = x.double()
    for l in range(s["layers"]):
        qkv = _rms(x, w[f"layers.{l}.input_layernorm"]) @ W(l, "qkv_proj")
        q, k, v = (t.reshape(len(x), -1, d) for t in torch.split(qkv, [H * d, KV * d, KV * d], -1))
        if s.get("rope", True):
            q, k = _rope(q, places), _rope(k, places)
        att = torch.cat([_attend(q[e - n: e], k[e - n: e], v[e - n: e], 0 if causal else None) for n, e in zip(lens, ends)])
        x = x + att.reshape(len(x), -1) @ W(l, "o_proj")
        gate, up = (_rms(x, w[f"layers.{l}.post_attention_layernorm"]) @ W(l, "gate_up_proj")).chunk(2, -1)
        x = x + (torch.nn.functional.silu(gate) * up) @ W(l, "down_proj")
    return _rms(x, w["norm"])


def _linear(x, w, name, bias=True):
    y = x @ w[f"{name}.weight"].double().t()
    return y + w[f"{name}.bias"].double() if bias else y


def _span():
    """The sampler's times: linspace(1, 0) swayed by cos(pi t / 2) - 1 + t, in float32."""
    f = np.float32
    step = f(-1) / f(TIMESTEPS)
    n = TIMESTEPS + 1
    t = np.array([f(1) + step * f(i) if i < n // 2 else -(step * f(n - i - 1)) for i in range(n)], dtype=f)
    return t + (np.cos(f(math.pi / 2) * t).astype(f) - f(1) + t)


def _time_tokens(w, t):
    def mlp(prefix, at):
        half = 512
        rate = np.float32(-(math.log(10000.0) / (half - 1)))
        angle = np.float32(np.float32(at) * np.float32(1000)) * np.exp(np.arange(half, dtype=np.float32) * rate)
        angle = torch.from_numpy(angle).cuda().double()
        return _linear(torch.nn.functional.silu(_linear(torch.cat([torch.sin(angle), torch.cos(angle)]), w, f"{prefix}.linear_1")),
                       w, f"{prefix}.linear_2")

    return mlp("time_mlp", t) + mlp("delta_time_mlp", 0.0)


def _sample(mu, cond, noise, guidance):
    w, rows = _weights("dit"), len(noise)
    T = 3 + 2 * FRAMES
    frames = lambda v, name: _linear(v.double().transpose(1, 2), w, name)  # noqa: E731
    state = noise.double().clone()
    tokens = torch.zeros(rows, 2, T, 1024, dtype=torch.float64, device="cuda")
    tokens[:, 0, :2] = mu.double().reshape(rows, 2, 1024)
    tokens[:, :, 3: 3 + FRAMES] = frames(cond, "cond_proj")[:, None]
    span = _span()
    t, dt = span[0], np.float32(span[0] - span[1])
    for step in range(1, len(span)):
        if step > max(1, int(len(span) * 0.04)):
            tokens[:, :, 2] = _time_tokens(w, t)
            tokens[:, :, 3 + FRAMES:] = frames(state, "in_proj")[:, None]
            out = _stack("dit", tokens.reshape(-1, 1024), [T] * (2 * rows), causal=False).reshape(rows, 2, T, 1024)
            vel = _linear(out[:, :, 3 + FRAMES:], w, "out_proj").transpose(2, 3).reshape(rows, 2, -1)
            c, u = vel[:, 0], vel[:, 1]
            scaled = u * ((c * u).sum(-1, keepdim=True) / ((u * u).sum(-1, keepdim=True) + 1e-8))
            state = state - float(dt) * (scaled + guidance * (c - scaled)).reshape(state.shape)
        t = np.float32(t - dt)
        if step < len(span) - 1:
            dt = np.float32(t - span[step + 1])
    return state


def _encode(patches):
    w, rows = _weights("encoder"), len(patches)
    tokens = torch.empty(rows, 1 + FRAMES, 1024, dtype=torch.float64, device="cuda")
    tokens[:, 0] = w["special_token"].double()
    tokens[:, 1:] = _linear(patches.double().transpose(1, 2), w, "in_proj")
    return _stack("encoder", tokens.reshape(-1, 1024), [1 + FRAMES] * rows, causal=False).reshape(rows, 1 + FRAMES, 1024)[:, 0]


def _behind(stack, prompt, lens, steps):
    """The last positions' outputs, [steps][rows][hidden], of the stack over each prompt with `steps`
    ([rows][hidden] each) behind it."""
    prompts = torch.split(prompt.double(), lens)
    x = torch.cat([torch.cat([p, torch.stack([s[i].double() for s in steps])]) for i, p in enumerate(prompts)])
    whole = [n + len(steps) for n in lens]
    return torch.stack([o[-len(steps):] for o in torch.split(_stack(stack, x, whole), whole)], 1)


def exact(case, seed):
    got, kind = _inputs(case, seed), case["kind"]
    if kind == "decode":
        return list(_behind(case["stack"], got["prompt"], got["lens"], list(got["x"])))
    if kind == "prefill":
        lens, starts = got["lens"], got["starts"]
        whole = [n + s for n, s in zip(lens, starts)]
        x = torch.cat([v for pair in zip(torch.split(got["prompt"], starts), torch.split(got["x"], lens)) for v in pair])
        return torch.cat([o[-n:] for o, n in zip(torch.split(_stack(case["stack"], x, whole), whole), lens)])
    if kind == "sample":
        return _sample(got["mu"], got["cond"], got["noise"], case["guidance"])
    if kind == "encode":
        return _encode(got["patches"])
    w, out, embeds, residuals, cond = _weights("heads"), [], [], [], got["cond"]
    for t in range(case["steps"]):
        embeds.append(_linear(_encode(cond), w, "enc_to_lm_proj"))
        base = _behind("backbone", got["prompt"], got["lens"], embeds)[-1]
        levels = torch.round(torch.tanh(_linear(base, w, "fsq_layer.in_proj")) * LEVELS) / LEVELS
        hidden = _linear(levels, w, "fsq_layer.out_proj")
        residuals.append(_linear(torch.cat([hidden, embeds[-1]], -1), w, "fusion_concat_proj"))
        residual = _behind("residual", got["residual_prompt"], got["lens"], residuals)[-1]
        mu = torch.stack([_linear(hidden, w, "lm_to_dit_proj"), _linear(residual, w, "res_to_dit_proj")], 1)
        stop = _linear(torch.nn.functional.silu(_linear(hidden, w, "stop_proj")), w, "stop_head", bias=False)
        cond = _sample(mu, cond, got["noise"][t], 2.0)
        out += [cond, stop]
    return out
