"""The work that this framework's speed is judged by: calls of its public entry points at the sizes its models, its tests and its
benchmark use, each with the inputs such a call meets, its result in 64 bits, and what it cannot do without.

`listed()` are the cases by name, `draw(rng)` makes others over the same ranges.  A case is a dict of plain values whose "kind" names
one of the functions below:

  generate            scoring of given tokens by the Based-360m: prompt, then one token at a time from the recorded graph
  linear_prefill      Taylor linear attention over prompts, decode state written (bfloat16, or float32 as the CPU reference runs it)
  linear_step         one decoding step of it, states updated in place
  sliding_prefill     sliding-window attention of the released Based models: packed qkv, rotary, cache fill
  recurrent_prefill   gated linear recurrent unit of Sozilix over prompts
  delta_prefill       gated delta rule of Sozilix over prompts
  window_prefill      grouped window attention of Sozilix over prompts, cache fill
  decay_prefill       linear attention with a decay per channel of Peponex over prompts
  experts             mixture of experts of Peponex: prompts, and the few tokens of a decoding step
  latent_step         one decoding step of Peponex's latent attention
"""
import math

import torch

from based_amd import ops
from based_amd.stack import GPTLMHeadModel, based_360m_released_config

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DTYPES = {"bf16": BF16, "f32": F32}
SIZES = {"bf16": 2, "f32": 4}


def listed():
    return [
        # Four requests answered by the released 360M model: the launches of a whole decoding step, one after the other.
        {"name": "generate", "kind": "generate", "B": 4, "L": 128, "new": 8},
        # A large batch of full-length prompts through one Based layer; the projections' (B, L, H * d) layout.
        {"name": "linear_prefill", "kind": "linear_prefill", "B": 32, "H": 16, "L": 4096, "dv": 64, "dtype": "bf16"},
        # The single float32 layer that the published implementation can run on a CPU: evaluation and debugging in full precision.
        {"name": "linear_prefill_f32", "kind": "linear_prefill", "B": 1, "H": 16, "L": 1024, "dv": 64, "dtype": "f32"},
        # Decoding of a large batch: every state read and written once a token.
        {"name": "linear_step", "kind": "linear_step", "B": 128, "H": 16, "dv": 64},
        # The window layer of the released 360M model over a batch of full-length prompts.
        {"name": "sliding_prefill", "kind": "sliding_prefill", "B": 8, "H": 16, "L": 4096, "D": 64, "w_left": 128},
        # A recurrent block of the 27-layer Sozilix model, a batch of prompts of 2048 tokens.
        {"name": "recurrent_prefill", "kind": "recurrent_prefill", "B": 4, "L": 2048, "W": 1024, "blocks": 8, "dtype": "bf16"},
        # The two halves of a parallel layer of the same model, the same prompts.
        {"name": "delta_prefill", "kind": "delta_prefill", "B": 4, "L": 2048, "H": 8, "d": 64, "dv": 128, "dtype": "bf16"},
        {"name": "window_prefill", "kind": "window_prefill", "B": 4, "L": 2048, "H": 16, "G": 4, "d": 64, "window": 129, "dtype": "bf16"},
        # A float32 replay of one request of ragged length.
        {"name": "window_prefill_f32", "kind": "window_prefill", "B": 1, "L": 777, "H": 16, "G": 4, "d": 64, "window": 129, "dtype": "f32"},
        # A time-mixing layer of the Peponex model, four prompts of 2048 tokens.
        {"name": "decay_prefill", "kind": "decay_prefill", "B": 4, "L": 2048, "H": 16, "d": 64, "dtype": "bf16"},
        # Its mixture of two of eight experts behind the same prompts.
        {"name": "experts", "kind": "experts", "n": 8192, "E": 8, "top": 2, "ff": 1024, "dtype": "bf16"},
        # One token of four requests with a full window: the smallest of the calls.
        {"name": "latent_step", "kind": "latent_step", "B": 4, "H": 16, "d": 64, "rot": 32, "R": 256, "window": 512, "dtype": "bf16"},
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _prompts(rng, tokens, longest):
    """Batch and length of a portion of up to `tokens` tokens, lengths of every kind: a few tokens, whole tiles, one more or less."""
    B = _spread(rng, 1, 32)
    L = _spread(rng, 3, min(longest, max(3, tokens // B)))
    if L >= 64 and rng.random() < 0.4:
        L = L // 64 * 64 + rng.choice((0, 0, 1, -1))
    return B, L


def draw(rng):
    kind = rng.choice(["generate", "linear_prefill", "linear_prefill", "linear_step", "sliding_prefill", "recurrent_prefill", "recurrent_prefill",
                       "delta_prefill", "delta_prefill", "window_prefill", "window_prefill", "decay_prefill", "decay_prefill", "experts",
                       "experts", "latent_step"])
    dtype = rng.choice(("bf16", "bf16", "bf16", "f32"))
    case = {"kind": kind}
    if kind == "generate":
        return {**case, "B": rng.randint(1, 4), "L": _spread(rng, 8, 128), "new": rng.randint(3, 8)}
    if kind == "linear_prefill":
        # float32 is a format of single requests here
        B, L = _prompts(rng, 2048, 1024) if dtype == "f32" else _prompts(rng, 65536, 8192)
        return {**case, "B": B, "H": 16, "L": L, "dv": rng.choice((64, 64, 112, 128)), "dtype": dtype}
    if kind == "linear_step":
        return {**case, "B": _spread(rng, 1, 128), "H": 16, "dv": rng.choice((64, 64, 112))}
    if kind == "sliding_prefill":
        B, L = _prompts(rng, 32768, 4096)
        return {**case, "B": B, "H": 16, "L": L, "D": rng.choice((64, 64, 112)), "w_left": rng.choice((64, 128))}
    if kind == "recurrent_prefill":
        B, L = _prompts(rng, 4096 if dtype == "f32" else 32768, 4096)
        return {**case, "B": B, "L": L, **rng.choice(({"W": 1024, "blocks": 8}, {"W": 768, "blocks": 12}, {"W": 1536, "blocks": 6})), "dtype": dtype}
    if kind == "delta_prefill":
        B, L = _prompts(rng, 4096 if dtype == "f32" else 16384, 4096)
        return {**case, "B": B, "L": L, "H": rng.choice((4, 8, 16)), "d": rng.choice((64, 128)), "dv": rng.choice((64, 128)), "dtype": dtype}
    if kind == "window_prefill":
        B, L = _prompts(rng, 2048 if dtype == "f32" else 16384, 4096)
        return {**case, "B": B, "L": L, "H": 16, "G": rng.choice((2, 4, 16)), "d": 64, "window": rng.choice((129, 129, 513, 1024)), "dtype": dtype}
    if kind == "decay_prefill":
        B, L = _prompts(rng, 2048 if dtype == "f32" else 16384, 4096)
        return {**case, "B": B, "L": L, **rng.choice(({"H": 16, "d": 64}, {"H": 8, "d": 128}, {"H": 12, "d": 64})), "dtype": dtype}
    if kind == "experts":
        n = _spread(rng, 1, 256 if dtype == "f32" else 8192)
        return {**case, "n": n, **rng.choice(({"E": 8, "top": 2, "ff": 1024}, {"E": 8, "top": 1, "ff": 2048}, {"E": 16, "top": 4, "ff": 512})),
                "dtype": dtype}
    return {**case, "B": _spread(rng, 1, 128), "H": 16, "d": 64, "rot": 32, "R": 256, "window": rng.choice((129, 512, 1024)), "dtype": dtype}


# ---- inputs ----
WIDTH = 1024       # width of the expert layers
EPS = 1e-5
CACHE_ROWS = 2048  # rows of a latent cache
MODEL_VOCAB = 50277


class _Random:
    """Tensors made on the GPU from one seed, in the order they are asked for."""

    def __init__(self, seed):
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.device).manual_seed(int(seed))

    def normal(self, *shape, dtype=F32, std=1.0, mean=0.0):
        return torch.empty(shape, device=self.device, dtype=F32).normal_(mean, std, generator=self.g).to(dtype)

    def integers(self, hi, *shape, lo=0):
        return torch.randint(lo, hi, shape, generator=self.g, device=self.device)


def _angles(rows, dims, device):
    """cos and sin of position * 10000^(-2i/dims), float32 (rows, dims / 2)."""
    a = torch.outer(torch.arange(rows, device=device, dtype=F64), 10000.0 ** (-torch.arange(0, dims, 2, device=device, dtype=F64) / dims))
    return a.cos().float().contiguous(), a.sin().float().contiguous()


def _model(seed):
    """The released Based-360m with weights drawn as its initialisation draws them."""
    r = _Random(seed)
    model = GPTLMHeadModel(based_360m_released_config(), device=r.device, dtype=BF16).eval()
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name or "ln_f" in name:
                p.copy_(1 + 0.1 * r.normal(*p.shape))
            elif "conv.conv.weight" in name:
                p.copy_(r.normal(*p.shape, std=0.5))
            else:
                p.copy_(r.normal(*p.shape, std=0.02))
    return model, r


def _inputs(case, seed):
    """What a case computes with, by name."""
    kind, r = case["kind"], _Random(seed)
    t = DTYPES[case.get("dtype", "bf16")]
    if kind == "linear_prefill":
        B, H, L, dv = case["B"], case["H"], case["L"], case["dv"]
        std = 1.0 if t == BF16 else 0.5
        return {"q": r.normal(B, L, H, 16, dtype=t, std=std).transpose(1, 2), "k": r.normal(B, L, H, 16, dtype=t, std=std).transpose(1, 2),
                "v": r.normal(B, L, H, dv, dtype=t).transpose(1, 2)}
    if kind == "linear_step":
        B, H, dv = case["B"], case["H"], case["dv"]
        keys = r.normal(H, 64, 16)  # the sums over the keys and values of a prompt of 64 tokens, another mixture of them in each request
        mix = torch.rand(B, 64, device=r.device, generator=r.g)
        phi = _features(keys)
        values = r.normal(H, dv, 64)
        kv = torch.stack([(values * mix[b]) @ phi for b in range(B)])
        ks = (mix @ phi.transpose(0, 1).reshape(64, -1)).view(B, H, -1)
        proj = r.normal(B, H * (32 + dv), dtype=BF16)
        return {"q": proj[:, :H * 16].view(B, H, 1, 16), "k": proj[:, H * 16:H * 32].view(B, H, 1, 16), "v": proj[:, H * 32:].view(B, H, 1, dv),
                "kv": kv.view(B, H, 1, dv, -1).contiguous(), "ks": ks.view(B, H, 1, 1, -1).contiguous()}
    if kind == "sliding_prefill":
        B, H, L, D = case["B"], case["H"], case["L"], case["D"]
        cos, sin = _angles(L, D, r.device)
        return {"qkv": r.normal(B, L, 3, H, D, dtype=BF16), "cos": cos, "sin": sin}
    if kind == "recurrent_prefill":
        B, L, W, n = case["B"], case["L"], case["W"], case["W"] // case["blocks"]
        gates = [r.normal(case["blocks"], n, n, dtype=t, std=n ** -0.5), r.normal(W, dtype=t), r.normal(case["blocks"], n, n, dtype=t, std=n ** -0.5),
                 r.normal(W, dtype=t), r.normal(W, dtype=t, std=1.5, mean=-3.0)]
        return {"u": r.normal(B, L, W, dtype=t), "y": r.normal(B, L, 2 * W, dtype=t)[..., :W], "gates": gates}
    if kind == "delta_prefill":
        B, L, H, d, dv = case["B"], case["L"], case["H"], case["d"], case["dv"]
        x = torch.nn.functional.silu(r.normal(B, L, H * (2 * d + dv))).to(t)
        ab = r.normal(B, L, 2 * H, dtype=t)
        return {"q": x[..., :H * d], "k": x[..., H * d:2 * H * d], "v": x[..., 2 * H * d:], "a": ab[..., :H], "b": ab[..., H:],
                "a_log": r.normal(H, dtype=t, mean=-2.0), "dt_bias": r.normal(H, dtype=t, std=0.7, mean=-2.0)}
    if kind == "window_prefill":
        B, L, H, G, d = case["B"], case["L"], case["H"], case["G"], case["d"]
        x = r.normal(B, L, (H + 2 * G) * d, dtype=t)
        cos, sin = _angles(L, 32, r.device)
        return {"q": x[..., :H * d], "k": x[..., H * d:(H + G) * d], "v": x[..., (H + G) * d:], "cos": cos, "sin": sin}
    if kind == "decay_prefill":
        B, L, H, d = case["B"], case["L"], case["H"], case["d"]
        # slow and fast channels, and tokens that forget more than others
        rate = r.normal(H * d, std=2.0, mean=-3.0) + r.normal(B, L, H * d)
        return {"q": r.normal(B, L, H * d, dtype=t), "k": r.normal(B, L, H * d, dtype=t), "v": r.normal(B, L, H * d, dtype=t),
                "log2": -rate.exp() * math.log2(math.e), "u": r.normal(H, d, dtype=t)}
    if kind == "experts":
        E, ff = case["E"], case["ff"]
        # tokens carry a mark of every expert, in an order of their own: a choice is no matter of the last digit
        marks = torch.linalg.qr(r.normal(WIDTH, E))[0].T
        order = torch.rand(case["n"], E, device=r.device, generator=r.g).argsort(-1)
        strength = torch.linspace(2.0, -2.0, E, device=r.device)[order] * WIDTH ** 0.5
        h = 0.7 * r.normal(case["n"], WIDTH) + (strength * 0.8) @ marks
        return {"h": h.to(t), "router": (marks * 3.0 * WIDTH ** -0.5).to(t), "w1": r.normal(E, 2 * ff, WIDTH, dtype=t, std=WIDTH ** -0.5),
                "w2": r.normal(E, WIDTH, ff, dtype=t, std=ff ** -0.5)}
    if kind == "latent_step":
        B, H, d, rot, R = case["B"], case["H"], case["d"], case["rot"], case["R"]
        cos, sin = _angles(CACHE_ROWS, rot, r.device)
        return {"q": r.normal(B, H * (rot + d), dtype=t), "x": r.normal(B, R + rot, dtype=t), "norm": r.normal(R, dtype=t, std=0.2, mean=1.0),
                "weight": r.normal(H * (rot + 2 * d), R + rot, dtype=t, std=R ** -0.5), "cache": r.normal(B, CACHE_ROWS, R + rot, dtype=t),
                "pos": r.integers(CACHE_ROWS, B, lo=CACHE_ROWS // 2).to(torch.int32), "cos": cos, "sin": sin}
    raise ValueError(kind)


def prepare(case, seed):
    if case["kind"] == "generate":
        model, r = _model(seed)
        tokens = r.integers(MODEL_VOCAB, case["B"], case["L"] + case["new"])
        state = {"case": case, "model": model, "prompt": tokens[:, :case["L"]].contiguous(), "tokens": tokens}
        run(state)  # a serving program has its graph recorded before requests come
        return state
    state = {"case": case, **_inputs(case, seed)}
    kind, B = case["kind"], case.get("B")
    if kind == "sliding_prefill":
        qkv = state["qkv"]
        state["cache"] = qkv.new_zeros(B, case["L"] + 64, 2, case["H"], case["D"])
    elif kind == "recurrent_prefill":
        state["state"] = torch.zeros(B, case["W"], device=state["u"].device)
        state["out"] = torch.empty_like(state["u"])
    elif kind == "delta_prefill":
        state["state"] = torch.zeros(B, case["H"], case["d"], case["dv"], device=state["q"].device)
    elif kind == "window_prefill":
        state["cache"] = state["q"].new_zeros(B, case["L"], case["G"], 2 * case["d"])
        state["out"] = torch.empty_like(state["q"], memory_format=torch.contiguous_format)
    elif kind == "decay_prefill":
        state["state"] = torch.zeros(B, case["H"], case["d"], case["d"], device=state["q"].device)
    elif kind == "latent_step":
        state["out"] = state["q"].new_empty(B, case["H"] * case["d"])
    return state


@torch.inference_mode()
def run(state):
    case = state["case"]
    kind, s = case["kind"], state
    if kind == "generate":
        out = s["model"].generate(s["prompt"], max_length=case["L"] + case["new"], cg=True, teacher_outputs=s["tokens"],
                                  return_dict_in_generate=True, output_scores=True)
        return {"sequences": out.sequences, "scores": out.scores}
    if kind == "linear_prefill":
        return ops.linear_attn_prefill(s["q"], s["k"], s["v"], return_state=True)
    if kind == "linear_step":
        return ops.linear_attn_step(s["q"], s["k"], s["v"], s["kv"], s["ks"]), s["kv"], s["ks"]
    if kind == "sliding_prefill":
        q, k, v = s["qkv"].unbind(2)
        return ops.swa_prefill(q, k, v, w_left=case["w_left"], rope=(s["cos"], s["sin"]), kv_cache=s["cache"]), s["cache"]
    if kind == "recurrent_prefill":
        return ops.rglru_prefill(s["u"], s["y"], *s["gates"], s["state"], 8.0, True, out=s["out"]), s["state"]
    if kind == "delta_prefill":
        o = ops.gated_delta_scan(s["q"], s["k"], s["v"], s["a"], s["b"], s["a_log"], s["dt_bias"], s["state"], case["H"], case["H"], True)
        return o, s["state"]
    if kind == "window_prefill":
        ops.window_attn_prefill(s["q"], s["k"], s["v"], s["cache"], case["H"], case["G"], case["window"], case["d"] ** -0.5, 0,
                                rope=(s["cos"], s["sin"], True), value_norm_eps=EPS, out=s["out"])
        return s["out"], s["cache"]
    if kind == "decay_prefill":
        return ops.decay_scan(s["q"], s["k"], s["v"], s["state"], case["H"], channel_log2=s["log2"], bonus=s["u"], fresh=True), s["state"]
    if kind == "experts":
        return ops.experts(s["h"], s["router"], s["w1"], s["w2"], case["top"])
    ops.latent_step(s["q"], s["x"], s["norm"], s["weight"], s["cache"], case["H"], case["d"], case["window"], (case["d"] + case["rot"]) ** -0.5,
                    s["pos"], EPS, (s["cos"], s["sin"], False), out=s["out"])
    return s["out"], s["cache"]


def work(case):
    kind, e = case["kind"], SIZES[case.get("dtype", "bf16")]
    if kind == "generate":
        # every weight once a token (tied embedding included), two operations each for every token
        params, tokens = 363e6, case["B"] * (case["L"] + case["new"])
        return {"bytes": int(params * 2 * case["new"]), "flops": int(2 * params * tokens)}
    if kind == "experts":
        used = min(case["E"], case["n"] * case["top"])
        flops = case["n"] * (case["top"] * 6 * case["ff"] * WIDTH + 2 * case["E"] * WIDTH)
        return {"bytes": e * (2 * case["n"] * WIDTH + used * 3 * case["ff"] * WIDTH + case["E"] * WIDTH), "flops": flops}
    B, H, L = case["B"], case.get("H", 1), case.get("L", 1)
    N = B * L
    if kind == "linear_prefill":
        dv = case["dv"]
        return {"bytes": N * H * (32 + 2 * dv) * e + B * H * 273 * (dv + 1) * 4, "flops": N * H * 4 * 273 * (dv + 1)}
    if kind == "linear_step":
        dv = case["dv"]
        return {"bytes": B * H * (2 * 273 * (dv + 1) * 4 + (32 + 2 * dv) * 2), "flops": B * H * 4 * 273 * (dv + 1)}
    if kind == "sliding_prefill":
        D, seen = case["D"], _seen(L, case["w_left"] + 1)
        return {"bytes": N * H * D * 6 * 2 + L * D * 4, "flops": B * H * seen * 4 * D}
    if kind == "recurrent_prefill":
        W, n = case["W"], case["W"] // case["blocks"]
        return {"bytes": N * W * 3 * e + 2 * W * n * e + B * W * 4, "flops": N * W * (4 * n + 30)}
    if kind == "delta_prefill":
        d, dv = case["d"], case["dv"]
        return {"bytes": N * H * ((2 * d + dv + 2) * e + dv * 4) + B * H * d * dv * 4, "flops": N * H * 6 * d * dv}
    if kind == "window_prefill":
        G, d = case["G"], case["d"]
        return {"bytes": N * (2 * H + 4 * G) * d * e + L * 32 * 4, "flops": B * H * _seen(L, case["window"]) * 4 * d}
    if kind == "decay_prefill":
        d = case["d"]
        return {"bytes": N * H * d * (4 * e + 4) + B * H * d * d * 4, "flops": N * H * 4 * d * d}
    d, rot, R, window = case["d"], case["rot"], case["R"], min(case["window"], CACHE_ROWS // 2)
    return {"bytes": e * (B * window * (R + rot) + B * H * (rot + 2 * d) + H * 2 * d * R),
            "flops": 2 * B * H * (2 * d * R + window * (2 * R + rot))}


def _seen(L, window):
    """Pairs of a query and a key that it sees."""
    full = max(0, L - window)
    short = L - full
    return full * window + short * (short + 1) // 2


def tolerance(case):
    # About four times what the kernels show against `exact` over the declared ranges (in brackets).
    kind = case["kind"]
    if kind == "generate":
        return {"rel": 0.12}    # (3e-2) 27 layers of bf16 activations
    if kind == "delta_prefill":
        return {"rel": 1.5e-6}  # (2.3e-7) outputs and states are 32-bit sums for both types of inputs
    if case.get("dtype", "bf16") == "f32":
        return {"rel": 1.5e-5}  # (3.5e-6) products of thousands of 32-bit decays
    return {"rel": 1.2e-2}      # (3.1e-3) bf16 results of matrix products with bf16 operands


# ---- results in 64 bits ----
def _features(x):
    """1, x / d^(1/4), x_i x_j / sqrt(2 d) of rows of 16."""
    d = x.shape[-1]
    second = (x[..., :, None] * x[..., None, :]).flatten(-2) / math.sqrt(2.0 * d)
    return torch.cat([torch.ones_like(x[..., :1]), x / d ** 0.25, second], -1)


def _linear_attention(q, k, v, eps=1e-12):
    """One request: q, k (H, L, 16), v (H, L, dv) in 64 bits."""
    L, y = q.shape[1], []
    for at in range(0, L, 1024):
        end = min(at + 1024, L)
        s = q[:, at:end] @ k[:, :end].transpose(1, 2) / 4
        a = torch.tril(1 + s + s * s / 2, diagonal=at)
        y.append(a @ v[:, :end] / (a.sum(-1, keepdim=True) + eps))
    return torch.cat(y, 1)


def _turn(x, cos, sin, interleaved):
    """x (..., L, heads, D): the first 2 * cos.shape[1] channels turned; cos, sin (L, pairs)."""
    n, out = cos.shape[-1], x.clone()
    c, s = cos.to(x.dtype)[:, None], sin.to(x.dtype)[:, None]
    first, second = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if interleaved else (slice(0, n), slice(n, 2 * n))
    out[..., first] = x[..., first] * c - x[..., second] * s
    out[..., second] = x[..., second] * c + x[..., first] * s
    return out


def _window_attention(q, k, v, window, scale):
    """One request: q (L, H, d), k (L, G, d), v (L, G, dv) in 64 bits; position i sees i - window + 1 .. i."""
    L, H, G, out = q.shape[0], q.shape[1], k.shape[1], []
    for at in range(0, L, 512):
        end, lo = min(at + 512, L), max(0, at - window + 1)
        kk, vv = (x[lo:end].repeat_interleave(H // G, 1).transpose(0, 1) for x in (k, v))
        gap = torch.arange(at, end, device=q.device)[:, None] - torch.arange(lo, end, device=q.device)[None]
        s = (q[at:end].transpose(0, 1) @ kk.transpose(1, 2) * scale).masked_fill((gap < 0) | (gap >= window), float("-inf"))
        out.append((s.softmax(-1) @ vv).transpose(0, 1))
    return torch.cat(out)


def _rms(x, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()


def _exact_model(model, tokens):
    """Logits of the Based-360m for every position of tokens (B, T), from its named weights."""
    c, F = model.config, torch.nn.functional
    w = {name: p.detach() for name, p in model.named_parameters()}
    get = lambda name: w[name].to(F64)

    def linear(x, name):
        y = x @ get(name + ".weight").T
        return y + get(name + ".bias") if name + ".bias" in w else y

    eps, H, D = c.layer_norm_epsilon, c.n_head, c.n_embd
    x = get("transformer.embeddings.word_embeddings.weight")[tokens]
    B, T = tokens.shape
    cos, sin = _angles(T, D // H, tokens.device)
    for i in range(c.n_layer):
        p = f"transformer.layers.{i}."
        h = _rms(x, eps) * get(p + "norm1.weight")
        m = p + "mixer."
        if m + "in_proj.weight" in w:
            u, gate = linear(h, m + "in_proj").chunk(2, -1)
            taps = get(m + "conv.conv.weight")[:, 0]
            past = F.pad(u, (0, 0, taps.shape[1] - 1, 0))
            y = sum(past[:, j:j + T] * taps[:, j] for j in range(taps.shape[1]))
            if m + "conv.conv.bias" in w:
                y = y + get(m + "conv.conv.bias")
            y = F.silu(y) * gate
        elif m + "proj_q.weight" in w:
            q, k, v = (linear(h, m + f"proj_{n}").view(B, T, H, -1).transpose(1, 2) for n in "qkv")
            y = torch.stack([_linear_attention(q[b], k[b], v[b], 1e-6) for b in range(B)]).transpose(1, 2).reshape(B, T, D)
        else:
            qkv = linear(h, m + "Wqkv").view(B, T, 3, H, -1)
            q, k, v = _turn(qkv[:, :, 0], cos, sin, False), _turn(qkv[:, :, 1], cos, sin, False), qkv[:, :, 2]
            window = c.alt_mixer_2["window_size"] // 2 + 1
            y = torch.stack([_window_attention(q[b], k[b], v[b], window, (D // H) ** -0.5) for b in range(B)]).reshape(B, T, D)
        x = x + linear(y, m + "out_proj")
        h = _rms(x, eps) * get(p + "norm2.weight")
        up, gate = linear(h, p + "mlp.fc1").chunk(2, -1)
        x = x + linear(up * F.silu(gate), p + "mlp.fc2")
    return (_rms(x, eps) * get("transformer.ln_f.weight")) @ get("transformer.embeddings.word_embeddings.weight").T


@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    if kind == "generate":
        model, r = _model(seed)
        tokens = r.integers(MODEL_VOCAB, case["B"], case["L"] + case["new"])
        logits = _exact_model(model, tokens[:, :-1])
        return {"sequences": tokens, "scores": tuple(logits[:, case["L"] - 1 + i] for i in range(case["new"]))}
    s = _inputs(case, seed)
    d64 = lambda name: s[name].to(F64)
    if kind == "linear_prefill":
        y, kv, ks = [], [], []
        for b in range(case["B"]):
            q, k, v = (s[n][b].to(F64) for n in "qkv")
            y.append(_linear_attention(q, k, v).to(F32))
            phi = [_features(part) for part in k.split(4096, 1)]
            kv.append(sum(vp.transpose(1, 2) @ f for vp, f in zip(v.split(4096, 1), phi)))
            ks.append(sum(f.sum(1) for f in phi))
        return torch.stack(y), torch.stack(kv)[:, :, None], torch.stack(ks)[:, :, None, None]
    if kind == "linear_step":
        phi = _features(d64("k"))
        kv = d64("kv") + d64("v")[..., None] * phi[:, :, :, None]
        ks = d64("ks") + phi[:, :, :, None]
        fq = _features(d64("q"))
        y = (kv @ fq[..., None])[..., 0] / ((ks @ fq[..., None])[..., 0] + 1e-12)
        return y, kv, ks
    if kind == "sliding_prefill":
        out, L = [], case["L"]
        cache = torch.zeros(case["B"], L + 64, 2, case["H"], case["D"], dtype=F32, device=s["qkv"].device)
        for b in range(case["B"]):
            q, k, v = s["qkv"][b].to(F64).unbind(1)
            q, k = _turn(q, s["cos"], s["sin"], False), _turn(k, s["cos"], s["sin"], False)
            cache[b, :L, 0], cache[b, :L, 1] = k, v
            out.append(_window_attention(q, k, v, case["w_left"] + 1, case["D"] ** -0.5).to(F32))
        return torch.stack(out), cache
    if kind == "recurrent_prefill":
        ra, rb, ri, ib, lam = (g.to(F64) for g in s["gates"])
        u = d64("u")
        parts = u.view(*u.shape[:2], case["blocks"], -1)
        r = torch.sigmoid(torch.einsum("blkn,kmn->blkm", parts, ra).flatten(2) + rb)
        i = torch.sigmoid(torch.einsum("blkn,kmn->blkm", parts, ri).flatten(2) + ib)
        log_a = -8.0 * r * torch.nn.functional.softplus(lam)
        a, x = log_a.exp(), (-torch.expm1(2 * log_a)).sqrt() * i * u
        S, out = torch.zeros_like(u[:, 0]), torch.empty_like(u)
        for t in range(case["L"]):
            S = a[:, t] * S + x[:, t]
            out[:, t] = S
        return out * torch.nn.functional.gelu(d64("y"), approximate="tanh"), S
    if kind == "delta_prefill":
        B, L, H, d, dv = (case[n] for n in ("B", "L", "H", "d", "dv"))
        unit = lambda x: x / (x.square().sum(-1, keepdim=True) + 1e-6).sqrt()
        q, k, v = unit(d64("q").view(B, L, H, d)) * d ** -0.5, unit(d64("k").view(B, L, H, d)), d64("v").view(B, L, H, dv)
        beta = torch.sigmoid(d64("b"))
        g = torch.exp(-torch.exp(d64("a_log")) * torch.nn.functional.softplus(d64("a") + d64("dt_bias")))
        S, out = torch.zeros(B, H, d, dv, dtype=F64, device=q.device), torch.empty(B, L, H, dv, dtype=F64, device=q.device)
        for t in range(L):
            S = S * g[:, t, :, None, None]
            u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S)[:, :, 0])
            S = S + k[:, t, :, :, None] * u[:, :, None]
            out[:, t] = (q[:, t, :, None] @ S)[:, :, 0]
        return out, S
    if kind == "window_prefill":
        B, L, H, G, d = (case[n] for n in ("B", "L", "H", "G", "d"))
        q = _turn(d64("q").view(B, L, H, d), s["cos"], s["sin"], True)
        k, v = _turn(d64("k").view(B, L, G, d), s["cos"], s["sin"], True), _rms(d64("v").view(B, L, G, d), EPS)
        out = torch.stack([_window_attention(q[b], k[b], v[b], case["window"], d ** -0.5) for b in range(B)])
        return out.view(B, L, H * d), torch.cat([k, v], -1)
    if kind == "decay_prefill":
        B, L, H, d = (case[n] for n in ("B", "L", "H", "d"))
        q, k, v, w = (x.view(B, L, H, d) for x in (d64("q"), d64("k"), d64("v"), d64("log2").exp2()))
        bonus = (q * d64("u") * k).sum(-1, keepdim=True) * v
        S, out = torch.zeros(B, H, d, d, dtype=F64, device=q.device), torch.empty(B, L, H, d, dtype=F64, device=q.device)
        for t in range(L):  # by value channel: S[.., value, key]
            out[:, t] = (S @ q[:, t, :, :, None])[..., 0]
            S = S * w[:, t, :, None] + v[:, t, :, :, None] * k[:, t, :, None]
        return (out + bonus).view(B, L, H * d), S
    if kind == "experts":
        h, router = d64("h"), d64("router")
        score, pick = torch.sigmoid(h @ router.T).topk(case["top"], -1)
        y = torch.zeros_like(h)
        for e in range(case["E"]):
            row, choice = (pick == e).nonzero(as_tuple=True)
            if row.numel():
                up, gate = (score[row, choice, None] * h[row] @ s["w1"][e].to(F64).T).chunk(2, -1)
                y.index_add_(0, row, (up * torch.nn.functional.silu(gate)) @ s["w2"][e].to(F64).T)
        return y
    B, H, d, rot, R = (case[n] for n in ("B", "H", "d", "rot", "R"))
    cache, at, out = d64("cache"), s["pos"].tolist(), []
    weight = d64("weight").view(H, rot + 2 * d, -1)[..., :R]
    for b, p in enumerate(at):
        turn = lambda x: _turn(x[None], s["cos"][p:p + 1], s["sin"][p:p + 1], False)[0]
        x = s["x"][b].to(F64)
        cache[b, p] = torch.cat([_rms(x[:R], EPS) * d64("norm"), turn(x[None, R:])[0]])
        rows = cache[b, max(0, p - case["window"] + 1):p + 1]
        q = s["q"][b].to(F64).view(H, rot + d)
        q = torch.cat([turn(q[:, :rot]), q[:, rot:]], -1)
        k = torch.cat([rows[:, R:].expand(H, -1, -1), rows[:, :R] @ weight[:, rot:rot + d].transpose(1, 2)], -1)
        weights = ((k @ q[..., None])[..., 0] * (d + rot) ** -0.5).softmax(-1)
        out.append((weights[:, None] @ (rows[:, :R] @ weight[:, rot + d:].transpose(1, 2)))[:, 0])
    return torch.stack(out).view(B, H * d), cache
