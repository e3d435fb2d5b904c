"""The work this library does for a speech-to-text server, as cases to time.

Every case is one pass through a public entry point with the inputs a server
has in hand at that moment: attention modules called on activations whose
sizes change from batch to batch (prompt passes, SenseVoice's utterances;
eager, as the model code calls them), and work of fixed sizes replayed from a
captured graph (decoder steps, as the decoders run them, and Whisper's encoder
attention, always 1500 frames).  ``listed()`` names
the cases, ``draw`` gives more of the same ranges, ``exact`` computes a
case's outputs in float64 with plain torch.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from asrback_amd import attention, gemma4, qwen3_asr, sensevoice, whisper
from asrback_amd.attention import KeyPrefix
from asrback_amd.transcription import CapturedGraph

# Whisper sizes: width, attention heads (head_dim 64), decoder layers.
WHISPER = {"tiny": (384, 6, 4), "base": (512, 8, 6), "small": (768, 12, 12), "turbo": (1280, 20, 4)}
FRAMES = 1500  # encoder frames of a 30 s window
VOCAB = 51865
KV_BUCKETS = (64, 128, 256, 448)
# Qwen3-1.7B's attention: 16 query heads over 8 kv heads of 128.
QWEN3 = {"hidden_size": 2048, "head_dim": 128, "num_attention_heads": 16, "num_key_value_heads": 8,
         "rms_norm_eps": 1e-6, "rope_theta": 1e6, "num_hidden_layers": 1}
SLOTS = qwen3_asr.CACHE_LENGTH
PAGE = 64
# SenseVoiceSmall's SAN-M: width 512, 4 heads, FSMN filters of 11 frames.
SANM = (512, 4, 11)
# Gemma 4's text attention: 8 query heads over 4 kv heads, sliding layers of
# head_dim 256 within 512 keys, full layers of head_dim 512.
GEMMA = {"hidden_size": 2048, "head_dim": 256, "global_head_dim": 512, "num_attention_heads": 8,
         "num_key_value_heads": 4, "sliding_window": 512, "rms_norm_eps": 1e-6,
         "rope_parameters": {
             "sliding_attention": {"rope_type": "default", "rope_theta": 1e4},
             "full_attention": {"rope_type": "proportional", "rope_theta": 1e6, "partial_rotary_factor": 0.25}}}


def listed() -> list[dict]:
    return [
        # One live stream on the smallest model in float32: a whole decoder
        # step (4 layers, the head, the greedy choice).  Latency and launches.
        {"name": "decoder-step-f32-1", "kind": "decoder_step", "size": "tiny", "rows": 1, "last": 200},
        # Whisper-small at the server's default batch: the attention of a step,
        # self (cache write included) and cross over the window's frames.
        {"name": "whisper-step-16", "kind": "whisper_step", "size": "small", "rows": 16, "last": 223, "dtype": "bf16"},
        # Qwen3-ASR decoding few windows from a paged cache (light load).
        {"name": "qwen3-step-paged-4", "kind": "qwen3_step", "rows": 4, "low": 400, "high": 560, "paged": True,
         "layers": 28},
        # The same model at its full batch over the slab cache.
        {"name": "qwen3-step-64", "kind": "qwen3_step", "rows": 64, "low": 400, "high": 560, "paged": False,
         "layers": 7},
        # Admission of eight Whisper windows: the four-token prompt attends
        # over every window's frames.
        {"name": "whisper-prompt-8", "kind": "whisper_prompt", "size": "small", "rows": 8, "tokens": 4,
         "dtype": "bf16"},
        # Qwen3-ASR's prompt pass over eight 30 s windows packed back to back.
        {"name": "qwen3-prompt-8", "kind": "qwen3_prompt", "rows": 8, "low": 400, "high": 430},
        # Encoder attention (four layers' calls) of one window (latency) and of
        # a full batch (throughput; the largest case), large-v3-turbo's width.
        {"name": "whisper-encoder-1", "kind": "whisper_encoder", "size": "turbo", "rows": 1, "layers": 4,
         "dtype": "bf16"},
        {"name": "whisper-encoder-16", "kind": "whisper_encoder", "size": "turbo", "rows": 16, "layers": 4,
         "dtype": "bf16"},
        # The same in float32 at the smallest width.
        {"name": "whisper-encoder-f32-1", "kind": "whisper_encoder", "size": "tiny", "rows": 1, "layers": 4,
         "dtype": "f32"},
        # SenseVoice: a ragged batch of 32 utterances, and a single one.
        {"name": "sensevoice-32", "kind": "sensevoice", "rows": 32, "low": 104, "high": 504},
        {"name": "sensevoice-1", "kind": "sensevoice", "rows": 1, "low": 300, "high": 300},
        # Gemma 4's prompt pass of two windows on a sliding layer.
        {"name": "gemma4-prompt-2", "kind": "gemma4_prompt", "rows": 2, "low": 800, "high": 840, "full": False,
         "dtype": "bf16"},
    ]


def _spread(rng, low: int, high: int) -> int:
    """A whole number of [low, high], spread over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.5))))))


def draw(rng) -> dict:
    kind = rng.choice(["decoder_step", "whisper_step", "qwen3_step", "whisper_prompt", "qwen3_prompt",
                       "whisper_encoder", "sensevoice", "gemma4_prompt"])
    case: dict = {"kind": kind}
    if kind == "decoder_step":
        case.update(size="tiny", rows=_spread(rng, 1, 6), last=_spread(rng, 5, 447))
    elif kind == "whisper_step":
        case.update(size=rng.choice(list(WHISPER)), rows=_spread(rng, 1, 16), last=_spread(rng, 5, 447),
                    dtype=rng.choice(["bf16", "bf16", "f32"]))
    elif kind == "qwen3_step":
        low = _spread(rng, 20, 600)
        case.update(rows=_spread(rng, 1, 64), low=low, high=min(SLOTS - 1, low + rng.randint(1, 300)),
                    paged=rng.random() < 0.5, layers=7)
    elif kind == "whisper_prompt":
        case.update(size=rng.choice(list(WHISPER)), rows=_spread(rng, 1, 16), tokens=_spread(rng, 2, 64),
                    dtype=rng.choice(["bf16", "bf16", "f32"]))
    elif kind == "qwen3_prompt":
        low = _spread(rng, 20, 400)
        case.update(rows=_spread(rng, 1, 12), low=low, high=low + rng.randint(1, 80))
    elif kind == "whisper_encoder":
        size, dtype = rng.choice([("tiny", "bf16"), ("tiny", "f32"), ("base", "f32"), ("base", "bf16"),
                                  ("small", "bf16"), ("turbo", "bf16")])
        case.update(size=size, dtype=dtype, rows=_spread(rng, 1, 3 if dtype == "f32" else 15),
                    layers=rng.choice([2, 3] if dtype == "f32" else [2, 3, 5]))
    elif kind == "sensevoice":
        low = _spread(rng, 24, 400)
        case.update(rows=_spread(rng, 1, 32), low=low, high=min(504, low + rng.randint(1, 400)))
    else:
        dtype = rng.choice(["bf16", "bf16", "f32"])
        low = _spread(rng, 100, 400 if dtype == "f32" else 800)
        case.update(rows=1 if dtype == "f32" else _spread(rng, 1, 4), low=low, high=low + rng.randint(1, 40),
                    full=rng.random() < 0.25, dtype=dtype)
    return case


# --- inputs ---------------------------------------------------------------


class _Rng:
    """Seeded values on the GPU."""

    def __init__(self, seed: int) -> None:
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std: float = 1.0) -> torch.Tensor:
        x = torch.empty(shape, dtype=dtype, device="cuda")
        return x.normal_(0.0, std, generator=self.g)

    def ints(self, low: int, high: int, *shape) -> torch.Tensor:
        return torch.randint(low, high + 1, shape, device="cuda", generator=self.g)


def _dtype(case: dict) -> torch.dtype:
    return torch.float32 if case.get("dtype") == "f32" or case["kind"] == "decoder_step" else torch.bfloat16


def _lengths(case: dict, seed: int) -> list[int]:
    """Sequence lengths of the case's rows: low to high in even steps (the
    same total for every seed), in an order of the seed's."""
    low, high, rows = case["low"], case["high"], case["rows"]
    n = [high - (high - low) * i // max(1, rows - 1) for i in range(rows)]
    order = torch.randperm(rows, generator=torch.Generator().manual_seed(seed + 1)).tolist()
    return [n[i] for i in order]


# Queries and keys are projected with this gain, for attention that picks
# some keys over others (scores of standard deviation ~2).
_PEAK = 1.5


def _fill(module: torch.nn.Module, rng: _Rng) -> torch.nn.Module:
    """Seeded weights: matrices of variance 1 / inputs (queries and keys with
    the gain above), norm weights near one, biases near zero."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if "norm" in name and name.endswith("weight"):
                p.normal_(1.0, 0.1, generator=rng.g)
            elif name.endswith("bias"):
                p.normal_(0.0, 0.1, generator=rng.g)
            elif "embed" in name:
                p.normal_(0.0, 0.3, generator=rng.g)
            elif "fsmn" in name:
                p.normal_(0.0, 0.3, generator=rng.g)
            else:
                gain = _PEAK if any(s in name for s in ("q_proj", "k_proj")) and "qkv" not in name else 1.0
                p.normal_(0.0, gain * p.shape[-1] ** -0.5, generator=rng.g)
    return module.requires_grad_(False).eval()


def _whisper_config(size: str) -> dict:
    width, heads, layers = WHISPER[size]
    return {"d_model": width, "encoder_attention_heads": heads, "decoder_attention_heads": heads,
            "encoder_layers": 0, "decoder_layers": layers, "encoder_ffn_dim": 4 * width, "decoder_ffn_dim": 4 * width,
            "vocab_size": VOCAB, "num_mel_bins": 80, "max_source_positions": FRAMES, "max_target_positions": 448}


def _bucket(case: dict) -> int:
    """The key bucket a decoder takes for rows up to position ``last``."""
    return next(b for b in KV_BUCKETS if b > case["last"])


def _positions(case: dict, rng: _Rng) -> torch.Tensor:
    """Positions past a four-token prompt; row 0 is the furthest."""
    positions = rng.ints(4, case["last"], case["rows"])
    positions[0] = case["last"]
    return positions


def _inputs(case: dict, seed: int) -> dict:
    rng = _Rng(seed)
    kind, dtype, rows = case["kind"], _dtype(case), case["rows"]
    s: dict = {"case": case}
    if kind == "decoder_step":
        with torch.device("cuda"):
            model = whisper.WhisperForConditionalGeneration(_whisper_config(case["size"]))
        s["model"] = _fill(model, rng)
        width, heads, layers = WHISPER[case["size"]]
        shape = (layers, rows, heads, KV_BUCKETS[-1], 64)
        cross = (layers, rows, heads, FRAMES, 64)
        cache = whisper.DecoderCache(*(rng.normal(*c, dtype=dtype) for c in (shape, shape, cross, cross)))
        s["cache"] = cache.narrow(rows, _bucket(case))
        s["tokens"] = rng.ints(0, VOCAB - 1, rows, 1)
        s["positions"] = _positions(case, rng)
        s["suppress"] = torch.zeros(VOCAB, dtype=torch.bool, device="cuda")
        s["suppress"][rng.ints(0, VOCAB - 1, 90)] = True
    elif kind == "whisper_step":
        width, heads, layers = WHISPER[case["size"]]
        s["layers"] = layers
        s["q"] = rng.normal(layers, 2, rows, heads, 64, dtype=dtype, std=_PEAK)
        s["new"] = rng.normal(layers, 2, rows, heads, 64, dtype=dtype)
        s["self"] = rng.normal(layers, 2, rows, heads, KV_BUCKETS[-1], 64, dtype=dtype)[..., : _bucket(case), :]
        s["cross"] = rng.normal(layers, 2, rows, heads, FRAMES, 64, dtype=dtype)
        s["positions"] = _positions(case, rng)
    elif kind == "qwen3_step":
        hd, hq, hkv = QWEN3["head_dim"], QWEN3["num_attention_heads"], QWEN3["num_key_value_heads"]
        layers = case["layers"]
        n = _lengths(case, seed)
        s["positions"] = torch.tensor(n, device="cuda")
        s["qkv"] = rng.normal(layers, rows, (hq + 2 * hkv) * hd, dtype=dtype)
        s["norms"] = rng.normal(layers, 2, hd, dtype=torch.float32, std=0.1).add_(1.0).to(dtype)
        cos, sin = qwen3_asr.rope_tables(QWEN3, SLOTS, torch.device("cuda"), dtype)
        s["cos"], s["sin"] = cos[s["positions"]], sin[s["positions"]]
        if case["paged"]:
            used = [-(-(x + 1) // PAGE) for x in n]
            pool = rows * SLOTS // PAGE
            order = torch.randperm(pool, generator=torch.Generator().manual_seed(seed + 2)).to(torch.int32)
            table = torch.full((rows, SLOTS // PAGE), -1, dtype=torch.int32)
            at = 0
            for b, count in enumerate(used):
                table[b, :count] = order[at : at + count]
                at += count
            s["pages"] = attention.PageTable(table.cuda(), SLOTS)
            s["kv"] = rng.normal(layers, 2, pool, PAGE, hkv, hd, dtype=dtype)
        else:
            s["pages"] = None
            s["kv"] = rng.normal(layers, 2, rows, SLOTS, hkv, hd, dtype=dtype)
    elif kind == "whisper_prompt":
        width, heads, _ = WHISPER[case["size"]]
        with torch.device("cuda"):
            module = whisper.MultiHeadAttention(width, heads)
        s["module"] = _fill(module.to(dtype), rng)
        s["x"] = rng.normal(rows, case["tokens"], width, dtype=dtype)
        s["key"], s["value"] = (rng.normal(rows, heads, FRAMES, 64, dtype=dtype) for _ in range(2))
    elif kind == "whisper_encoder":
        # Each layer's projections, (rows, frames, width), viewed as heads.
        width, heads, _ = WHISPER[case["size"]]
        s["q"] = rng.normal(case["layers"], rows, FRAMES, width, dtype=dtype, std=_PEAK)
        s["k"], s["v"] = (rng.normal(case["layers"], rows, FRAMES, width, dtype=dtype) for _ in range(2))
    elif kind == "qwen3_prompt":
        with torch.device("cuda"):
            module = qwen3_asr.TextAttention(QWEN3)
        s["module"] = _fill(module.to(dtype), rng)
        n = _lengths(case, seed)
        s["lengths"] = n
        s["x"] = rng.normal(sum(n), QWEN3["hidden_size"], dtype=dtype)
        shape = (rows, SLOTS, QWEN3["num_key_value_heads"], QWEN3["head_dim"])
        s["keys"], s["values"] = (torch.zeros(shape, dtype=dtype, device="cuda") for _ in range(2))
        s["rows"] = torch.repeat_interleave(torch.arange(rows), torch.tensor(n)).cuda()
        s["positions"] = torch.cat([torch.arange(k) for k in n]).cuda()
        s["segments"] = qwen3_asr.Segments.from_lengths(n, torch.device("cuda"))
        cos, sin = qwen3_asr.rope_tables(QWEN3, SLOTS, torch.device("cuda"), dtype)
        s["cos"], s["sin"] = cos[s["positions"]], sin[s["positions"]]
    elif kind == "sensevoice":
        size, heads, taps = SANM
        with torch.device("cuda"):
            module = sensevoice.SANMAttention(size, size, heads, taps)
        s["module"] = _fill(module.to(dtype), rng)
        n = _lengths(case, seed)
        s["x"] = rng.normal(rows, max(n), size, dtype=dtype)
        s["lengths"] = s["mask"] = None
        if rows > 1:
            s["lengths"] = torch.tensor(n, dtype=torch.int32, device="cuda")
            s["mask"] = torch.arange(max(n), device="cuda")[None, :] < s["lengths"][:, None]
    else:
        layer_type = "full_attention" if case["full"] else "sliding_attention"
        with torch.device("cuda"):
            module = gemma4.TextAttention(GEMMA, layer_type, shared=False)
        s["module"] = _fill(module.to(dtype), rng)
        # Queries and keys leave their norms with unit variance and there is
        # no 1 / sqrt(head_dim): trained norm weights hold the scores down.
        with torch.no_grad():
            module.q_norm.weight.mul_(2.0 * module.head_dim**-0.5)
        n = _lengths(case, seed)
        length = max(n)
        s["lengths"] = torch.tensor(n, dtype=torch.int32, device="cuda")
        s["x"] = rng.normal(rows, length, GEMMA["hidden_size"], dtype=dtype)
        cos, sin = (t.to("cuda", dtype) for t in gemma4.rotary_tables(GEMMA, layer_type, module.head_dim, length))
        s["cos"], s["sin"] = cos, sin
        shape = (rows, SLOTS, GEMMA["num_key_value_heads"], module.head_dim)
        s["cache"] = gemma4.LayerKV(*(torch.zeros(shape, dtype=dtype, device="cuda") for _ in range(2)))
        s["rows"] = torch.arange(rows, device="cuda")
    return s


# --- the passes -----------------------------------------------------------


@torch.inference_mode()
def prepare(case: dict, seed: int) -> dict:
    s = _inputs(case, seed)
    step = _STEPS.get(case["kind"])
    if step is not None:
        # Captured once per bucket, the split partials in a buffer the program
        # owns.
        need = _workspace_bytes(case)
        s["workspace"] = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")

        def call() -> None:
            with attention.workspace(s["workspace"]):
                s["out"] = step(s)

        s["graph"] = CapturedGraph(call)
    return s


@torch.inference_mode()
def run(s: dict):
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    return _CALLS[s["case"]["kind"]](s)


def _workspace_bytes(case: dict) -> int:
    size = attention.decode_workspace_size
    rows, dtype = case["rows"], _dtype(case)
    if case["kind"] == "whisper_encoder":
        return 0
    if case["kind"] == "qwen3_step":
        return size(rows, QWEN3["num_attention_heads"], QWEN3["num_key_value_heads"], QWEN3["head_dim"], SLOTS, dtype)
    heads = WHISPER[case["size"]][1]
    need = max(size(rows, heads, heads, 64, n, dtype) for n in (_bucket(case), FRAMES))
    return max(need, attention.choice_workspace_size(rows, VOCAB))


def _decoder_step(s: dict) -> tuple:
    hidden = s["model"].decode(s["tokens"], s["positions"], s["cache"])
    logits = s["model"].logits(hidden[:, -1]).float()
    token, logprob = whisper.choose(logits, s["suppress"])
    return logits, logprob, token, s["cache"].self_keys, s["cache"].self_values


def _whisper_step(s: dict) -> tuple:
    out = []
    for layer in range(s["layers"]):
        q, new, own, cross = s["q"][layer], s["new"][layer], s["self"][layer], s["cross"][layer]
        out.append(attention.decode_append(q[0], new[0], new[1], own[0].transpose(1, 2), own[1].transpose(1, 2),
                                           s["positions"]))
        out.append(attention.sdpa(q[1][:, :, None], cross[0], cross[1]))
    return out, s["self"]


def _qwen3_step(s: dict) -> tuple:
    hd, hq, hkv = QWEN3["head_dim"], QWEN3["num_attention_heads"], QWEN3["num_key_value_heads"]
    out = []
    for qkv, norms, kv in zip(s["qkv"], s["norms"], s["kv"]):
        q, k, v = qkv.split([hq * hd, hkv * hd, hkv * hd], dim=-1)
        out.append(attention.decode_append(
            q.view(-1, hq, hd), k.view(-1, hkv, hd), v.view(-1, hkv, hd), kv[0], kv[1], s["positions"],
            q_norm=norms[0], k_norm=norms[1], eps=QWEN3["rms_norm_eps"], cos=s["cos"], sin=s["sin"], pages=s["pages"]))
    return out, s["kv"]


def _whisper_prompt(s: dict) -> torch.Tensor:
    return s["module"].attend(s["x"], s["key"], s["value"])


def _whisper_encoder(s: dict) -> list:
    heads = WHISPER[s["case"]["size"]][1]
    return [attention.sdpa(*(t.view(*t.shape[:2], heads, 64).transpose(1, 2) for t in layer))
            for layer in zip(s["q"], s["k"], s["v"])]


def _qwen3_prompt(s: dict) -> tuple:
    out = s["module"].prefill(s["x"], s["keys"], s["values"], s["rows"], s["positions"], s["segments"], s["cos"],
                              s["sin"])
    return out, s["keys"], s["values"]


def _sensevoice(s: dict) -> torch.Tensor:
    return s["module"](s["x"], s["mask"], s["lengths"])


def _gemma4_prompt(s: dict) -> tuple:
    kv: dict = {}
    out = s["module"].prefill(s["x"], s["cache"], s["rows"], kv, KeyPrefix(lengths=s["lengths"]), s["cos"], s["sin"])
    return out, s["cache"].keys, s["cache"].values


_STEPS = {"decoder_step": _decoder_step, "whisper_step": _whisper_step, "qwen3_step": _qwen3_step,
          "whisper_encoder": _whisper_encoder}
_CALLS = {"whisper_prompt": _whisper_prompt, "qwen3_prompt": _qwen3_prompt, "sensevoice": _sensevoice,
          "gemma4_prompt": _gemma4_prompt}


# --- what a pass cannot do without ----------------------------------------


def work(case: dict) -> dict:
    kind, rows = case["kind"], case["rows"]
    es = 4 if _dtype(case) == torch.float32 else 2
    mean = (case["low"] + case["high"]) / 2 if "low" in case else 0.0
    if kind == "decoder_step":
        width, heads, layers = WHISPER[case["size"]]
        weights = layers * (8 * width * width + 8 * width * width) + VOCAB * width - 2 * layers * width * width
        keys = (4 + case["last"]) / 2 + FRAMES
        kv = 2 * layers * rows * keys * width
        return {"bytes": es * (weights + kv) + 4 * rows * VOCAB, "flops": 2 * rows * weights + 2 * kv}
    if kind == "whisper_step":
        width, heads, layers = WHISPER[case["size"]]
        keys = (4 + case["last"]) / 2 + FRAMES
        kv = 2 * layers * rows * keys * width
        return {"bytes": es * (kv + 8 * layers * rows * width), "flops": 2 * kv}
    if kind == "qwen3_step":
        hd, hq, hkv = QWEN3["head_dim"], QWEN3["num_attention_heads"], QWEN3["num_key_value_heads"]
        kv = 2 * case["layers"] * rows * mean * hkv * hd
        small = case["layers"] * rows * (2 * hq + 4 * hkv) * hd
        return {"bytes": es * (kv + small), "flops": 2 * kv * hq / hkv}
    if kind == "whisper_prompt":
        width, _, _ = WHISPER[case["size"]]
        tokens = rows * case["tokens"]
        return {"bytes": es * (2 * rows * FRAMES * width + 2 * tokens * width + 2 * width * width),
                "flops": 4 * tokens * FRAMES * width + 4 * tokens * width * width}
    if kind == "whisper_encoder":
        width, _, _ = WHISPER[case["size"]]
        tokens = case["layers"] * rows * FRAMES
        return {"bytes": es * 4 * tokens * width, "flops": 4 * tokens * FRAMES * width}
    if kind == "qwen3_prompt":
        hd, hq, hkv = QWEN3["head_dim"], QWEN3["num_attention_heads"], QWEN3["num_key_value_heads"]
        width, tokens = QWEN3["hidden_size"], rows * mean
        weights = width * (2 * hq + 2 * hkv) * hd
        return {"bytes": es * (2 * tokens * width + weights + 2 * tokens * hkv * hd),
                "flops": 2 * tokens * weights + 2 * tokens * mean * hq * hd}
    if kind == "sensevoice":
        size, _, taps = SANM
        tokens = rows * case["high"]  # padded frames pass through the projections too
        return {"bytes": es * (2 * tokens * size + 4 * size * size),
                "flops": 8 * tokens * size * size + 4 * rows * mean * mean * size + 2 * tokens * size * taps}
    hd = GEMMA["global_head_dim"] if case["full"] else GEMMA["head_dim"]
    hq, hkv, width = GEMMA["num_attention_heads"], GEMMA["num_key_value_heads"], GEMMA["hidden_size"]
    tokens, weights = rows * case["high"], width * (2 * hq + 2 * hkv) * hd
    w = GEMMA["sliding_window"]
    visible = mean * mean / 2 if case["full"] or mean <= w else w * w / 2 + (mean - w) * w
    return {"bytes": es * (2 * tokens * width + weights + 2 * tokens * hkv * hd),
            "flops": 2 * tokens * weights + 4 * rows * visible * hq * hd}


def tolerance(case: dict) -> dict:
    # float32: sums of up to 1536 products and 1500 keys in another order
    # (through four layers and the head in the whole decoder step).  bf16:
    # outputs rounded to 8 bits, and one or two rounded intermediates.
    if _dtype(case) == torch.float32:
        return {"rel": 2e-5, "max": 1e-3, "differ": 0.0}
    # Gemma 4's scores (no 1 / sqrt(head_dim)) magnify the rounding of its
    # normalized, rotated queries and keys: 0.8% off float64.
    return {"rel": 2e-2 if case["kind"] == "gemma4_prompt" else 1e-2, "max": 0.2}


# --- float64 --------------------------------------------------------------


def _attend(q, k, v, scale, visible=None):
    """float64 attention of q (rows, heads, n, d) over k, v (rows, kv heads, m,
    d), a row of the batch at a time; visible: (rows or 1, n, m) or None."""
    group = q.shape[1] // k.shape[1]
    out = []
    for b in range(q.shape[0]):
        kb, vb = (t[b].double().repeat_interleave(group, 0) for t in (k, v))
        score = (q[b].double() @ kb.transpose(1, 2).contiguous()) * scale
        if visible is not None:
            score = score.masked_fill(~visible[b if visible.shape[0] > 1 else 0][None], -math.inf)
        out.append(score.softmax(-1) @ vb)
    return torch.stack(out)


def _linear(layer, x):
    return F.linear(x, layer.weight.double(), None if layer.bias is None else layer.bias.double())


def _layer_norm(layer, x):
    return F.layer_norm(x, layer.normalized_shape, layer.weight.double(), layer.bias.double(), layer.eps)


def _rms(x, weight, eps):
    x = x * (x.square().mean(-1, keepdim=True) + eps).rsqrt()
    return x if weight is None else x * weight.double()


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), -1) * sin


def _heads(x, heads):
    return x.unflatten(-1, (heads, -1)).transpose(-3, -2)


def _write(cache, rows, positions, new):
    """The cache in float64 with each row's new token at its position; cache
    (rows, heads, length, d), new (rows, heads, d)."""
    cache = cache.double()
    cache[rows, :, positions] = new
    return cache


@torch.inference_mode()
def exact(case: dict, seed: int):
    s = _inputs(case, seed)
    kind, rows = case["kind"], case["rows"]
    every = torch.arange(rows, device="cuda")
    if kind == "decoder_step":
        model, cache = s["model"], s["cache"]
        decoder = model.model.decoder
        heads = WHISPER[case["size"]][1]
        pos = s["positions"]
        x = (decoder.embed_tokens.weight[s["tokens"]] + decoder.embed_positions.weight[pos][:, None]).double()
        seen = (torch.arange(_bucket(case), device="cuda") <= pos[:, None])[:, None, :]
        keys, values = [], []
        for i, layer in enumerate(decoder.layers):
            h = _layer_norm(layer.self_attn_layer_norm, x)
            at = layer.self_attn
            q, k, v = (_heads(_linear(p, h), heads) for p in (at.q_proj, at.k_proj, at.v_proj))
            keys.append(_write(cache.self_keys[i], every, pos, k[:, :, 0]))
            values.append(_write(cache.self_values[i], every, pos, v[:, :, 0]))
            y = _attend(q, keys[-1], values[-1], 0.125, seen if rows > 1 else seen[:1])
            x = x + _linear(at.out_proj, y.transpose(1, 2).flatten(2))
            at = layer.encoder_attn
            h = _layer_norm(layer.encoder_attn_layer_norm, x)
            y = _attend(_heads(_linear(at.q_proj, h), heads), cache.cross_keys[i], cache.cross_values[i], 0.125)
            x = x + _linear(at.out_proj, y.transpose(1, 2).flatten(2))
            x = x + _linear(layer.fc2, F.gelu(_linear(layer.fc1, _layer_norm(layer.final_layer_norm, x))))
        logits = _layer_norm(decoder.layer_norm, x)[:, -1] @ decoder.embed_tokens.weight.double().T.contiguous()
        kept = logits.masked_fill(s["suppress"], -math.inf)
        logprob, token = kept.log_softmax(-1).max(-1)
        return logits, logprob, token, torch.stack(keys), torch.stack(values)
    if kind == "whisper_step":
        out, pos = [], s["positions"]
        seen = (torch.arange(_bucket(case), device="cuda") <= pos[:, None])[:, None, :]
        own = s["self"].double()
        for i in range(s["layers"]):
            for j in range(2):
                own[i, j] = _write(own[i, j], every, pos, s["new"][i, j].double())
            out.append(_attend(s["q"][i, 0][:, :, None], own[i, 0], own[i, 1], 0.125, seen)[:, :, 0])
            out.append(_attend(s["q"][i, 1][:, :, None], s["cross"][i, 0], s["cross"][i, 1], 0.125).transpose(1, 2))
        return out, own
    if kind == "qwen3_step":
        hd, hq, hkv = QWEN3["head_dim"], QWEN3["num_attention_heads"], QWEN3["num_key_value_heads"]
        eps, pos, out = QWEN3["rms_norm_eps"], s["positions"], []
        cos, sin = s["cos"].double()[:, None], s["sin"].double()[:, None]
        for i in range(case["layers"]):
            q, k, v = (t.unflatten(-1, (-1, hd)) for t in s["qkv"][i].double().split([hq * hd, hkv * hd, hkv * hd], -1))
            q = _rotate(_rms(q, s["norms"][i, 0], eps), cos, sin)
            k = _rotate(_rms(k, s["norms"][i, 1], eps), cos, sin)
            layer = []
            for b, n in enumerate(pos.tolist()):
                if case["paged"]:
                    pages = s["pages"].block_table[b, : -(-(n + 1) // PAGE)].long()
                    kv = s["kv"][i][:, pages].flatten(1, 2)[:, : n + 1].double()
                else:
                    kv = s["kv"][i][:, b, : n + 1].double()
                kv[0, n], kv[1, n] = k[b], v[b]
                layer.append(_attend(q[b][None, :, None], kv[0].transpose(0, 1)[None], kv[1].transpose(0, 1)[None],
                                     hd**-0.5)[0, :, 0])
            out.append(torch.stack(layer))
        return out, None
    if kind == "whisper_encoder":
        heads = WHISPER[case["size"]][1]
        return [_attend(*(_heads(t, heads) for t in layer), 0.125).transpose(1, 2)
                for layer in zip(s["q"], s["k"], s["v"])]
    if kind == "whisper_prompt":
        at, x = s["module"], s["x"].double()
        y = _attend(_heads(_linear(at.q_proj, x), at.heads), s["key"], s["value"], 0.125)
        return _linear(at.out_proj, y.transpose(1, 2).flatten(2))
    if kind == "qwen3_prompt":
        at, hd, eps = s["module"], QWEN3["head_dim"], QWEN3["rms_norm_eps"]
        q, k, v = (t.unflatten(-1, (-1, hd)) for t in _linear(at.qkv_proj, s["x"].double()).split(at.sizes, -1))
        cos, sin = s["cos"].double()[:, None], s["sin"].double()[:, None]
        q = _rotate(_rms(q, at.q_norm.weight, eps), cos, sin)
        k = _rotate(_rms(k, at.k_norm.weight, eps), cos, sin)
        keys, values = s["keys"].double(), s["values"].double()
        keys[s["rows"], s["positions"]], values[s["rows"], s["positions"]] = k, v
        out, first = [], 0
        for n in s["lengths"]:
            part = slice(first, first + n)
            seen = torch.ones(1, n, n, dtype=torch.bool, device="cuda").tril()
            y = _attend(*(t[part].transpose(0, 1)[None] for t in (q, k, v)), hd**-0.5, seen)
            out.append(y[0].transpose(0, 1).flatten(1))
            first += n
        return _linear(at.o_proj, torch.cat(out)), keys, values
    if kind == "sensevoice":
        at, x = s["module"], s["x"].double()
        size, heads, taps = SANM
        q, k, v = _linear(at.linear_q_k_v, x).split(size, -1)
        length = x.shape[1]
        n = torch.full((rows,), length, device="cuda") if s["lengths"] is None else s["lengths"]
        keep = torch.arange(length, device="cuda") < n[:, None]
        y = _attend(*(_heads(t, heads) for t in (q, k, v)), (size // heads) ** -0.5, keep[:, None, :])
        y = y.transpose(1, 2).flatten(2) * keep[..., None]
        inside = (v * keep[..., None]).transpose(1, 2)
        padded = F.pad(inside, ((taps - 1) // 2, taps // 2))
        memory = F.conv1d(padded, at.fsmn_block.weight.double(), groups=size) + inside
        return _linear(at.linear_out, y) + memory.transpose(1, 2) * keep[..., None]
    at, eps = s["module"], GEMMA["rms_norm_eps"]
    hd = at.head_dim
    q, k, v = (t.unflatten(-1, (-1, hd)) for t in _linear(at.qkv_proj, s["x"].double()).split(at.sizes, -1))
    cos, sin = s["cos"].double()[:, None], s["sin"].double()[:, None]
    q = _rotate(_rms(q, at.q_norm.weight, eps), cos, sin)
    k = _rotate(_rms(k, at.k_norm.weight, eps), cos, sin)
    v = _rms(v, None, eps)
    length = q.shape[1]
    keys, values = s["cache"].keys.double(), s["cache"].values.double()
    keys[:, :length], values[:, :length] = k, v
    i = torch.arange(length, device="cuda")
    seen = (i[None, :, None] >= i) & (i < s["lengths"][:, None, None])
    if at.window:
        seen &= i[:, None] - i < at.window
        # Padding rows past the window of their last real key see no key.
        seen[:, :, 0] |= ~seen.any(-1)
    y = _attend(*(t.transpose(1, 2) for t in (q, k, v)), 1.0, seen).transpose(1, 2).flatten(2)
    if at.window:
        y[i >= s["lengths"][:, None] + at.window - 1] = 0.0
    return _linear(at.o_proj, y), keys, values
