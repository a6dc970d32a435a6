"""The work of this framework that its speed is measured on.

A speech server built on the two libraries does five things, each a `kind`
here: it prefills a prompt (`prefill`), generates codec frames for one session
(`frame`) or for a lockstep batch of sessions (`frames`), decodes codec frames
to PCM (`codec`), and, where it drives the layers itself, calls the int8 GEMVs
of decoder layers directly (`gemv`).  Geometry, sampling settings and input
distributions are those of bench.py and the tests; weights are random.

The int8 decode of one session and of a batch keeps its bits (greedy or
sampled, one other token changes everything after it), so those kinds compare
exactly; the others compare with what their data types give.
"""
import ctypes as C
import math
import os
import pathlib
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "qwen3-tts-native_amd"))
import qwen3_tts_codec_hip as codec_hip  # noqa: E402
import qwen3_tts_hip as hip  # noqa: E402

DEVICE = "cuda"
HEAD = 128
MAX_SEQUENCE = 1024  # KV capacity of every session, as bench.py's
PREFILL_LAYERS = 8   # depth of the prefill kind's model: rounding travels through the layers
# (hidden, intermediate, query width, key/value width) of the two decoders
WIDTHS = {"talker": (2048, 6144, 2048, 1024), "predictor": (1024, 3072, 2048, 1024)}
HISTORY = 80         # frames a codec stream has decoded before the measured packet: its 72-frame window is full
LARGEST_CONTEXT = 700


def listed():
    return [
        # one code-predictor layer's four GEMVs for one session: the smallest
        # calls of the decode path, where launching counts
        {"name": "gemv_predictor_b1", "kind": "gemv", "width": "predictor", "layers": 1, "rows": 1},
        # talker layers for one session: weights streamed from HBM once per token
        {"name": "gemv_talker_b1", "kind": "gemv", "width": "talker", "layers": 6, "rows": 1},
        # the same for a full lockstep batch of eight sessions
        {"name": "gemv_talker_b8", "kind": "gemv", "width": "talker", "layers": 6, "rows": 8},
        # one session early in an utterance, and late in a long one
        {"name": "frame_early", "kind": "frame", "context": 97},
        {"name": "frame_late", "kind": "frame", "context": LARGEST_CONTEXT},
        # eight sessions of different ages in lockstep: a busy server
        {"name": "frames_b8", "kind": "frames", "sessions": 8, "shortest": 33, "longest": LARGEST_CONTEXT},
        # a short sentence; a long voice description; a prompt beyond the
        # 512 rows up to which attention runs as matrix products
        {"name": "prefill_33", "kind": "prefill", "rows": 33},
        {"name": "prefill_512", "kind": "prefill", "rows": 512},
        {"name": "prefill_801", "kind": "prefill", "rows": 801},
        # the first packet of a low-latency stream; the steady four-frame
        # packet; six listeners served together
        {"name": "codec_1", "kind": "codec", "streams": 1, "frames": 1},
        {"name": "codec_4", "kind": "codec", "streams": 1, "frames": 4},
        {"name": "codec_4_b6", "kind": "codec", "streams": 6, "frames": 4},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    shapes = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    case = _drawn(rng)
    while case in shapes:
        case = _drawn(rng)
    return case


def _drawn(rng):
    kind = rng.choice(["gemv", "gemv", "frame", "frames", "prefill", "prefill", "prefill", "codec", "codec"])
    if kind == "gemv":
        return {"kind": kind, "width": rng.choice(["talker", "predictor"]), "layers": rng.randint(1, 6),
                "rows": rng.randint(1, 8)}
    if kind == "frame":
        return {"kind": kind, "context": _log_int(rng, 16, LARGEST_CONTEXT)}
    if kind == "frames":
        return {"kind": kind, "sessions": rng.randint(2, 8), "shortest": _log_int(rng, 16, 60),
                "longest": _log_int(rng, 61, LARGEST_CONTEXT)}
    if kind == "prefill":
        return {"kind": kind, "rows": _log_int(rng, 9, 801)}
    return {"kind": kind, "streams": rng.randint(1, 6), "frames": rng.randint(1, 4)}


# ---------------------------------------------------------------------------
# random numbers: made on the GPU, from a seed alone
# ---------------------------------------------------------------------------
class _Random:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(int(seed))

    def normal(self, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        return torch.empty(shape, device=DEVICE).normal_(mean, std, generator=self.g).to(dtype)

    def uniform(self, shape, low, high):
        return torch.empty(shape, device=DEVICE).uniform_(low, high, generator=self.g)

    def integers(self, shape, low, high, dtype):
        return torch.randint(low, high, shape, device=DEVICE, generator=self.g).to(dtype)


def _host_bf16(count, read):
    """`count` bf16 values that `read(pointer, bytes)` copies to the host."""
    raw = np.empty(count, np.int16)
    read(raw.ctypes.data, raw.nbytes)
    return torch.from_numpy(raw).view(torch.bfloat16)


# ---------------------------------------------------------------------------
# models: loaded once per process, as a server does; sessions and inputs are
# what the seed makes
# ---------------------------------------------------------------------------
_MODELS = {}
_WEIGHTS_SEED = 20260


def _config(layers):
    c = hip.default_config()
    c.talker_layers = layers
    return c


def _talker_shapes(cfg):
    """(name, shape, mean, std) of every tensor of the talker checkpoint."""
    shapes = []

    def layer(prefix, d):
        h, i, qw, kw = d
        for name, shape in (("input_layernorm", (h,)), ("self_attn.q_proj", (qw, h)), ("self_attn.k_proj", (kw, h)),
                            ("self_attn.v_proj", (kw, h)), ("self_attn.o_proj", (h, qw)),
                            ("self_attn.q_norm", (HEAD,)), ("self_attn.k_norm", (HEAD,)),
                            ("post_attention_layernorm", (h,)), ("mlp.gate_proj", (i, h)), ("mlp.up_proj", (i, h)),
                            ("mlp.down_proj", (h, i))):
            mean, std = (1.0, 0.05) if len(shape) == 1 else (0.0, 0.02)
            shapes.append((f"{prefix}.{name}.weight", shape, mean, std))

    hidden, p = cfg.talker_hidden, cfg.predictor_hidden
    shapes += [("talker.model.codec_embedding.weight", (cfg.talker_vocabulary, hidden), 0.0, 1.0),
               ("talker.model.text_embedding.weight", (cfg.text_vocabulary, hidden), 0.0, 1.0),
               ("talker.text_projection.linear_fc1.weight", (hidden, hidden), 0.0, 0.02),
               ("talker.text_projection.linear_fc1.bias", (hidden,), 0.0, 0.02),
               ("talker.text_projection.linear_fc2.weight", (hidden, hidden), 0.0, 0.02),
               ("talker.text_projection.linear_fc2.bias", (hidden,), 0.0, 0.02),
               ("talker.model.norm.weight", (hidden,), 1.0, 0.05),
               ("talker.codec_head.weight", (cfg.talker_vocabulary, hidden), 0.0, 0.02),
               ("talker.code_predictor.small_to_mtp_projection.weight", (p, hidden), 0.0, 0.02),
               ("talker.code_predictor.small_to_mtp_projection.bias", (p,), 0.0, 0.02),
               ("talker.code_predictor.model.norm.weight", (p,), 1.0, 0.05)]
    for index in range(cfg.talker_layers):
        layer(f"talker.model.layers.{index}", WIDTHS["talker"])
    for index in range(cfg.predictor_layers):
        layer(f"talker.code_predictor.model.layers.{index}", WIDTHS["predictor"])
    for index in range(15):
        shapes += [(f"talker.code_predictor.model.codec_embedding.{index}.weight", (cfg.predictor_vocabulary, hidden), 0.0, 1.0),
                   (f"talker.code_predictor.lm_head.{index}.weight", (cfg.predictor_vocabulary, p), 0.0, 0.02)]
    return shapes


def _talker_weight(cfg, index, name, shape, mean, std):
    w = _Random(_WEIGHTS_SEED + index).normal(shape, std, mean)
    if name == "talker.codec_head.weight":
        w[cfg.codec_eos_token] = 0  # an utterance of random weights must not end by chance
    return w


def _talker_model(layers):
    key = ("talker", layers)
    if key not in _MODELS:
        cfg, handle = _config(layers), C.c_void_p()
        hip.call("qwen3_tts_model_create_with_config", 0, C.byref(cfg), C.byref(handle))
        for index, (name, shape, mean, std) in enumerate(_talker_shapes(cfg)):
            w = _talker_weight(cfg, index, name, shape, mean, std)
            torch.cuda.synchronize()
            hip.call("qwen3_tts_model_upload_tensor", handle, name.encode(), w.data_ptr(), 2 * w.numel(), len(shape),
                     (C.c_uint64 * len(shape))(*shape))
        hip.call("qwen3_tts_model_finalize", handle, C.byref(hip.ModelMemory()))
        _MODELS[key] = handle, cfg
    return _MODELS[key]


def _codec_weights():
    """{name: fp32 tensor} of the decoder, with activations of order one throughout."""
    out = {}
    for index, (name, shape) in enumerate(codec_hip.tensor_shapes().items()):
        r = _Random(_WEIGHTS_SEED + 5000 + index)
        fan_in = math.prod(shape[1:]) if len(shape) > 1 else 1
        if name.endswith("cluster_usage"):
            w = r.uniform(shape, 0.5, 2.0)
        elif name.endswith(("scale", "gamma")):
            w = r.uniform(shape, 0.05, 0.2)
        elif name.endswith("norm.weight"):
            w = r.normal(shape, 0.1, 1.0, torch.float32)
        elif name.endswith(("alpha", "beta")):
            w = r.normal(shape, 0.3, 0.0, torch.float32)
        elif len(shape) == 1:
            w = r.normal(shape, 0.05, 0.0, torch.float32)
        elif name.endswith("embedding_sum"):
            w = r.normal(shape, 1.0, 0.0, torch.float32)
        elif name.endswith("rvq_rest.output_proj.weight"):
            w = r.normal(shape, 1.0 / math.sqrt(256 * 15), 0.0, torch.float32)
        elif ".block.1.conv.weight" in name or (name.startswith("decoder.upsample") and name.endswith("0.conv.weight")):
            w = r.normal(shape, 1.0 / math.sqrt(2 * shape[0]), 0.0, torch.float32)  # [in][out][taps], two taps an output
        elif name == "decoder.decoder.6.conv.weight":
            w = r.normal(shape, 0.25 / math.sqrt(fan_in), 0.0, torch.float32)
        elif ".conv1.conv.weight" in name or ".conv2.conv.weight" in name:
            w = r.normal(shape, 0.5 / math.sqrt(fan_in), 0.0, torch.float32)
        else:
            w = r.normal(shape, 1.0 / math.sqrt(fan_in), 0.0, torch.float32)
        out[name] = w
    return out


def _codec_model():
    if "codec" not in _MODELS:
        _MODELS["codec"] = codec_hip.SharedModel({k: v.cpu().numpy() for k, v in _codec_weights().items()})
    return _MODELS["codec"]


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Session:
    """A talker session; destroyed with the state that holds it."""

    def __init__(self, model, seed):
        self.handle = C.c_void_p()
        self.destroy = hip.load().qwen3_tts_session_destroy
        hip.call("qwen3_tts_session_create", model, MAX_SEQUENCE, seed, C.byref(self.handle), C.byref(hip.SessionMemory()))
        self.semantic = C.c_uint16()
        self.position = 0

    def __del__(self):
        if self.handle:
            self.destroy(self.handle)
            self.handle = None

    def prefill(self, text, semantic_ids, count, sampling):
        result = hip.PrefillResult()
        p = C.POINTER(C.c_int32)
        hip.call("qwen3_tts_session_prefill", self.handle, text.ctypes.data_as(p), semantic_ids.ctypes.data_as(p), count,
                 sampling, C.byref(result))
        self.semantic.value = result.first_semantic_token
        self.position = count

    def last_hidden(self):
        return _host_bf16(2048, lambda p, n: hip.call("qwen3_tts_session_read_last_hidden_v1", self.handle, p, n))


def _prompt(seed, count, cfg):
    r = np.random.default_rng(seed)
    text = r.integers(0, cfg.text_vocabulary, count).astype(np.int32)
    codes = r.integers(0, 2048, count).astype(np.int32)
    text[1::7] = -1  # positions with codec input only, and with text only
    codes[np.where((np.arange(count) % 5 == 2) & (text >= 0))] = -1
    return text, codes


TALKER_SAMPLING = (1, 50, 1.0, 0.9, 1.05)
PREDICTOR_SAMPLING = (1, 50, 1.0, 0.9, 1.0)


def _started_session(model, cfg, seed, context):
    """A session `context` positions into its utterance.  Its prompt runs
    through the int8 decode step, the numerics its frames have."""
    s = _Session(model, seed + 1)
    s.text, s.codes = _prompt(seed, context, cfg)
    s.trailing = int(np.random.default_rng(seed + 7).integers(0, cfg.text_vocabulary))
    before = os.environ.get("QWEN3_TTS_PREFILL")
    os.environ["QWEN3_TTS_PREFILL"] = "decode"
    try:
        s.prefill(s.text, s.codes, context, hip.sampling(*TALKER_SAMPLING))
    finally:
        if before is None:
            del os.environ["QWEN3_TTS_PREFILL"]
        else:
            os.environ["QWEN3_TTS_PREFILL"] = before
    return s


def _contexts(case):
    n = case["sessions"]
    low, high = case["shortest"], case["longest"]
    return [int(round(low * (high / low) ** (i / max(1, n - 1)))) for i in range(n)]


def _gemv_layer(r, width, rows):
    """One decoder layer's four GEMVs: weights, inputs and outputs on the GPU."""
    hidden, intermediate, qw, kvw = WIDTHS[width]
    add = hip.EPI_ADD_ROUNDED if rows == 1 else hip.EPI_ADD_FMA
    silu = hip.EPI_SILU_ROUNDED if rows == 1 else hip.EPI_SILU_FUSED
    calls = []
    for inputs, outputs, epilogue, norm in ((hidden, qw + 2 * kvw, hip.EPI_STORE, True), (qw, hidden, add, False),
                                            (hidden, intermediate, silu, True), (intermediate, hidden, add, False)):
        weight_rows = 2 * outputs if epilogue == silu else outputs
        t = {"weight": r.integers((weight_rows, inputs), -127, 128, torch.int8),
             "scales": r.uniform((weight_rows,), 1e-3, 2e-2),
             "input": r.normal((rows, inputs)),
             "gain": r.normal((inputs,), 0.1, 1.0) if norm else None,
             "out": r.normal((rows, outputs))}
        a = hip.Int8GemvV1()
        a.struct_size = C.sizeof(a)
        a.in_features, a.out_features, a.rows = inputs, outputs, rows
        a.epilogue, a.mode, a.norm_epsilon = epilogue, hip.MODE_AUTO, 1e-6
        a.weight, a.scales, a.input, a.out16 = (t[k].data_ptr() for k in ("weight", "scales", "input", "out"))
        a.norm_weight = t["gain"].data_ptr() if norm else None
        calls.append((a, t))
    return calls


def _codec_codes(case, seed):
    count = HISTORY + case["frames"]
    return np.random.default_rng(seed).integers(0, 2048, (case["streams"], count, 16)).astype(np.uint16)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        r = _Random(seed)
        calls = [c for _ in range(case["layers"]) for c in _gemv_layer(r, case["width"], case["rows"])]
        return {"kind": kind, "calls": calls, "outputs": [t["out"] for _, t in calls]}
    if kind in ("frame", "frames"):
        model, cfg = _talker_model(28)
        contexts = [case["context"]] if kind == "frame" else _contexts(case)
        sessions = [_started_session(model, cfg, seed * 64 + i, c) for i, c in enumerate(contexts)]
        return {"kind": kind, "model": model, "sessions": sessions, "talker": hip.sampling(*TALKER_SAMPLING),
                "predictor": hip.sampling(*PREDICTOR_SAMPLING)}
    if kind == "prefill":
        model, cfg = _talker_model(PREFILL_LAYERS)
        text, codes = _prompt(seed, case["rows"], cfg)
        return {"kind": kind, "session": _Session(model, seed + 1), "text": text, "codes": codes, "rows": case["rows"],
                "sampling": hip.sampling(*TALKER_SAMPLING)}
    model = _codec_model()
    codes = _codec_codes(case, seed)
    sessions = [model.session() for _ in range(case["streams"])]
    for at in range(0, HISTORY, 4):
        codec_hip.process_batch(sessions, [c[at:at + 4] for c in codes])
    return {"kind": kind, "sessions": sessions, "codes": [np.ascontiguousarray(c[HISTORY:]) for c in codes]}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _restart_full(state):
    """A session whose cache is full begins its next utterance."""
    for s in state["sessions"]:
        if s.position >= MAX_SEQUENCE:
            hip.call("qwen3_tts_session_reset", s.handle, 1)
            s.prefill(s.text, s.codes, len(s.text), state["talker"])


def _run_frame(state):
    _restart_full(state)
    s = state["sessions"][0]
    codes, following, info = (C.c_uint16 * 16)(), C.c_uint16(), hip.CodecFrameInfo()
    hip.call("qwen3_tts_session_next_frame", s.handle, s.semantic, s.trailing, state["talker"], state["predictor"], codes, 16,
             C.byref(following), C.byref(info))
    s.semantic.value = following.value
    s.position += 1
    return {"codes": np.array(codes, np.int32), "next": int(following.value), "hidden": s.last_hidden()}


def _run_frames(state):
    _restart_full(state)
    sessions = state["sessions"]
    n = len(sessions)
    handles = (C.c_void_p * n)(*[s.handle for s in sessions])
    trailing = (C.c_int32 * n)(*[s.trailing for s in sessions])
    talker = (hip.SamplingConfig * n)(*[state["talker"]] * n)
    predictor = (hip.SamplingConfig * n)(*[state["predictor"]] * n)
    views = (hip.DeviceFrameViewV2 * n)(*[hip.DeviceFrameViewV2(C.sizeof(hip.DeviceFrameViewV2))] * n)
    hip.call("qwen3_tts_model_batch_next_frame_begin_v2", state["model"], handles, n, trailing, talker, predictor, views)
    out = []
    for s, view in zip(sessions, views):
        following, info = C.c_uint16(), hip.CodecFrameInfo()
        hip.call("qwen3_tts_session_next_frame_finish_v2", s.handle, view.lease_id, None, C.byref(following), C.byref(info))
        codes = np.empty(16, np.uint16)
        hip.call("qwen3_tts_device_memcpy", codes.ctypes.data, view.device_codes, codes.nbytes)
        s.semantic.value = following.value
        s.position += 1
        out.append({"codes": codes.astype(np.int32), "next": int(following.value), "hidden": s.last_hidden()})
    return out


def run(state):
    kind = state["kind"]
    if kind == "gemv":
        for a, _ in state["calls"]:
            hip.call("qwen3_tts_int8_gemv_v1", C.byref(a), None)
        return state["outputs"]
    if kind == "frame":
        return _run_frame(state)
    if kind == "frames":
        return _run_frames(state)
    if kind == "prefill":
        s, rows = state["session"], state["rows"]
        s.prefill(state["text"], state["codes"], rows, state["sampling"])
        # the state the frames start from: the last hidden row, and the
        # deepest layer's keys of every prompt row
        keys = _host_bf16(rows * 1024, lambda p, n: hip.call("qwen3_tts_session_read_talker_cache_v1", s.handle,
                                                             PREFILL_LAYERS - 1, 0, rows, p, n))
        return {"hidden": s.last_hidden(), "keys": keys.view(rows, 1024)}
    if len(state["sessions"]) == 1:
        packets = [state["sessions"][0].packet(state["codes"][0])]
    else:
        packets = codec_hip.process_batch(state["sessions"], state["codes"])
    return [pcm.astype(np.float32) / 32767.0 for pcm, _ in packets]  # audio as a mixer takes it


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _layer_parameters(width):
    hidden, intermediate, qw, kvw = WIDTHS[width]
    return hidden * (qw + 2 * kvw) + qw * hidden + 3 * hidden * intermediate


def _frame_work(contexts):
    rows = len(contexts)
    talker, predictor = 28 * _layer_parameters("talker"), 5 * _layer_parameters("predictor")
    text, head, into = 2 * 2048 * 2048, 3072 * 2048, 1024 * 2048
    heads = 15 * 2048 * 1024
    kv = sum(28 * 2 * 1024 * 2 * (c + 1) for c in contexts)
    flops = rows * 2 * (talker + text + head + 16 * (predictor + into) + heads)
    flops += sum(28 * 4 * 2048 * (c + 1) for c in contexts)
    return {"bytes": talker + text + head + predictor + into + heads + kv, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        hidden, intermediate, qw, kvw = WIDTHS[case["width"]]
        rows, n = case["rows"], case["layers"]
        weights = _layer_parameters(case["width"])
        scales = 4 * (qw + 2 * kvw + 2 * hidden + 2 * intermediate)
        values = 2 * rows * (hidden + (qw + 2 * kvw) + qw + 2 * hidden + hidden + intermediate + intermediate + 2 * hidden)
        return {"bytes": n * (weights + scales + values + 4 * hidden), "flops": n * 2 * rows * weights}
    if kind == "frame":
        return _frame_work([case["context"]])
    if kind == "frames":
        return _frame_work(_contexts(case))
    if kind == "prefill":
        rows = case["rows"]
        weights = PREFILL_LAYERS * _layer_parameters("talker")
        head, text = 3072 * 2048, 2 * 2048 * 2048
        flops = 2 * rows * (weights + text) + 2 * head + PREFILL_LAYERS * 2 * 2048 * rows * (rows + 1)
        return {"bytes": 2 * (weights + head) + text + 2 * rows * 2 * 2048 + PREFILL_LAYERS * rows * 2 * 2 * 1024, "flops": flops}
    frames, streams = case["frames"], case["streams"]
    weights = 4 * (114323137 - 16 * 2048 * 257)
    macs = 512 * 512 + 1024 * 512 * 3 + 2 * 512 * 1024 + 8 * (3 * 1024 * 512 + 512 * 1024 + 3 * 1024 * 512)
    for scale in (1, 2):
        macs += scale * 1024 * 2048 + 2 * scale * (7 * 1024 + 2 * 1024 * 4096)
    macs += 4 * 1536 * 7 * 1024
    positions = 4
    for into, out, stride in zip((1536, 768, 384, 192), (768, 384, 192, 96), (8, 5, 4, 3)):
        macs += positions * 2 * into * stride * out
        positions *= stride
        macs += positions * 3 * 8 * out * out
    macs += positions * 7 * 96
    return {"bytes": weights + streams * frames * (2 * 1920 + 32), "flops": 2 * macs * frames * streams}


def tolerance(case):
    """About four times what the path shows against itself with its sums in
    another order (matrix cores against the exact order, other tiles and
    slices of K) or, for the decoder, against 64 bits."""
    kind = case["kind"]
    if kind == "gemv":
        # one row: the summation order is part of the interface; more rows:
        # fp32 sums in any order, rounded to bf16 (seen: 3e-5, 4e-3)
        return "exact" if case["rows"] == 1 else {"rel": 1.5e-4, "max": 1.5e-2}
    if kind in ("frame", "frames"):
        return "exact"
    if kind == "prefill":
        return {"rel": 3e-2, "max": 2.5e-1}  # bf16 activations through eight layers (seen: 1.1e-2, 6e-2)
    return {"rel": 8e-5, "max": 3e-4}  # fp32 throughout, then 16-bit PCM, whose step alone is 2e-5 and 7e-5


# ---------------------------------------------------------------------------
# the same in 64 bits, by plain torch
# ---------------------------------------------------------------------------
def _rms64(x, gain, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gain


def _silu64(x):
    return x / (1.0 + torch.exp(-x))


def _exact_gemv(case, seed):
    r = _Random(seed)
    out = []
    for _ in range(case["layers"]):
        for a, t in _gemv_layer(r, case["width"], case["rows"]):
            x = t["input"].double()
            if t["gain"] is not None:
                x = _rms64(x, t["gain"].double(), 1e-6)
            y = x @ (t["weight"].double() * t["scales"].double()[:, None]).T
            if a.epilogue in (hip.EPI_SILU_FUSED, hip.EPI_SILU_ROUNDED):
                half = y.shape[1] // 2
                y = _silu64(y[:, :half]) * y[:, half:]
            elif a.epilogue != hip.EPI_STORE:
                y = y + t["out"].double()
            out.append(y)
    return out


def _exact_prefill(case, seed):
    cfg = _config(PREFILL_LAYERS)
    names = {name: (i, name, shape, mean, std) for i, (name, shape, mean, std) in enumerate(_talker_shapes(cfg))}

    def weight(name):
        return _talker_weight(cfg, *names[name]).double()

    def quantized(name):
        w = weight(name)
        scale = (w.abs().amax(1, keepdim=True) / 127.0).float().double()
        return torch.clamp(torch.round(w / scale), -127, 127) * scale

    rows = case["rows"]
    text, codes = (torch.from_numpy(v).to(DEVICE).long() for v in _prompt(seed, rows, cfg))
    p = "talker.text_projection.linear_"
    table = _talker_weight(cfg, *names["talker.model.text_embedding.weight"])
    x = table[text.clamp(min=0)].double()
    del table
    x = _silu64(x @ quantized(p + "fc1.weight").T + weight(p + "fc1.bias"))
    x = x @ quantized(p + "fc2.weight").T + weight(p + "fc2.bias")
    h = torch.where((text >= 0)[:, None], x, 0.0)
    h = h + torch.where((codes >= 0)[:, None], weight("talker.model.codec_embedding.weight")[codes.clamp(min=0)], 0.0)
    half = HEAD // 2
    angle = torch.arange(rows, device=DEVICE, dtype=torch.float64)[:, None] * (
        float(cfg.rope_theta) ** (-torch.arange(half, device=DEVICE, dtype=torch.float64) / half))[None]
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
    causal = torch.ones(rows, rows, dtype=torch.bool, device=DEVICE).tril()

    def rotated(v, gain):
        v = _rms64(v, gain, cfg.rms_epsilon)
        a, b = v[..., :half], v[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for index in range(PREFILL_LAYERS):
        w = f"talker.model.layers.{index}."
        a = _rms64(h, weight(w + "input_layernorm.weight"), cfg.rms_epsilon)
        q = (a @ weight(w + "self_attn.q_proj.weight").T).view(rows, 16, HEAD)
        k = (a @ weight(w + "self_attn.k_proj.weight").T).view(rows, 8, HEAD)
        v = (a @ weight(w + "self_attn.v_proj.weight").T).view(rows, 8, HEAD)
        q, k = rotated(q, weight(w + "self_attn.q_norm.weight")), rotated(k, weight(w + "self_attn.k_norm.weight"))
        heads = []
        for head in range(16):
            s = q[:, head] @ k[:, head // 2].T / math.sqrt(HEAD)
            heads.append(torch.softmax(s.masked_fill(~causal, -math.inf), -1) @ v[:, head // 2])
        h = h + torch.cat(heads, 1) @ weight(w + "self_attn.o_proj.weight").T
        a = _rms64(h, weight(w + "post_attention_layernorm.weight"), cfg.rms_epsilon)
        a = _silu64(a @ weight(w + "mlp.gate_proj.weight").T) * (a @ weight(w + "mlp.up_proj.weight").T)
        h = h + a @ weight(w + "mlp.down_proj.weight").T
    return {"hidden": _rms64(h[-1], weight("talker.model.norm.weight"), cfg.rms_epsilon), "keys": k.reshape(rows, 1024)}


def _exact_codec(case, seed):
    w = {k: v.double() for k, v in _codec_weights().items()}
    codes = torch.from_numpy(_codec_codes(case, seed).astype(np.int64)).to(DEVICE)

    def conv(x, weight, bias, dilation=1):  # causal, [time][channels], weight [out][in][taps]
        taps = weight.shape[2]
        x = torch.cat([x.new_zeros((taps - 1) * dilation, x.shape[1]), x])
        time = x.shape[0] - (taps - 1) * dilation
        return sum(x[t * dilation:t * dilation + time] @ weight[:, :, t].T for t in range(taps)) + bias

    def transposed(x, weight, bias, stride):  # weight [in][out][taps]; the tail of the last frame is cut
        taps, time = weight.shape[2], x.shape[0]
        y = x.new_zeros(time * stride + taps - stride, weight.shape[1])
        for t in range(taps):
            y[t:t + stride * time:stride] += x @ weight[:, :, t]
        return y[:time * stride] + bias

    def snake(x, prefix):
        return x + torch.sin(x * torch.exp(w[prefix + "alpha"])) ** 2 / (torch.exp(w[prefix + "beta"]) + 1e-9)

    def transformer(x):
        t = "decoder.pre_transformer."
        n = x.shape[0]
        h = x @ w[t + "input_proj.weight"].T + w[t + "input_proj.bias"]
        angle = torch.arange(n, device=DEVICE, dtype=torch.float64)[:, None] / 10000.0 ** (
            torch.arange(32, device=DEVICE, dtype=torch.float64) / 32)[None]
        cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
        i = torch.arange(n, device=DEVICE)
        window = (i[None] <= i[:, None]) & (i[None] > i[:, None] - 72)

        def rotated(v):
            a, b = v[..., :32], v[..., 32:]
            return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

        for index in range(8):
            p = f"{t}layers.{index}."
            a = _rms64(h, w[p + "input_layernorm.weight"], 1e-5)
            q, k, v = ((a @ w[p + f"self_attn.{c}_proj.weight"].T).view(n, 16, 64) for c in "qkv")
            q, k = rotated(q), rotated(k)
            heads = []
            for head in range(16):
                s = (q[:, head] @ k[:, head].T / 8.0).masked_fill(~window, -math.inf)
                heads.append(torch.softmax(s, -1) @ v[:, head])
            h = h + torch.cat(heads, 1) @ w[p + "self_attn.o_proj.weight"].T * w[p + "self_attn_layer_scale.scale"]
            a = _rms64(h, w[p + "post_attention_layernorm.weight"], 1e-5)
            a = _silu64(a @ w[p + "mlp.gate_proj.weight"].T) * (a @ w[p + "mlp.up_proj.weight"].T)
            h = h + a @ w[p + "mlp.down_proj.weight"].T * w[p + "mlp_layer_scale.scale"]
        return _rms64(h, w[t + "norm.weight"], 1e-5) @ w[t + "output_proj.weight"].T + w[t + "output_proj.bias"]

    def decode(code):
        q = "decoder.quantizer."
        parts = []
        for part, books in (("rvq_first", range(1)), ("rvq_rest", range(1, 16))):
            total = 0.0
            for at, book in enumerate(books):
                p = f"{q}{part}.vq.layers.{at}._codebook."
                table = w[p + "embedding_sum"] / w[p + "cluster_usage"].clamp(min=1e-5)[:, None]
                total = total + table[code[:, book]]
            parts.append(total @ w[f"{q}{part}.output_proj.weight"].reshape(512, 256).T)
        x = conv(parts[0] + parts[1], w["decoder.pre_conv.conv.weight"], w["decoder.pre_conv.conv.bias"])
        x = transformer(x)
        for u in range(2):
            p = f"decoder.upsample.{u}."
            y = transposed(x, w[p + "0.conv.weight"], w[p + "0.conv.bias"], 2)
            d = w[p + "1.dwconv.conv.weight"].reshape(1024, 7)
            padded = torch.cat([y.new_zeros(6, 1024), y])
            z = sum(padded[t:t + y.shape[0]] * d[:, t] for t in range(7)) + w[p + "1.dwconv.conv.bias"]
            z = z - z.mean(-1, keepdim=True)
            z = z / torch.sqrt((z * z).mean(-1, keepdim=True) + 1e-6) * w[p + "1.norm.weight"] + w[p + "1.norm.bias"]
            z = z @ w[p + "1.pwconv1.weight"].T + w[p + "1.pwconv1.bias"]
            z = 0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0)))
            x = y + (z @ w[p + "1.pwconv2.weight"].T + w[p + "1.pwconv2.bias"]) * w[p + "1.gamma"]
        x = conv(x, w["decoder.decoder.0.conv.weight"], w["decoder.decoder.0.conv.bias"])
        for b, stride in enumerate((8, 5, 4, 3)):
            p = f"decoder.decoder.{b + 1}.block."
            x = transposed(snake(x, p + "0."), w[p + "1.conv.weight"], w[p + "1.conv.bias"], stride)
            for u, dilation in enumerate((1, 3, 9)):
                r = f"{p}{u + 2}."
                y = conv(snake(x, r + "act1."), w[r + "conv1.conv.weight"], w[r + "conv1.conv.bias"], dilation)
                x = x + conv(snake(y, r + "act2."), w[r + "conv2.conv.weight"], w[r + "conv2.conv.bias"])
        x = conv(snake(x, "decoder.decoder.5."), w["decoder.decoder.6.conv.weight"], w["decoder.decoder.6.conv.bias"])
        return x[:, 0].clamp(-1.0, 1.0)[HISTORY * 1920:]

    return [decode(c) for c in codes]


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "gemv":
            return _exact_gemv(case, seed)
        if case["kind"] == "prefill":
            return _exact_prefill(case, seed)
        if case["kind"] == "codec":
            return _exact_codec(case, seed)
    return None  # sampled tokens, and hidden states that follow from them
