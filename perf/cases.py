"""The calls whose time this library is judged by, each through its public
Python entry points: the mel front end, the encoder, single-stream and batched
decoding, a long prompt, and the per-op kernel calls.

Sizes are the published checkpoints' (whispereacp_amd.synthetic's
WORKLOADS and ENCODER_WORKLOADS); the deeper models are cut to a few of their
identical layers, so that inputs stay quick to make. Weights are random:
projections, biases and embeddings N(0, 0.02), LayerNorm gamma near one.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from whispereacp_amd import _native as N
from whispereacp_amd import synthetic as S
from whispereacp_amd.decoder import BatchedDecoder, Decoder, KernelContext
from whispereacp_amd.encoder import Encoder, EncoderWeights
from whispereacp_amd.mel import MelSpectrogram

_BYTES = {"F32": 4, "F16": 2, "BF16": 2}
_TORCH = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}
_CODE = {"F32": N.WSP_F32, "F16": N.WSP_F16, "BF16": N.WSP_BF16}
_MAX_POSITIONS = 448
_WINDOW = 1500


def listed():
    return [
        # Every transcription starts here: 30 s of 16 kHz samples, 11 s of
        # them audio and the rest the zero padding of the window.
        dict(name="mel-80", kind="mel", bands=80, seconds=11.0),
        # The whole tiny.en encoder over one window, the fp16 projections
        # OpenAI's checkpoints carry: the low-latency transcriber.
        dict(name="encoder-tiny.en-f16", kind="encoder", bands=80, width=384, layers=4, positions=1500, dtype="F16"),
        # The whole base.en encoder from an fp32 checkpoint.
        dict(name="encoder-base.en-f32", kind="encoder", bands=80, width=512, layers=6, positions=1500, dtype="F32"),
        # Four of large-v3's 32 encoder layers behind its convolutions, bf16
        # projections: the dense work of an accurate transcriber.
        dict(name="encoder-large-v3-bf16", kind="encoder", bands=128, width=1280, layers=4, positions=1500,
             dtype="BF16"),
        # The whole tiny.en decode of a short clip: the cross projection, the
        # two-token prompt and 25 greedy steps, one stream.
        dict(name="decode-tiny.en-f16", kind="decode", width=384, layers=4, vocab=51864, dtype="F16", rows=1500,
             prompt=2, steps=25),
        # The small decoder, one stream, the multilingual four-token prefix.
        dict(name="decode-small-f16", kind="decode", width=768, layers=12, vocab=51865, dtype="F16", rows=1500,
             prompt=4, steps=32),
        # One stream of large-v3 (four of its 32 layers), bf16.
        dict(name="decode-large-v3-bf16", kind="decode", width=1280, layers=4, vocab=51866, dtype="BF16", rows=1500,
             prompt=4, steps=24),
        # The small decoder given the previous window's text as its prompt.
        dict(name="prefill-small-f16", kind="decode", width=768, layers=12, vocab=51865, dtype="F16", rows=1500,
             prompt=96, steps=4),
        # 16 streams of medium (four of its 24 layers) advancing together.
        dict(name="batch-medium-f16", kind="batch", width=1024, layers=4, vocab=51865, dtype="F16", rows=1500,
             streams=16, prompt=4, steps=32),
        # 32 streams of large-v3 (four of its 32 layers).
        dict(name="batch-large-v3-bf16", kind="batch", width=1280, layers=4, vocab=51866, dtype="BF16", rows=1500,
             streams=32, prompt=4, steps=32),
        # One feed-forward block through the per-op calls, one token's rows:
        # three small launches (norm, fc1 with GELU, fc2 into the residual).
        dict(name="mlp-small-f16", kind="mlp", width=768, rows=1, dtype="F16"),
        # One token's cross attention through the per-op call (base.en).
        dict(name="attention-base.en", kind="attention", width=512, queries=1, keys=1500, causal=False),
    ]


_WIDTHS = [384, 512, 768, 1024, 1280]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["mel", "encoder", "encoder", "decode", "decode", "batch", "mlp", "attention"])
    if kind == "mel":
        return dict(kind="mel", bands=rng.choice([80, 128]), seconds=round(rng.uniform(1.0, 30.0), 2))
    width = rng.choice(_WIDTHS)
    if kind == "encoder":
        # From a reduced audio context of a second or two to the whole window.
        dtype = rng.choice(["F16", "BF16", "F16", "BF16", "F32"])
        return dict(kind="encoder", bands=128 if width == 1280 else 80, width=width, layers=rng.randint(1, 3),
                    positions=rng.choice([1500, _log_int(rng, 64, 1500)]), dtype=dtype)
    if kind == "decode":
        dtype = rng.choice(["F16", "BF16", "F32"])
        prompt = rng.choice([1, 2, 4, _log_int(rng, 5, 224)])
        return dict(kind="decode", width=width, layers=rng.randint(1, 4), vocab=51864 + rng.randint(0, 2), dtype=dtype,
                    rows=rng.choice([1500, _log_int(rng, 64, 1500)]), prompt=prompt, steps=_log_int(rng, 4, 48))
    if kind == "batch":
        return dict(kind="batch", width=width, layers=rng.randint(1, 3), vocab=51864 + rng.randint(0, 2),
                    dtype=rng.choice(["F16", "BF16"]), rows=rng.choice([1500, _log_int(rng, 64, 1500)]),
                    streams=_log_int(rng, 2, 32), prompt=rng.randint(1, 4), steps=_log_int(rng, 4, 32))
    if kind == "mlp":
        return dict(kind="mlp", width=width, rows=_log_int(rng, 1, 1500), dtype=rng.choice(["F16", "BF16", "F32"]))
    causal = rng.random() < 0.5
    queries = rng.choice([1, _log_int(rng, 2, 224)])
    return dict(kind="attention", width=width, queries=queries,
                keys=rng.randint(queries, _MAX_POSITIONS) if causal else _log_int(rng, 64, 1500), causal=causal)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Draws:
    """Seeded normal values, made on the GPU."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda")
        self.generator.manual_seed(int(seed) * 7919 + 17)

    def normal(self, extents, std, dtype="F32"):
        values = torch.randn(extents, generator=self.generator, device="cuda", dtype=torch.float32)
        return (values * std).to(_TORCH[dtype])


def _stored(name, tensor, dtype):
    data = tensor.contiguous().cpu()
    array = data.view(torch.int16).numpy().view(np.uint16) if dtype == "BF16" else data.numpy()
    return S.StoredTensor(name, dtype, tuple(tensor.shape), array)


def _weight(draws, name, extents, dtype):
    if S.is_norm_weight(name):
        return (1.0 + draws.normal(extents, 0.1)).to(_TORCH[dtype])
    return draws.normal(extents, 0.02, dtype)


def _encoder_shape(case):
    width = case["width"]
    return S.EncoderShape(case["bands"], width, width // 64, case["layers"], 4 * width, 2 * _WINDOW)


def _decoder_shape(case):
    width = case["width"]
    return S.DecoderShape(width, width // 64, case["layers"], 4 * width, case["vocab"], _MAX_POSITIONS, _WINDOW)


def _encoder_tensors(case, draws):
    """The projections in the case's storage, everything else fp32."""
    shape = _encoder_shape(case)
    for name in S.encoder_canonical_names(shape.layers):
        dtype = case["dtype"] if S.is_projection(name) else "F32"
        yield name, _weight(draws, name, S.encoder_tensor_extents(shape, name), dtype), dtype


def _decoder_tensors(case, draws):
    shape = _decoder_shape(case)
    for name in S.file_order(shape.layers):
        yield name, _weight(draws, name, S.tensor_extents(shape, name), case["dtype"]), case["dtype"]


def _audio(case, seed):
    """Voiced and noisy stretches of sound, then the window's zero padding."""
    shape = S.MelShape(mel_count=case["bands"])
    draws = _Draws(seed)
    n = min(shape.sample_count, int(case["seconds"] * 16000))
    t = torch.arange(n, device="cuda", dtype=torch.float64) / 16000
    pitch = 90 + 8 * (int(seed) % 16)
    phase = 2 * math.pi * (pitch * t + 3 * torch.sin(2 * math.pi * 0.7 * t))
    voice = sum(torch.sin(k * phase) / k for k in range(1, 20))
    loud = 0.55 + 0.45 * torch.sin(2 * math.pi * 1.3 * t)
    samples = torch.zeros(shape.sample_count, device="cuda", dtype=torch.float32)
    samples[:n] = (0.2 * loud * voice).float() + draws.normal((n,), 0.01)
    filters = torch.from_numpy(S.triangular_filters(case["bands"], shape.bin_count)).cuda()
    return shape, samples, filters


def _mel_rows(case, draws):
    return draws.normal((case["bands"], 2 * _WINDOW), 0.5).clamp_(-1.5, 1.5)


def _prompt(case, seed, count):
    return torch.from_numpy(np.random.RandomState(int(seed) % 2 ** 31).randint(0, case["vocab"], count).astype(np.int32))


def _mlp_inputs(case, seed):
    draws, d, f = _Draws(seed), case["width"], 4 * case["width"]
    dtype = case["dtype"]
    return dict(x=draws.normal((case["rows"], d), 1.0), gamma=1.0 + draws.normal((d,), 0.1),
                beta=draws.normal((d,), 0.02), fc1=draws.normal((f, d), 0.02, dtype), fc1_bias=draws.normal((f,), 0.02),
                fc2=draws.normal((d, f), 0.02, dtype), fc2_bias=draws.normal((d,), 0.02))


def _attention_inputs(case, seed):
    draws, d = _Draws(seed), case["width"]
    return dict(q=draws.normal((case["queries"], d), 1.0), k=draws.normal((case["keys"], d), 1.0),
                v=draws.normal((case["keys"], d), 1.0))


def _op_context(width):
    return KernelContext(S.DecoderShape(width, width // 64, 1, 4 * width, 51864, _MAX_POSITIONS, _WINDOW))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mel":
        shape, samples, filters = _audio(case, seed)
        return dict(kind=kind, front=MelSpectrogram(shape), samples=samples, filters=filters,
                    out=torch.empty((shape.mel_count, shape.frame_count), device="cuda"))
    if kind == "encoder":
        shape, draws = _encoder_shape(case), _Draws(seed)
        file = {name: _stored(name, t, dtype) for name, t, dtype in _encoder_tensors(case, draws)}
        return dict(kind=kind, encoder=Encoder(shape), weights=EncoderWeights(shape, file), mel=_mel_rows(case, draws),
                    positions=case["positions"], out=torch.empty((case["positions"], shape.width), device="cuda"))
    if kind in ("decode", "batch"):
        shape, draws = _decoder_shape(case), _Draws(seed)
        file = {name: _stored(name, t, dtype) for name, t, dtype in _decoder_tensors(case, draws)}
        prompt, steps, vocab = case["prompt"], case["steps"], shape.vocabulary_size
        if kind == "batch":
            streams = case["streams"]
            ring = torch.zeros((_MAX_POSITIONS + 1, streams), dtype=torch.int32, device="cuda")
            return dict(kind=kind, decoder=BatchedDecoder(shape, file, streams), rows=case["rows"],
                        encoded=draws.normal((streams, case["rows"], shape.width), 1.0),
                        tokens=_prompt(case, seed, streams * prompt).reshape(streams, prompt).cuda(), ring=ring,
                        prompt=prompt, steps=steps, prompt_logits=torch.empty((streams * prompt, vocab), device="cuda"),
                        logits=torch.empty((streams, vocab), device="cuda"))
        slots = torch.zeros(prompt + steps + 1, dtype=torch.int32, device="cuda")
        slots[:prompt] = _prompt(case, seed, prompt)
        logits = torch.empty((prompt + steps, vocab), device="cuda")
        packing = "Float" if case["dtype"] == "F32" else "ExactHalf"
        return dict(kind=kind, decoder=Decoder(shape, file, packing), rows=case["rows"],
                    encoded=draws.normal((case["rows"], shape.width), 1.0), slots=slots, logits=logits, prompt=prompt,
                    vocab=vocab, views=[(slots[p:p + 1], logits[p:p + 1], slots[p + 1:p + 2])
                                        for p in range(prompt, prompt + steps)])
    if kind == "mlp":
        inputs = _mlp_inputs(case, seed)
        rows, d = inputs["x"].shape
        return dict(kind=kind, context=_op_context(d), dtype=_CODE[case["dtype"]], h=torch.empty((rows, d), device="cuda"),
                    normed=torch.empty((rows, d), device="cuda"), ff=torch.empty((rows, 4 * d), device="cuda"), **inputs)
    inputs = _attention_inputs(case, seed)
    return dict(kind=kind, context=_op_context(case["width"]), causal=case["causal"],
                out=torch.empty((case["queries"], case["width"]), device="cuda"), **inputs)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    s, kind = state, state["kind"]
    if kind == "mel":
        s["front"].encode(s["samples"], s["filters"], s["out"])
        return s["out"]
    if kind == "encoder":
        s["encoder"].encode(s["mel"], s["weights"], s["out"], s["positions"])
        return s["out"]
    if kind == "decode":
        decoder, prompt = s["decoder"], s["prompt"]
        decoder.begin_sequence(s["encoded"], s["rows"])
        decoder.step(s["slots"][:prompt], prompt, s["logits"][:prompt])
        decoder.argmax(s["logits"][prompt - 1:prompt], 1, s["vocab"], None, s["slots"][prompt:prompt + 1])
        for token, logits, slot in s["views"]:
            decoder.step_and_sample(token, logits, None, slot)
        return s["logits"], s["slots"]
    if kind == "batch":
        decoder, prompt, ring = s["decoder"], s["prompt"], s["ring"]
        decoder.begin(s["encoded"], s["rows"])
        decoder.step(s["tokens"], prompt, s["prompt_logits"], None, ring[prompt])
        for _ in range(s["steps"]):
            decoder.ring_step(ring, s["logits"])
        return s["prompt_logits"], s["logits"], ring[prompt:prompt + s["steps"] + 1]
    context = s["context"]
    if kind == "mlp":
        rows, d = s["x"].shape
        f = 4 * d
        s["h"].copy_(s["x"])
        context.layernorm(s["h"], s["gamma"], s["beta"], s["normed"], rows, d)
        context.linear(s["normed"], rows, d, s["fc1"], s["dtype"], s["fc1_bias"], s["ff"], f, N.WSP_LINEAR_GELU)
        context.linear(s["ff"], rows, f, s["fc2"], s["dtype"], s["fc2_bias"], s["h"], d, N.WSP_LINEAR_RESIDUAL)
        return s["h"]
    queries, width = s["q"].shape
    context.attention(s["q"], queries, s["k"], s["v"], s["k"].shape[0], width, width // 64, s["causal"], 0.125, s["out"])
    return s["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "mel":
        # A real transform of each frame, its power and the filterbank's
        # triangles (each bin is in two of them).
        bins = 201
        return {"bytes": 4.0 * (480000 + bins * case["bands"] + 3000 * case["bands"]),
                "flops": 3000.0 * (2.5 * 400 * math.log2(400) + 3 * bins + 4 * bins + case["bands"])}
    d = case["width"]
    f = 4 * d
    if kind == "encoder":
        t, size = case["positions"], _BYTES[case["dtype"]]
        frames = 2 * t
        flops = 2.0 * frames * 3 * case["bands"] * d + 2.0 * t * 3 * d * d
        flops += case["layers"] * (2.0 * t * (4 * d * d + 2 * d * f) + 4.0 * t * t * d)
        weights = 4.0 * (3 * case["bands"] * d + 3 * d * d + t * d) + case["layers"] * (4 * d * d + 2 * d * f) * size
        return {"bytes": weights + 4.0 * frames * case["bands"] + 4.0 * t * d, "flops": flops}
    if kind in ("decode", "batch"):
        streams = case.get("streams", 1)
        size, layers, rows, vocab = _BYTES[case["dtype"]], case["layers"], case["rows"], case["vocab"]
        projections = layers * (6 * d * d + 2 * d * f) * size + vocab * d * size
        moved = streams * rows * d * 4.0 + layers * 2.0 * d * d * size + 2.0 * streams * layers * rows * d * 4
        flops = streams * layers * 4.0 * rows * d * d
        position = 0
        for tokens in [case["prompt"]] + [1] * case["steps"]:
            keys = position + tokens
            moved += projections + streams * (layers * 2.0 * (rows + keys) * d * 4 + tokens * vocab * 4.0)
            per_token = layers * (2.0 * (6 * d * d + 2 * d * f) + 4.0 * (rows + keys) * d) + 2.0 * vocab * d
            flops += streams * tokens * per_token
            position += tokens
        return {"bytes": moved, "flops": flops}
    if kind == "mlp":
        rows = case["rows"]
        return {"bytes": 2.0 * d * f * _BYTES[case["dtype"]] + 8.0 * rows * d, "flops": 4.0 * rows * d * f}
    q, k = case["queries"], case["keys"]
    return {"bytes": 8.0 * (q + k) * d, "flops": 4.0 * q * k * d}


# ---------------------------------------------------------------------------
# what the results are held to
# ---------------------------------------------------------------------------

# Every path accumulates in fp32 and keeps its operands to about 2^-22: against
# 64 bits the listed and drawn cases measure rel 1e-7 to 1.3e-6 and max 4e-7 to
# 8e-6 (the deepest chains the most), and these are about four times that.
# Whole numbers (sampled tokens) have to be equal.
_TOLERANCES = {
    "mel": {"rel": 1.5e-6, "max": 1e-5},
    "encoder": {"rel": 5e-6, "max": 3e-5},
    "decode": {"rel": 5e-6, "max": 3e-5},
    "batch": {"rel": 4e-6, "max": 2e-5},
    "mlp": {"rel": 2e-6, "max": 1.5e-5},
    "attention": {"rel": 1.2e-6, "max": 1.6e-5},
}


def tolerance(case):
    return _TOLERANCES[case["kind"]]


def _wide(tensor):
    return tensor.double()


def _norm(x, gamma, beta):
    centred = x - x.mean(-1, keepdim=True)
    return centred / torch.sqrt((centred * centred).mean(-1, keepdim=True) + 1e-5) * gamma + beta


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _heads(x):
    """[..., rows, width] to [..., heads, rows, 64]."""
    return x.reshape(*x.shape[:-1], -1, 64).transpose(-2, -3).contiguous()


def _attend(q, k, v, hidden=None):
    """q, k, v [..., rows, width]; `hidden` marks the keys a query does not see."""
    scores = torch.matmul(_heads(q), _heads(k).transpose(-1, -2).contiguous()) * 0.125
    if hidden is not None:
        scores = scores.masked_fill(hidden, -math.inf)
    rows = torch.matmul(torch.softmax(scores, -1), _heads(v))
    return rows.transpose(-2, -3).reshape(q.shape)


def _future(queries, keys):
    """Which of `keys` positions the last `queries` of them do not see."""
    own = torch.arange(keys - queries, keys, device="cuda")[:, None]
    return torch.arange(keys, device="cuda")[None, :] > own


def _exact_mel(case, seed):
    shape, samples, filters = _audio(case, seed)
    x = np.pad(samples.double().cpu().numpy(), shape.fft_length // 2, mode="reflect")
    n = np.arange(shape.fft_length)
    window = 0.5 * (1.0 - np.cos(2.0 * np.pi * n / shape.fft_length))
    frames = x[np.arange(shape.frame_count)[:, None] * shape.hop_length + n[None, :]] * window
    spectrum = np.fft.rfft(frames, axis=1)
    power = spectrum.real ** 2 + spectrum.imag ** 2
    mel = np.log10(np.maximum(filters.double().cpu().numpy() @ power.T, 1e-10))
    return (np.maximum(mel, mel.max() - 8.0) + 4.0) / 4.0


def _taps(x, stride):
    """[channels, frames] to [out frames, channels * 3]: kernel 3, padding 1."""
    padded = torch.nn.functional.pad(x, (1, 1))
    return padded.unfold(1, 3, stride).permute(1, 0, 2).reshape(-1, 3 * x.shape[0])


def _exact_encoder(case, seed):
    draws = _Draws(seed)
    w = {name: _wide(t) for name, t, _ in _encoder_tensors(case, draws)}
    mel = _wide(_mel_rows(case, draws))[:, :2 * case["positions"]]
    conv = [w[n] for n in S.ENCODER_MODEL_NAMES[:4]]
    x = _gelu(_taps(mel, 1) @ conv[0].flatten(1).T + conv[1])
    h = _gelu(_taps(x.T, 2) @ conv[2].flatten(1).T + conv[3])
    h = h + w[S.ENCODER_MODEL_NAMES[4]][:h.shape[0]]
    for layer in range(case["layers"]):
        p = {s: w[S.encoder_layer_name(layer, s)] for s in S.ENCODER_LAYER_SUFFIXES}
        y = _norm(h, p["self_attn_layer_norm.weight"], p["self_attn_layer_norm.bias"])
        att = _attend(y @ p["self_attn.q_proj.weight"].T + p["self_attn.q_proj.bias"], y @ p["self_attn.k_proj.weight"].T,
                      y @ p["self_attn.v_proj.weight"].T + p["self_attn.v_proj.bias"])
        h = h + att @ p["self_attn.out_proj.weight"].T + p["self_attn.out_proj.bias"]
        y = _norm(h, p["final_layer_norm.weight"], p["final_layer_norm.bias"])
        h = h + _gelu(y @ p["fc1.weight"].T + p["fc1.bias"]) @ p["fc2.weight"].T + p["fc2.bias"]
    return _norm(h, w[S.ENCODER_MODEL_NAMES[5]], w[S.ENCODER_MODEL_NAMES[6]])


def _exact_decode(case, seed):
    """Greedy decoding of all streams ([streams, rows, width] throughout)."""
    draws, streams = _Draws(seed), case.get("streams", 1)
    w = {name: _wide(t) for name, t, _ in _decoder_tensors(case, draws)}
    encoded = _wide(draws.normal((streams, case["rows"], case["width"]), 1.0))
    layers = [{s: w[S.layer_name(i, s)] for s in S.LAYER_SUFFIXES} for i in range(case["layers"])]
    cross = [(encoded @ p["encoder_attn.k_proj.weight"].T,
              encoded @ p["encoder_attn.v_proj.weight"].T + p["encoder_attn.v_proj.bias"]) for p in layers]
    cache = [None] * len(layers)
    tokens = _prompt(case, seed, streams * case["prompt"]).reshape(streams, -1).cuda().long()
    position, sampled, logits = 0, [], []
    for _ in range(case["steps"] + 1):
        count = tokens.shape[1]
        h = w[S.MODEL_NAMES[0]][tokens] + w[S.MODEL_NAMES[1]][position:position + count]
        for i, p in enumerate(layers):
            y = _norm(h, p["self_attn_layer_norm.weight"], p["self_attn_layer_norm.bias"])
            k = y @ p["self_attn.k_proj.weight"].T
            v = y @ p["self_attn.v_proj.weight"].T + p["self_attn.v_proj.bias"]
            if cache[i] is not None:
                k, v = torch.cat([cache[i][0], k], 1), torch.cat([cache[i][1], v], 1)
            cache[i] = (k, v)
            att = _attend(y @ p["self_attn.q_proj.weight"].T + p["self_attn.q_proj.bias"], k, v,
                          _future(count, k.shape[1]))
            h = h + att @ p["self_attn.out_proj.weight"].T + p["self_attn.out_proj.bias"]
            y = _norm(h, p["encoder_attn_layer_norm.weight"], p["encoder_attn_layer_norm.bias"])
            att = _attend(y @ p["encoder_attn.q_proj.weight"].T + p["encoder_attn.q_proj.bias"], *cross[i])
            h = h + att @ p["encoder_attn.out_proj.weight"].T + p["encoder_attn.out_proj.bias"]
            y = _norm(h, p["final_layer_norm.weight"], p["final_layer_norm.bias"])
            h = h + _gelu(y @ p["fc1.weight"].T + p["fc1.bias"]) @ p["fc2.weight"].T + p["fc2.bias"]
        position += count
        logits.append(_norm(h, w[S.MODEL_NAMES[2]], w[S.MODEL_NAMES[3]]) @ w[S.MODEL_NAMES[0]].T)
        tokens = logits[-1][:, -1].argmax(-1, keepdim=True)
        sampled.append(tokens.int())
        if case["kind"] == "batch" and len(logits) > 2:
            logits[-2] = None
    if case["kind"] == "batch":
        return logits[0].flatten(0, 1), logits[-1].flatten(0, 1), torch.cat(sampled, 1).T.contiguous()
    prompt = _prompt(case, seed, case["prompt"]).cuda()
    return torch.cat(logits, 1)[0], torch.cat([prompt] + [t[0] for t in sampled])


def exact(case, seed):
    kind = case["kind"]
    if kind == "mel":
        return _exact_mel(case, seed)
    if kind == "encoder":
        return _exact_encoder(case, seed)
    if kind in ("decode", "batch"):
        return _exact_decode(case, seed)
    if kind == "mlp":
        p = {n: _wide(t) for n, t in _mlp_inputs(case, seed).items()}
        y = _gelu(_norm(p["x"], p["gamma"], p["beta"]) @ p["fc1"].T + p["fc1_bias"])
        return p["x"] + y @ p["fc2"].T + p["fc2_bias"]
    p = {n: _wide(t) for n, t in _attention_inputs(case, seed).items()}
    return _attend(p["q"], p["k"], p["v"], _future(case["queries"], case["keys"]) if case["causal"] else None)
