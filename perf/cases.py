"""Performance cases: the work a program does through this framework, from one RMSNorm to a
whole 40-step sampling run, with float64 results to compare against.

A case is a dict of plain values.  `listed` holds the fixed ones, `draw` one more of the same
ranges, `prepare` makes what a program has in hand before the call (inputs from the seed, the
engine / encoder / codec with its weights), `run` is one pass through the public entry points,
`work` the bytes and operations it cannot do without, `tolerance` how far another correct
implementation at the same precision may be, and `exact` the same pass in float64 torch.

The model shapes are the package's own configurations; text holds up to 256 tokens, the
reference audio up to 375 latent frames, an utterance up to 750 latent frames (30 s).
"""
import functools
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "irodori-tts-burn_amd"))
import irodori_hip as ih  # noqa: E402
from irodori_hip import _lib  # noqa: E402
from irodori_hip.engine import ops  # noqa: E402

DEV = "cuda"
F64 = torch.float64
BACKEND = {"bf16": ih.InferenceBackendKind.HIP_BF16, "f32": ih.InferenceBackendKind.HIP_F32,
           "fp8": ih.InferenceBackendKind.HIP_FP8}
TORCH_TYPE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
OP_TYPE = {"f32": _lib.DTYPE_F32, "bf16": _lib.DTYPE_BF16, "f16": _lib.DTYPE_F16}


# ---- the cases ----------------------------------------------------------------------------
def listed():
    return [
        # The smallest call: one norm over a few rows, where the launch is all there is.
        dict(name="rms_norm_rows4", kind="rms_norm", rows=4, dim=1024),
        # The modulated norm of one block over both guidance rows of a 30 s utterance.
        dict(name="adaln_2x750", kind="adaln", batch=2, seq=750, dim=1024),
        # The attention operator at the published model's heads and a 30 s utterance, masked keys.
        dict(name="sdpa_bf16_750x950", kind="sdpa", dtype="bf16", batch=1, heads=20, sq=750, skv=950, dh=64, masked=True),
        # The same operator as an f32 program calls it, on a 15 s utterance.
        dict(name="sdpa_f32_375x631", kind="sdpa", dtype="f32", batch=2, heads=16, sq=375, skv=631, dh=64, masked=False),
        # The attention half of a block: head norms, RoPE, latent + text + speaker keys, gate.
        dict(name="joint_attention_2x750", kind="joint_attention", dtype="bf16", batch=2, seq=750, t_text=256, t_aux=375),
        # The MLP half of a block on 1500 tokens.
        dict(name="swiglu_mlp_2x750", kind="swiglu_mlp", dtype="bf16", batch=2, seq=750),
        # One fp8 projection (quantize, multiply) of two utterances' guidance rows.
        dict(name="fp8_linear_3000", kind="fp8_linear", m=3000, n=5632, k=1024),
        # A request's text through the 14-layer text encoder.
        dict(name="encode_text_256", kind="encode", dtype="bf16", which="text", batch=1, seq=256),
        # A program with its own integrator: the context of a new request, then one model forward.
        dict(name="context_and_forward_750", kind="first_eval", dtype="bf16", seq=750, t_text=256, t_aux=375),
        # A short utterance (4 s, odd length) with the default guidance (text and speaker dropped
        # in turn, the second half of the steps unguided).
        dict(name="sample_short_101", kind="sample", dtype="bf16", mode="independent", utterances=1, seq=101, steps=40,
             t_text=37, t_aux=125),
        # The headline run: 30 s, joint guidance on every one of 40 steps.
        dict(name="sample_joint_750", kind="sample", dtype="bf16", mode="joint", utterances=1, seq=750, steps=40,
             t_text=256, t_aux=375),
        # The waveform of a 30 s utterance from its latent.
        dict(name="codec_decode_750", kind="codec", dtype="bf16", batch=1, frames=750),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["rms_norm", "adaln", "sdpa", "sdpa", "joint_attention", "swiglu_mlp", "fp8_linear", "encode",
                       "encode", "first_eval", "sample", "sample", "codec"])
    if kind == "rms_norm":
        return dict(kind=kind, rows=_log_int(rng, 1, 24000), dim=rng.choice([96, 256, 1000, 1024, 1280, 2048]))
    if kind == "adaln":
        return dict(kind=kind, batch=_log_int(rng, 1, 32), seq=_log_int(rng, 1, 750),
                    dim=rng.choice([96, 256, 1024, 1280, 2048]))
    if kind == "sdpa":
        return dict(kind=kind, dtype=rng.choice(["f32", "bf16", "f16"]), batch=rng.randint(1, 3),
                    heads=rng.choice([2, 10, 16, 20]), sq=_log_int(rng, 1, 1500), skv=_log_int(rng, 1, 1500),
                    dh=rng.choice([64, 64, 128]), masked=rng.random() < 0.5)
    if kind == "joint_attention":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f32"]), batch=rng.randint(1, 4), seq=_log_int(rng, 3, 750),
                    t_text=_log_int(rng, 4, 256), t_aux=_log_int(rng, 1, 375))
    if kind == "swiglu_mlp":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]), batch=rng.randint(1, 4),
                    seq=_log_int(rng, 3, 750))
    if kind == "fp8_linear":
        n, k = rng.choice([(5632, 1024), (4096, 1024), (1024, 2816), (1024, 1024)])
        return dict(kind=kind, m=_log_int(rng, 1, 12000), n=n, k=k)
    if kind == "encode":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]), which=rng.choice(["text", "speaker"]),
                    batch=rng.randint(1, 2), seq=_log_int(rng, 4, 375))
    if kind == "first_eval":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f32"]), seq=_log_int(rng, 8, 750),
                    t_text=_log_int(rng, 4, 256), t_aux=_log_int(rng, 1, 375))
    if kind == "sample":
        utt = rng.randint(1, 2)
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "fp8"]), mode=rng.choice(["joint", "independent"]),
                    utterances=utt, seq=_log_int(rng, 8, 750 // utt), steps=rng.choice([4, 8, 16, 24, 40]),
                    t_text=_log_int(rng, 4, 256), t_aux=_log_int(rng, 1, 375))
    batch = rng.randint(1, 2)
    return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]), batch=batch,
                frames=_log_int(rng, 2, 750 // (2 * batch)))


# ---- model handles: the weights a program loads once ---------------------------------------
@functools.lru_cache(maxsize=None)
def _dit_cfg(layers):
    cfg = ih.cfg_full_rf()
    cfg.num_layers = layers
    return cfg


@functools.lru_cache(maxsize=None)
def _dit_weights(layers):
    return ih.DitWeights.random(_dit_cfg(layers), seed=11, std=0.02, norm_jitter=0.1)


@functools.lru_cache(maxsize=None)
def _ctx_proj(layers):
    return ih.CtxProjWeights.random(_dit_cfg(layers), 1280, 1280, seed=12)


@functools.lru_cache(maxsize=None)
def _encoder(which):
    # The default encoders; a vocabulary of 8192 keeps the embedding table small (a token
    # costs one row of it at any vocabulary).
    cfg = ih.enc_text_default() if which == "text" else ih.enc_speaker_default()
    if which == "text":
        cfg.vocab_size = 8192
    return cfg, ih.EncoderWeights.random(cfg, seed=13, std=0.02, norm_jitter=0.1)


@functools.lru_cache(maxsize=None)
def _codec():
    cfg = ih.codec_default()
    return cfg, ih.CodecWeights.random(cfg, seed=14)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 * seed + 17)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)


def _guidance(case):
    """Joint: one scale on every step; independent: the defaults (text 3, speaker 5, guided
    while t >= 0.5)."""
    if case["mode"] == "joint":
        g = ih.GuidanceConfig(mode=ih.CfgGuidanceMode.JOINT, scale_text=3.0, scale_speaker=3.0, min_t=0.0)
    else:
        g = ih.GuidanceConfig()
    return ih.SamplerParams(num_steps=case["steps"], guidance=g)


def _roles(case):
    return ["cond", "uncond"] if case["mode"] == "joint" else ["cond", "no_text", "no_aux"]


def _context(case, seed, roles, utterances, layers):
    return ih.make_role_context(_dit_cfg(layers), utterances, case["t_text"], case["t_aux"], roles, seed=1000 + seed)


# ---- prepare ------------------------------------------------------------------------------
def prepare(case, seed):
    st = _PREPARE[case["kind"]](case, seed)
    st["case"] = case
    torch.cuda.synchronize()
    return st


def _inputs_rms(case, seed):
    g = _gen(seed)
    x = _randn(g, case["rows"], case["dim"])
    w = 1 + 0.1 * _randn(g, case["dim"])
    return x, w


def _prepare_rms(case, seed):
    x, w = _inputs_rms(case, seed)
    return dict(x=x, w=w)


def _inputs_adaln(case, seed):
    g = _gen(seed)
    x = _randn(g, case["batch"], case["seq"], case["dim"])
    scale, shift = 0.1 * _randn(g, case["batch"], case["dim"]), 0.1 * _randn(g, case["batch"], case["dim"])
    return x, scale, shift


def _prepare_adaln(case, seed):
    x, scale, shift = _inputs_adaln(case, seed)
    return dict(x=x, scale=scale, shift=shift)


def _inputs_sdpa(case, seed):
    g = _gen(seed)
    B, H, dh = case["batch"], case["heads"], case["dh"]
    t = TORCH_TYPE[case["dtype"]]
    q = _randn(g, B, H, case["sq"], dh).to(t)
    k = _randn(g, B, H, case["skv"], dh).to(t)
    v = _randn(g, B, H, case["skv"], dh).to(t)
    mask = None
    if case["masked"]:  # the text's padding: the last keys of each row
        n = torch.randint((case["skv"] + 1) // 2, case["skv"] + 1, (B, 1), generator=g, device=DEV)
        mask = (torch.arange(case["skv"], device=DEV)[None] < n).float()
    return q, k, v, mask


def _prepare_sdpa(case, seed):
    q, k, v, mask = _inputs_sdpa(case, seed)
    return dict(q=q, k=k, v=v, mask=mask)


def _inputs_joint(case, seed):
    g = _gen(seed)
    B, S, H = case["batch"], case["seq"], _dit_cfg(1).num_heads
    q, k, v = (_randn(g, B, S, H, 64) for _ in range(3))
    gate = _randn(g, B, S, H * 64)
    roles = ["cond", "uncond", "no_text", "no_aux"][:B]
    return q, k, v, gate, _context(case, seed, roles, 1, 1)


def _block_engine(case, t_ctx):
    eng = ih.HipInferenceEngine(_dit_cfg(1), BACKEND[case["dtype"]], max_rows=case["batch"], max_seq=case["seq"],
                                max_ctx=t_ctx)
    eng.load_weights(_dit_weights(1))
    return eng


def _prepare_joint(case, seed):
    q, k, v, gate, ctx = _inputs_joint(case, seed)
    eng = _block_engine(case, ctx.t_ctx)
    eng.set_context_kv(ctx)
    return dict(q=q, k=k, v=v, gate=gate, eng=eng, stream=torch.cuda.Stream())


def _inputs_mlp(case, seed):
    g = _gen(seed)
    B, S, D = case["batch"], case["seq"], _dit_cfg(1).model_dim
    x = _randn(g, B, S, D)
    shift, scale = 0.1 * _randn(g, B, D), 0.1 * _randn(g, B, D)
    gate = torch.tanh(0.5 * _randn(g, B, D))
    return x, shift, scale, gate


def _prepare_mlp(case, seed):
    x, shift, scale, gate = _inputs_mlp(case, seed)
    return dict(x=x, shift=shift, scale=scale, gate=gate, eng=_block_engine(case, 1), stream=torch.cuda.Stream())


def _inputs_fp8(case, seed):
    g = _gen(seed)
    x = _randn(g, case["m"], case["k"])
    w = 0.02 * _randn(g, case["n"], case["k"])  # the layer's weight: e4m3 codes, one scale a row
    ws = w.abs().amax(1) / 448.0
    return x, (w / ws[:, None]).to(torch.float8_e4m3fn).view(torch.uint8), ws


def _prepare_fp8(case, seed):
    x, w8, ws = _inputs_fp8(case, seed)
    return dict(x=x, w8=w8, ws=ws)


def _inputs_encode(case, seed):
    rng = np.random.default_rng(seed)
    cfg, _ = _encoder(case["which"])
    B, S = case["batch"], case["seq"]
    mask = np.ones((B, S), np.uint8)
    if B > 1:  # a batch is padded to its longest row
        mask[1, (S + 1) // 2 + int(rng.integers(0, S // 2 + 1)):] = 0
    if case["which"] == "text":
        return mask, dict(ids=rng.integers(0, cfg.vocab_size, (B, S)).astype(np.int32))
    return mask, dict(latent=rng.standard_normal((B, S, cfg.in_dim)).astype(np.float32))


def _prepare_encode(case, seed):
    mask, inp = _inputs_encode(case, seed)
    cfg, w = _encoder(case["which"])
    enc = ih.HipEncoder(cfg, BACKEND[case["dtype"]], max_rows=case["batch"], max_seq=case["seq"])
    enc.load_weights(w)
    return dict(enc=enc, mask=mask, inp=inp)


def _inputs_first_eval(case, seed):
    rng = np.random.default_rng(seed)
    text = rng.standard_normal((case["t_text"], 1280)).astype(np.float32)  # encoder states are RMS-normed
    aux = rng.standard_normal((case["t_aux"], 1280)).astype(np.float32)
    tm = np.zeros(case["t_text"], np.uint8)
    tm[:max(1, int(rng.integers(case["t_text"] // 2, case["t_text"] + 1)))] = 1
    am = np.ones(case["t_aux"], np.uint8)
    x = rng.standard_normal((1, case["seq"], 32)).astype(np.float32).repeat(2, 0)  # both guidance rows: one state
    t = np.full(2, rng.uniform(0.1, 0.95), np.float32)
    return text, tm, aux, am, x, t


def _prepare_first_eval(case, seed):
    layers = 12
    eng = ih.HipInferenceEngine(_dit_cfg(layers), BACKEND[case["dtype"]], max_rows=2, max_seq=case["seq"],
                                max_ctx=case["t_text"] + case["t_aux"])
    eng.load_weights(_dit_weights(layers))
    eng.load_ctx_proj_weights(_ctx_proj(layers))
    return dict(eng=eng, inp=_inputs_first_eval(case, seed))


def _inputs_sample(case, seed):
    x0 = np.random.default_rng(seed).standard_normal((case["utterances"], case["seq"], 32)).astype(np.float32)
    return x0, _context(case, seed, _roles(case), case["utterances"], 12)


def _prepare_sample(case, seed):
    x0, ctx = _inputs_sample(case, seed)
    eng = ih.HipInferenceEngine(_dit_cfg(12), BACKEND[case["dtype"]], max_rows=ctx.mask.shape[0], max_seq=case["seq"],
                                max_ctx=ctx.t_ctx)
    eng.load_weights(_dit_weights(12))
    eng.set_context_kv(ctx)
    return dict(eng=eng, x0=x0, params=_guidance(case))


def _inputs_codec(case, seed):
    return _randn(_gen(seed), case["batch"], case["frames"], 32)


def _prepare_codec(case, seed):
    cfg, w = _codec()
    codec = ih.HipDacVaeCodec(cfg, BACKEND[case["dtype"]], max_frames=case["frames"])
    codec.load_weights(w)
    return dict(codec=codec, latent=_inputs_codec(case, seed), hop=cfg.hop_length, stream=torch.cuda.Stream())


# ---- run ----------------------------------------------------------------------------------
def run(st):
    return _RUN[st["case"]["kind"]](st, st["case"])


def _current():
    return torch.cuda.current_stream().cuda_stream


def _on_stream(st, call):
    """call(stream handle) in order with torch's current stream.  The context and codec entry
    points read a null handle as their own stream, so a program on torch's default stream
    hands them one of its own."""
    cur = torch.cuda.current_stream()
    if cur.cuda_stream:
        call(cur.cuda_stream)
        return
    st["stream"].wait_stream(cur)
    call(st["stream"].cuda_stream)
    cur.wait_stream(st["stream"])


def _run_rms(st, case):
    y = torch.empty_like(st["x"])
    ops.rms_norm(st["x"].data_ptr(), st["w"].data_ptr(), case["rows"], case["dim"], 1e-6, y.data_ptr(), _current())
    return y


def _run_adaln(st, case):
    y = torch.empty_like(st["x"])
    ops.fused_adaln(st["x"].data_ptr(), st["scale"].data_ptr(), st["shift"].data_ptr(), case["batch"], case["seq"],
                    case["dim"], 1e-6, y.data_ptr(), _current())
    return y


def _run_sdpa(st, case):
    out = torch.empty(st["q"].shape, dtype=torch.float32, device=DEV)
    ops.sdpa(OP_TYPE[case["dtype"]], st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(),
             st["mask"].data_ptr() if case["masked"] else 0, case["batch"], case["heads"], case["sq"], case["skv"],
             case["dh"], case["dh"] ** -0.5, out.data_ptr(), _current())
    return out


def _run_joint(st, case):
    out = torch.empty_like(st["gate"])
    _on_stream(st, lambda s: st["eng"].joint_attention(0, case["batch"], case["seq"], st["q"].data_ptr(),
                                                       st["k"].data_ptr(), st["v"].data_ptr(), st["gate"].data_ptr(),
                                                       out.data_ptr(), s))
    return out


def _run_mlp(st, case):
    x = st["x"].clone()  # updated in place
    _on_stream(st, lambda s: st["eng"].swiglu_mlp(0, case["batch"], case["seq"], x.data_ptr(), st["shift"].data_ptr(),
                                                  st["scale"].data_ptr(), st["gate"].data_ptr(), s))
    return x


def _run_fp8(st, case):
    m, n, k = case["m"], case["n"], case["k"]
    q = torch.empty(m, k, dtype=torch.uint8, device=DEV)
    s = torch.empty(m, k // 32, dtype=torch.uint8, device=DEV)
    c = torch.empty(m, n, dtype=torch.float32, device=DEV)
    ops.mx_quantize(st["x"].data_ptr(), m, k, q.data_ptr(), s.data_ptr(), _current())
    ops.gemm_fp8(q.data_ptr(), s.data_ptr(), st["w8"].data_ptr(), st["ws"].data_ptr(), m, n, k, c.data_ptr(), _current())
    return c


def _run_encode(st, case):
    state, mask = st["enc"].forward(st["mask"], **st["inp"])
    return state, mask


def _run_first_eval(st, case):
    eng = st["eng"]
    text, tm, aux, am, x, t = st["inp"]
    eng.clear_context_kv()
    eng.build_context_kv(0, text, tm, aux, am)
    eng.build_context_kv(1, np.zeros_like(text), np.zeros_like(tm), np.zeros_like(aux), np.zeros_like(am))
    return eng.forward_with_cond_cached(x, t)


def _run_sample(st, case):
    return st["eng"].sample(st["x0"], st["params"], has_speaker=True, ctx_aux_start=case["t_text"])


def _run_codec(st, case):
    wav = torch.empty(case["batch"], 1, case["frames"] * st["hop"], dtype=torch.float32, device=DEV)
    _on_stream(st, lambda s: st["codec"].decode_device(st["latent"].data_ptr(), case["batch"], case["frames"],
                                                       wav.data_ptr(), s))
    return wav


# ---- work ---------------------------------------------------------------------------------
def work(case):
    b, f = _WORK[case["kind"]](case)
    return {"bytes": int(b), "flops": int(f)}


_SIZE = {"f32": 4, "bf16": 2, "f16": 2, "fp8": 1}


def _block_params(cfg):
    D = cfg.model_dim
    return 5 * D * D + 3 * D * cfg.mlp_hidden


def _dit_work(cfg, dtype, rows, seq, keys, evals):
    """Model forwards: weights once per forward, the latents in and out; keys = attended keys
    of every row, summed."""
    D, tok = cfg.model_dim, rows * seq
    flops = cfg.num_layers * (2 * tok * _block_params(cfg) + 4 * D * seq * keys)
    kv = cfg.num_layers * 2 * (keys - rows * seq) * D * 2
    return evals * (cfg.num_layers * _block_params(cfg) * _SIZE[dtype] + kv + 8 * tok * cfg.latent_dim), evals * flops


def _work_rms(c):
    return 8 * c["rows"] * c["dim"] + 4 * c["dim"], 4 * c["rows"] * c["dim"]


def _work_adaln(c):
    n = c["batch"] * c["seq"] * c["dim"]
    return 8 * n + 8 * c["batch"] * c["dim"], 5 * n


def _work_sdpa(c):
    bh = c["batch"] * c["heads"] * c["dh"]
    return bh * (_SIZE[c["dtype"]] * (c["sq"] + 2 * c["skv"]) + 4 * c["sq"]), 4 * bh * c["sq"] * c["skv"]


def _work_joint(c):
    D, T = _dit_cfg(1).model_dim, c["t_text"] + c["t_aux"]
    n = c["batch"] * c["seq"] * D
    # the guidance rows drop the text, the speaker or both
    keys = sum((c["seq"] + T, c["seq"], c["seq"] + c["t_aux"], c["seq"] + c["t_text"])[:c["batch"]])
    return 20 * n + 2 * (keys - c["batch"] * c["seq"]) * D * _SIZE[c["dtype"]], 4 * D * c["seq"] * keys


def _work_mlp(c):
    cfg = _dit_cfg(1)
    n, w = c["batch"] * c["seq"], 3 * cfg.model_dim * cfg.mlp_hidden
    return 8 * n * cfg.model_dim + w * _SIZE[c["dtype"]], 2 * n * w


def _work_fp8(c):
    return 4 * c["m"] * c["k"] + c["n"] * c["k"] + 4 * c["m"] * c["n"], 2 * c["m"] * c["n"] * c["k"]


def _work_encode(c):
    cfg, _ = _encoder(c["which"])
    E, tok = cfg.dim, c["batch"] * c["seq"]
    params = cfg.num_layers * (5 * E * E + 3 * E * cfg.mlp_hidden)
    return params * _SIZE[c["dtype"]] + 8 * tok * E, 2 * tok * params + cfg.num_layers * 4 * E * tok * c["seq"]


def _work_first_eval(c):
    cfg = _dit_cfg(12)
    T, D = c["t_text"] + c["t_aux"], cfg.model_dim
    b, f = _dit_work(cfg, c["dtype"], 2, c["seq"], 2 * c["seq"] + T, 1)
    proj = cfg.num_layers * 2 * 2 * 1280 * D  # text and speaker, K and V (zero states need no product)
    return b + proj * _SIZE[c["dtype"]] + 4 * T * 1280, f + proj * T


def _work_sample(c):
    cfg = _dit_cfg(12)
    U, S, T, n = c["utterances"], c["seq"], c["t_text"] + c["t_aux"], c["steps"]
    if c["mode"] == "joint":
        return _dit_work(cfg, c["dtype"], 2 * U, S, U * (2 * S + T), n)
    guided = sum(0.999 * (1 - i / n) >= 0.5 for i in range(n))
    a = _dit_work(cfg, c["dtype"], 3 * U, S, U * (3 * S + 2 * T), guided)
    b = _dit_work(cfg, c["dtype"], U, S, U * (S + T), n - guided)
    return a[0] + b[0], a[1] + b[1]


def _work_codec(c):
    cfg, _ = _codec()
    es, L = _SIZE[c["dtype"]], c["frames"]
    params = cfg.proj_dim * cfg.latent_dim + 7 * cfg.proj_dim * cfg.decoder_dim
    flops = 2 * L * params
    for i, r in enumerate(cfg.rates):
        cin, cout = cfg.block_dims(i)
        flops += 2 * L * cin * cout * 2 * r
        L *= r
        params += cin * cout * 2 * r + 3 * 8 * cout * cout
        flops += 2 * L * 3 * 8 * cout * cout
    flops += 2 * L * 7 * cfg.head_dim
    return params * es + c["batch"] * 4 * (c["frames"] * cfg.latent_dim + L), c["batch"] * flops


# ---- tolerance ----------------------------------------------------------------------------
def tolerance(case):
    kind, dtype = case["kind"], case.get("dtype", "f32")
    if kind == "encode":  # the speaker states are unbounded latents, the text states table rows
        kind = "encode_" + case["which"]
    return {"rel": _TOL[kind][dtype]}


# Four times the relative error measured against float64 over the ranges (in brackets): the
# rounding of the operands in 16 bits and fp8, that of the sums in f32.  The f32 rows of the
# joint attention and the models hold the f32 RoPE tables too.
_TOL = {
    "rms_norm": {"f32": 2.5e-7},                               # [6e-8]
    "adaln": {"f32": 2.5e-7},                                  # [6e-8]
    "sdpa": {"f32": 3e-6, "bf16": 1e-2, "f16": 1.2e-3},        # [7.5e-7, 2.4e-3, 2.9e-4]
    "joint_attention": {"bf16": 1.6e-2, "f32": 1e-5},          # [4.1e-3, 2.3e-6]
    "swiglu_mlp": {"bf16": 1.6e-3, "f32": 5.5e-7},             # [4.2e-4, 1.3e-7]
    "fp8_linear": {"f32": 6e-5},                               # [1.5e-5]
    "encode_text": {"bf16": 2.3e-2, "f32": 8e-6},              # [5.8e-3, 1.8e-6]
    "encode_speaker": {"bf16": 7.5e-2, "f32": 2.2e-5},         # [1.9e-2, 5.3e-6]
    "first_eval": {"bf16": 5.5e-3, "f32": 6.5e-6},             # [1.4e-3, 1.6e-6]
    "sample": {"bf16": 8e-3, "fp8": 0.11},                     # [1.9e-3, 2.8e-2]
    "codec": {"bf16": 5.3e-2, "f32": 2.3e-5},                  # [1.3e-2, 5.8e-6]
}


# ---- exact: the same in float64 torch --------------------------------------------------------
def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _t(a):
    return torch.as_tensor(a).to(DEV, F64)


def _rms(x, eps):
    return torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _exact_rms(case, seed):
    x, w = (a.double() for a in _inputs_rms(case, seed))
    return x / _rms(x, 1e-6) * w


def _exact_adaln(case, seed):
    x, scale, shift = (a.double() for a in _inputs_adaln(case, seed))
    return x / _rms(x, 1e-6) * (1 + scale[:, None]) + shift[:, None]


def _attend(q, k, v, mask, scale):
    """[B, H, S, Dh] attention; a row without a valid key gives 0."""
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) * scale
    if mask is not None:
        s = s.masked_fill(~mask[:, None, None, :], -math.inf)
    return torch.matmul(torch.nan_to_num(torch.softmax(s, -1)), v)


def _exact_sdpa(case, seed):
    q, k, v, mask = _inputs_sdpa(case, seed)
    return _attend(q.double(), k.double(), v.double(), None if mask is None else mask >= 0.5, case["dh"] ** -0.5)


def _rope(x):
    """Interleaved pairs of [B, S, H, Dh] rotated by their position."""
    B, S, H, Dh = x.shape
    freq = 10000.0 ** (-2.0 * torch.arange(Dh // 2, device=DEV, dtype=F64) / Dh)
    ang = torch.arange(S, device=DEV, dtype=F64)[:, None] * freq[None]
    c, s = torch.cos(ang)[None, :, None], torch.sin(ang)[None, :, None]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], -1).reshape(B, S, H, Dh)


def _joint(q, k, v, blk, ctx_k, ctx_v, ctx_mask, eps):
    """Head norms, half RoPE and attention over [latent | context] keys: [B, S, H * Dh]."""
    B, S, H, Dh = q.shape
    half = H // 2
    q = q / _rms(q, eps) * _t(blk["q_norm"])
    k = k / _rms(k, eps) * _t(blk["k_norm"])
    q = torch.cat([_rope(q[:, :, :half]), q[:, :, half:]], 2)
    k = torch.cat([_rope(k[:, :, :half]), k[:, :, half:]], 2)
    K, V = torch.cat([k, ctx_k], 1).transpose(1, 2), torch.cat([v, ctx_v], 1).transpose(1, 2)
    mask = torch.cat([torch.ones(B, S, device=DEV, dtype=torch.bool), ctx_mask], 1)
    o = _attend(q.transpose(1, 2).contiguous(), K.contiguous(), V.contiguous(), mask, Dh ** -0.5)
    return o.transpose(1, 2).reshape(B, S, H * Dh)


def _exact_joint(case, seed):
    q, k, v, gate, ctx = _inputs_joint(case, seed)
    o = _joint(q.double(), k.double(), v.double(), _dit_weights(1).blocks[0], _t(ctx.k[0]), _t(ctx.v[0]),
               torch.as_tensor(ctx.mask, device=DEV) > 0, _dit_cfg(1).norm_eps)
    return torch.sigmoid(gate.double()) * o


def _swiglu(h, w13, w2):
    u = h @ _t(w13)
    n = u.shape[-1] // 2
    return (F.silu(u[..., :n]) * u[..., n:]) @ _t(w2)


def _exact_mlp(case, seed):
    x, shift, scale, gate = (a.double() for a in _inputs_mlp(case, seed))
    blk = _dit_weights(1).blocks[0]
    h = x / _rms(x, _dit_cfg(1).norm_eps) * (1 + scale[:, None]) + shift[:, None]
    return x + gate[:, None] * _swiglu(h, blk["w13"], blk["w2"])


def _exact_fp8(case, seed):
    x, w8, ws = _inputs_fp8(case, seed)
    m, k = case["m"], case["k"]
    xb = x.view(m, k // 32, 32)
    amax = xb.abs().amax(2, keepdim=True).double()
    step = torch.exp2(torch.ceil(torch.log2(amax.clamp(min=2.0 ** -119) / 448.0)))
    xq = (xb.double() / step).to(torch.float32).to(torch.float8_e4m3fn).double() * step
    return (xq.view(m, k) @ w8.view(torch.float8_e4m3fn).double().t().contiguous()) * ws.double()


def _exact_encode(case, seed):
    mask, inp = _inputs_encode(case, seed)
    cfg, w = _encoder(case["which"])
    eps, H, E = cfg.norm_eps, cfg.num_heads, cfg.dim
    B, S = mask.shape
    valid = torch.as_tensor(mask, device=DEV) > 0
    m = valid.double()[..., None]
    if case["which"] == "text":
        x = _t(w.io["embedding"][inp["ids"]])
    else:
        x = (_t(inp["latent"]) @ _t(w.io["in_w"]) + _t(w.io["in_b"])) / 6.0
    x = x * m
    for blk in w.blocks:
        h = x / _rms(x, eps) * _t(blk["attn_norm"])
        q, k, v = ((h @ _t(blk[n])).view(B, S, H, E // H) for n in ("wq", "wk", "wv"))
        q = _rope(q / _rms(q, eps) * _t(blk["q_norm"]))
        k = _rope(k / _rms(k, eps) * _t(blk["k_norm"]))
        o = _attend(*(a.transpose(1, 2).contiguous() for a in (q, k, v)), valid, (E // H) ** -0.5)
        o = o.transpose(1, 2).reshape(B, S, E)
        x = x + (torch.sigmoid(h @ _t(blk["w_gate"])) * o) @ _t(blk["wo"])
        x = (x + _swiglu(x / _rms(x, eps) * _t(blk["mlp_norm"]), blk["w13"], blk["w2"])) * m
    state, out_mask = x / _rms(x, eps) * _t(w.io["out_norm"]), valid
    if cfg.mean_token:
        cnt = m.sum(1, keepdim=True)
        state = torch.cat([(state * m).sum(1, keepdim=True) / cnt.clamp(min=1.0), state], 1)
        out_mask = torch.cat([cnt[:, 0] > 0, out_mask], 1)
    return state.cpu().numpy(), out_mask.to(torch.uint8).cpu().numpy()


class _Dit:
    """The model in float64 on cached context keys / values [L, R, T, H, Dh]."""

    def __init__(self, layers):
        self.cfg, w = _dit_cfg(layers), _dit_weights(layers)
        self.io = {k: _t(a) for k, a in w.io.items()}
        self.blocks = [{k: ([[_t(a) for a in r] for r in v] if isinstance(v, list) else _t(v)) for k, v in b.items()}
                       for b in w.blocks]

    def _adaln(self, x, chunks, blk, i):
        shift, scale, gate = (F.silu(c) @ blk["ada_down"][i][n] @ blk["ada_up"][i][n] + blk["ada_up_b"][i][n] + c
                              for n, c in enumerate(chunks))
        h = x / _rms(x, self.cfg.norm_eps) * (1 + scale[:, None]) + shift[:, None]
        return h, torch.tanh(gate)[:, None]

    def __call__(self, x_t, t, ck, cv, mask):
        cfg, io = self.cfg, self.io
        B, S, _ = x_t.shape
        D, H, Dh = cfg.model_dim, cfg.num_heads, cfg.head_dim
        half = cfg.timestep_embed_dim // 2
        ang = t[:, None] * (1000.0 * torch.exp(-math.log(10000.0) * torch.arange(half, device=DEV, dtype=F64) / half))[None]
        c = torch.cat([torch.cos(ang), torch.sin(ang)], 1)
        c = F.silu(F.silu(c @ io["cond_w0"]) @ io["cond_w1"]) @ io["cond_w2"]
        chunks = [c[:, i * D:(i + 1) * D] for i in range(3)]
        x = x_t @ io["in_w"] + io["in_b"]
        for l, blk in enumerate(self.blocks):
            h, g = self._adaln(x, chunks, blk, 0)
            q, k, v = (a.reshape(B, S, H, Dh) for a in (h @ blk["w_qkv"]).split(H * Dh, -1))
            o = _joint(q, k, v, blk, ck[l], cv[l], mask, cfg.norm_eps)
            x = x + g * ((torch.sigmoid(h @ blk["w_gate"]) * o) @ blk["w_o"])
            h, g = self._adaln(x, chunks, blk, 1)
            x = x + g * _swiglu(h, blk["w13"], blk["w2"])
        return x / _rms(x, cfg.norm_eps) * io["out_norm_w"] @ io["out_w"] + io["out_b"]


def _exact_first_eval(case, seed):
    text, tm, aux, am, x, t = _inputs_first_eval(case, seed)
    net, eps = _Dit(12), _dit_cfg(12).norm_eps
    H, Dh = net.cfg.num_heads, net.cfg.head_dim
    ck, cv = [], []
    for blk, p in zip(net.blocks, _ctx_proj(12).layers):
        k, v = (torch.cat([_t(text) @ _t(p[n + "_text"]), _t(aux) @ _t(p[n + "_aux"])]).view(1, -1, H, Dh)
                for n in ("wk", "wv"))
        k = k / _rms(k, eps) * blk["k_norm"]
        ck.append(torch.cat([k, torch.zeros_like(k)]))
        cv.append(torch.cat([v, torch.zeros_like(v)]))
    m = np.concatenate([tm, am])
    mask = torch.as_tensor(np.stack([m, np.zeros_like(m)]), device=DEV) > 0
    return net(_t(x), _t(t), ck, cv, mask).cpu().numpy()


def _exact_sample(case, seed):
    x0, ctx = _inputs_sample(case, seed)
    net, p, U = _Dit(12), _guidance(case), case["utterances"]
    x, ck, cv = _t(x0), _t(ctx.k), _t(ctx.v)
    mask = torch.as_tensor(ctx.mask, device=DEV) > 0
    scales = [p.guidance.scale_text] if case["mode"] == "joint" else [p.guidance.scale_text, p.guidance.scale_speaker]
    n = case["steps"]
    ts = [float(np.float32(0.999) * (np.float32(1) - np.float32(i) / np.float32(n))) for i in range(n + 1)]
    for i in range(n):
        rows = U * (1 + len(scales)) if ts[i] >= p.guidance.min_t else U
        xin = x.repeat(rows // U, 1, 1)
        v = net(xin, torch.full((rows,), ts[i], device=DEV, dtype=F64), ck[:, :rows], cv[:, :rows], mask[:rows])
        v = v.view(rows // U, U, *v.shape[1:])
        step = v[0] + sum((v[0] - v[1 + j]) * scales[j] for j in range(rows // U - 1))
        x = x + step * (ts[i + 1] - ts[i])
    return x.cpu().numpy()


def _conv(x, w, b, dil=1):
    """Conv1d of [B, C, L] with zero padding (odd kernels), one matrix product per tap."""
    k, L = w.shape[2], x.shape[2]
    xp = F.pad(x, ((k - 1) * dil // 2,) * 2)
    y = sum(torch.matmul(w[:, :, j].contiguous(), xp[:, :, j * dil:j * dil + L].contiguous()) for j in range(k))
    return y + b[:, None]


def _conv_t(x, w, b, r):
    """ConvTranspose1d, kernel 2r, stride r, output length L * r: output i * r + tap - pad."""
    B, _, L = x.shape
    y = torch.zeros(B, w.shape[1], (L + 1) * r, device=DEV, dtype=F64)
    for tap in range(2 * r):
        part = torch.matmul(w[:, :, tap].t().contiguous(), x)
        first = tap // r
        y.view(B, -1, L + 1, r)[:, :, first:first + L, tap % r] += part
    pad = (r + 1) // 2
    return y[:, :, pad:pad + L * r] + b[:, None]


def _snake(x, alpha):
    a = _t(alpha)[:, None]
    return x + torch.sin(a * x).pow(2) / (a + 1e-9)


def _exact_codec(case, seed):
    cfg, w = _codec()
    outs = []
    for row in _inputs_codec(case, seed):
        x = row.double().t().contiguous()[None]
        x = _conv(x, _t(w.io["out_proj_w"]), _t(w.io["out_proj_b"]))
        x = _conv(x, _t(w.io["stem_w"]), _t(w.io["stem_b"]))
        for blk, r in zip(w.blocks, cfg.rates):
            x = _conv_t(_snake(x, blk["alpha"]), _t(blk["convt_w"]), _t(blk["convt_b"]), r)
            for u, d in enumerate((1, 3, 9)):
                y = _conv(_snake(x, blk["res_alpha0"][u]), _t(blk["res_conv_w"][u]), _t(blk["res_conv_b"][u]), d)
                x = x + _conv(_snake(y, blk["res_alpha1"][u]), _t(blk["res_pw_w"][u]), _t(blk["res_pw_b"][u]))
        outs.append(torch.tanh(_conv(_snake(x, w.io["head_alpha"]), _t(w.io["head_w"]), _t(w.io["head_b"]))))
    return torch.cat(outs)


_PREPARE = dict(rms_norm=_prepare_rms, adaln=_prepare_adaln, sdpa=_prepare_sdpa, joint_attention=_prepare_joint,
                swiglu_mlp=_prepare_mlp, fp8_linear=_prepare_fp8, encode=_prepare_encode,
                first_eval=_prepare_first_eval, sample=_prepare_sample, codec=_prepare_codec)
_RUN = dict(rms_norm=_run_rms, adaln=_run_adaln, sdpa=_run_sdpa, joint_attention=_run_joint, swiglu_mlp=_run_mlp,
            fp8_linear=_run_fp8, encode=_run_encode, first_eval=_run_first_eval, sample=_run_sample, codec=_run_codec)
_WORK = dict(rms_norm=_work_rms, adaln=_work_adaln, sdpa=_work_sdpa, joint_attention=_work_joint,
             swiglu_mlp=_work_mlp, fp8_linear=_work_fp8, encode=_work_encode, first_eval=_work_first_eval,
             sample=_work_sample, codec=_work_codec)
_EXACT = dict(rms_norm=_exact_rms, adaln=_exact_adaln, sdpa=_exact_sdpa, joint_attention=_exact_joint,
              swiglu_mlp=_exact_mlp, fp8_linear=_exact_fp8, encode=_exact_encode, first_eval=_exact_first_eval,
              sample=_exact_sample, codec=_exact_codec)
