"""The block's hot kernels in isolation (irodori_op_joint_attention / irodori_op_swiglu_mlp)
at the isolated-kernel configurations, through the C ABI, against oracle compositions of
the pinned operators (head RMSNorm, half RoPE, SDPA with the joint key mask, adaLN,
SwiGLU) in float64.

- Joint attention, B = 2 x 16 heads x 64, 750 latent queries; keys = 750 latent (RoPE'd
  and head-normed with the layer's weights) + 256 text (valid length U[32, 256] per row) +
  375 speaker, Q/K/V ~ N(0, 1), sigmoid output gate (attention.rs:328-425).
- SwiGLU MLP half of a block, 1500 tokens (B = 2 x 750) x 1024 -> 2816 -> 1024, weights
  N(0, 0.02), activations N(0, 1), shift / scale / gate per batch row ~ N(0, 0.1), RMSNorm
  eps 1e-6 (diffusion.rs:101-104).
Bars: f32 1e-4 relative L2; bf16 1e-2 (the MLP's increment on its own 2e-2).
"""
import dataclasses

import numpy as np
import pytest
import torch

import irodori_hip as ih
from conftest import rel_l2

pytestmark = pytest.mark.gpu

BF16, F32 = ih.InferenceBackendKind.HIP_BF16, ih.InferenceBackendKind.HIP_F32
TOL = {BF16: 1e-2, F32: 1e-4}


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda")


def one_layer(eps=1e-5):
    return dataclasses.replace(ih.cfg_full_rf(), num_layers=1, norm_eps=eps)


def joint_attention_ref(orc, cfg, blk, q, k, v, gate, ck, cv, cmask):
    """attention.rs:328-425 composed from the oracle's pinned operators."""
    B, S, H, Dh = q.shape
    qn = orc.head_rms_norm(q, blk["q_norm"], cfg.norm_eps)
    kn = orc.head_rms_norm(k, blk["k_norm"], cfg.norm_eps)
    cs, sn = orc.rope_tables(S, Dh, cfg.rope_theta)
    qr, kr = orc.rope_half(qn, cs, sn), orc.rope_half(kn, cs, sn)
    K = np.concatenate([kr, ck], axis=1).transpose(0, 2, 1, 3)
    V = np.concatenate([v, cv], axis=1).transpose(0, 2, 1, 3)
    mask = np.concatenate([np.ones((B, S), np.float32), cmask.astype(np.float32)], axis=1)
    o = orc.sdpa(qr.transpose(0, 2, 1, 3), K, V, mask, Dh ** -0.5).transpose(0, 2, 1, 3)
    g = 1.0 / (1.0 + np.exp(-gate.astype(np.float64)))
    return (o.reshape(B, S, H * Dh) * g).astype(np.float64)


@pytest.mark.parametrize("backend", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("roles", [["cond"], ["cond", "uncond"]], ids=["two-utterances", "cond+uncond"])
def test_joint_attention_op_config2(oracle64, backend, roles):
    cfg = one_layer()
    w = ih.DitWeights.random(cfg, 7, norm_jitter=0.1)
    U = 2 if roles == ["cond"] else 1
    ctx = ih.make_role_context(cfg, U, 256, 375, roles, seed=8)  # 2 rows either way
    B, S, H, Dh = 2, 750, cfg.num_heads, cfg.head_dim
    rng = np.random.default_rng(9)
    q, k, v = (rng.standard_normal((B, S, H, Dh)).astype(np.float32) for _ in range(3))
    gate = rng.standard_normal((B, S, H * Dh)).astype(np.float32)
    out = torch.empty((B, S, H * Dh), dtype=torch.float32, device="cuda")
    with ih.HipInferenceEngine(cfg, backend, max_rows=B, max_seq=S, max_ctx=ctx.t_ctx) as e:
        e.load_weights(w)
        e.set_context_kv(ctx)
        dq, dk, dv, dg = dev(q), dev(k), dev(v), dev(gate)
        e.joint_attention(0, B, S, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dg.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        # No gate: sigmoid(gate) replaced by 1.
        e.joint_attention(0, B, S, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), 0, out.data_ptr())
        torch.cuda.synchronize()
        got_ng = out.cpu().numpy()
    ref = joint_attention_ref(oracle64, cfg, w.blocks[0], q, k, v, gate, ctx.k[0], ctx.v[0], ctx.mask)
    ref_ng = joint_attention_ref(oracle64, cfg, w.blocks[0], q, k, v, np.full_like(gate, 60.0), ctx.k[0],
                                 ctx.v[0], ctx.mask)
    err, err_ng = rel_l2(got, ref), rel_l2(got_ng, ref_ng)
    print(backend.value, roles, "joint attention op rel L2 %.2e / ungated %.2e" % (err, err_ng))
    assert err < TOL[backend] and err_ng < TOL[backend]


def test_joint_attention_op_rejects_missing_context():
    cfg = one_layer()
    with ih.HipInferenceEngine(cfg, BF16, max_rows=2, max_seq=64, max_ctx=16) as e:
        e.load_weights(ih.DitWeights.random(cfg, 1))
        ctx = ih.make_context_kv(cfg, 1, 8, 8, seed=2)
        e.set_context_kv(ih.ContextKV(ctx.k[:, :1], ctx.v[:, :1], ctx.mask[:1]))  # row 0 only
        z = torch.zeros((2, 64, cfg.model_dim), device="cuda")
        with pytest.raises(ih.IrodoriError) as ei:
            e.joint_attention(0, 2, 64, z.data_ptr(), z.data_ptr(), z.data_ptr(), 0, z.data_ptr())
        assert ei.value.kind == "NotLoaded"


@pytest.mark.parametrize("backend", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("B", [2, 1])
def test_swiglu_mlp_op_config3(oracle64, backend, B):
    cfg = one_layer(eps=1e-6)
    w = ih.DitWeights.random(cfg, 3)
    S, D = 750, cfg.model_dim
    rng = np.random.default_rng(4)
    x = rng.standard_normal((B, S, D)).astype(np.float32)
    shift, scale, gate = ((0.1 * rng.standard_normal((B, D))).astype(np.float32) for _ in range(3))
    # Keep every device tensor referenced until the call completes (a temporary's block
    # would go back to torch's cache and be handed to the next allocation).
    dx, dsh, dsc, dg = dev(x), dev(shift), dev(scale), dev(gate)
    with ih.HipInferenceEngine(cfg, backend, max_rows=B, max_seq=S, max_ctx=1) as e:
        e.load_weights(w)
        e.swiglu_mlp(0, B, S, dx.data_ptr(), dsh.data_ptr(), dsc.data_ptr(), dg.data_ptr())
        torch.cuda.synchronize()
    got = dx.cpu().numpy()
    h = oracle64.fused_adaln(x.reshape(B * S, D), scale, shift, B, S, 1e-6)
    m = oracle64.swiglu(h, w.blocks[0]["w13"], w.blocks[0]["w2"]).reshape(B, S, D).astype(np.float64)
    ref = x + gate[:, None, :].astype(np.float64) * m
    err, inc = rel_l2(got, ref), rel_l2(got - x, ref - x)
    print(backend.value, "B=%d swiglu mlp op rel L2 %.2e, increment %.2e" % (B, err, inc))
    assert err < TOL[backend] and inc < 2 * TOL[backend]


@pytest.mark.parametrize("backend", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("S", [1, 31, 33, 64, 97])
def test_joint_attention_op_ragged(oracle64, backend, S):
    # Lengths around the staging kernel's 32-token blocks and the 64-key tiles; the operands
    # at an odd float, the least alignment that the entry point's types promise; no gate, too.
    cfg = one_layer()
    w = ih.DitWeights.random(cfg, 7, norm_jitter=0.1)
    B, H, Dh = 3, cfg.num_heads, cfg.head_dim
    ctx = ih.make_role_context(cfg, B, 40, 30, ["cond"], seed=8)
    rng = np.random.default_rng(S)
    ops = [rng.standard_normal((B, S, H, Dh)).astype(np.float32) for _ in range(3)]
    ops.append(rng.standard_normal((B, S, H * Dh)).astype(np.float32))
    n = B * S * H * Dh
    bufs = [dev(np.concatenate([np.zeros(1, np.float32), a.ravel()])) for a in ops]
    out = torch.full((n + 2,), 7.0, dtype=torch.float32, device="cuda")
    ptrs = [b.data_ptr() + 4 for b in bufs]
    with ih.HipInferenceEngine(cfg, backend, max_rows=B, max_seq=S, max_ctx=ctx.t_ctx) as e:
        e.load_weights(w)
        e.set_context_kv(ctx)
        for gate in (True, False):
            e.joint_attention(0, B, S, *ptrs[:3], ptrs[3] if gate else 0, out.data_ptr() + 4)
            torch.cuda.synchronize()
            g = ops[3] if gate else np.full_like(ops[3], 60.0)
            ref = joint_attention_ref(oracle64, cfg, w.blocks[0], *ops[:3], g, ctx.k[0], ctx.v[0], ctx.mask)
            o = out.cpu().numpy()
            assert o[0] == 7.0 and o[-1] == 7.0
            assert rel_l2(o[1:-1].reshape(ref.shape), ref) < TOL[backend]


@pytest.mark.parametrize("backend", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("B,S", [(3, 1), (3, 31), (2, 33), (3, 130)])
def test_swiglu_mlp_op_rows_on_their_own_vectors(oracle64, backend, B, S):
    # Rows shorter than, and not a multiple of, a GEMM tile's row block, so that one block of
    # the residual epilogue spans two or three rows' gates; vectors at an odd float.
    cfg = one_layer(eps=1e-6)
    w = ih.DitWeights.random(cfg, 3)
    D = cfg.model_dim
    rng = np.random.default_rng(5)
    x = rng.standard_normal((B, S, D)).astype(np.float32)
    vec = [rng.standard_normal((B, D)).astype(np.float32) for _ in range(3)]
    dx = dev(x)
    bufs = [dev(np.concatenate([np.zeros(1, np.float32), a.ravel()])) for a in vec]
    with ih.HipInferenceEngine(cfg, backend, max_rows=B, max_seq=S, max_ctx=1) as e:
        e.load_weights(w)
        e.swiglu_mlp(0, B, S, dx.data_ptr(), *[b.data_ptr() + 4 for b in bufs])
        torch.cuda.synchronize()
    got = dx.cpu().numpy()
    shift, scale, gate = vec
    h = oracle64.fused_adaln(x.reshape(B * S, D), scale, shift, B, S, 1e-6)
    m = oracle64.swiglu(h, w.blocks[0]["w13"], w.blocks[0]["w2"]).reshape(B, S, D).astype(np.float64)
    ref = x + gate[:, None, :].astype(np.float64) * m
    assert rel_l2(got, ref) < TOL[backend] and rel_l2(got - x, ref - x) < 2 * TOL[backend]


@pytest.mark.parametrize("backend", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("T", [4097, 4796, 16200])
def test_joint_attention_op_key_tiles_beyond_one_list_word(oracle64, backend, T):
    # More than 64 context key tiles: the bf16 kernel's tile list spans several words per lane.  Row 0
    # drops whole tiles from the first word (and, when present, later ones) so that later entries shift
    # down; row 1 has a partial mask in every tile.
    cfg = dataclasses.replace(ih.cfg_tiny(), num_layers=1)
    w = ih.DitWeights.random(cfg, 7, norm_jitter=0.1)
    B, S, H, Dh = 2, 70, cfg.num_heads, cfg.head_dim
    rng = np.random.default_rng(T)
    ctx = ih.ContextKV(*(rng.standard_normal((1, B, T, H, Dh)).astype(np.float32) for _ in range(2)),
                       np.ones((B, T), np.uint8))
    ctx.mask[0, 640:1600] = 0
    ctx.mask[0, 4160:4300] = 0
    ctx.mask[0, 9000:9999] = 0
    ctx.mask[1, ::7] = 0
    ops = [rng.standard_normal((B, S, H, Dh)).astype(np.float32) for _ in range(3)]
    ops.append(rng.standard_normal((B, S, H * Dh)).astype(np.float32))
    bufs = [dev(a) for a in ops]
    out = torch.full((B, S, H * Dh), 7.0, dtype=torch.float32, device="cuda")
    with ih.HipInferenceEngine(cfg, backend, max_rows=B, max_seq=S, max_ctx=T) as e:
        e.load_weights(w)
        e.set_context_kv(ctx)
        e.joint_attention(0, B, S, *(b.data_ptr() for b in bufs), out.data_ptr())
        torch.cuda.synchronize()
    ref = joint_attention_ref(oracle64, cfg, w.blocks[0], *ops, ctx.k[0], ctx.v[0], ctx.mask)
    assert rel_l2(out.cpu().numpy(), ref) < TOL[backend]
