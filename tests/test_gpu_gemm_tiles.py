"""The block GEMMs' tile shapes: a row's result must not depend on how many rows it is launched
with, which is what picks the tile (64x64, 64x128, 128x64, 32x64, 128x128 or 192x128).  Every output is
the same MFMA sequence over k in each shape, so the comparison is exact; the 128x128 and 64x64
results themselves are held to the oracle elsewhere."""
import numpy as np
import pytest

import irodori_hip as ih

pytestmark = pytest.mark.gpu

KIND = {"bf16": ih.InferenceBackendKind.HIP_BF16, "f32": ih.InferenceBackendKind.HIP_F32,
        "fp8": ih.InferenceBackendKind.HIP_FP8}


@pytest.mark.parametrize("backend", ["bf16", "f32", "fp8"])
def test_rows_do_not_depend_on_the_launch_size(backend):
    # d1024, F 2816: 37-frame rows, odd so that tiles start inside a row.  Rows per launch 2, 5,
    # 8, 11 and 22 are 74, 185, 296, 407 and 814 tokens: 64x64 tiles for every projection, then
    # one after another the 64x128, 128x64 and 128x128 ones and the 32x64 -> 64x64 step; 45 are
    # 1665 and 62 2294, the 192x128 tiles of W1|W3 (in f32 at 1665, 128x128 at 2294) and the
    # eight-wavefront 128x128 ones of the residuals.
    cfg = ih.cfg_full_rf()
    cfg.num_layers = 1
    S, T, R = 37, 20, 62
    w = ih.DitWeights.random(cfg, seed=3, norm_jitter=0.1)
    one = ih.make_role_context(cfg, 1, 12, 8, ["cond"], seed=4)
    ctx = ih.ContextKV(*(np.repeat(a, R, axis) for a, axis in ((one.k, 1), (one.v, 1), (one.mask, 0))))
    x = np.repeat(ih.make_noise(1, S, cfg.latent_dim, 5), R, 0)
    with ih.HipInferenceEngine(cfg, KIND[backend], max_rows=R, max_seq=S, max_ctx=T) as e:
        e.load_weights(w)
        e.set_context_kv(ctx)
        want = None
        for rows in (2, 5, 8, 11, 22, 45, 62):
            v, dbg = e.forward_with_cond_cached(x[:rows], np.full(rows, 0.4, np.float32), debug=True)
            want = dbg[:, 0] if want is None else want
            assert np.isfinite(dbg).all()
            for r in range(rows):
                assert np.array_equal(dbg[:, r], want), (rows, r)
            assert np.array_equal(v, np.repeat(v[:1], rows, 0))


@pytest.mark.parametrize("backend", ["bf16", "f32"])
def test_encoder_rows_do_not_depend_on_the_launch_size(backend):
    # E 512: 35-token rows, the first a copy in every batch.  70, 700, 1400, 2800 and 4550 tokens:
    # QKV+gate in 64x64, 64x128 and 128x128 tiles, the residual projections in 32x64, 64x64, 128x64
    # and 128x128.
    ecfg = ih.EncoderConfig(dim=512, num_layers=1, num_heads=8, mlp_hidden=192, vocab_size=50)
    S, R = 35, 130
    ids = np.tile(np.random.default_rng(1).integers(0, 50, (1, S)).astype(np.int32), (R, 1))
    mask = np.ones((R, S), bool)
    mask[:, 30:] = False
    with ih.HipEncoder(ecfg, KIND[backend], max_rows=R, max_seq=S) as enc:
        enc.load_weights(ih.EncoderWeights.random(ecfg, 2))
        want = None
        for rows in (2, 20, 40, 80, 130):
            out = enc.forward(mask[:rows], ids=ids[:rows])
            out = np.asarray(out[0] if isinstance(out, tuple) else out)
            want = out[0] if want is None else want
            assert np.isfinite(out).all()
            for r in range(rows):
                assert np.array_equal(out[r], want), (rows, r)
