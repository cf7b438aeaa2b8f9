"""The block GEMMs' tile shapes: a row's result must not depend on how many rows it is launched
with, which is what picks the tile (64x64, 64x128, 128x64, 32x64 or 128x128).  Every output is
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
    # one after another the 64x128, 128x64 and 128x128 ones and the 32x64 -> 64x64 step.
    cfg = ih.cfg_full_rf()
    cfg.num_layers = 1
    S, T, R = 37, 20, 22
    w = ih.DitWeights.random(cfg, seed=3, norm_jitter=0.1)
    one = ih.make_role_context(cfg, 1, 12, 8, ["cond"], seed=4)
    ctx = ih.ContextKV(*(np.repeat(a, R, axis) for a, axis in ((one.k, 1), (one.v, 1), (one.mask, 0))))
    x = np.repeat(ih.make_noise(1, S, cfg.latent_dim, 5), R, 0)
    with ih.HipInferenceEngine(cfg, KIND[backend], max_rows=R, max_seq=S, max_ctx=T) as e:
        e.load_weights(w)
        e.set_context_kv(ctx)
        want = None
        for rows in (2, 5, 8, 11, 22):
            v, dbg = e.forward_with_cond_cached(x[:rows], np.full(rows, 0.4, np.float32), debug=True)
            want = dbg[:, 0] if want is None else want
            assert np.isfinite(dbg).all()
            for r in range(rows):
                assert np.array_equal(dbg[:, r], want), (rows, r)
            assert np.array_equal(v, np.repeat(v[:1], rows, 0))
