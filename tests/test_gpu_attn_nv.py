"""The SDPA operator on row-major K / V (16-bit: kernels_attn_nv.hip, f32: kernels_attn.hip) against
the float64 oracle, at the edges of its tiles, key parities or halves, tile words and workgroup shapes.

Tolerance: the scores and sums are f32, so the error is the rounding of the probabilities to the
operand dtype, at most half a unit in the last place of each (2^-9 in bf16, 2^-12 in f16) on
terms of random sign: the relative L2 stays below twice that.  In f32 the scores, up to about
6 |mul| in log2 units, carry a rounding of 2^-24 from each of a few steps, which the exponential makes a
relative error of under 2^-19 |mul|, and the sums add about as much: 2^-17 max(1, |mul|)."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from irodori_hip import _lib as L
from irodori_hip.engine import ops

pytestmark = pytest.mark.gpu

TYPES = {"bf16": (L.DTYPE_BF16, torch.bfloat16, 2.0 ** -8), "f16": (L.DTYPE_F16, torch.float16, 2.0 ** -11),
         "f32": (L.DTYPE_F32, torch.float32, 2.0 ** -17)}
# B, H, Sq, Skv, Dh, mask, scale / Dh^-1/2.  Masks: None, "tail" (ragged rows), "holes" (whole
# tiles and single keys dropped), "none valid" in the last row.
CASES = [
    (1, 1, 1, 1, 64, None, 1.0), (1, 2, 33, 65, 64, None, 1.0), (2, 3, 64, 128, 64, "tail", 1.0),
    (3, 2, 65, 129, 64, "holes", 1.0), (1, 2, 40, 4100, 64, "holes", 1.0), (2, 2, 37, 200, 64, "empty", 1.0),
    (1, 1, 1, 1, 128, None, 1.0), (1, 2, 31, 64, 128, "tail", 1.0), (2, 3, 65, 193, 128, "holes", 1.0),
    (1, 2, 40, 4161, 128, "holes", 1.0), (2, 2, 37, 200, 128, "empty", 1.0),
    (2, 16, 641, 70, 128, "tail", 1.0),                               # four query blocks per workgroup
    (4, 32, 500, 70, 64, "tail", 1.0), (2, 2, 33, 32, 64, None, 1.0),  # 32 queries a wavefront; an empty key half (f32)
    (1, 2, 50, 150, 64, "tail", -3.0), (1, 2, 50, 150, 128, "tail", 0.0), (1, 2, 50, 150, 64, "holes", 40.0),
]


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("B,H,Sq,Skv,Dh,mask,mul", CASES)
def test_row_major_attention(oracle64, dtype, B, H, Sq, Skv, Dh, mask, mul):
    code, tdt, tol = TYPES[dtype]
    rng = np.random.default_rng(Sq * 7 + Skv)
    dq, dk, dv = (torch.from_numpy(rng.standard_normal((B, H, n, Dh)).astype(np.float32)).to("cuda").to(tdt)
                  for n in (Sq, Skv, Skv))
    m = np.ones((B, Skv), np.float32)
    if mask == "tail":
        for b in range(B):
            m[b, max(1, Skv - 1 - 67 * b):] = 0
    elif mask == "holes":
        m[:, 64:min(Skv, 4000):3] = 0
        m[0, 70:max(71, Skv - 66)] = 0
    elif mask == "empty":
        m[-1] = 0
    out = torch.full((B, H, Sq, Dh), 7.0, dtype=torch.float32, device="cuda")
    scale = mul * Dh ** -0.5
    dm = torch.from_numpy(m).to("cuda")
    ops.sdpa(code, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), 0 if mask is None else dm.data_ptr(), B, H, Sq, Skv,
             Dh, scale, out.data_ptr())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    want = oracle64.sdpa(*(a.float().cpu().numpy() for a in (dq, dk, dv)), m, scale)
    assert np.isfinite(got).all()
    if mask == "empty":
        assert not got[-1].any()
    err = rel_l2(got, want)
    print("%s %s: rel L2 %.2e" % (dtype, (B, H, Sq, Skv, Dh, mask, mul), err))
    assert err < (tol * max(1.0, abs(mul)) if dtype == "f32" else tol)


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("Sq,Skv,Dh", [(1, 1, 64), (33, 200, 64), (40, 4161, 64), (65, 193, 128)])
def test_operands_at_any_element_alignment(dtype, Sq, Skv, Dh):
    # The same operands and output one, two or four elements past a 16-byte boundary: the same bits.
    code, tdt, _ = TYPES[dtype]
    B, H = 2, 3
    rng = np.random.default_rng(Skv)
    arrs = [rng.standard_normal(B * H * n * Dh).astype(np.float32) for n in (Sq, Skv, Skv)]
    m = np.ones((B, Skv), np.float32)
    m[0, Skv // 2 + 1:] = 0
    dm = torch.from_numpy(m).to("cuda")
    got = []
    for off in (0, 1, 2, 4):
        bufs = [torch.from_numpy(np.concatenate([np.zeros(off, np.float32), a])).to("cuda").to(tdt) for a in arrs]
        out = torch.full((off + B * H * Sq * Dh + 1,), 7.0, dtype=torch.float32, device="cuda")
        ops.sdpa(code, *[b[off:].data_ptr() for b in bufs], dm.data_ptr(), B, H, Sq, Skv, Dh, Dh ** -0.5,
                 out[off:].data_ptr())
        torch.cuda.synchronize()
        out = out.cpu().numpy()
        assert (out[:off] == 7.0).all() and out[-1] == 7.0
        got.append(out[off:-1])
    assert np.isfinite(got[0]).all()
    for g in got[1:]:
        assert np.array_equal(g, got[0])


@pytest.mark.parametrize("Dh", [64, 128])
@pytest.mark.parametrize("Skv", [31, 70, 150])
def test_f32_rows_do_not_depend_on_the_launch_size(Dh, Skv):
    # Few heads take one query block per wavefront and two wavefronts per tile; many take two query
    # blocks, and with 64 dims both key halves in one wavefront: the same arithmetic, so the same bits.
    Sq, many = 130, 300
    rng = np.random.default_rng(Skv)
    q, k, v = (torch.from_numpy(rng.standard_normal((1, 1, n, Dh)).astype(np.float32)).to("cuda")
               for n in (Sq, Skv, Skv))
    m = torch.ones((1, Skv), device="cuda")
    m[0, 5:9] = 0
    got = []
    for H in (1, many):
        qq, kk, vv = (a.expand(1, H, -1, -1).contiguous() for a in (q, k, v))
        out = torch.full((1, H, Sq, Dh), 7.0, dtype=torch.float32, device="cuda")
        ops.sdpa(L.DTYPE_F32, qq.data_ptr(), kk.data_ptr(), vv.data_ptr(), m.data_ptr(), 1, H, Sq, Skv, Dh, Dh ** -0.5,
                 out.data_ptr())
        torch.cuda.synchronize()
        got.append(out.cpu().numpy()[0])
    assert np.isfinite(got[0]).all() and np.array_equal(got[1], np.repeat(got[0], many, 0))


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("Dh", [64, 128])
def test_scores_of_minus_infinity(oracle64, dtype, Dh):
    # A query whose first tiles hold only scores of -inf (k = -inf where q > 0) and whose other scores are
    # far below zero: its reference must come from the first finite score, or every p underflows.
    # Queries with q[0] = 0 would see 0 * inf, so the last one has q[0] < 0: scores of +inf, a NaN row.
    code, tdt, tol = TYPES[dtype]
    B, H, Sq, Skv = 1, 2, 35, 330
    rng = np.random.default_rng(Dh)
    q, k, v = (rng.standard_normal((B, H, n, Dh)).astype(np.float32) for n in (Sq, Skv, Skv))
    q[..., 0], q[..., 1] = 1.0, 16.0
    q[:, :, -1, 0] = -1.0
    k[:, :, :192, 0] = -np.inf
    k[:, :, 192:, 1] = -160.0
    dq, dk, dv = (torch.from_numpy(a).to("cuda").to(tdt) for a in (q, k, v))
    out = torch.full((B, H, Sq, Dh), 7.0, dtype=torch.float32, device="cuda")
    ops.sdpa(code, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), 0, B, H, Sq, Skv, Dh, Dh ** -0.5, out.data_ptr())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    # The keys at -inf take no part in a finite row: the oracle on the other ones.
    qq, kk, vv = (a.float().cpu().numpy() for a in (dq, dk, dv))
    want = oracle64.sdpa(qq, kk[:, :, 192:], vv[:, :, 192:], np.ones((B, Skv - 192), np.float32), Dh ** -0.5)
    assert np.isfinite(got[:, :, :-1]).all() and np.isnan(got[:, :, -1]).all()
    assert rel_l2(got[:, :, :-1], want[:, :, :-1]) < tol


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("Dh", [64, 128])
def test_nan_and_infinite_operands(dtype, Dh):
    # A masked key's NaN or infinite K row changes nothing; a valid key's makes every row it enters NaN
    # (an infinite V element only its column).  One query block's NaN row leaves the others alone.
    code, tdt, _ = TYPES[dtype]
    B, H, Sq, Skv = 1, 2, 40, 200
    rng = np.random.default_rng(Dh + 1)
    q, k, v = (torch.from_numpy(rng.standard_normal((B, H, n, Dh)).astype(np.float32)).to(tdt)
               for n in (Sq, Skv, Skv))
    m = torch.ones((B, Skv))
    m[0, 70:75] = 0

    def run(qq, kk, vv):
        dq, dk, dv, dm = (a.to("cuda") for a in (qq, kk, vv, m))
        out = torch.full((B, H, Sq, Dh), 7.0, dtype=torch.float32, device="cuda")
        ops.sdpa(code, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dm.data_ptr(), B, H, Sq, Skv, Dh, Dh ** -0.5,
                 out.data_ptr())
        torch.cuda.synchronize()
        return out.cpu().numpy()

    clean = run(q, k, v)
    assert np.isfinite(clean).all()
    bad = k.clone()
    bad[:, :, 71], bad[:, :, 72], bad[:, :, 73] = float("nan"), float("inf"), float("-inf")
    assert np.array_equal(run(q, bad, v), clean)
    for key in (3, 150):
        bad = k.clone()
        bad[:, 0, key, 5] = float("nan")
        got = run(q, bad, v)
        assert np.isnan(got[:, 0]).all() and np.array_equal(got[:, 1], clean[:, 1])
    bad = q.clone()
    bad[:, :, 7] = float("nan")
    got = run(bad, k, v)
    rest = np.arange(Sq) != 7
    assert np.isnan(got[:, :, 7]).all() and np.array_equal(got[:, :, rest], clean[:, :, rest])
    bad = v.clone()
    bad[:, :, 9, 11] = float("inf")
    got = run(q, k, bad)
    rest = np.arange(Dh) != 11
    assert (got[..., 11] == np.inf).all() and np.array_equal(got[..., rest], clean[..., rest])


def test_operands_above_four_gib_per_head():
    # 2^24 + 1 keys of 128 dims: a tile's byte window taken from all remaining keys wraps at 2^32.  One key
    # holds all the weight: key 5 of the first tile, whose window would end after key 0.
    Skv, Dh = 2 ** 24 + 1, 128
    q = torch.zeros((1, 1, 1, Dh), dtype=torch.bfloat16, device="cuda")
    k, v = (torch.zeros((1, 1, Skv, Dh), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    q[..., 0], k[0, 0, 5, 0], v[0, 0, 5] = 64.0, 64.0, 3.0
    out = torch.empty((1, 1, 1, Dh), dtype=torch.float32, device="cuda")
    ops.sdpa(L.DTYPE_BF16, q.data_ptr(), k.data_ptr(), v.data_ptr(), 0, 1, 1, 1, Skv, Dh, 1.0, out.data_ptr())
    torch.cuda.synchronize()
    assert (out == 3.0).all()
