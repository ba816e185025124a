"""GPU: the staged LM-head GEMM on direct LDS loads (csrc/lm_head_ring.hip)
at the edges of its tiles, against the oracle: batch rows around each row
count it is built for, one to several K stages (H = 64 has one, 192 three:
fewer and more than the ring's slots), vocabularies of one partial tile, of
more blocks than rows, and of two tiles per block with a remainder
(V > 256 x 256), bf16, f16, and f32 activations on bf16 weights (three
terms per value, 64 rows per pass)."""
import numpy as np
import pytest
import torch

import nvjsel
from nvjsel import _lib
from oracle import selection as sel
from tests.gpu_helpers import check_fused_sampled, check_greedy, engine_keys, keys_tensor

pytestmark = pytest.mark.gpu

SHAPES = [(3, 64, 5), (31, 192, 257), (33, 64, 66000), (64, 320, 2055), (65, 128, 66000), (128, 192, 4099),
          (129, 64, 70001), (256, 192, 1000), (257, 64, 300), (18, 2048, 300)]


def _inputs(B, H, V, dt, seed=0):
    rng = np.random.default_rng(B * 1009 + H + V + seed)
    h = torch.from_numpy(rng.standard_normal((B, H)).astype(np.float32)).cuda().to(dt)
    w = torch.from_numpy((rng.standard_normal((V, H)) * 0.3).astype(np.float32)).cuda()
    w = w.to(torch.bfloat16 if dt == torch.float32 else dt)
    z = sel.lm_head_logits(h.float().cpu().numpy(), w.float().cpu().numpy())
    return rng, h, w, z, {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dt]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,H,V", SHAPES)
def test_greedy_and_logits(B, H, V, dt):
    _, h, w, z, rc = _inputs(B, H, V, dt)
    ids, best = nvjsel.lm_head_greedy_top1_hip(h, w, weight_layout="vh", return_best=True)
    logits = nvjsel.lm_head_logits_hip(h, w, weight_layout="vh")
    torch.cuda.synchronize()
    check_greedy(ids.cpu().numpy(), z, rc, f"ring greedy {dt} {B} {H} {V}")
    got = logits.float().cpu().numpy().astype(np.float64)
    # fp32 sums of H products (H 2^-24 sum |h w| <= H 2^-24 |h| |w|) and one
    # rounding to the 16-bit type (within an ulp: 2^-8 bf16, 2^-11 f16, f32 as summed)
    hn = np.linalg.norm(h.float().cpu().numpy(), axis=1)[:, None]
    wn = np.linalg.norm(w.float().cpu().numpy(), axis=1)[None, :]
    tol = H * 2.0 ** -24 * hn * wn * 2 + np.abs(z) * {0: 2.0 ** -24, 1: 2.0 ** -8, 2: 2.0 ** -11}[rc] + 1e-7
    assert (np.abs(got - z) <= tol).all()
    # the winning logit is the row's largest stored logit, at its first index
    np.testing.assert_array_equal(best.cpu().numpy(), logits.float().max(dim=1).values.cpu().numpy())
    np.testing.assert_array_equal(ids.cpu().numpy().reshape(-1), got.argmax(axis=1))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V,stride,base", [(516, 516, 0), (516, 520, 4), (516, 517, 0), (516, 518, 0), (516, 516, 1),
                                           (516, 516, 2), (514, 516, 0), (515, 515, 0), (2052, 2053, 3)])
def test_logits_row_stride_and_base(V, stride, base, dt):
    """16-bit logits leave 8 bytes per lane only where every row's quads allow
    it; other strides and bases store the same values, and nothing is written
    between the rows.  base: elements past a 256-byte boundary."""
    B, H = 45, 64
    _, h, w, z, rc = _inputs(B, H, V, dt, 2)
    code = _lib.BF16 if dt == torch.bfloat16 else _lib.F16
    buf = torch.full((base + B * stride + 8,), -777.0, device="cuda", dtype=dt)
    _lib.call("nvjsel_lm_head_logits", h.data_ptr(), code, w.data_ptr(), code, _lib.W_VH, B, H, V, rc,
              buf.data_ptr() + 2 * base, code, stride, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    rows = buf[base:base + B * stride].view(B, stride)
    assert bool((buf[:base] == -777.0).all()) and bool((buf[base + B * stride:] == -777.0).all())
    assert bool((rows[:, V:] == -777.0).all())
    torch.testing.assert_close(rows[:, :V], nvjsel.lm_head_logits_hip(h, w, weight_layout="vh"), rtol=0, atol=0)
    hn = np.linalg.norm(h.float().cpu().numpy(), axis=1)[:, None]
    wn = np.linalg.norm(w.float().cpu().numpy(), axis=1)[None, :]
    tol = H * 2.0 ** -23 * hn * wn + np.abs(z) * {1: 2.0 ** -8, 2: 2.0 ** -11}[rc] + 1e-7  # as above
    assert (np.abs(rows[:, :V].float().cpu().numpy().astype(np.float64) - z) <= tol).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,H,V", [s for s in SHAPES if s[0] <= 128 or s[0] == 257])
def test_sample(B, H, V, dt):
    rng, h, w, z, rc = _inputs(B, H, V, dt, 1)
    T = [float(x) for x in rng.choice([0.0, 0.3, 0.7, 1.0, 1.7], B)]
    keys = engine_keys(B, 7)
    ids = nvjsel.lm_head_sample_token_ids(h, w, temperatures=torch.tensor(T).cuda(), rng_keys=keys_tensor(keys),
                                          weight_layout="vh")
    torch.cuda.synchronize()
    namb = check_fused_sampled(ids.cpu().numpy(), z, T, keys, rc, f"ring sample {dt} {B} {H} {V}")
    assert namb <= max(2, B // 8)


@pytest.mark.parametrize("reduce_cast", [0, 1])
def test_ties_nan_and_infinities(reduce_cast):
    """First index among equal rounded logits, first NaN, +inf and all -inf
    rows; the unrounded comparison too."""
    B, H, V = 40, 64, 66000
    rng = np.random.default_rng(5)
    h = np.zeros((B, H), np.float32)
    h[:, 0] = 1.0
    w = np.zeros((V, H), np.float32)
    w[:, 0] = rng.integers(-40, 40, V) / 8.0  # many exact ties
    w[300, 0], w[65999, 0] = 7.0, 7.0
    big = 3.0e38
    h[1, 1] = h[1, 2] = big  # row 1: inf - inf = NaN at 777 and 65900, +inf at 5
    w[[777, 65900], 1], w[[777, 65900], 2] = big, -big
    w[5, 1] = big
    h[2] = 0.0
    h[2, 3] = big  # row 2: -inf everywhere
    w[:, 3] = -big
    hb = torch.from_numpy(h).cuda().to(torch.bfloat16)
    wb = torch.from_numpy(w).cuda().to(torch.bfloat16)
    ids = nvjsel.lm_head_greedy_top1_hip(hb, wb, weight_layout="vh", reduce_cast=reduce_cast).cpu().numpy().reshape(-1)
    assert ids[0] == 300 and (ids[3:] == 300).all()
    assert ids[2] == 0
    assert ids[1] == 777


@pytest.mark.parametrize("B,H,V,layout", [
    (20, 2048, 300, "vh"), (33, 64, 66000, "vh"), (64, 192, 257, "vh"),  # three terms in the staged GEMM
    (200, 64, 515, "vh"),                                                # ... in the blocked GEMM
    (20, 64, 1027, "hv"), (70, 128, 515, "hv"), (130, 64, 1027, "hv"), (200, 64, 520, "hv")])
def test_f32_activations_keep_infinities(B, H, V, layout):
    """f32 activations on bf16 weights give the logits of fp32 products where
    an operand is infinite, a finite value rounds to bf16's infinity, or an
    infinite weight meets a value whose lower terms are zero."""
    rng = np.random.default_rng(B + H + V)
    h = rng.standard_normal((B, H)).astype(np.float32)
    w = (rng.standard_normal((V, H)) * 0.3).astype(np.float32)
    h[0, 1] = np.inf
    w[::7, 1] = 0.0  # inf * 0
    h[1, 2] = -np.inf
    h[2, 3] = 3.4e38
    w[:, 3] *= 1e-3
    h[3, 4], h[4, 4], h[5, 4], h[6, 4] = 1.0, 1.1, -0.7, 0.0
    w[5, 4], w[9, 4] = np.inf, -np.inf
    h[7, 5] = np.nan
    wb = torch.from_numpy(w).cuda().to(torch.bfloat16)
    hb = torch.from_numpy(h).cuda()
    wo = wb if layout == "vh" else wb.T.contiguous()
    h64, w64 = h.astype(np.float64), wb.float().cpu().numpy().astype(np.float64)
    with np.errstate(invalid="ignore"):
        z = h64 @ w64.T
        A = np.abs(h64) @ np.abs(w64).T
    got = nvjsel.lm_head_logits_hip(hb, wo, weight_layout=layout).cpu().numpy().astype(np.float64)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(z))
    fin = np.isfinite(z)
    np.testing.assert_array_equal(got[~fin], z[~fin])
    # fp32 sums of three products per element: 3 H 2^-24 sum |h w| at most
    assert (np.abs(got[fin] - z[fin]) <= 3 * H * 2.0 ** -24 * A[fin]).all()
    exp = np.where(np.isnan(z).any(axis=1), np.isnan(z).argmax(axis=1), np.nan_to_num(z, nan=0.0).argmax(axis=1))
    ids, best = nvjsel.lm_head_greedy_top1_hip(hb, wo, weight_layout=layout, return_best=True)
    np.testing.assert_array_equal(ids.cpu().numpy().reshape(-1), exp)  # (every row's best is not finite)
    np.testing.assert_array_equal(best.cpu().numpy().astype(np.float64), z[np.arange(B), exp])
    T = torch.tensor([float(b % 2) for b in range(B)]).cuda()
    ids = nvjsel.lm_head_sample_token_ids(hb, wo, temperatures=T, rng_keys=keys_tensor(engine_keys(B, 3)),
                                          weight_layout=layout)
    np.testing.assert_array_equal(ids.cpu().numpy(), exp)  # an infinity or a NaN wins whatever the draw


@pytest.mark.parametrize("B,H,layout", [(80, 64, "vh"), (40, 1024, "vh"), (20, 64, "hv"), (140, 64, "vh")])
def test_sample_extreme_temperatures_and_nan(B, H, layout):
    """Tiny and huge temperatures (products with 1 / T' out of the float range
    are divided instead), a NaN temperature and a NaN logit row, in every
    kernel that scores with the product."""
    V = 3001
    rng = np.random.default_rng(9)
    h = rng.standard_normal((B, H)).astype(np.float32)
    w = (rng.standard_normal((V, H)) * 0.3).astype(np.float32)
    hb = torch.from_numpy(h).cuda().to(torch.bfloat16)
    wb = torch.from_numpy(w).cuda().to(torch.bfloat16)
    wo = wb if layout == "vh" else wb.T.contiguous()
    T = [float(x) for x in rng.choice([1e-7, 1e-3, 0.5, 50.0, 1e30], B)]
    keys = engine_keys(B, 3)
    ids = nvjsel.lm_head_sample_token_ids(hb, wo, temperatures=torch.tensor(T).cuda(), rng_keys=keys_tensor(keys),
                                          weight_layout=layout).cpu().numpy()
    z = sel.lm_head_logits(hb.float().cpu().numpy(), wb.float().cpu().numpy())
    check_fused_sampled(ids, z, T, keys, 1, "ring sample extreme T")
    hb[4, 0] = float("nan")
    T[9] = float("nan")
    ids = nvjsel.lm_head_sample_token_ids(hb, wo, temperatures=torch.tensor(T).cuda(), rng_keys=keys_tensor(keys),
                                          weight_layout=layout).cpu().numpy()
    assert ids[4] == 0 and ids[9] == 0  # every score a NaN: the first
    ok = [b for b in range(B) if b not in (4, 9)]
    check_fused_sampled(ids[ok], z[ok], [T[b] for b in ok], keys[ok], 1, "ring sample beside NaN rows")
