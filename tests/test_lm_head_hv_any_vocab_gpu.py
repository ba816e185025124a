"""GPU: [H, V] weights whose vocabulary is not a multiple of 8, where every
weight row starts at another alignment, and f16 weights in that layout, against
the oracle.

The streaming kernel takes calls of up to 8 rows: on a vocabulary of 512 columns
for more than half of the CUs (V > 65,536 on 256 CUs; f16 up to two rows), where
the hidden size is not a multiple of 64 (H = 40, 72: passes of 8 rows whatever
the batch), and for operands of two types.  Its two-product body runs bf16
activations (H % 8 == 0), the plain one the rest.  The blocked GEMM takes the
other calls (H % 64 == 0; f32 activations at 65-128 rows: 64-row passes, then
streaming ones)."""
import numpy as np
import pytest
import torch

import nvjsel
from oracle import selection as sel
from tests.gpu_helpers import check_fused_sampled, check_greedy, engine_keys, keys_tensor

pytestmark = pytest.mark.gpu

VOCABS = [8, 9, 15, 257, 511, 514, 1023, 1027]


def _case(B, H, V, act, wdt, seed=0):
    rng = np.random.default_rng(B * 31 + H + V * 7 + seed)
    h = torch.from_numpy(rng.standard_normal((B, H)).astype(np.float32)).cuda().to(act)
    w = torch.from_numpy((rng.standard_normal((H, V)) * 0.3).astype(np.float32)).cuda().to(wdt)
    z = sel.lm_head_logits(h.float().cpu().numpy(), w.float().cpu().numpy().T)
    rc = 1 if act == wdt == torch.bfloat16 else 2 if act == wdt == torch.float16 else 0
    return rng, h, w, z, rc


@pytest.mark.parametrize("act,wdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16),
                                     (torch.float16, torch.float16), (torch.float32, torch.float16)])
@pytest.mark.parametrize("B,H", [(1, 40), (2, 64), (4, 72), (8, 64), (9, 64), (64, 128), (70, 64), (130, 64)])
@pytest.mark.parametrize("V", VOCABS)
def test_greedy_and_logits(V, B, H, act, wdt):
    _, h, w, z, rc = _case(B, H, V, act, wdt)
    ids = nvjsel.lm_head_greedy_top1_hip(h, w, weight_layout="hv")
    logits = nvjsel.lm_head_logits_hip(h, w, weight_layout="hv")
    torch.cuda.synchronize()
    check_greedy(ids.cpu().numpy(), z, rc, f"hv any V greedy {act} {wdt} B={B} H={H} V={V}")
    got = logits.float().cpu().numpy().astype(np.float64)
    hn = np.linalg.norm(h.float().cpu().numpy(), axis=1)[:, None]
    wn = np.linalg.norm(w.float().cpu().numpy(), axis=0)[None, :]
    ulp = {0: 2.0 ** -24, 1: 2.0 ** -8, 2: 2.0 ** -11}[rc]
    assert (np.abs(got - z) <= H * 2.0 ** -23 * hn * wn + np.abs(z) * ulp + 1e-7).all()


@pytest.mark.parametrize("act,wdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16),
                                     (torch.float16, torch.float16)])
@pytest.mark.parametrize("B,H,V", [(4, 768, 1001), (8, 64, 9), (20, 64, 1027), (64, 128, 515),
                                   (1, 72, 1027), (2, 72, 515), (3, 136, 1001), (8, 72, 1023), (11, 72, 257)])
def test_sample(B, H, V, act, wdt):
    rng, h, w, z, rc = _case(B, H, V, act, wdt, 1)
    T = [float(x) for x in rng.choice([0.0, 0.7, 1.0], B)]
    keys = engine_keys(B, 5)
    ids = nvjsel.lm_head_sample_token_ids(h, w, temperatures=torch.tensor(T).cuda(), rng_keys=keys_tensor(keys),
                                          weight_layout="hv")
    torch.cuda.synchronize()
    namb = check_fused_sampled(ids.cpu().numpy(), z, T, keys, rc, f"hv any V sample {act} {wdt} B={B} V={V}")
    assert namb <= max(2, B // 8)


@pytest.mark.parametrize("B,H", [(3, 64), (40, 64), (1, 72), (2, 72), (3, 72), (8, 72)])  # GEMM; streaming
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("part", [1, 2, 3, 4, 5, 6, 7])
def test_winner_in_the_last_partial_group(part, dt, B, H):
    """The last columns' last k-row: the load that would pass the weight's end,
    for every length of the last group."""
    V = 1024 + part
    h = torch.zeros(B, H, device="cuda", dtype=dt)
    h[:, H - 1] = 1.0
    for col in range(1024, V):
        w = torch.zeros(H, V, device="cuda", dtype=dt)
        w[H - 1] = -1.0
        w[H - 1, col] = 2.0
        ids, best = nvjsel.lm_head_greedy_top1_hip(h, w, weight_layout="hv", return_best=True)
        assert (ids.cpu().numpy() == col).all() and (best.cpu().numpy() == 2.0).all(), col


@pytest.mark.parametrize("act,wdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16),
                                     (torch.float16, torch.float16)])
@pytest.mark.parametrize("B", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("H,V", [(64, 70001), (128, 70008)])
def test_streaming_of_a_wide_vocabulary(H, V, B, act, wdt):
    """V > 65,536: up to 8 rows stream at H % 64 == 0 too (f16 up to two)."""
    rng, h, w, z, rc = _case(B, H, V, act, wdt, 3)
    ids, best = nvjsel.lm_head_greedy_top1_hip(h, w, weight_layout="hv", return_best=True)
    logits = nvjsel.lm_head_logits_hip(h, w, weight_layout="hv")
    T = [float(x) for x in rng.choice([0.0, 0.7, 1.0], B)]
    keys = engine_keys(B, 6)
    sids = nvjsel.lm_head_sample_token_ids(h, w, temperatures=torch.tensor(T).cuda(), rng_keys=keys_tensor(keys),
                                           weight_layout="hv")
    torch.cuda.synchronize()
    ctx = f"hv wide V {act} {wdt} B={B} H={H} V={V}"
    check_greedy(ids.cpu().numpy(), z, rc, ctx)
    assert check_fused_sampled(sids.cpu().numpy(), z, T, keys, rc, ctx) <= 2
    got = logits.float().cpu().numpy().astype(np.float64)
    hn = np.linalg.norm(h.float().cpu().numpy(), axis=1)[:, None]
    wn = np.linalg.norm(w.float().cpu().numpy(), axis=0)[None, :]
    ulp = {0: 2.0 ** -24, 1: 2.0 ** -8, 2: 2.0 ** -11}[rc]
    assert (np.abs(got - z) <= H * 2.0 ** -23 * hn * wn + np.abs(z) * ulp + 1e-7).all()
    np.testing.assert_array_equal(best.cpu().numpy(), logits.float().max(dim=1).values.cpu().numpy())


@pytest.mark.parametrize("act,wdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16),
                                     (torch.float16, torch.float16)])
@pytest.mark.parametrize("B,H,V", [(3, 72, 1024), (8, 72, 1027), (3, 64, 1024), (20, 64, 1027), (70, 64, 1024)])
def test_weight_at_an_odd_element(B, H, V, act, wdt):
    """A weight that starts 2, 6 or 14 bytes past a 16-byte boundary, rows whole
    vectors long or not, at the end of its allocation."""
    rng, h, w, z, rc = _case(B, H, V, act, wdt, 4)
    T = [float(x) for x in rng.choice([0.0, 0.7, 1.0], B)]
    keys = engine_keys(B, 8)
    for off in (1, 3, 7):
        flat = torch.empty(off + H * V, device="cuda", dtype=wdt)
        flat[off:] = w.reshape(-1)
        wo = flat[off:].view(H, V)
        ids = nvjsel.lm_head_greedy_top1_hip(h, wo, weight_layout="hv")
        sids = nvjsel.lm_head_sample_token_ids(h, wo, temperatures=torch.tensor(T).cuda(), rng_keys=keys_tensor(keys),
                                               weight_layout="hv")
        torch.cuda.synchronize()
        ctx = f"hv base +{off} {act} {wdt} B={B} H={H} V={V}"
        check_greedy(ids.cpu().numpy(), z, rc, ctx)
        assert check_fused_sampled(sids.cpu().numpy(), z, T, keys, rc, ctx) <= max(2, B // 8)


@pytest.mark.parametrize("B", [65, 66, 72, 73, 128])
@pytest.mark.parametrize("V", [136, 129])
def test_f32_rows_past_the_streaming_kernels_lds(V, B):
    """H = 5120: eight streaming rows do not fit the LDS, so 65-128 f32 rows
    have no streaming pass to end on and one GEMM pass takes them all."""
    H = 5120
    _, h, w, z, rc = _case(B, H, V, torch.float32, torch.bfloat16, 2)
    ids = nvjsel.lm_head_greedy_top1_hip(h, w, weight_layout="hv")
    logits = nvjsel.lm_head_logits_hip(h, w, weight_layout="hv")
    torch.cuda.synchronize()
    check_greedy(ids.cpu().numpy(), z, rc, f"hv f32 B={B} H={H} V={V}")
    # fp32 sums of three products per element: 3 H 2^-24 sum |h w| at most, sum |h w| <= |h| |w|
    hn = np.linalg.norm(h.float().cpu().numpy(), axis=1)[:, None]
    wn = np.linalg.norm(w.float().cpu().numpy(), axis=0)[None, :]
    assert (np.abs(logits.cpu().numpy().astype(np.float64) - z) <= 3 * H * 2.0 ** -24 * hn * wn).all()
