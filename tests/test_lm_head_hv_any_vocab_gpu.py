"""GPU: [H, V] weights whose vocabulary is not a multiple of 8, where every
weight row starts at another alignment, and f16 weights in that layout, through
the streaming kernel (up to 8 rows) and the blocked GEMM (from 9 rows; f32
activations at 65-128 rows mix the two), against the oracle."""
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
@pytest.mark.parametrize("B,H,V", [(4, 768, 1001), (8, 64, 9), (20, 64, 1027), (64, 128, 515)])
def test_sample(B, H, V, act, wdt):
    rng, h, w, z, rc = _case(B, H, V, act, wdt, 1)
    T = [float(x) for x in rng.choice([0.0, 0.7, 1.0], B)]
    keys = engine_keys(B, 5)
    ids = nvjsel.lm_head_sample_token_ids(h, w, temperatures=torch.tensor(T).cuda(), rng_keys=keys_tensor(keys),
                                          weight_layout="hv")
    torch.cuda.synchronize()
    namb = check_fused_sampled(ids.cpu().numpy(), z, T, keys, rc, f"hv any V sample {act} {wdt} B={B} V={V}")
    assert namb <= max(2, B // 8)


@pytest.mark.parametrize("B", [3, 40])
@pytest.mark.parametrize("col", [1024, 1025, 1026])
def test_winner_in_the_last_partial_group(B, col):
    """The last columns' last k-row: the load that would pass the weight's end."""
    H, V = 64, 1027
    h = torch.zeros(B, H, device="cuda", dtype=torch.bfloat16)
    h[:, H - 1] = 1.0
    w = torch.zeros(H, V, device="cuda", dtype=torch.bfloat16)
    w[H - 1] = -1.0
    w[H - 1, col] = 2.0
    ids, best = nvjsel.lm_head_greedy_top1_hip(h, w, weight_layout="hv", return_best=True)
    assert (ids.cpu().numpy() == col).all() and (best.cpu().numpy() == 2.0).all()


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
