"""GPU: every LM-head route at the batch sizes on both sides of its
thresholds, against the oracle.

[V, H] weights.  Streaming GEMV: greedy / logits up to 2 rows, 4 for fp32
activations; sampling one fp32 row.  bf16 activations: the MFMA tile kernel up
to 64 rows, and sampling in 64-row passes up to 128 (where the blocks' shares
of W fill the staged GEMM's tiles, that one takes such calls: test_share_routes);
the staged GEMM for greedy above 64 rows, 256 per pass; the blocked GEMM for
sampling above 128, 256 per pass, but for 161-192 rows (tile passes).  fp32
activations: 16-row passes of the tile kernel up to 16 rows, the staged GEMM on
three terms in 64-row passes up to 192 (a rest of at most 16 rows in the tile
kernel, of one or two in the GEMV), the blocked GEMM above, 256 per pass.

[H, V] weights.  On this vocabulary (few 512-column strips) the blocked GEMM
takes bf16 activations from 2 rows (sampled 3), the streaming kernel fewer; its
narrow layout up to 64 rows, the one that idles padding waves up to 192.  fp32
activations: streaming up to 8 rows, the blocked GEMM above; at 65-128 rows
64-row passes of its narrow layout, then 8-row streaming passes.

Each
case checks greedy ids (check_greedy: first index of the maximum of the
rounded logits, rows within the fp32-summation flip accepted) or sampled ids
(check_fused_sampled: the oracle's Gumbel-max scores) on a vocabulary that is
not a multiple of any tile (V % 256 = 8)."""
import numpy as np
import pytest
import torch

import nvjsel
from oracle import selection as sel
from tests.gpu_helpers import bf16_tensor, check_fused_sampled, check_greedy, engine_keys, keys_tensor

pytestmark = pytest.mark.gpu

H, V = 1024, 4104
BATCHES = [1, 2, 3, 4, 9, 17, 33, 57, 65, 66, 81, 96, 97, 128, 129, 160, 161, 193, 257]


@pytest.fixture(scope="module")
def weights():
    rng = np.random.default_rng(2024)
    Wvh = bf16_tensor(rng.standard_normal((V, H)) * 0.05)
    return Wvh, Wvh.T.contiguous(), Wvh.float().cpu().numpy()


@pytest.mark.parametrize("layout", ["vh", "hv"])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B", BATCHES)
def test_greedy_routes(weights, layout, act, B):
    Wvh, Whv, wf = weights
    rng = np.random.default_rng(31 * B + (act == torch.float32))
    h = torch.from_numpy(rng.standard_normal((B, H)).astype(np.float32)).cuda().to(act)
    if layout == "vh":
        ids = nvjsel.lm_head_greedy_top1_hip(h, Wvh, weight_layout="vh")
    else:
        ids = nvjsel.lm_head_greedy_top1_hip(h, Whv)
    torch.cuda.synchronize()
    rc = 1 if act == torch.bfloat16 else 0
    z = sel.lm_head_logits(h.float().cpu().numpy(), wf)
    check_greedy(ids.cpu().numpy().reshape(-1), z, rc, f"route greedy {layout} {act} B={B}")


@pytest.mark.parametrize("layout", ["vh", "hv"])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B", BATCHES)
def test_sample_routes(weights, layout, act, B):
    Wvh, Whv, wf = weights
    rng = np.random.default_rng(37 * B + (act == torch.float32))
    h = torch.from_numpy(rng.standard_normal((B, H)).astype(np.float32)).cuda().to(act)
    T = [float(x) for x in rng.choice([0.0, 0.8, 1.0], B)]
    keys = engine_keys(B, 101 + B)
    Tt = torch.tensor(T).cuda()
    if layout == "vh":
        ids = nvjsel.lm_head_sample_token_ids(h, Wvh, temperatures=Tt, rng_keys=keys_tensor(keys), weight_layout="vh")
    else:
        ids = nvjsel.lm_head_sample_token_ids(h, Whv, temperatures=Tt, rng_keys=keys_tensor(keys))
    torch.cuda.synchronize()
    rc = 1 if act == torch.bfloat16 else 0
    z = sel.lm_head_logits(h.float().cpu().numpy(), wf)
    namb = check_fused_sampled(ids.cpu().numpy(), z, T, keys, rc, f"route sample {layout} {act} B={B}")
    # every exempt row is within a one-ulp logit flip of the oracle's best
    # score and is reported; the count bound catches a systematic error (B =
    # 66, bf16: 5 such rows, the same ids from the [V, H] tile passes and the
    # [H, V] blocked GEMM)
    assert namb <= max(2, B // 8)


@pytest.mark.parametrize("mode,B", [("greedy", 16), ("greedy", 49), ("logits", 8), ("logits", 9), ("logits", 40),
                                    ("sample", 65), ("sample", 97)])
def test_share_routes(mode, B):
    """bf16 calls that the tile kernel and the staged GEMM both take, on a
    vocabulary whose shares fill the staged GEMM's tiles on 256 CUs (248 of 256
    rows): greedy above 48 rows, logits above 8 and sampled above 64 go there."""
    v = 62470
    rng = np.random.default_rng(B)
    h = bf16_tensor(rng.standard_normal((B, H)))
    w = bf16_tensor(rng.standard_normal((v, H)) * 0.05)
    z = sel.lm_head_logits(h.float().cpu().numpy(), w.float().cpu().numpy())
    ctx = f"share route {mode} B={B}"
    if mode == "sample":
        T = [float(x) for x in rng.choice([0.0, 0.8, 1.0], B)]
        keys = engine_keys(B, 11)
        ids = nvjsel.lm_head_sample_token_ids(h, w, temperatures=torch.tensor(T).cuda(), rng_keys=keys_tensor(keys),
                                              weight_layout="vh")
        assert check_fused_sampled(ids.cpu().numpy(), z, T, keys, 1, ctx) <= B // 8
    elif mode == "greedy":
        check_greedy(nvjsel.lm_head_greedy_top1_hip(h, w, weight_layout="vh").cpu().numpy(), z, 1, ctx)
    else:
        got = nvjsel.lm_head_logits_hip(h, w, weight_layout="vh").float().cpu().numpy().astype(np.float64)
        # fp32 sums of H products and one rounding to bf16
        hn = np.linalg.norm(h.float().cpu().numpy(), axis=1)[:, None]
        wn = np.linalg.norm(w.float().cpu().numpy(), axis=1)[None, :]
        assert (np.abs(got - z) <= H * 2.0 ** -23 * hn * wn + np.abs(z) * 2.0 ** -8 + 1e-7).all()
