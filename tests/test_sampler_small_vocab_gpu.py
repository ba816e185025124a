"""GPU: top-k rows of vocabularies of a few scan chunks, where a chunk holds
more of the row's top k than its first candidate tier: the candidates' second
tier and the row floor from all published lane maximums, against the oracle."""
import numpy as np
import pytest
import torch

import nvjsel
from tests.gpu_helpers import check_sampled, engine_keys, keys_tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [300, 1000, 8192, 16385, 37888, 50257, 65536, 131072])
def test_top_k_rows(V, dtype):
    rng = np.random.default_rng(V)
    ks = [20, 100, 100, 128, 200, 256]
    B = len(ks)
    l = (rng.exponential(1.2, (B, V)) + rng.standard_normal((B, V))).astype(np.float32)
    l[2] = np.round(l[2] * 2) / 2  # ties at the k-th largest
    l[4, : V // 2] += 8.0  # the row's top k in some of the chunks
    t = torch.from_numpy(l).cuda().to(dtype)
    T = [0.7, 1.0, 0.9, 0.6, 1.3, 0.7]
    P = [1.0, 0.95, 0.8, 1.0, 0.9, 1.0]
    keys = engine_keys(B, 11)
    ids = nvjsel.sample_token_ids(t, torch.tensor(T).cuda(), keys_tensor(keys),
                                  top_k=torch.tensor(ks, dtype=torch.int32).cuda(), top_p=torch.tensor(P).cuda())
    torch.cuda.synchronize()
    check_sampled(ids.cpu().numpy(), t.float().cpu().numpy(), T, ks, P, keys, ctx=f"small vocab {dtype} V={V}")
