"""CPU: the sizes at which a top-k row of the sampler publishes more lane
maximums or lists more candidates (csrc/route_rules.h), against a model of the
lists on random logits: a row that settles without tier B must not pay for it,
and where more of either settles every row the rules take it."""
import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "nano-vllm-jax_amd" / "csrc"
EPT, WAVES, CAP = 32, 4, 512  # f32 elements per lane of a chunk, waves, survivors
LISTED = 360  # of a list's 512 entries: room for the spread between rows


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text('#include "route_rules.h"\nextern "C" {\n'
                             "int tier_b(int nc, int k, int fill) { return nvjsel::topk_tier_b(nc, k, fill); }\n"
                             "int more_tops(int nc, int k) { return nvjsel::topk_more_tops(nc, k); }\n}\n")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", str(CSRC), str(d / "r.cpp"), "-o", str(d / "r.so")],
                   check=True)
    return ctypes.CDLL(str(d / "r.so"))


def _settles(logits, k, published, tier_b):
    """Whether the lists of one row settle its top k: logits [chunks, 4 waves,
    64 lanes, EPT]; the scan's floors and tiers, then select's row floor."""
    lanes = -np.sort(-logits.max(axis=3), axis=2)  # per wave, descending
    theta = lanes[:, :, -(-k // WAVES) - 1].min(axis=1)  # each chunk's floor
    tier_a = np.maximum(lanes[:, :, 7].min(axis=1), theta)
    tops = -np.sort(-lanes[:, :, :published].reshape(-1))
    floor = max(theta.max(), tops[k - 1] if len(tops) >= k else -np.inf)
    chunks = logits.reshape(len(logits), -1)
    n = int((chunks >= floor).sum())
    if not k <= n <= CAP:
        return False
    for c, ta, th in zip(chunks, tier_a, theta):
        if floor < ta and not tier_b:
            return False
        if (c >= (ta if floor >= ta else th)).sum() > LISTED:
            return False
    return True


@pytest.mark.parametrize("fill", [2, 5, 8])
@pytest.mark.parametrize("k", [16, 32, 33, 48, 64, 100, 128, 160, 200, 256])
@pytest.mark.parametrize("nc", [1, 2, 3, 4, 5, 6, 7, 9, 10, 12, 16, 20, 31])
def test_top_k_rules(rules, nc, k, fill):
    rng = np.random.default_rng((nc * 257 + k) * 9 + fill)
    rows = [rng.exponential(1.2, (nc, WAVES, 64, EPT)).astype(np.float32) for _ in range(10)]
    for r in rows:  # the last chunk's vectors beyond `fill` eighths hold no element
        r[-1, :, :, EPT * fill // 8:] = -np.inf
    plain = sum(_settles(r, k, 4, False) for r in rows)
    more, tier_b = bool(rules.more_tops(nc, k)), bool(rules.tier_b(nc, k, fill))
    if tier_b:  # it costs a row that settles without
        assert more and plain < 10, plain
    best = max(sum(_settles(r, k, 8, b) for r in rows) for b in (False, True))
    ruled = sum(_settles(r, k, 8 if more else 4, tier_b) for r in rows)
    # the rows that miss set the time of a call: where something settles all, the rule does
    if best == 10:
        assert ruled >= 9, (plain, ruled, best)
    assert ruled >= plain
