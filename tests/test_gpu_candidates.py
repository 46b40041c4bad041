"""The candidates of the split transform (orc_transform_probs with T > 0 and
1 <= top_k <= 128): rows whose top_k a slice's or the row's group maxima bound
well, rows where they do not (the largest logits next to each other, ties,
fewer positive probabilities than top_k) and top_k on both sides of the line
(72), against the oracle's transform (Sampler::sample, core/sampler.cpp:29-76):
the same kept set, and probabilities within 2e-6 (of at most 1: the scaled
logit and the row maximum, below 32 here, are rounded at 2^-24 each, so e^l is
off by at most 64 * 2^-24 = 3.8e-6 relative for p near 0 and by 2e-6 absolute
where p (1 - p) bounds it, as the error of the largest p falls on all)."""
import numpy as np
import pytest

from test_gpu_spec_sampling import _check_transform

pytestmark = pytest.mark.gpu


def _rows(kind, V, rng):
    lg = rng.normal(0, 2, (2, V)).astype(np.float32)
    if kind == "sorted":  # the largest next to each other, in the first slice
        lg = -np.sort(-lg, axis=1)
    elif kind == "stripe":  # the largest in the slices of one wave of the last launch
        at = (np.arange(V) // 4096) % 16 == 3
        lg[:, at] += 6
    elif kind == "ties":  # hundreds of equal candidates over the row
        lg = (np.round(lg * 6) / 6).astype(np.float32)
    elif kind == "few":  # fewer positive probabilities than top_k, side by side
        lg -= 500
        lg[:, V // 2: V // 2 + 20] += 500
    return lg


@pytest.mark.parametrize("V,K,kind", [(1, 2, "plain"), (63, 64, "plain"), (4095, 40, "sorted"), (8193, 72, "plain"),
                                      (8193, 73, "plain"), (50000, 64, "sorted"), (50000, 128, "sorted"),
                                      (152064, 40, "sorted"), (152064, 40, "stripe"), (152064, 72, "ties"),
                                      (152064, 40, "few"), (152064, 1, "ties"), (196608, 64, "stripe"),
                                      (196608, 128, "ties")])
def test_candidates_match_oracle(dev, oracle, V, K, kind):
    print(f"[gpu] candidates V={V} top_k={K} {kind}", flush=True)
    rng = np.random.default_rng(V + K)
    hist, extra = rng.integers(0, V, 80).astype(np.int32), rng.integers(0, V, 4).astype(np.int32)
    _check_transform(dev, oracle, _rows(kind, V, rng), 0.9, 0.95, K, 1.1, 64, hist, extra, 1)
