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

import oracle_lib as ol
from test_gpu_spec_sampling import _check_transform, _uniform

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


def _subnormal_row(V):
    """One large logit, and 4096 ascending ones whose p are subnormal (exp(-95)
    is some 4000 units of 2^-149): neighbours tie, the lower index first,
    though their logits differ."""
    rng = np.random.default_rng(3)
    lg = np.full(V, -0.01, np.float32)
    lg[:4096] = np.sort(rng.normal(0, 2e-4, 4096)).astype(np.float32)
    lg[V - 5] = 95 * 0.9
    return lg


@pytest.mark.parametrize("V,K,P,kind", [(50000, 40, 1.5, "subnormal"), (50000, 100, 1.5, "subnormal"),
                                        (50000, 40, 0.95, "mask"), (152064, 128, 1.5, "mask")])
def test_candidates_of_masked_and_subnormal_rows(dev, oracle, V, K, P, kind):
    """Slices whose logits say nothing about their p: all masked by a low value
    (their e are zero and tie), or p below 2^-100, where the k-th p ties with
    smaller logits. Same kept set as the oracle (top_p above 1 keeps all)."""
    print(f"[gpu] candidates V={V} top_k={K} {kind}", flush=True)
    if kind == "subnormal":
        lg = np.stack([_subnormal_row(V)] * 2)
    else:
        rng = np.random.default_rng(K)
        lg = np.full((2, V), [[-1e30], [np.finfo(np.float32).min]], np.float32)
        ids = rng.choice(V, 30, replace=False)
        lg[:, ids] = rng.normal(0, 2, 30).astype(np.float32)
    none = np.zeros(1, np.int32)
    _check_transform(dev, oracle, lg, 0.9, P, K, 1.0, 64, none, none, 0)


def test_draw_after_a_redone_row(dev, oracle):
    """A row that the last launch hands to the one-workgroup transform draws
    with one uniform: it takes the large logit, and the next row's draw is the
    oracle's second."""
    L, V, K = dev.L, 50000, 40
    print("[gpu] draw after a redone row", flush=True)
    state, dp, do = dev.alloc(L.orc_sampler_state_bytes()), dev.alloc(V * 4), dev.alloc(8)
    dev.check(L.orc_sampler_init(state.ptr, 0.9, 1.5, K, 1.0, 64, 31, None, 0, None))
    s = oracle.L.orco_sampler_new(0.9, 1.5, K, 1.0, 64, 31)
    for lg in (_subnormal_row(V), np.random.default_rng(1).normal(0, 2, V).astype(np.float32)):
        dl = dev.upload(lg)
        dev.check(L.orc_transform_draw(state.ptr, dl.ptr, V, None, 0, dp.ptr, do.ptr, None, None))
        p = dp.read(np.float32)
        assert int(do.read(np.int32, 1)[0]) == oracle.L.orco_pick(ol.fptr(p), V, _uniform(oracle, s))
    oracle.L.orco_sampler_free(s)
