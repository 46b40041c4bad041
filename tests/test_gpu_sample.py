"""orc_sample (Sampler::sample, core/sampler.cpp:91-97) split over workgroups
(T > 0, 1 <= top_k <= 128, up to 196608 logits) against the oracle's sampler:
draw after draw the same id (the same mt19937 uniform against the same sorted
kept set) and the row left holding the probabilities, in float64: the scaled
logits l and their maximum m are rounded (2^-24 of each, an error of the
exponent, and so relative), then e, the sum and the product (8 more roundings
with the sum's order), twice over."""
import numpy as np
import pytest

from oracle_lib import fptr

pytestmark = pytest.mark.gpu


def _logits(kind, V, rng):
    lg = rng.normal(0, 3, V).astype(np.float32)
    if kind == "grid":  # many exact ties, at the k-th largest too
        lg = (np.round(lg * 2) / 2).astype(np.float32)
    elif kind == "tied":  # more candidates in a slice than it passes on: the row is redone whole
        lg[: min(V, 9000)] = 5.0
    elif kind == "peaked":  # the tail underflows to zero probability
        lg[V // 3] = 300.0
    elif kind == "masked":  # all but a few tokens masked out
        keep = rng.integers(0, V, 5)
        row = np.full(V, -np.inf, np.float32)
        row[keep] = lg[keep]
        row[rng.integers(0, V)] = np.finfo(np.float32).min
        lg = row
    return lg


@pytest.mark.parametrize("V,K,kind", [(1, 40, "plain"), (100, 128, "plain"), (4096, 40, "grid"), (4097, 1, "plain"),
                                      (32000, 128, "grid"), (40000, 40, "tied"), (50000, 40, "peaked"),
                                      (9000, 40, "masked"), (152064, 40, "plain"), (196608, 100, "plain")])
def test_sample_matches_oracle(dev, oracle, V, K, kind):
    print(f"[gpu] sample V={V} top_k={K} {kind}", flush=True)
    L, T, P, pen, last, seed = dev.L, 0.8, 0.95, 1.1, 64, 1234 + V
    rng = np.random.default_rng(V + K)
    hist = rng.integers(0, V, 70).astype(np.int32)
    hist[:20] = rng.integers(0, min(V, 9), 20)  # repeats compound
    state, dh, do = dev.alloc(L.orc_sampler_state_bytes()), dev.upload(hist), dev.alloc(4)
    dev.check(L.orc_sampler_init(state.ptr, T, P, K, pen, last, seed, dh.ptr, hist.size, None))
    s = oracle.L.orco_sampler_new(T, P, K, pen, last, seed)
    for h in hist:
        oracle.L.orco_sampler_record(s, int(h))
    dl, recorded = dev.alloc(4 * V), hist.tolist()
    for i in range(12):
        lg = _logits(kind, V, rng)
        x = lg.astype(np.float64)
        for t in recorded[-last:]:
            x[t] = x[t] / np.float32(pen) if x[t] > 0 else x[t] * np.float32(pen)
        x *= 1.0 / np.float32(T)
        e = np.exp(x - x.max())
        p = e / e.sum()
        want = oracle.L.orco_sampler_sample(s, fptr(lg.copy()), V)
        recorded.append(want)
        dl.write(lg)
        dev.check(L.orc_sample(state.ptr, dl.ptr, V, do.ptr, None))
        assert int(do.read(np.int32)[0]) == want, i
        got = dl.read(np.float32)
        rel = 2.0 ** -23 * (np.minimum(np.abs(x), 1e30) + abs(x.max()) + 8)
        assert np.all(np.abs(got - p) <= rel * p + 1e-37), i
    oracle.L.orco_sampler_free(s)
