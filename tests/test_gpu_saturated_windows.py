"""GPU: rows whose history holds all of their top ids many times over (a long
generation's own draws), so the first threshold leaves no survivor and the
K-th value that no penalty touches lies in a dense part of the row: the
register path's proven threshold, its split bin and its scan in several
rounds, against the oracle, with no row handed over."""
import numpy as np
import pytest

from oracle import oracle
from scriptonait_amd.workloads import make_params

pytestmark = pytest.mark.gpu


# K past 384, whose threshold comes from the chunks' maxima (and its scan, in
# rounds, lists more than the small-K kernel ranks), up to 1024 and just past it,
# where the per-slot narrowing takes over.
LARGE_K = [(8191, 1500, 5), (16384, 2500, 4), (32000, 1000, 12), (32000, 4000, 3), (32768, 3000, 5)]


@pytest.mark.parametrize("V,top,reps", LARGE_K)
@pytest.mark.parametrize("K", [385, 700, 1024, 1025])
@pytest.mark.parametrize("masked", [False, True])
def test_every_top_id_penalized_at_large_k(sampler, V, top, reps, K, masked):
    test_every_top_id_penalized(sampler, V, top, reps, K, masked)


@pytest.mark.parametrize("V,top,reps", [(4096, 300, 12), (8191, 500, 12), (16384, 700, 9), (32000, 400, 12),
                                        (32000, 1000, 12), (32768, 1500, 12), (32000, 2500, 7)])
@pytest.mark.parametrize("K", [1, 20, 40, 64, 100, 380])
@pytest.mark.parametrize("masked", [False, True])
def test_every_top_id_penalized(sampler, V, top, reps, K, masked):
    rs = np.random.default_rng(V + top + K)
    B = 8
    x = (np.where(np.arange(B) % 2 == 0, 3.0, 0.7)[:, None] * rs.standard_normal((B, V))).astype(np.float32)
    order = np.argsort(-x, axis=1)[:, :top]
    hist = np.tile(order, (1, reps)).astype(np.uint32)
    hist[:, ::5] = rs.integers(0, V, hist[:, ::5].shape)
    offs = (np.arange(B + 1) * hist.shape[1]).astype(np.uint32)
    allowed = (rs.random(V) < 0.7).astype(np.uint8) if masked else None
    prm = make_params(0.7, K, 0.98, 0.0, 1.3)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    sampler.status()
    g = sampler.sample_host(x, prm, seeds, hist.reshape(-1), offs, allowed=allowed, V=V)
    st = sampler.status()
    o = oracle.sample_batch(x, prm, seeds, hist.reshape(-1), offs, allowed=allowed, V=V, threads=8)
    assert np.array_equal(g.ids, o.ids)
    assert np.array_equal(g.kept, o.kept)
    assert np.array_equal(g.rng_state, o.rng_state)
    assert st.handovers == 0
