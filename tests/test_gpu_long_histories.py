"""GPU: histories at the length from which a u16 multiplicity could overflow.
The register path hands such rows to the sorting path, and the host entry
copies their inputs to the device (it reads the others in pinned memory)."""
import numpy as np
import pytest

from oracle import oracle
from scriptonait_amd.workloads import PARAMS_DTYPE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,handed", [([8191, 65535], 0), ([65536, 3], 1), ([100000, 0, 65537], 2)])
@pytest.mark.parametrize("top_k,T,rp", [(40, 0.8, 1.1), (40, 0.8, 1.0), (40, 0.8, 0.9), (0, 0.0, 0.9), (0, 0.8, 1.1)])
def test_host_rows_with_long_histories(sampler, lengths, handed, top_k, T, rp):
    rs = np.random.default_rng(sum(lengths) + top_k)
    B, V = len(lengths), 32000
    x = (rs.standard_normal((B, V)) * 2).astype(np.float32)
    # A hot id in each history: its count alone passes 16 bits.
    hist = np.concatenate([np.where(rs.random(n) < 0.9, 7 + b, rs.integers(0, V, n)) for b, n in enumerate(lengths)])
    x[np.arange(B), 7 + np.arange(B)] = 30.0
    hist, offs = hist.astype(np.uint32), np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint32)
    prm = np.zeros(1, dtype=PARAMS_DTYPE)
    prm["temperature"], prm["top_k"], prm["top_p"], prm["repetition_penalty"] = T, top_k, 0.95, rp
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    sampler.status()
    g = sampler.sample_host(x, prm, seeds, hist, offs, V=V)
    st = sampler.status()
    o = oracle.sample_batch(x, prm, seeds, hist, offs, V=V, threads=8)
    assert np.array_equal(g.ids, o.ids)
    assert np.array_equal(g.kept, o.kept)
    assert np.array_equal(g.rng_state, o.rng_state)
    assert st.flags == 0
    if top_k == 40 and rp >= 1.0:
        assert st.handovers == (handed if rp != 1.0 else 0)
