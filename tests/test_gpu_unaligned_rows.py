"""GPU: rows that start at any float (odd strides, an offset base), whose
length is not a multiple of 4: the register, greedy, streaming and
full-vocabulary kernels' 16-byte loads against the oracle.

Each row's largest values include its first and its last ones, so a value
lost or moved at either end changes the ids."""
import numpy as np
import pytest

from oracle import oracle
from scriptonait_amd.workloads import PARAMS_DTYPE

pytestmark = pytest.mark.gpu


def _params(B):
    prm = np.zeros(B, dtype=PARAMS_DTYPE)
    prm["temperature"] = np.where(np.arange(B) % 3 == 2, 0.0, 0.8)
    prm["top_k"] = np.where(np.arange(B) % 2 == 0, 3, np.where(np.arange(B) == 3, 0, 100))
    prm["top_p"] = 0.95
    prm["min_p"] = 0.0
    prm["repetition_penalty"] = 1.2
    return prm


@pytest.mark.parametrize("V,pad,off", [
    (1, 0, 1), (2, 1, 0), (3, 0, 2), (4, 0, 3), (5, 0, 1), (6, 1, 1), (7, 2, 3), (255, 0, 1), (257, 0, 0), (1023, 0, 3),
    (4095, 0, 1), (4097, 0, 2), (8190, 1, 1), (8193, 2, 2), (16383, 0, 3), (16387, 0, 0), (32765, 0, 1), (32766, 1, 0),
    (32767, 0, 2), (32768, 1, 3), (32769, 0, 1), (32770, 0, 0), (32771, 3, 2), (32772, 1, 1), (49151, 0, 3),
    (50257, 0, 1), (65535, 0, 2), (65539, 0, 0)])
@pytest.mark.parametrize("masked", [False, True])
def test_rows_at_any_float(sampler, V, pad, off, masked):
    import torch

    rs = np.random.default_rng(V * 8 + off)
    B, ld = 7, V + pad
    x = rs.standard_normal((B, V)).astype(np.float32)
    ends = np.unique(np.clip(np.r_[0:4, V - 5:V], 0, V - 1))
    x[:, ends] += rs.uniform(4.0, 6.0, size=(B, ends.size)).astype(np.float32)
    # What lies between the rows must not be seen.
    flat = np.full(off + B * ld, np.float32(1e30))
    for b in range(B):
        flat[off + b * ld: off + b * ld + V] = x[b]
    dev = torch.device("cuda:0")
    logits = torch.from_numpy(flat).to(dev)[off:].view(B, ld)
    H = 16
    hist = rs.choice(ends, size=(B, H)).astype(np.uint32)
    hist[:, ::3] = rs.integers(0, V, size=(B, (H + 2) // 3))
    offs = (np.arange(B + 1) * H).astype(np.uint32)
    allowed = (rs.random(V) < 0.8).astype(np.uint8) if masked else None
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    prm = _params(B)
    rng = torch.from_numpy(seeds.view(np.int64).copy()).to(dev)
    ids = torch.full((B,), -1, dtype=torch.int32, device=dev)
    kept = torch.full((B,), -1, dtype=torch.int32, device=dev)
    sampler.status()
    sampler.sample_device(logits, prm, rng, ids, V=V, hist=torch.from_numpy(hist.view(np.int32).reshape(-1)).to(dev),
                          hist_offsets=torch.from_numpy(offs.view(np.int32)).to(dev),
                          allowed=None if allowed is None else torch.from_numpy(allowed).to(dev), out_kept=kept)
    torch.cuda.synchronize()
    assert sampler.status().flags == 0
    o = oracle.sample_batch(np.ascontiguousarray(x), prm, seeds, hist.reshape(-1), offs, allowed=allowed, V=V)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), o.ids)
    assert np.array_equal(kept.cpu().numpy().view(np.uint32), o.kept)
    assert np.array_equal(rng.cpu().numpy().view(np.uint64), o.rng_state)
