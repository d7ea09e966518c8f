"""GPU: the allowed mask on the register path (V <= 32768: greedy, top_k <= 64
and larger rows), as bytes at any address and as bits, covering part of the
vocabulary, all of it or more, against the oracle. Nearly half of each row's
largest values are masked, so a bit off by one changes the ids."""
import numpy as np
import pytest

from oracle import oracle
from scriptonait_amd.workloads import PARAMS_DTYPE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,mlen,eos", [
    (4, 3, 0), (300, 1, 7), (1000, 3, 2), (1000, 5, 258), (4096, 4095, 4095), (4097, 4097, 33), (8191, 8190, 0),
    (8192, 9001, 8191), (12345, 12343, 12000), (16384, 16384, 16383), (20000, 6, 5), (31999, 31998, 31998),
    (32000, 32000, 258), (32768, 32768, 32767), (32768, 40000, 99999)])
@pytest.mark.parametrize("kind", ["bits", "bytes0", "bytes1", "bytes3"])
def test_mask_edges(sampler, V, mlen, eos, kind):
    import torch

    rs = np.random.default_rng(V + mlen)
    B = 9
    x = rs.standard_normal((B, V)).astype(np.float32)
    top = np.argsort(-x, axis=1)[:, :max(1, min(V, 40) // 2)]
    allowed = np.zeros(mlen, dtype=np.uint8)
    allowed[rs.random(mlen) < 0.6] = rs.integers(1, 256)  # any nonzero byte allows
    for row in top:
        inside = row[row < mlen]
        allowed[inside[::2]] = 0
    ends = np.array([i for i in (0, 1, 2, mlen - 1, mlen - 2, mlen, mlen + 1, V - 1, eos) if 0 <= i < V])
    x[:, ends] += 3.0
    prm = np.zeros(B, dtype=PARAMS_DTYPE)
    prm["temperature"] = np.where(np.arange(B) % 3 == 0, 0.0, 0.9)
    prm["top_k"] = np.minimum(np.where(np.arange(B) % 3 == 1, 20, 200), max(1, V - 1))
    prm["top_p"] = 0.97
    prm["repetition_penalty"] = 1.15
    H = 24
    hist = np.concatenate([np.resize(t, H) for t in top]).astype(np.uint32)
    offs = (np.arange(B + 1) * H).astype(np.uint32)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    dev = torch.device("cuda:0")
    ids = torch.full((B,), -1, dtype=torch.int32, device=dev)
    kept = torch.full((B,), -1, dtype=torch.int32, device=dev)
    rng = torch.from_numpy(seeds.view(np.int64).copy()).to(dev)
    kw = {}
    if kind == "bits":
        words = np.zeros((mlen + 31) // 32 * 4, dtype=np.uint8)
        words[:(mlen + 7) // 8] = np.packbits(allowed != 0, bitorder="little")
        kw = dict(allowed_bits=torch.from_numpy(words.view(np.int32)).to(dev), allowed_len=mlen)
    else:
        off = int(kind[5:])
        buf = np.full(off + mlen, 1, dtype=np.uint8)
        buf[off:] = allowed
        kw = dict(allowed=torch.from_numpy(buf).to(dev)[off:])
    sampler.status()
    sampler.sample_device(torch.from_numpy(x).to(dev), prm, rng, ids,
                          hist=torch.from_numpy(hist.view(np.int32)).to(dev),
                          hist_offsets=torch.from_numpy(offs.view(np.int32)).to(dev), eos_id=eos, out_kept=kept, **kw)
    torch.cuda.synchronize()
    assert sampler.status().flags == 0
    o = oracle.sample_batch(x, prm, seeds, hist, offs, allowed=allowed, V=V, eos_id=eos)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), o.ids)
    assert np.array_equal(kept.cpu().numpy().view(np.uint32), o.kept)
    assert np.array_equal(rng.cpu().numpy().view(np.uint64), o.rng_state)
