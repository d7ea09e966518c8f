"""GPU: llmhip_sample_tied_head_device against the oracle.

The reference's decode step computes logits = final_normed @ embed^T with
ops::linear_fwd (crates/llm-core/src/model.rs:396-397, ops/linear.rs:
19-32, 110-125) and samples them with sample_with. The GPU entry must give
the same logits bit for bit (compared with ==, where -0.0 == +0.0: the sign
of a zero logit changes nothing downstream) and the same ids, kept counts
and RNG states as the oracle's linear_fwd followed by its sample_with.
"""
import numpy as np
import pytest

from oracle import oracle
from scriptonait_amd.workloads import make_params

pytestmark = pytest.mark.gpu


def _case(rs, B, V, h, scale=0.02):
    hidden = rs.standard_normal((B, h)).astype(np.float32)
    embed = (scale * rs.standard_normal((V, h))).astype(np.float32)
    return hidden, embed


def _run(sampler, hidden, embed, prm, seeds, hist=None, offs=None, take_logits=True, ldh=None):
    import torch

    dev = torch.device("cuda:0")
    B, h = hidden.shape
    V = embed.shape[0]
    if ldh is not None:  # rows at a stride that is not a multiple of 4 floats
        padded = np.zeros((B, ldh), dtype=np.float32)
        padded[:, :h] = hidden
        d_hidden = torch.from_numpy(padded).to(dev)[:, :h]
    else:
        d_hidden = torch.from_numpy(hidden).to(dev)
    d_embed = torch.from_numpy(embed).to(dev)
    rng = torch.from_numpy(seeds.view(np.int64).copy()).to(dev)
    ids = torch.zeros(B, dtype=torch.int32, device=dev)
    kept = torch.zeros(B, dtype=torch.int32, device=dev)
    lg = torch.full((B, V), float("nan"), dtype=torch.float32, device=dev) if take_logits else None
    hs = os_ = None
    if hist is not None:
        hs = torch.from_numpy(hist.view(np.int32)).to(dev)
        os_ = torch.from_numpy(offs.view(np.int32)).to(dev)
    sampler.sample_tied_head_device(d_hidden, d_embed, prm, rng, ids, hist=hs, hist_offsets=os_, out_kept=kept,
                                    out_logits=lg)
    torch.cuda.synchronize()
    return (ids.cpu().numpy().view(np.uint32), rng.cpu().numpy().view(np.uint64), kept.cpu().numpy().view(np.uint32),
            None if lg is None else lg.cpu().numpy())


def _check(got, hidden, embed, prm, seeds, hist=None, offs=None):
    ids, rng, kept, lg = got
    want_lg = oracle.linear_fwd(hidden, embed, threads=8)
    if lg is not None:
        bad = np.nonzero(~(lg == want_lg))
        assert bad[0].size == 0, f"logits differ at {list(zip(*bad))[:5]}"
    o = oracle.sample_batch(want_lg, prm, seeds, hist, offs, V=embed.shape[0], threads=8)
    assert np.array_equal(ids, o.ids)
    assert np.array_equal(rng, o.rng_state)
    assert np.array_equal(kept, o.kept)


@pytest.mark.parametrize("h", [256, 512])
def test_config3_shape(sampler, h):
    """V = 32000, B = 64, config 3's filters and a 1024-token history."""
    rs = np.random.default_rng(h)
    B, V = 64, 32000
    hidden, embed = _case(rs, B, V, h)
    H = 1024
    hist = rs.integers(0, V, size=B * H).astype(np.uint32)
    offs = (np.arange(B + 1) * H).astype(np.uint32)
    prm = make_params(0.7, 64, 0.95, 0.05, 1.15)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    got = _run(sampler, hidden, embed, prm, seeds, hist, offs)
    _check(got, hidden, embed, prm, seeds, hist, offs)


@pytest.mark.parametrize("B,V,h", [(45, 1000, 257), (3, 130, 5), (33, 4099, 64), (1, 8192, 3)])
def test_ragged_shapes(sampler, B, V, h):
    """B and V off the tile sizes, h off the chunk sizes (the remainder
    fold), tiny h."""
    rs = np.random.default_rng(B * 7 + h)
    hidden, embed = _case(rs, B, V, h, scale=0.5)
    prm = make_params(0.9, 40, 0.9, 0.02, 1.0)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    _check(_run(sampler, hidden, embed, prm, seeds), hidden, embed, prm, seeds)


def test_unaligned_rows_and_context_logits(sampler):
    """Hidden rows 257 floats apart (no 16-byte loads), and the same call
    with the logits kept in the context: the same ids."""
    rs = np.random.default_rng(11)
    B, V, h = 40, 5000, 256
    hidden, embed = _case(rs, B, V, h, scale=0.1)
    prm = make_params(1.0, 50, 0.9, 0.1, 1.0)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    got = _run(sampler, hidden, embed, prm, seeds, ldh=257)
    _check(got, hidden, embed, prm, seeds)
    ids2, rng2, _, _ = _run(sampler, hidden, embed, prm, seeds, take_logits=False)
    assert np.array_equal(ids2, got[0]) and np.array_equal(rng2, got[1])


def test_full_vocabulary_rows(sampler):
    """top_k = 0: the head feeds the full-vocabulary kernel."""
    rs = np.random.default_rng(12)
    B, V, h = 24, 50257, 128
    hidden, embed = _case(rs, B, V, h, scale=0.15)
    prm = make_params(1.0, 0, 0.98, 0.0, 1.0)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    _check(_run(sampler, hidden, embed, prm, seeds, take_logits=False), hidden, embed, prm, seeds)


def test_one_hot_hidden_rows_select_embedding_columns(sampler):
    """hidden = e_j: every logit is embed[o][j] exactly, so greedy picks the
    argmax of column j."""
    rs = np.random.default_rng(13)
    B, V, h = 16, 3000, 64
    embed = rs.standard_normal((V, h)).astype(np.float32)
    hidden = np.zeros((B, h), dtype=np.float32)
    cols = rs.integers(0, h, size=B)
    hidden[np.arange(B), cols] = 1.0
    prm = make_params(0.0, 64, 0.95, 0.05, 1.0)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    ids, _, _, lg = _run(sampler, hidden, embed, prm, seeds)
    assert np.array_equal(lg, embed[:, cols].T)
    assert np.array_equal(ids, np.argmax(embed[:, cols], axis=0).astype(np.uint32))


# Both sides of every line the launch draws (rows, 16- and 32-row tiles, the
# GEMV's output limit) and of every tile: rows, outputs and chunks.
@pytest.mark.parametrize("B,V,h", [
    (1, 33, 0), (1, 31, 4), (1, 16385, 129), (2, 1000, 1027), (2, 33, 127), (3, 16384, 36), (3, 16388, 40), (4, 65, 1156),
    (4, 16385, 32), (5, 64, 33), (16, 65, 35), (17, 63, 64), (32, 129, 31), (33, 4100, 68), (48, 32768, 12),
    (49, 32768, 8), (63, 32769, 37), (64, 32767, 100), (65, 70001, 5), (96, 2049, 64), (128, 16353, 63),
    (8, 65535, 16), (8, 65536, 16), (7, 80000, 4), (33, 16001, 3), (64, 31249, 17), (64, 31250, 17), (63, 40000, 48),
    (97, 20641, 48), (65, 32769, 49), (255, 62500, 64), (256, 62500, 64), (8, 600001, 5), (33000, 64, 4),
    (63, 32769, 165), (65, 70001, 160), (65, 70001, 159), (65, 40000, 65), (65, 40001, 65), (66, 39997, 64), (128, 16353, 191), (64, 32767, 228)])
def test_kernel_boundaries(sampler, B, V, h):
    rs = np.random.default_rng(B * 131 + V + h)
    hidden, embed = _case(rs, B, V, h, scale=0.3)
    prm = make_params(0.9, 20, 0.9, 0.02, 1.0)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    _check(_run(sampler, hidden, embed, prm, seeds), hidden, embed, prm, seeds)


@pytest.mark.parametrize("B", [1, 4, 20, 64])
def test_rows_off_16_byte_alignment_and_extreme_products(sampler, B):
    """Both operands start 4 bytes past a 16-byte boundary with odd strides,
    and the values span products that are denormal, underflow to zero or are
    of denormal inputs: every kernel's products round as binary32 multiplies."""
    import torch

    rs = np.random.default_rng(77 + B)
    V, h = 33000, 130
    ex = lambda n: np.ldexp(rs.standard_normal(n), rs.integers(-80, -55, size=n)).astype(np.float32)  # noqa: E731
    hidden, embed = ex((B, h)), ex((V, h))
    hidden[:, ::7] = np.ldexp(hidden[:, ::7], -75)  # denormals
    embed[:, ::7] = np.ldexp(embed[:, ::7], 120)
    dev = torch.device("cuda:0")

    def place(x, ld):
        buf = torch.zeros(1 + x.shape[0] * ld, dtype=torch.float32, device=dev)
        view = buf[1:].view(x.shape[0], ld)[:, :x.shape[1]]
        view.copy_(torch.from_numpy(x))
        return view

    d_hidden, d_embed = place(hidden, h + 1), place(embed, h + 3)
    seeds = rs.integers(0, 2**63, size=B, dtype=np.uint64)
    rng = torch.from_numpy(seeds.view(np.int64).copy()).to(dev)
    ids = torch.zeros(B, dtype=torch.int32, device=dev)
    lg = torch.empty(B, V, dtype=torch.float32, device=dev)
    sampler.sample_tied_head_device(d_hidden, d_embed, make_params(0.0, 1, 1.0, 0.0, 1.0), rng, ids, out_logits=lg)
    torch.cuda.synchronize()
    want = oracle.linear_fwd(hidden, embed, threads=8)
    assert np.count_nonzero(want) > 0
    assert np.array_equal(lg.cpu().numpy(), want)


# One of each kernel: the GEMV, 16 x 16 tiles, 32 x 32 tiles, vector multiplies.
KERNELS = [(1, 20000, 36), (4, 9000, 36), (20, 9000, 36), (64, 33000, 164), (64, 33000, 12)]


def _logits(sampler, hidden, embed):
    seeds = np.arange(hidden.shape[0], dtype=np.uint64)
    return _run(sampler, hidden, embed, make_params(0.0, 1, 1.0, 0.0, 1.0), seeds)


@pytest.mark.parametrize("B,V,h", KERNELS)
def test_products_over_random_bit_patterns(sampler, B, V, h):
    """One nonzero element per row, of any bit pattern (denormals, infinities
    and NaNs among them): each logit is one product, rounded as binary32
    multiplies round."""
    rs = np.random.default_rng(h * V + B)
    bits = lambda n: rs.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32).view(np.float32)  # noqa: E731
    hidden, embed = np.zeros((B, h), dtype=np.float32), np.zeros((V, h), dtype=np.float32)
    k = int(rs.integers(0, h))
    hidden[:, k], embed[:, k] = bits(B), bits(V)
    hidden[0, k] = np.float32(1e-42)  # a denormal among any number of rows
    embed[:4, k] = np.inf, -np.inf, np.nan, np.float32(3e-45)
    lg = _logits(sampler, hidden, embed)[3]
    with np.errstate(all="ignore"):
        want = hidden[:, k][:, None] * embed[:, k][None, :]
    # (0 * inf and 0 * NaN stay in the column's own accumulator: no other
    # element of a row is infinite.)
    assert np.array_equal(np.isnan(lg), np.isnan(want))
    assert np.array_equal(lg[~np.isnan(lg)], want[~np.isnan(want)])


@pytest.mark.parametrize("B,V,h", KERNELS)
def test_infinities_and_nans_stay_in_their_rows(sampler, B, V, h):
    """Infinite and NaN elements of some hidden and embedding rows: those rows'
    and outputs' logits are the oracle's, and so are the greedy ids."""
    rs = np.random.default_rng(h + V + B)
    hidden, embed = _case(rs, B, V, h, scale=0.3)
    hidden[::3, rs.integers(0, h)] = np.inf
    hidden[2::5, rs.integers(0, h)] = -np.inf
    hidden[4::7, rs.integers(0, h)] = np.nan
    at = rs.choice(V, 60, replace=False)
    embed[at[:20], rs.integers(0, h)] = np.inf
    embed[at[20:40], rs.integers(0, h)] = -np.inf
    embed[at[40:], rs.integers(0, h)] = np.nan
    ids, _, _, lg = _logits(sampler, hidden, embed)
    want = oracle.linear_fwd(hidden, embed, threads=8)
    assert np.array_equal(lg, want, equal_nan=True)
    o = oracle.sample_batch(want, make_params(0.0, 1, 1.0, 0.0, 1.0), np.arange(B, dtype=np.uint64), V=V, threads=8)
    assert np.array_equal(ids, o.ids)
