"""GPU: unmasked FLASH_ATTN_EXT of many query rows (the DiT, src/dit.h:221-222)
where the DMA kernel's tiles and units end: key counts round the 32-key unit,
the 64-key tile and the 4-tile ring, ragged query tiles, one workgroup and
more, grouped KV heads, strided K / V.

Tolerance: the f16 roundings of Q (a score error of at most 2^-11 |s|) and of
P (2^-11 of each weight) move the output by at most 2^-11 (|s| + 1) of the
weighted |V|: 0.017 with |s| <= 6 and |V| <= 5 if every rounding went the same
way.  They are independent, so 2e-3, the bound of the other attention tests,
holds by far."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def oracle(q, k, v, s):
    G = q.shape[1] // k.shape[1]
    k, v = (np.repeat(np.repeat(t.astype(np.float64), G, 1), q.shape[0] // t.shape[0], 0) for t in (k, v))
    a = np.einsum("bhqd,bhkd->bhqk", q.astype(np.float64), k) * s
    p = np.exp(a - a.max(-1, keepdims=True))
    return np.einsum("bhqk,bhkd->bqhd", p / p.sum(-1, keepdims=True), v)


def run(mm, q, k, v, s):
    return mm.flash_attn_ext(torch.from_numpy(q).cuda(), k if isinstance(k, torch.Tensor) else torch.from_numpy(k).cuda(),
                             v if isinstance(v, torch.Tensor) else torch.from_numpy(v).cuda(), None, s).cpu().numpy()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("nq,nkv", [(9, 1), (32, 31), (33, 32), (127, 63), (128, 64), (129, 65), (40, 127), (130, 129),
                                    (60, 191), (257, 193), (31, 256), (96, 257), (250, 321), (20, 700)])
def test_edges(mm, D, nq, nkv):
    rng = np.random.default_rng(1000 * D + 7 * nq + nkv)
    q = rng.standard_normal((2, 6, nq, D)).astype(np.float32)
    k = rng.standard_normal((1, 3, nkv, D)).astype(np.float16)
    v = rng.standard_normal((1, 3, nkv, D)).astype(np.float16)
    s = float(np.float32(1 / np.sqrt(D)))
    out = run(mm, q, k, v, s)
    assert np.abs(out - oracle(q, k, v, s)).max() < 2e-3


@pytest.mark.parametrize("D", [64, 128])
def test_running_max_moves(mm, D):
    """Scores that rise and fall by hundreds from tile to tile: every tile's
    maximum moves the running one, or leaves earlier keys far behind."""
    rng = np.random.default_rng(5)
    nq, nkv = 70, 330
    q = np.abs(rng.standard_normal((1, 2, nq, D))).astype(np.float32)
    k = rng.standard_normal((1, 2, nkv, D)).astype(np.float16)
    k += (np.sin(np.arange(nkv) / 23.0) * 3)[None, None, :, None].astype(np.float16)
    v = rng.standard_normal((1, 2, nkv, D)).astype(np.float16)
    q16 = q.astype(np.float16).astype(np.float32)
    s = 0.5
    # queries that f16 holds exactly: the kernel rounds only their scaled form
    out = run(mm, q16, k, v, s)
    ref = oracle(q16, k, v, s)
    # scaled-query rounding: 2^-11 of each of D products of a score of up to ~200, summed
    # in quadrature: 200 / sqrt(D) 2^-11 sqrt(2) < 0.02 of a probability, times |V| < 4
    assert np.abs(out - ref).max() < 0.08
    assert np.abs(out - ref).mean() < 4e-3


def test_last_value_row_infinite(mm):
    """An infinite last value row gives infinities, not NaN, past a ragged end."""
    rng = np.random.default_rng(6)
    q = rng.standard_normal((1, 2, 40, 64)).astype(np.float32)
    k = rng.standard_normal((1, 2, 70, 64)).astype(np.float16)
    v = rng.standard_normal((1, 2, 70, 64)).astype(np.float16)
    v[:, :, -1] = np.inf
    assert np.isposinf(run(mm, q, k, v, 0.125)).all()


def test_strided_heads(mm):
    """K and V as [nkv, Hkv, D] rows viewed per head, Q as [nq, Hq, D]."""
    rng = np.random.default_rng(7)
    q = torch.from_numpy(rng.standard_normal((1, 200, 4, 64)).astype(np.float32)).cuda().permute(0, 2, 1, 3)
    k = torch.from_numpy(rng.standard_normal((1, 150, 4, 64)).astype(np.float16)).cuda().permute(0, 2, 1, 3)
    v = torch.from_numpy(rng.standard_normal((1, 150, 4, 64)).astype(np.float16)).cuda().permute(0, 2, 1, 3)
    out = mm.flash_attn_ext(q, k, v, None, 0.125).cpu().numpy()
    ref = oracle(q.cpu().numpy(), k.cpu().numpy(), v.cpu().numpy(), 0.125)
    assert np.abs(out - ref).max() < 2e-3
