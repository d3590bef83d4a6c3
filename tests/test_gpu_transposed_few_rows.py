"""Transposed weights, two to four rows (sbvr_row_deq_few_kernel): plane bits turned by a matrix product, the coefficients on the
activations' side.  Taken where the launch that decodes every weight has more workgroups than the chip has CUs."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _sums(x, bvr, idx, cache, G):
    """The selected coefficients alone, in 64 bits."""
    bits = ((bvr[:, :, None, :] >> np.arange(32, dtype=np.uint32)[None, None, :, None]) & 1).astype(bool)   # (N/32, K, 32, S)
    line = np.repeat(cache.astype(np.float64)[idx.astype(np.int64)], G // 32, axis=0)                      # (N/32, K, S)
    out = np.zeros((x.shape[0], bvr.shape[0] * 32))
    with np.errstate(invalid="ignore"):
        for m in range(x.shape[0]):
            out[m] = np.where(bits, (x[m].astype(np.float64)[None, :, None] * line)[:, :, None, :], 0.0).sum(axis=(1, 3)).ravel()
    return out


def _call(x, bvr, idx, cache, G, bias=None):
    import sbvr
    from sbvr import hip
    dev = torch.device("cuda:0")
    none = torch.zeros(0, dtype=torch.float16) if bias is None else torch.from_numpy(bias)
    args = [torch.from_numpy(a).to(dev) for a in (x, bvr, idx, cache)] + [none.to(dev)]
    y = sbvr._sbvr_row_deq_mm_T(*args, 0, bvr_len=G)
    assert hip.row_deq_last()[0] == hip.ROW_DEQ_ROWS
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert hip.row_deq_last_turned()
    assert torch.equal(y.view(torch.int16), sbvr._sbvr_row_deq_mm_T(*args, 0, bvr_len=G).view(torch.int16))
    assert int(hip._workspace(8 * y.numel(), dev).count_nonzero()) == 0
    return y.float().cpu().numpy().astype(np.float64), hip.row_deq_last()[1]


def _encoding(N, K, S, G, L, seed):
    from sbvr import synth
    return [t.numpy() for t in synth.random_encoding(K, N, S, G, L, seed=seed)]


@pytest.mark.parametrize("M,N,K,S,G,L,bias", [
    (2, 8256, 1410, 4, 64, 256, False),         # the last tile of K two rows
    (3, 8256, 1409, 3, 64, 300, True),          # one row in it, uint16 indices
    (4, 16448, 1537, 2, 16448, 16, False),      # one group
    (4, 8320, 129, 4, 128, 256, True),          # two tiles, one of one row, K whole
    (4, 14336, 127, 3, 128, 256, False),        # less than a tile
    (3, 4096, 4096, 4, 256, 768, False),        # K in parts
    (4, 2048, 8200, 2, 128, 256, True),         # parts of different lengths
])
def test_against_sums_in_64_bits(M, N, K, S, G, L, bias):
    """Within 2 fp16 ulps: the fp32 additions and the one rounding."""
    bvr, idx, cache = _encoding(N, K, S, G, L, N + K)
    rng = np.random.default_rng(K)
    # rows of very different size, and a row that ends in zeros
    x = (rng.standard_normal((M, K)) * np.array([1.0, 1e-3, 100.0, 1.0])[:M, None]).astype(np.float16)
    x[M - 1, K // 2:] = 0
    b = (rng.standard_normal(N) * 0.1).astype(np.float16) if bias else None
    y, _ = _call(x, bvr, idx, cache, G, b)
    want = _sums(x, bvr, idx, cache, G) + (b.astype(np.float64) if bias else 0.0)
    rms = np.sqrt(np.mean(want ** 2, axis=1, keepdims=True))
    err = np.abs(y - want) / (np.maximum(np.maximum(np.abs(want), rms), 2.0 ** -14) * 2.0 ** -10)
    assert err.max() <= 2.0, err.max()


@pytest.mark.parametrize("N,K,S,G", [(4096, 4100, 4, 128), (8192, 1500, 2, 128), (2048, 12032, 3, 256)])
def test_as_exact_as_fp32_sums(N, K, S, G):
    """The sums before their rounding to fp16 (a bias takes all but a rounding's remainder away; only columns count whose
    remainder's own rounding does not show), against the row by itself on the lanes launch: exact products added up in fp32."""
    import sbvr
    from sbvr import hip
    dev = torch.device("cuda:0")
    bvr, idx, cache = _encoding(N, K, S, G, 256, N + K)
    x = torch.randn((1, K), generator=torch.Generator().manual_seed(K)).to(torch.float16)
    want = _sums(x.numpy(), bvr, idx, cache, G)[0]
    bias = (-want).astype(np.float16)
    rest, rms = want + bias.astype(np.float64), np.sqrt(np.mean(want ** 2))
    near = np.abs(rest) < 2.0 ** -14 * rms
    assert near.sum() > 200
    args = [torch.from_numpy(a).to(dev) for a in (bvr, idx, cache, bias)]
    error = {}
    for M in (1, 3):
        y = sbvr._sbvr_row_deq_mm_T(x.to(dev).repeat(M, 1), *args, 0, bvr_len=G).float().cpu().numpy().astype(np.float64)
        assert hip.row_deq_last()[0] in ((hip.ROW_DEQ_LANES,) if M == 1 else (hip.ROW_DEQ_ROWS,))
        if M > 1 and torch.cuda.get_device_properties(dev).multi_processor_count == 256:
            assert hip.row_deq_last_turned()
        error[M] = np.sqrt(np.mean((y - rest)[:, near] ** 2))
    assert error[3] <= error[1], (error[3] / rms, error[1] / rms)


def test_values_that_are_not_finite():
    """Infinite and NaN activations, an infinite coefficient, weights beyond fp16: outputs that do not select them stay finite."""
    M, N, K, S, G, L = 4, 8256, 1500, 3, 64, 40
    bvr, idx, cache = _encoding(N, K, S, G, L, 12)
    cache = cache.copy()
    cache[7, 1] = np.inf
    cache[9] = [60000, 40000, 50000]
    rng = np.random.default_rng(12)
    idx = np.where(np.isin(idx, (7, 9)), 1, idx).astype(idx.dtype)
    idx[:2, 3], idx[2:4, 800] = 7, 9
    x = (rng.standard_normal((M, K)) * 0.01).astype(np.float16)
    x[0, 5], x[1, 1499], x[1, 5], x[2, 300] = np.inf, -np.inf, np.inf, np.nan
    y, parts = _call(x, bvr, idx, cache, G)
    want = _sums(x, bvr, idx, cache, G)
    want = np.where(np.abs(want) >= 65520.0, np.sign(want) * np.inf, want)
    assert np.array_equal(np.isnan(y), np.isnan(want))
    assert np.array_equal(np.isposinf(y), np.isposinf(want)) and np.array_equal(np.isneginf(y), np.isneginf(want))
    finite = np.isfinite(want)
    assert finite[:3].any(axis=1).all() and not finite[:3].all(axis=1).any()
    rms = np.sqrt(np.mean(want[finite] ** 2))
    assert (np.abs(y[finite] - want[finite]) <= 2.0 ** -9 * np.maximum(np.abs(want[finite]), min(rms, 1.0))).all()
