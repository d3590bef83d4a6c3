"""Activations encoded on the fly, more than 64 (row, plane) pairs: the product through the activations as fp16 numbers
(sbvr_online_product_kernel) against the planes' own, `_online_mm_T_general`, and sums in 64 bits."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _weight(N, K, S, G, L, Sl, seed, lines_sigma=1.0):
    import sbvr
    from sbvr import synth
    dev = torch.device("cuda:0")
    enc = sbvr.sbvr.from_parts(*(t.to(dev) for t in synth.random_encoding(N, K, S, G, L, seed=seed)), G)
    enc.input_num_sums = Sl
    enc.input_coeff = torch.nn.Parameter(synth.make_lines(K // G, Sl, lines_sigma, seed + 1).to(dev), requires_grad=False)
    return enc


def _dense(bvr, idx, cache, G):
    """(rows, K) of an encoding in 64 bits: the coefficients whose bit is set."""
    bvr, idx, cache = bvr.cpu().numpy(), idx.cpu().numpy().astype(np.int64), cache.cpu().numpy().astype(np.float64)
    bits = ((bvr[:, None, :, :] >> np.arange(32, dtype=np.uint32)[None, :, None, None]) & 1).astype(np.float64)      # (K/32, 32, rows, S)
    line = np.repeat(cache[idx], G // 32, axis=0)                                                                    # (K/32, rows, S)
    return np.einsum("wbns,wns->nwb", bits, line).reshape(bvr.shape[1], -1)


def _taken(enc, x, G):
    """Whether the call goes that way: scratch memory is what it asks for."""
    from sbvr import hip
    lib, (K, N) = hip._load(), (x.shape[1], enc.bvr.shape[1])
    ask = lib.sbvr_hip_online_mm_T_scratch
    ask.restype, ask.argtypes = ctypes.c_size_t, [ctypes.c_void_p] * 2 + [ctypes.c_int] * 6
    return ask(enc.bvr.data_ptr(), enc.coeff_cache.data_ptr(), x.shape[0], N, K, enc.input_coeff.shape[1], enc.bvr.shape[2], G) > 0


def _sums(enc, x, G):
    l_bvr, l_idx, l_cache = enc._online_tranfrom(x)
    return _dense(l_bvr, l_idx, l_cache, G) @ _dense(enc.bvr.data, enc.coeff_idx.data, enc.coeff_cache.data, G).T


@pytest.mark.parametrize("M,N,K,S,Sl,G,L,bias", [
    (9, 3057, 128, 4, 8, 128, 16, False),        # one sub-group, a column over
    (16, 4096, 4096, 4, 8, 128, 256, False),
    (17, 1600, 384, 3, 8, 128, 300, True),       # a second row tile of one row, 16-bit indices
    (33, 1027, 2304, 2, 6, 256, 256, False),     # an odd number of row tiles
    (64, 4100, 768, 6, 8, 256, 16, True),        # two row tiles a workgroup
    (40, 8211, 384, 8, 5, 128, 256, False),      # the same, the second tile of the last not there
    (22, 1700, 640, 8, 8, 128, 256, False),
    (15, 14336, 1152, 4, 5, 128, 256, False),    # eight waves
])
def test_against_sums_in_64_bits(M, N, K, S, Sl, G, L, bias):
    """Within 2 fp16 ulps: fp32 sums and one rounding (and the bias's)."""
    enc = _weight(N, K, S, G, L, Sl, N + K)
    gen = torch.Generator().manual_seed(M)
    x = torch.randn((M, K), generator=gen).to(torch.float16).to("cuda:0")
    b = (torch.randn(N, generator=gen) * 0.1).to(torch.float16).to("cuda:0") if bias else None
    assert _taken(enc, x, G)
    y = enc.online_mm_T(x, b)
    assert torch.equal(y, enc.online_mm_T(x, b))
    want = _sums(enc, x, G) + (b.cpu().numpy().astype(np.float64) if bias else 0.0)
    rms = np.sqrt(np.mean(want ** 2))
    err = np.abs(y.float().cpu().numpy() - want) / (np.maximum(np.abs(want), rms) * 2.0 ** -10)
    assert err.max() <= (3.0 if bias else 2.0), err.max()


@pytest.mark.parametrize("N,K,S,Sl,G,sigma", [(4096, 4096, 4, 8, 128, 1.0), (4096, 1024, 3, 8, 256, 1e-3), (2048, 8192, 2, 6, 128, 100.0)])
def test_as_exact_as_plane_by_plane(N, K, S, Sl, G, sigma):
    """Activations and lines of any size: the outputs are no further from 64 bits than those of the planes' own product (both are
    rounded to fp16 once, which is most of it: 1e-3 of it is what rounding one sum in 1000 the other way makes)."""
    enc = _weight(N, K, S, G, 256, Sl, N + K, sigma)
    x = (torch.randn((32, K), generator=torch.Generator().manual_seed(K)) * sigma).to(torch.float16).to("cuda:0")
    assert _taken(enc, x, G)
    want = _sums(enc, x, G)
    error = [np.sqrt(np.mean((y.double().cpu().numpy() - want) ** 2) / np.mean(want ** 2)) for y in (enc.online_mm_T(x), enc._online_mm_T_general(x, None))]
    assert error[0] <= error[1] * 1.001, error


def test_lines_that_are_not_finite():
    """A group whose input coefficients hold an infinity: every output is finite, infinite or NaN as in the planes' own product
    (NaN, all of them).  Without it, activations of which one is infinite and one NaN: finite outputs."""
    enc = _weight(3100, 768, 4, 128, 64, 8, 5)
    lines = enc.input_coeff.data.clone()
    lines[2, 3] = float("inf")
    enc.input_coeff = torch.nn.Parameter(lines, requires_grad=False)
    x = torch.randn((16, 768), generator=torch.Generator().manual_seed(1)).to(torch.float16).to("cuda:0")
    x[3, 5], x[4, 7] = float("inf"), float("nan")
    assert _taken(enc, x, 128) and not _taken(enc, x[:8], 128)
    y, want = enc.online_mm_T(x), enc._online_mm_T_general(x, None)
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isposinf(), want.isposinf()) and torch.equal(y.isneginf(), want.isneginf())
    lines[2, 3] = 1.0
    y, want = enc.online_mm_T(x), enc._online_mm_T_general(x, None)
    assert want.isfinite().all() and (y.float() - want.float()).abs().max() <= 2.0 ** -9 * max(1.0, want.float().abs().max().item())


@pytest.mark.parametrize("M,N,K,S,G", [(16, 3100, 768, 4, 128), (33, 3100, 768, 2, 256), (20, 3100, 512, 8, 256)])
def test_weights_that_are_not_finite(M, N, K, S, G):
    """A line of the weight's table with an infinity, one with NaN and one with an infinity whose plane has no bits in the second half
    of a group, which only some columns use: these outputs are infinite or NaN as in the planes' own product, which adds up 128
    elements at a time; all others finite and as exact."""
    enc = _weight(N, K, S, G, 64, 8, 5)
    cache, idx, bvr = enc.coeff_cache.data.clone(), enc.coeff_idx.data.clone(), enc.bvr.data.clone()
    cache[5, 1], cache[9, 0], cache[12, 1] = float("inf"), float("nan"), float("inf")
    idx[idx == 5], idx[idx == 9], idx[idx == 12] = 1, 1, 1
    idx[1, 100:2000:7], idx[0, 103:2000:70], idx[1, 3::9] = 5, 9, 12
    if G > 128:
        bvr.view(torch.int32)[(G + 128) // 32:2 * G // 32, 3::9, 1] = 0
    enc.coeff_cache, enc.coeff_idx, enc.bvr = (torch.nn.Parameter(t, requires_grad=False) for t in (cache, idx, bvr))
    enc.input_coeff = torch.nn.Parameter(enc.input_coeff.data.abs(), requires_grad=False)           # (of both signs: NaN, not infinite)
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(1)).abs().to(torch.float16).to("cuda:0")
    assert _taken(enc, x, G)
    y, want = enc.online_mm_T(x), enc._online_mm_T_general(x, None)
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isposinf(), want.isposinf()) and torch.equal(y.isneginf(), want.isneginf())
    assert 0 < want.isinf().sum() < want.numel() / 2 and 0 < want.isnan().sum() < want.numel() / 2
    finite = want.isfinite()
    rms = want[finite].float().pow(2).mean().sqrt().item()
    assert (y[finite].float() - want[finite].float()).abs().max() <= 2.0 ** -9 * max(rms, want[finite].float().abs().max().item())


@pytest.mark.parametrize("M,K,taken", [(2048, 16384, True), (2049, 16384, False), (4096, 8192, True), (4096, 8320, False)])
def test_memory_of_the_call_is_bounded(M, K, taken):
    """The activations as fp16 numbers take 128 MiB at most; beyond, the planes' own product needs their planes alone."""
    from sbvr import hip
    ask = hip._load().sbvr_hip_online_mm_T_scratch
    ask.restype, ask.argtypes = ctypes.c_size_t, [ctypes.c_void_p] * 2 + [ctypes.c_int] * 6
    need = ask(64, 64, M, 4096, K, 8, 4, 128)
    assert (need > 0) == taken and need <= (128 << 20) + M * K + 4 * K
