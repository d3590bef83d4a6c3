"""Activations encoded on the fly, many rows: the sums in front of the output's rounding to fp16, which hides a thousand times what
they are off.  Seen through the outputs that almost cancel: their own rounding is as small as they are."""
import numpy as np
import pytest
import torch

from test_gpu_online_product import _sums, _taken, _weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("one_sign", [False, True])
@pytest.mark.parametrize("M,N,K,S,Sl,G", [(64, 14336, 1024, 4, 8, 128), (64, 14336, 2048, 2, 8, 256), (48, 14336, 1024, 6, 6, 128), (64, 12288, 1024, 3, 7, 256)])
def test_sums_as_exact_as_plane_by_plane(M, N, K, S, Sl, G, one_sign):
    """No further from 64 bits than the planes' own product (exact popcounts, fp32 sums of their products), in the root mean square
    over outputs below 2^-11 of the RMS output.  (Rounding adds at most 2^-23 / sqrt(12) of it to either side; some 300 outputs tell
    a root mean square to 4 %, hence the tenth.)"""
    enc = _weight(N, K, S, G, 256, Sl, N + K)
    enc.coeff_cache = torch.nn.Parameter(enc.coeff_cache.data * 64, requires_grad=False)         # (outputs whose 2^-11 is a normal number)
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(K)).to(torch.float16).to("cuda:0")
    if one_sign:
        enc.input_coeff = torch.nn.Parameter(enc.input_coeff.data.abs(), requires_grad=False)
        x = x.abs()
    assert _taken(enc, x, G)
    want = _sums(enc, x, G)
    rms = np.sqrt(np.mean(want ** 2))
    near = np.abs(want) < 2.0 ** -11 * rms
    assert near.sum() > 200 and rms > 16.0
    error = [np.sqrt(np.mean((y.double().cpu().numpy() - want)[near] ** 2)) / rms for y in (enc.online_mm_T(x), enc._online_mm_T_general(x, None))]
    print(f"{error[0]:.2e} {error[1]:.2e} {near.sum()}")
    assert error[0] <= error[1] * 1.1, error
