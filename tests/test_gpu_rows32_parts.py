"""The table look-up kernel of up to 32 rows with K in parts: numbers of them that are no power of two, parts and waves of
different lengths, waves without a word pair, both sides of two workgroups a CU."""
import numpy as np
import pytest
import torch

import parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,S,G,L,bias,parts", [
    (9, 32, 28672, 4, 128, 256, False, 14),         # one block of columns, the most parts
    (17, 600, 20480, 3, 256, 300, True, 10),        # uint16 indices, bias
    (32, 601, 14272, 2, 64, 256, False, 7),         # 223 word pairs: an odd number, the last part shorter
    (24, 1300, 10240, 8, 128, 256, True, 5),
    (12, 2399, 6144, 4, 128, 256, False, 3),
    (12, 4096, 14336, 3, 128, 256, False, 2),       # one workgroup a CU, though four parts come out nearly the same
    (16, 3000, 20480, 4, 64, 768, False, 5),        # two workgroups on most CUs
    (31, 5000, 4096, 3, 128, 256, True, 1),         # 157 blocks, whole
    (6, 200, 4096, 6, 64, 256, False, 4),           # two word pairs a wave
    (20, 513, 576, 8, 64, 16, False, 1),            # 9 pairs, taken by twos: three waves without one
])
def test_k_in_parts(M, N, K, S, G, L, bias, parts):
    """Against the products with decode()'s weights in 64 bits, as every call's; the accumulators left clean."""
    import sbvr
    from sbvr import hip, synth
    dev = torch.device("cuda:0")
    bvr, idx, cache = (t.to(dev) for t in synth.random_encoding(N, K, S, G, L, seed=N + K))
    gen = torch.Generator().manual_seed(M)
    x = torch.randn((M, K), generator=gen).to(torch.float16).to(dev)
    b = (torch.randn(N, generator=gen) * 0.3).to(torch.float16).to(dev) if bias else None
    y = sbvr._sbvr_linear_f16(x, bvr, idx, cache, b, bvr_len=G)
    assert hip.last_kernel() == 3                   # the 32-row kernel
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert hip.last_parts() == parts
    assert torch.equal(y, sbvr._sbvr_linear_f16(x, bvr, idx, cache, b, bvr_len=G))
    weight = sbvr.sbvr.from_parts(bvr, idx, cache, G).decode()
    want = x.double() @ weight.double().t()
    if bias:
        want += b.double()
    got, want = y.double().cpu().numpy(), want.cpu().numpy()
    (parity.tight if S <= 4 and not bias else parity.loose)(got, want, f"{M} x {N}, K {K}, {S} planes, groups of {G}")
    assert np.isfinite(got).all()
