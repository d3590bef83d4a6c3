"""Prefill with five to eight row blocks a workgroup (prefill_ops.hip) where its steps, tiles and stores end: odd numbers of
steps, one and two of them, columns and rows that are no multiple of anything, K in parts, groups of 64, all plane counts.  Shapes
with tiles for most of the chip, which is where the plan takes that many row blocks."""
import numpy as np
import pytest
import torch

import parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,S,G,L,bias,kernel", [
    (512, 28672, 64, 4, 64, 256, False, 4),            # one step
    (500, 28001, 128, 4, 128, 256, True, 4),           # two, odd width
    (481, 28665, 192, 4, 64, 300, False, 4),           # three: no second of a pair
    (300, 28672, 448, 3, 64, 256, True, 4),            # five row blocks, seven steps
    (380, 28679, 512, 2, 256, 16, False, 4),           # six
    (430, 28610, 256, 4, 128, 768, True, 4),           # seven, uint16 indices
    (700, 28417, 320, 6, 64, 256, False, 4),
    (512, 28433, 384, 8, 128, 256, True, 4),
    (512, 28672, 320, 8, 64, 256, False, 4),
    (1458, 3075, 12800, 8, 256, 256, True, 5),         # K in parts, fp32 partial results at an odd width
    (1983, 1644, 2816, 8, 64, 256, False, 5),          # seven row blocks
    (1388, 2144, 4608, 4, 64, 256, False, 5),          # five
    (403, 16386, 12544, 4, 256, 256, False, 5),        # parts that begin inside a group
    (700, 5100, 11008, 3, 128, 256, False, 5),         # the last part shorter, three and two planes
    (1400, 2050, 12288, 2, 64, 256, True, 5),
    (400, 9000, 10240, 6, 128, 256, False, 5),
    (2048, 1001, 8192, 4, 128, 256, True, 5),          # (parts of three and four row blocks, which sbvr_hip.hip's kernel takes)
    (1009, 2050, 6144, 3, 256, 256, False, 5),
    (1300, 1025, 5376, 2, 64, 256, False, 5),
])
def test_where_steps_and_tiles_end(M, N, K, S, G, L, bias, kernel):
    """Against the products with decode()'s weights in 64 bits: what tests/parity.py allows fp16 results of fp32 sums."""
    import sbvr
    from sbvr import hip, synth
    dev = torch.device("cuda:0")
    bvr, idx, cache = (t.to(dev) for t in synth.random_encoding(N, K, S, G, L, seed=N + K))
    gen = torch.Generator().manual_seed(M)
    x = torch.randn((M, K), generator=gen).to(torch.float16).to(dev)
    b = (torch.randn(N, generator=gen) * 0.3).to(torch.float16).to(dev) if bias else None
    y = sbvr._sbvr_linear_f16(x, bvr, idx, cache, b, bvr_len=G)
    assert hip.last_kernel() == kernel
    assert (hip.last_row_blocks() >= 5) == ((M, N) not in ((2048, 1001), (1009, 2050), (1300, 1025)))
    assert torch.equal(y, sbvr._sbvr_linear_f16(x, bvr, idx, cache, b, bvr_len=G))
    weight = sbvr.sbvr.from_parts(bvr, idx, cache, G).decode()
    want = x.double() @ weight.double().t()
    if bias:
        want += b.double()
    got, want = y.double().cpu().numpy(), want.cpu().numpy()
    (parity.tight if S <= 4 and not bias else parity.loose)(got, want, f"{M} x {N}, K {K}, {S} planes, groups of {G}")
    assert np.isfinite(got).all()
