"""decode() whatever the number of workgroups, which are dealt out in eight runs: fewer than eight, no multiple of it, several along
K, ragged edges."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,S,G", [
    (8, 64, 4, 64), (49, 256, 2, 256), (64, 1024, 3, 128), (100, 1280, 4, 256), (1000, 3072, 4, 128), (333, 2048, 8, 64),
    (2056, 1088, 2, 64), (17, 9216, 3, 128), (77, 1280, 6, 128),
])
def test_every_workgroup_finds_its_weights(N, K, S, G):
    """Bit for bit the subset sums in fp32, plane by plane, rounded once."""
    import sbvr
    from sbvr import synth
    bvr, idx, cache = synth.random_encoding(N, K, S, G, 256, seed=N + K)
    got = sbvr.sbvr.from_parts(*(t.to("cuda:0") for t in (bvr, idx, cache)), G).decode().cpu().numpy()
    assert np.array_equal(got.view(np.uint16), _sums(bvr, idx, cache, N, K, S, G).view(np.uint16))


@pytest.mark.parametrize("S", [5, 6, 7, 8])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_more_planes_whatever_the_coefficients(S, dtype):
    """Columns whose coefficients lie near each other (sums of them are exact in fp32), ten and eleven binades apart, further,
    subnormal, zero and not finite, in waves of their own and mixed: the same fp32 sums, their order showing where it counts."""
    import sbvr
    from sbvr import synth
    N, K, G, L = 264, 512, 64, 256
    bvr, idx, cache = synth.random_encoding(N, K, S, G, L, seed=S)
    gen = torch.Generator().manual_seed(S)
    lines = torch.randn((L, S), generator=gen) * 0.02
    lines[0] = torch.exp2(torch.arange(S) % 2 * 10.0 - 6) * (1 + torch.rand(S, generator=gen))       # 10 binades
    lines[1] = torch.exp2(torch.arange(S) % 2 * 11.0 - 6) * (1 + torch.rand(S, generator=gen))
    lines[2] = torch.exp2(torch.linspace(-14, 15, S)) * (1 + torch.rand(S, generator=gen) * 0.9) * (torch.randint(0, 2, (S,), generator=gen) * 2 - 1)
    lines[3] = torch.exp2(torch.linspace(-24, -15, S))
    lines[4], lines[5, 0], lines[6, S - 1], lines[7, 1], lines[8] = 0.0, float("inf"), float("nan"), 0.0, 60000.0
    lines[9, 2] = -0.0
    cache = lines.to(torch.float16)
    which = torch.randint(0, 10, idx.shape, generator=gen)
    which[:, :80] = torch.arange(80)[None, :] // 8                   # (eight columns to a wave)
    which[:, 80:160] = torch.randint(10, L, (idx.shape[0], 80), generator=gen)
    idx = which.to(torch.uint8)
    enc = sbvr.sbvr.from_parts(*(t.to("cuda:0") for t in (bvr, idx, cache)), G)
    enc.original_dtype = dtype
    got = enc.decode().cpu()
    want = torch.from_numpy(_sums(bvr, idx, cache, N, K, S, G)).to(dtype)
    assert got.dtype == dtype and torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.nan_to_num(got.float(), 0.5, 1e9, -1e9), torch.nan_to_num(want.float(), 0.5, 1e9, -1e9))


def _sums(bvr, idx, cache, N, K, S, G):
    bits = (bvr.numpy()[:, None] >> np.arange(32, dtype=np.uint32)[None, :, None, None]) & 1              # (K/32, 32, N, S)
    line = np.repeat(cache.numpy().astype(np.float32)[idx.numpy().astype(np.int64)], G, axis=0).reshape(K // 32, 32, N, S)
    want = np.zeros(line.shape[:3], np.float32)
    with np.errstate(invalid="ignore", over="ignore"):
        for q in range(S):
            want += bits[..., q].astype(np.float32) * line[..., q]
        return np.ascontiguousarray(want.reshape(K, N).T.astype(np.float16))
