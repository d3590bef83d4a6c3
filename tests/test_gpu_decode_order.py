"""decode() whatever the number of workgroups, which are dealt out in eight runs: fewer than eight, no multiple of it, several along
K, ragged edges."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,S,G", [
    (8, 64, 4, 64), (49, 256, 2, 256), (64, 1024, 3, 128), (100, 1280, 4, 256), (1000, 3072, 4, 128), (333, 2048, 8, 64),
    (2056, 1088, 2, 64), (17, 9216, 3, 128),
])
def test_every_workgroup_finds_its_weights(N, K, S, G):
    """Bit for bit the subset sums in fp32, plane by plane, rounded once."""
    import sbvr
    from sbvr import synth
    bvr, idx, cache = synth.random_encoding(N, K, S, G, 256, seed=N + K)
    got = sbvr.sbvr.from_parts(*(t.to("cuda:0") for t in (bvr, idx, cache)), G).decode().cpu().numpy()
    bits = (bvr.numpy()[:, None] >> np.arange(32, dtype=np.uint32)[None, :, None, None]) & 1              # (K/32, 32, N, S)
    line = np.repeat(cache.numpy().astype(np.float32)[idx.numpy().astype(np.int64)], G, axis=0).reshape(K // 32, 32, N, S)
    want = np.zeros(line.shape[:3], np.float32)
    for q in range(S):
        want += np.where(bits[..., q] != 0, line[..., q], np.float32(0))
    want = want.reshape(K, N).T.astype(np.float16)
    assert np.array_equal(got.view(np.uint16), np.ascontiguousarray(want).view(np.uint16))
