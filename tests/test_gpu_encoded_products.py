"""The matrix-core product of two encoded operands, the dense weight back from an encoding, and activations encoded
from their input coefficients, each against the CPU oracle at the sizes where its tiling has edges."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _enc(rng, rows, K, S, G, L, oracle, scale=0.5):
    sel = rng.integers(0, 1 << S, size=rows * K).astype(np.int32)
    bvr = oracle.C.planes_to_default(oracle.C.sel_to_planes(sel, S, 32), rows, K)
    idx = rng.integers(0, L, size=(K // G, rows)).astype(np.uint8 if L <= 256 else np.uint16)
    return bvr, idx, (rng.standard_normal((L, S)) * scale).astype(np.float16)


def _dev(*arrays):
    return [torch.from_numpy(a).to("cuda:0") for a in arrays]


# (left row, plane) pairs on both sides of the 16-pair tiles and of the 64-pair workgroups; ragged N; one sub-group
# of K, fewer sub-groups than waves, several per wave; groups of one and of three sub-groups; and, on 256 CUs, every
# pair of row tiles and waves that the launch picks
@pytest.mark.parametrize("M,N,K,Sl,Sr,G,Ll,Lr", [
    (2, 1, 128, 8, 4, 128, 3, 9), (15, 17, 384, 1, 2, 384, 300, 7), (3, 100, 1024, 5, 3, 128, 9, 300),
    (4, 4100, 4096, 4, 4, 256, 16, 256), (5, 33, 2304, 7, 6, 128, 5, 70), (11, 250, 512, 6, 8, 256, 4, 5),
    (16, 520, 4352, 8, 4, 128, 40, 256), (17, 130, 2176, 8, 3, 128, 300, 16), (33, 64, 256, 4, 8, 128, 8, 8),
    (64, 1030, 1280, 8, 2, 128, 16, 700), (1, 300, 7168, 8, 4, 256, 28, 256), (1, 40, 256, 16, 4, 128, 2, 3),
    # four row tiles, eight waves, the last block of rows ragged
    (19, 4099, 256, 8, 3, 128, 5, 9), (19, 4099, 256, 8, 4, 128, 5, 9), (19, 4099, 384, 8, 6, 128, 5, 9), (19, 4099, 256, 8, 8, 256, 5, 9),
    (70, 4099, 256, 3, 4, 128, 5, 300),
    # two row tiles, sixteen waves: up to 32 pairs, and more of them where the columns are few
    (4, 4099, 256, 8, 3, 128, 5, 9), (5, 4099, 2304, 6, 8, 128, 5, 9), (17, 1000, 384, 8, 4, 128, 5, 9), (17, 1000, 256, 8, 6, 128, 5, 9),
    # two row tiles, eight waves
    (3, 8200, 256, 8, 4, 128, 5, 9), (3, 8200, 256, 8, 8, 128, 5, 9), (7, 8200, 384, 4, 6, 128, 5, 9), (7, 8200, 256, 4, 3, 128, 5, 300),
    # one row tile, eight waves
    (2, 8200, 256, 8, 4, 128, 5, 9), (2, 8200, 1408, 5, 6, 128, 5, 9)])
def test_mm_T_any_rows(oracle, M, N, K, Sl, Sr, G, Ll, Lr):
    import sbvr
    rng = np.random.default_rng(M * 1000 + N)
    left, right = _enc(rng, M, K, Sl, G, Ll, oracle), _enc(rng, N, K, Sr, G, Lr, oracle)
    bias = rng.standard_normal(N).astype(np.float16)
    none = torch.zeros(0, dtype=torch.float16, device="cuda:0")
    y = sbvr._sbvr_mm_T(*_dev(*left, *right), none, bvr_len=G).cpu().numpy()
    _, yd = oracle.C.mm_T(*left, *right, G)
    # exact popcounts and fp32 sums of K / 128 * Sl * Sr terms, then one rounding to fp16: within 2 fp16 ulps
    rms = float(np.sqrt(np.mean(yd ** 2)))
    assert (np.abs(y.astype(np.float64) - yd) / (np.maximum(np.abs(yd), rms) * 2.0 ** -10)).max() <= 2.0
    # the bias is added to the rounded sum
    yb = sbvr._sbvr_mm_T(*_dev(*left, *right, bias), bvr_len=G).cpu().numpy()
    assert np.array_equal(yb, (y.astype(np.float32) + bias.astype(np.float32)).astype(np.float16))


@pytest.mark.parametrize("N,K,S,G,L,cols,dtype", [
    (1, 32, 4, 32, 1, 32, torch.float16), (9, 288, 4, 96, 300, 288, torch.bfloat16), (7, 256, 3, 64, 5, 250, torch.float16),
    (65, 1280, 2, 256, 256, 1280, torch.float32), (130, 512, 3, 128, 700, 505, torch.float32), (40, 544, 6, 32, 17, 544, torch.float16),
    (24, 256, 8, 128, 256, 248, torch.bfloat16), (8, 256, 1, 256, 4, 256, torch.float16), (16, 2048, 4, 128, 256, 2048, torch.float64),
    (33, 64, 5, 64, 9, 64, torch.float16)])
def test_decode_weight(oracle, N, K, S, G, L, cols, dtype):
    import sbvr
    rng = np.random.default_rng(N * 100 + K)
    bvr, idx, cache = _enc(rng, N, K, S, G, L, oracle, 0.02)
    # coefficients that are multiples of 2^-14 below 2^-3: every fp32 sum is exact, whatever its order
    cache = (np.round(cache.astype(np.float64) * 2 ** 14) / 2 ** 14).astype(np.float16)
    obj = sbvr.sbvr.from_parts(*_dev(bvr, idx, cache), G, original_shape=(N, cols), original_dtype=dtype)
    got = obj.decode()
    want = torch.from_numpy(oracle.C.decode(bvr, idx, cache, G)[:, :cols].astype(np.float16)).to(dtype)
    assert got.shape == (N, cols) and got.dtype == dtype and torch.equal(got.cpu(), want)


def _dense(bvr, idx, cache, G, oracle):
    return torch.from_numpy(oracle.C.decode(bvr, idx, cache, G).astype(np.float16))


def test_decode_takes_every_form_it_took_on_the_cpu(oracle):
    """Strides, types and shapes beside those that the one launch reads: the same values as on the CPU, on the GPU."""
    import sbvr
    rng = np.random.default_rng(8)
    N, K, S, G, L = 6, 256, 4, 64, 9
    bvr, idx, cache = _enc(rng, N, K, S, G, L, oracle, 0.02)
    cache = (np.round(cache.astype(np.float64) * 2 ** 14) / 2 ** 14).astype(np.float16)
    want = _dense(bvr, idx, cache, G, oracle)
    db, di, dc = _dev(bvr, idx, cache)
    strided_idx = di.t().contiguous().t()
    strided_cache = torch.cat((dc, dc), dim=1)[:, :S]
    strided_bvr = torch.cat((db.view(torch.int32), db.view(torch.int32)), dim=2)[:, :, :S].view(torch.uint32)
    assert not (strided_idx.is_contiguous() or strided_cache.is_contiguous() or strided_bvr.is_contiguous())
    for b, i, c in ((db, di, dc), (db, strided_idx, dc), (db, di, strided_cache), (strided_bvr, di, dc), (db, di.to(torch.int64), dc),
                    (db, di.to(torch.int32), dc), (db, di, dc.float()), (db, di, dc.double())):
        got = sbvr.sbvr.from_parts(b, i, c, G).decode()
        assert got.dtype == torch.float16 and torch.equal(got.cpu(), want), (i.dtype, i.stride(), c.dtype, c.stride(), b.stride())
    # leading dimensions; no rows
    assert torch.equal(sbvr.sbvr.from_parts(db, di, dc, G, original_shape=(2, 3, K)).decode().cpu(), want.view(2, 3, K))
    assert torch.equal(sbvr.sbvr.from_parts(db[:, :1].contiguous(), di[:, :1].contiguous(), dc, G, original_shape=(K - 5,)).decode().cpu(),
                       want[0, :K - 5])
    empty = sbvr.sbvr.from_parts(db[:, :0].contiguous(), di[:, :0].contiguous(), dc, G).decode()
    assert empty.shape == (0, K) and empty.dtype == torch.float16


@pytest.mark.parametrize("S,L,dtype", [(2, 5, torch.float16), (3, 300, torch.bfloat16), (4, 16, torch.float32), (6, 17, torch.float16)])
def test_decode_shows_an_index_beyond_the_table(oracle, S, L, dtype):
    """A group whose index is not below the number of lines decodes to NaN, and nothing else does."""
    import sbvr
    rng = np.random.default_rng(S)
    N, K, G = 11, 512, 64
    bvr, idx, cache = _enc(rng, N, K, S, G, L, oracle, 0.02)
    cache = (np.round(cache.astype(np.float64) * 2 ** 14) / 2 ** 14).astype(np.float16)
    bad = rng.random(idx.shape) < 0.3
    bad[0, 0] = True
    marked = np.where(bad, L + rng.integers(0, 200, size=idx.shape), idx).astype(idx.dtype)
    got = sbvr.sbvr.from_parts(*_dev(bvr, marked, cache), G, original_dtype=dtype).decode().cpu()
    want = _dense(bvr, idx, cache, G, oracle).to(dtype)
    want[torch.from_numpy(np.repeat(bad.T, G, axis=1))] = float("nan")
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize("S,dtype", [(2, torch.float16), (3, torch.float32), (4, torch.bfloat16), (4, torch.float16), (1, torch.float16),
                                     (6, torch.float16)])
def test_decode_of_coefficients_that_are_not_finite(oracle, S, dtype):
    """Infinite and NaN coefficients, one and several of a line, and sums beyond fp16: as the torch expressions give
    them on the CPU (a coefficient counts as 0 * c where its bit is not set)."""
    import sbvr
    rng = np.random.default_rng(20 + S)
    N, K, G, L = 19, 512, 32, 12
    bvr, idx, cache = _enc(rng, N, K, S, G, L, oracle, 1.0)
    cache = (np.round(cache.astype(np.float64) * 2 ** 8) / 2 ** 8).astype(np.float16)
    cache[0, 0] = cache[1, S - 1] = np.inf
    cache[2, 0] = -np.inf
    cache[3, S // 2] = np.nan
    cache[4, 0], cache[4, S - 1] = np.inf, -np.inf
    cache[5] = np.inf
    cache[6] = 60000.0
    parts = [torch.from_numpy(a) for a in (bvr, idx, cache)]
    want = sbvr.sbvr.from_parts(*parts, G, original_dtype=dtype).decode()
    got = sbvr.sbvr.from_parts(*(p.to("cuda:0") for p in parts), G, original_dtype=dtype).decode().cpu()
    assert want.isnan().any() and want.isinf().any() and want.isfinite().any()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[~want.isnan()], want[~want.isnan()])


@pytest.mark.parametrize("shape", [(6, 100), (5, 256), (7, 256), (6, 512)])
def test_decode_refuses_a_shape_that_is_not_the_arrays(oracle, shape):
    """A shape that does not pad to the rows and columns of the arrays is an error, not a part of them."""
    import sbvr
    arrays = _dev(*_enc(np.random.default_rng(9), 6, 256, 4, 64, 9, oracle))
    with pytest.raises(RuntimeError):
        sbvr.sbvr.from_parts(*arrays, 64, original_shape=shape).decode()


@pytest.mark.parametrize("S,G,M,K", [(2, 32, 1, 32), (4, 96, 5, 288), (8, 128, 3, 512), (8, 256, 4, 67072), (1, 64, 9, 64)])
def test_online_encode_lines(S, G, M, K):
    """The same planes as from the table of subset sums, and every group's own number as its line."""
    from sbvr import hip, layout
    gen = torch.Generator().manual_seed(K + S)
    x = torch.randn((M, K), generator=gen).to(torch.float16).to("cuda:0")
    lines = (torch.randint(-1000, 1000, (K // G, S), generator=gen) / 512).to(torch.float16).to("cuda:0")
    points = (lines.float() @ layout.bin_combs(S, torch.float32, "cuda:0").T).to(torch.float16)   # (exact sums)
    bvr, idx = hip.online_encode_lines(x, lines, G)
    assert torch.equal(bvr.view(torch.int32), hip.online_encode(x, points, G).view(torch.int32))
    assert idx.dtype == (torch.uint8 if K // G <= 256 else torch.uint16)
    assert torch.equal(idx.to(torch.int64), torch.arange(K // G, device="cuda:0").view(-1, 1).expand(-1, M))


@pytest.mark.parametrize("N,K,Sl,Sr,decode_kernel", [
    (512, 14336, 4, 4, True), (600, 4096, 2, 3, True), (1024, 14336, 1, 8, True), (2048, 2048, 3, 3, True),     # few columns, long K
    (4112, 1024, 4, 4, True), (8192, 4096, 2, 2, True), (8200, 14336, 4, 6, True),                              # more columns than CUs x 16
    (4096, 1024, 1, 3, False), (640, 2048, 4, 2, False), (4096, 4096, 2, 8, False), (3072, 10240, 4, 4, False)])
def test_one_left_row_takes_the_kernel_that_is_faster_for_it(oracle, N, K, Sl, Sr, decode_kernel):
    """One left row of up to four planes: where the columns leave the chip idle or outnumber its workgroups the decode
    kernel (which splits K), otherwise the one that does not; the same bits on every call, the accumulators zero again."""
    import sbvr
    from sbvr import hip
    dev = torch.device("cuda:0")
    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        pytest.skip("the rule's columns are those of 256 CUs")
    rng = np.random.default_rng(N + K)
    left, right = _enc(rng, 1, K, Sl, 128, 16, oracle), _enc(rng, N, K, Sr, 128, 256, oracle)
    none = torch.zeros(0, dtype=torch.float16, device=dev)
    # (a launch of another kernel first: the report is of the last launch that makes one)
    w, wi, wc = _dev(*_enc(rng, 64, 256, 4, 128, 16, oracle))
    sbvr._sbvr_linear_f16(torch.zeros((40, 256), dtype=torch.float16, device=dev), w, wi, wc)
    assert hip.last_kernel() != hip.KERNEL_DECODE
    d = _dev(*left, *right)
    y = sbvr._sbvr_mm_T(*d, none, bvr_len=128)
    assert (hip.last_kernel() == hip.KERNEL_DECODE) == decode_kernel
    _, yd = oracle.C.mm_T(*left, *right, 128)
    rms = float(np.sqrt(np.mean(yd ** 2)))
    assert (np.abs(y.cpu().numpy().astype(np.float64) - yd) / (np.maximum(np.abs(yd), rms) * 2.0 ** -10)).max() <= 2.0
    for _ in range(3):                 # (words that a launch left behind would be in the next one's sums)
        assert torch.equal(y, sbvr._sbvr_mm_T(*d, none, bvr_len=128))


@pytest.mark.parametrize("M", [262140, 262141])
def test_left_rows_beyond_the_grid_go_on_to_the_portable_kernel(oracle, M):
    """16 left planes: 65535 blocks of four rows still fit the grid of the matrix-core kernel, one row more does not."""
    import sbvr
    K, N, Sl, Sr = 128, 16, 16, 2
    rng = np.random.default_rng(M)
    lb = rng.integers(0, 1 << 32, size=(K // 32, M, Sl), dtype=np.uint32)
    li = rng.integers(0, 5, size=(1, M)).astype(np.uint8)
    lc = (rng.standard_normal((5, Sl)) * 0.05).astype(np.float16)
    right = _enc(rng, N, K, Sr, 128, 7, oracle)
    none = torch.zeros(0, dtype=torch.float16, device="cuda:0")
    y = sbvr._sbvr_mm_T(*_dev(lb, li, lc, *right), none, bvr_len=128).cpu().numpy()
    some = np.r_[0:40, M // 2:M // 2 + 40, M - 40:M]
    _, yd = oracle.C.mm_T(np.ascontiguousarray(lb[:, some]), np.ascontiguousarray(li[:, some]), lc, *right, 128)
    rms = float(np.sqrt(np.mean(yd ** 2)))
    assert (np.abs(y[some].astype(np.float64) - yd) / (np.maximum(np.abs(yd), rms) * 2.0 ** -10)).max() <= 2.0
