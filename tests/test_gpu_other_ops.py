"""GPU parity of the reference-compatible alternates (both-encoded _sbvr_mm_T and
the trans=True _sbvr_row_deq_mm_T) and of SBVRLinear, against the CPU oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand_enc(rng, rows, K, S, G, L, oracle):
    sel = rng.integers(0, 1 << S, size=rows * K).astype(np.int32)
    bvr = oracle.C.planes_to_default(oracle.C.sel_to_planes(sel, S, 32), rows, K)
    idx = rng.integers(0, L, size=(K // G, rows)).astype(np.uint8 if L <= 256 else np.uint16)
    cache = (rng.standard_normal((L, S)) * 0.5).astype(np.float16)
    return bvr, idx, cache


def _close(y, yd, ulps=2.0):
    got = y.float().cpu().numpy().astype(np.float64)
    rms = float(np.sqrt(np.mean(yd ** 2))) + 1e-30
    assert (np.abs(got - yd) / np.maximum(np.abs(yd), 1e-2 * rms)).max() <= 1e-2
    assert (np.abs(got - yd) / (np.maximum(np.abs(yd), rms) * 2.0 ** -10)).max() <= ulps


@pytest.mark.parametrize("M,N,K,Sl,Sr,G,Ll,Lr", [(1, 64, 512, 4, 4, 256, 5, 9), (3, 40, 256, 2, 3, 128, 300, 7),
                                                 (2, 33, 512, 8, 6, 256, 4, 400),       # no popcount-kernel instance
                                                 (1, 1000, 160, 4, 4, 32, 16, 256),     # 5 words: a partial chunk
                                                 (1, 130, 4096, 4, 2, 64, 16, 300),     # 16 chunks, uint16 right index
                                                 (2, 200, 14336, 3, 4, 128, 16, 256),   # 7 chunks per wave
                                                 (1, 96, 512, 4, 4, 512, 8, 8),         # group longer than a chunk
                                                 # one left row of up to 4 planes at the decode kernel's shapes: the
                                                 # left planes are that kernel's batch rows
                                                 (1, 256, 1024, 4, 4, 128, 16, 256), (1, 1030, 2048, 3, 4, 128, 300, 300),
                                                 (1, 48, 512, 2, 3, 256, 7, 9), (1, 4096, 4096, 4, 4, 128, 16, 256),
                                                 (1, 14336, 4096, 4, 4, 128, 16, 256), (1, 1000, 1024, 1, 8, 128, 5, 40),
                                                 (1, 4096, 14336, 4, 4, 128, 16, 256),  # K split across workgroups
                                                 (1, 2048, 7168, 4, 2, 256, 16, 300), (1, 512, 4096, 4, 6, 128, 9, 256),
                                                 (1, 8192, 1024, 4, 2, 128, 16, 256), (1, 8200, 1024, 3, 3, 128, 16, 300),
                                                 (1, 8192, 2048, 2, 6, 256, 16, 256), (1, 9000, 1024, 4, 8, 128, 16, 256),
                                                 # groups of 32 and 64: the popcount kernel, by planes
                                                 (2, 100, 256, 2, 3, 32, 16, 256), (5, 130, 320, 3, 2, 64, 300, 9),
                                                 (1, 70, 512, 2, 4, 32, 9, 300), (3, 200, 192, 3, 3, 32, 9, 9),
                                                 (64, 33, 128, 2, 2, 64, 9, 9), (65, 33, 128, 3, 4, 64, 9, 9)])
def test_mm_T(oracle, M, N, K, Sl, Sr, G, Ll, Lr):
    import sbvr
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(M * 100 + N)
    lb, li, lc = _rand_enc(rng, M, K, Sl, G, Ll, oracle)
    rb, ri, rc = _rand_enc(rng, N, K, Sr, G, Lr, oracle)
    t = lambda a: torch.from_numpy(a).to(dev)
    y = sbvr._sbvr_mm_T(t(lb), t(li), t(lc), t(rb), t(ri), t(rc), torch.zeros(0, dtype=torch.float16, device=dev),
                        bvr_len=G)
    _, yd = oracle.C.mm_T(lb, li, lc, rb, ri, rc, G)
    _close(y, yd)
    bias = (rng.standard_normal(N)).astype(np.float16)
    yb = sbvr._sbvr_mm_T(t(lb), t(li), t(lc), t(rb), t(ri), t(rc), t(bias), bvr_len=G)
    want, _ = oracle.C.mm_T(lb, li, lc, rb, ri, rc, G, bias)
    d = np.abs(yb.float().cpu().numpy().astype(np.float64) - want.astype(np.float64))
    assert d.max() <= 2.0 ** -9 * max(np.abs(want.astype(np.float64)).max(), 1.0)


def test_mm_T_without_workspace_and_repeatable(oracle):
    """The reference-shaped entry point (no workspace) at a shape whose decode launch splits K across workgroups: it
    must still answer (through the matrix-core kernel, which does not split); and the split form, bit for bit on every
    call, its accumulators zero again."""
    import ctypes
    import sbvr
    from sbvr import hip
    dev = torch.device("cuda:0")
    M, N, K, S, G, L = 1, 4096, 14336, 4, 128, 256
    rng = np.random.default_rng(11)
    lb, li, lc = _rand_enc(rng, M, K, S, G, 16, oracle)
    rb, ri, rc_ = _rand_enc(rng, N, K, S, G, L, oracle)
    t = lambda a: torch.from_numpy(a).to(dev)
    d = [t(a) for a in (lb, li, lc, rb, ri, rc_)]
    out = torch.empty((M, N), dtype=torch.float16, device=dev)
    lib = hip._load()
    vp = ctypes.c_void_p
    rc = lib.sbvr_hip_mm_T(vp(d[0].data_ptr()), vp(d[1].data_ptr()), 1, vp(d[2].data_ptr()), vp(d[3].data_ptr()),
                           vp(d[4].data_ptr()), 1, vp(d[5].data_ptr()), None, vp(out.data_ptr()), M, N, K, S, S, G, 16, L,
                           vp(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    _, yd = oracle.C.mm_T(lb, li, lc, rb, ri, rc_, G)
    _close(out, yd)
    none = torch.zeros(0, dtype=torch.float16, device=dev)
    plan = (ctypes.c_int * 8)()
    assert lib.sbvr_hip_decode_plan(S, N, K, S, G, torch.cuda.get_device_properties(dev).multi_processor_count, plan) == 0
    assert plan[0] == 1 and plan[6] > 1                      # the left planes as four rows, K in parts
    first = sbvr._sbvr_mm_T(*d, none, bvr_len=G)
    assert hip.last_kernel() == hip.KERNEL_DECODE
    _close(first, yd)
    for _ in range(4):
        again = sbvr._sbvr_mm_T(*d, none, bvr_len=G)
        assert torch.equal(first, again)
    assert int(hip._workspace(8 * N, dev).count_nonzero()) == 0


def test_mm_T_with_a_table_of_less_alignment(oracle):
    """A right table that is not 16-byte aligned (a slice of a longer one): the popcount kernel at groups of 128 and
    256, and the portable one beyond its planes."""
    import sbvr
    dev = torch.device("cuda:0")
    for M, N, K, Sl, Sr, G in ((2, 130, 1024, 4, 4, 128), (1, 70, 512, 3, 2, 256), (3, 65, 256, 2, 3, 128), (2, 40, 256, 8, 4, 128)):
        rng = np.random.default_rng(N)
        left, right = _rand_enc(rng, M, K, Sl, G, 9, oracle), _rand_enc(rng, N, K, Sr, G, 30, oracle)
        d = [torch.from_numpy(a).to(dev) for a in (*left, *right)]
        d[5] = torch.cat((d[5][:1], d[5]))[1:]
        assert d[5].is_contiguous() and d[5].data_ptr() % 16 != 0
        y = sbvr._sbvr_mm_T(*d, torch.zeros(0, dtype=torch.float16, device=dev), bvr_len=G)
        _, yd = oracle.C.mm_T(*left, *right, G)
        _close(y, yd)


def test_mm_T_object_api(oracle, golden):
    """sbvr.mm_T(lhs, rhs, bias) on objects built from the reference's encodings."""
    import sbvr
    dev = torch.device("cuda:0")
    g = golden("default_s2")
    mk = lambda: sbvr.sbvr.from_parts(*(torch.from_numpy(g[k]).to(dev) for k in ("bvr", "coeff_idx", "coeff_cache")), 256)
    a, b = mk(), mk()
    y = sbvr.mm_T(a, b, None)
    _, yd = oracle.C.mm_T(g["bvr"], g["coeff_idx"], g["coeff_cache"], g["bvr"], g["coeff_idx"], g["coeff_cache"], 256)
    _close(y, yd)
    w = g["decoded"].astype(np.float64)
    assert np.abs(y.float().cpu().numpy() - w @ w.T).max() <= 1e-2 * np.abs(w @ w.T).max()


@pytest.mark.parametrize("M,N,K,S,G,L", [(1, 256, 64, 4, 256, 9), (2, 512, 40, 2, 128, 300),
                                         (3, 1024, 4096, 4, 128, 256), (1, 96, 1000, 3, 32, 700),
                                         (5, 64, 130, 8, 64, 40), (1, 4096, 2048, 6, 128, 256),
                                         (2, 14336, 512, 4, 128, 256), (1, 32, 1, 4, 32, 2),
                                         # four planes, K a multiple of 128, groups of 64 columns and more: the MFMA form
                                         (1, 64, 128, 4, 64, 5), (4, 256, 640, 4, 64, 300), (2, 192, 256, 4, 192, 9),
                                         (1, 14336, 4096, 4, 128, 256), (1, 4096, 14336, 4, 256, 256)])
def test_row_deq_mm_T(oracle, M, N, K, S, G, L):
    import sbvr
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(N + K)
    # the encoded tensor is W^T: K rows of N columns, groups along N
    bvr, idx, cache = _rand_enc(rng, K, N, S, G, L, oracle)         # (N/32, K, S), (N/G, K)
    x = rng.standard_normal((M, K)).astype(np.float16)
    bias = rng.standard_normal(N).astype(np.float16)
    t = lambda a: torch.from_numpy(a).to(dev)
    y = sbvr._sbvr_row_deq_mm_T(t(x), t(bvr), t(idx), t(cache), t(bias), 0, bvr_len=G)
    want = oracle.C.row_deq_mm_T(x, bvr, idx, cache, G, bias).astype(np.float64)
    d = np.abs(y.float().cpu().numpy().astype(np.float64) - want)
    assert d.max() <= 2.0 ** -9 * max(np.abs(want).max(), 1.0)


@pytest.mark.parametrize("M,N,K,S,G,L,bias", [
    (2, 8192, 705, 4, 64, 300, True),           # the last tile has 65 rows, K odd
    (33, 512, 1, 3, 32, 9, False),              # (short K on few columns: the one-row kernels)
    (32, 544, 127, 2, 32, 256, False),
    (17, 1024, 129, 4, 256, 40, True),
    (33, 14336, 1, 3, 32, 9, False),            # one row of the weight, two blocks of batch rows
    (32, 14336, 127, 2, 32, 256, False),        # one tile, one row short
    (17, 8192, 129, 4, 256, 40, True),          # a second tile with one row
    (3, 4096, 4096, 4, 256, 256, False),        # K in parts
    (8, 512, 4143, 2, 256, 768, True),          # K in parts of different lengths, uint16 indices
    (65, 256, 1001, 4, 128, 256, False),        # three blocks of batch rows
])
def test_row_deq_mm_T_of_several_rows(oracle, M, N, K, S, G, L, bias):
    """Every weight decoded once for all rows, as two fp16 values: within 2 fp16 ulps of the sums in 64 bits (the fp32 additions
    and one rounding), the same bits on a second call, the accumulators left zero."""
    import sbvr
    from sbvr import hip
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(N + K)
    bvr, idx, cache = _rand_enc(rng, K, N, S, G, L, oracle)
    x = rng.standard_normal((M, K)).astype(np.float16)
    b = rng.standard_normal(N).astype(np.float16) if bias else np.zeros(0, np.float16)
    args = [torch.from_numpy(a).to(dev) for a in (x, bvr, idx, cache, b)]
    y = sbvr._sbvr_row_deq_mm_T(*args, 0, bvr_len=G)
    assert hip.row_deq_last()[0] == (hip.ROW_DEQ_LANES if K <= 129 and N <= 1024 else hip.ROW_DEQ_ROWS)
    assert torch.equal(y, sbvr._sbvr_row_deq_mm_T(*args, 0, bvr_len=G))
    bits = (bvr[:, :, None, :] >> np.arange(32, dtype=np.uint32)[None, None, :, None]) & 1          # (N/32, K, 32, S)
    line = cache.astype(np.float64)[idx.astype(np.int64)]                                          # (N/G, K, S)
    w = np.einsum("nkbs,nks->nkb", bits.astype(np.float64), np.repeat(line, G // 32, axis=0))
    want = x.astype(np.float64) @ w.transpose(1, 0, 2).reshape(K, N) + (b.astype(np.float64) if bias else 0.0)
    rms = np.sqrt(np.mean(want ** 2))
    err = np.abs(y.float().cpu().numpy() - want) / (np.maximum(np.abs(want), rms) * 2.0 ** -10)
    assert err.max() <= 2.0, err.max()
    assert int(hip._workspace(8 * M * N, dev).count_nonzero()) == 0


@pytest.mark.parametrize("N,K,S,G", [(2048, 800, 2, 128), (4096, 4100, 4, 128), (2048, 12032, 3, 256)])
def test_row_deq_mm_T_of_several_rows_is_as_exact_as_fp32_sums(N, K, S, G):
    """The sums before their rounding to fp16: a bias takes all but a rounding's remainder away, and of the columns those count
    whose remainder is so small (2^-14 of the RMS output) that its own rounding, 2^-25, does not show.  Several rows, K in parts
    or not, against the row by itself on the lanes launch: exact products, added up in fp32."""
    import sbvr
    from sbvr import hip, synth
    dev = torch.device("cuda:0")
    bvr, idx, cache = synth.random_encoding(K, N, S, G, 256, seed=N + K)
    x = torch.randn((1, K), generator=torch.Generator().manual_seed(K)).to(torch.float16)
    want = _transposed_sums(x.numpy(), bvr.numpy(), idx.numpy(), cache.numpy(), G)[0][0]
    bias = (-want).astype(np.float16)
    rest, rms = want + bias.astype(np.float64), np.sqrt(np.mean(want ** 2))
    near = np.abs(rest) < 2.0 ** -14 * rms
    assert near.sum() > 200
    args = [t.to(dev) for t in (bvr, idx, cache, torch.from_numpy(bias))]
    error = {}
    for M in (1, 5):
        y = sbvr._sbvr_row_deq_mm_T(x.to(dev).repeat(M, 1), *args, 0, bvr_len=G).float().cpu().numpy().astype(np.float64)
        assert hip.row_deq_last()[0] == (hip.ROW_DEQ_LANES if M == 1 else hip.ROW_DEQ_ROWS)
        error[M] = np.sqrt(np.mean((y - rest)[:, near] ** 2))
    assert error[5] <= error[1], (error[5] / rms, error[1] / rms)


def test_row_deq_mm_T_of_several_rows_with_values_that_are_not_finite(oracle):
    """Infinite and NaN activations, an infinite coefficient and a weight beyond fp16 in the launch of several rows: every
    output is finite, infinite or NaN as in the launch of that row by itself, and the finite ones agree."""
    import sbvr
    dev = torch.device("cuda:0")
    M, N, K, S, G, L = 5, 8192, 790, 3, 128, 40
    rng = np.random.default_rng(12)
    bvr, idx, cache = _rand_enc(rng, K, N, S, G, L, oracle)
    cache[7, 1] = np.inf
    cache[9] = [60000, 40000, 50000]
    x = (rng.standard_normal((M, K)) * 0.01).astype(np.float16)
    x[0, 3], x[1, 789], x[2, 300], x[2, 301] = np.inf, -np.inf, np.nan, np.inf
    idx[:, 3] = idx[:, 300:302] = 0
    idx[:, 5:] = np.where(np.isin(idx[:, 5:], (7, 9)) & (rng.random(idx[:, 5:].shape) < 0.98), 1, idx[:, 5:])
    args = [torch.from_numpy(a).to(dev) for a in (bvr, idx, cache)]
    none = torch.zeros(0, dtype=torch.float16, device=dev)
    y = sbvr._sbvr_row_deq_mm_T(torch.from_numpy(x).to(dev), *args, none, 0, bvr_len=G).float().cpu().numpy()
    one = np.concatenate([sbvr._sbvr_row_deq_mm_T(torch.from_numpy(x[m:m + 1]).to(dev), *args, none, 0, bvr_len=G).float().cpu().numpy()
                          for m in range(M)])
    assert np.array_equal(np.isnan(y), np.isnan(one)) and np.array_equal(np.isposinf(y), np.isposinf(one))
    assert np.array_equal(np.isneginf(y), np.isneginf(one))
    finite = np.isfinite(one)
    assert 0 < finite.sum() < finite.size
    scale = np.sqrt(np.mean(one[finite].astype(np.float64) ** 2))
    assert (np.abs(y[finite] - one[finite]) <= 2.0 ** -9 * np.maximum(np.abs(one[finite]), scale)).all()


def _transposed_sums(x, bvr, idx, cache, G):
    """Per output the sum in 64 bits of the selected coefficients alone, and the largest magnitude its fp32 partial sums can
    reach (of the finite terms)."""
    bits = ((bvr[:, :, None, :] >> np.arange(32, dtype=np.uint32)[None, None, :, None]) & 1).astype(bool)   # (N/32, K, 32, S)
    line = np.repeat(cache.astype(np.float64)[idx.astype(np.int64)], G // 32, axis=0)                      # (N/32, K, S)
    out = np.zeros((x.shape[0], bvr.shape[0] * 32))
    peak = np.zeros_like(out)
    with np.errstate(invalid="ignore"):
        for m in range(x.shape[0]):
            z = np.where(bits, (x[m].astype(np.float64)[None, :, None] * line)[:, :, None, :], 0.0)
            out[m] = z.sum(axis=(1, 3)).ravel()
            peak[m] = np.where(np.isfinite(z), np.abs(z), 0.0).sum(axis=(1, 3)).ravel()
    return out, peak


def _same_class_and_close(y, want, peak):
    """NaN, +inf and -inf where the sums in 64 bits have them (beyond fp16: infinite), finite values within 2 fp16 ulps
    and the fp32 rounding inside parts that the accumulators hold (two of up to 130000; eight MFMAs a tile, four tiles and four waves
    a part at most, 36 roundings and the last one's; an output with larger parts is summed in 64 bits)."""
    want = np.where(np.abs(want) >= 65520.0, np.sign(want) * np.inf, want)
    assert np.array_equal(np.isnan(y), np.isnan(want))
    assert np.array_equal(np.isposinf(y), np.isposinf(want)) and np.array_equal(np.isneginf(y), np.isneginf(want))
    finite = np.isfinite(want)
    rms = np.sqrt(np.mean(want[finite] ** 2))
    bound = 2.0 ** -9 * np.maximum(np.abs(want), min(rms, 10.0)) + 40 * 2.0 ** -24 * np.minimum(peak, 260000.0)
    assert (np.abs(y[finite] - want[finite]) <= bound[finite]).all()
    return finite


@pytest.mark.parametrize("M,N,K,S,G,L", [(8, 2048, 4096, 4, 256, 256), (8, 512, 4143, 2, 256, 768), (7, 1024, 2100, 3, 32, 40)])
def test_row_deq_mm_T_with_values_that_the_accumulators_cannot_hold(oracle, M, N, K, S, G, L):
    """K in parts: NaN, infinities of one and of both signs in different parts, partial sums beyond the fixed point's range
    that cancel and that do not, an infinite coefficient."""
    import sbvr
    from sbvr import hip
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(N + K)
    bvr, idx, cache = _rand_enc(rng, K, N, S, G, L, oracle)
    cache[7 % L] = [8] * S
    cache[9 % L, S - 1] = np.inf
    far = K - 30
    idx[:] = np.where(np.isin(idx, (7 % L, 9 % L)), 1, idx)
    idx[:, [5, far]] = 7 % L
    bvr[:, far] = bvr[:, 5]
    idx[:1, 77] = 9 % L                                        # (the first columns only)
    x = (rng.standard_normal((M, K)) * 0.1).astype(np.float16)
    x[:, [5, far]] = 0
    x[1, 300] = np.nan
    x[2, 400] = np.inf
    x[3, 400], x[3, far - 1] = np.inf, -np.inf
    x[4, 5], x[4, far] = 30000, -29000                         # up to 960000 in one part, 928000 back in the last
    x[5, 5] = -60000
    args = [torch.from_numpy(a).to(dev) for a in (bvr, idx, cache)]
    none = torch.zeros(0, dtype=torch.float16, device=dev)
    y = sbvr._sbvr_row_deq_mm_T(torch.from_numpy(x).to(dev), *args, none, 0, bvr_len=G)
    kernel, parts = hip.row_deq_last()
    assert kernel == hip.ROW_DEQ_ROWS and parts > 1
    want, peak = _transposed_sums(x, bvr, idx, cache, G)
    finite = _same_class_and_close(y.float().cpu().numpy().astype(np.float64), want, peak)
    assert finite[0, -32:].all() and finite[4, -32:].all() and not finite[1:4].all(axis=1).any()
    assert np.abs(np.where(finite[4], peak[4], 0)).max() > 4 * 130000
    assert int(hip._workspace(8 * M * N, dev).count_nonzero()) == 0


@pytest.mark.parametrize("M,N,K,S,G,kernel,parts", [(3, 2048, 1024, 4, 128, 3, 1), (2, 4096, 1024, 4, 128, 3, 1),      # many column workgroups
                                                    (1, 2048, 1024, 4, 128, 3, 2), (2, 1024, 1024, 4, 128, 3, 2),
                                                    (3, 4096, 4096, 6, 128, 2, 1),                                    # no launch that splits
                                                    (4, 14336, 2048, 3, 128, 4, 2), (3, 4096, 4096, 4, 256, 4, 4),
                                                    # both sides of the line between the two launches
                                                    (2, 1024, 2048, 4, 128, 3, 4), (3, 2048, 1280, 4, 128, 3, 1), (3, 2048, 2048, 4, 128, 4, 4),
                                                    (4, 512, 704, 3, 128, 2, 1), (4, 512, 705, 3, 128, 4, 1)])
def test_row_deq_mm_T_splits_where_it_asks_for_the_accumulators(M, N, K, S, G, kernel, parts):
    """K in parts only where the call's own rule says so, not wherever a caller brings accumulators: those of a call that is not
    split stay as they are (here: not zero), and it asks for none."""
    import ctypes
    import sbvr
    from sbvr import hip, synth
    dev = torch.device("cuda:0")
    lib, vp = hip._load(), ctypes.c_void_p
    db, di, dc = (t.to(dev) for t in synth.random_encoding(K, N, S, G, 256, seed=N + M))
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(M)).to(torch.float16).to(dev)
    ws = torch.full((M * N,), 0 if parts > 1 else 1 << 40, dtype=torch.int64, device=dev)
    outs = []
    for w in (ws, None):
        out = torch.empty((M, N), dtype=torch.float16, device=dev)
        rc = lib.sbvr_hip_row_deq_mm_T_ws(vp(x.data_ptr()), vp(db.data_ptr()), vp(di.data_ptr()), 1, vp(dc.data_ptr()), None, vp(out.data_ptr()),
                                          M, N, K, S, G, 256, vp(w.data_ptr()) if w is not None else None, 8 * M * N if w is not None else 0,
                                          vp(torch.cuda.current_stream().cuda_stream))
        assert rc == 0 and hip.row_deq_last()[1] == (parts if w is not None else 1)
        assert hip.row_deq_last()[0] == kernel or (w is None and parts > 1)        # (which launch is the faster one may hang on the parts)
        outs.append(out)
    need = lib.sbvr_hip_row_deq_mm_T_workspace_for(M, N, K, S, G)
    assert (need > 0) == (parts > 1) and need in (0, 8 * M * N) and lib.sbvr_hip_row_deq_mm_T_workspace(M, N) >= need
    assert bool((ws == (0 if parts > 1 else 1 << 40)).all())
    if parts == 1:
        assert torch.equal(*outs)


def test_row_deq_mm_T_without_workspace_and_repeatable(oracle):
    """The reference-shaped entry point (no workspace: K is never split across workgroups) against the oracle at a
    shape the binding would split, and the split form twice: the fixed-point accumulators make it repeatable."""
    import ctypes
    import sbvr
    from sbvr import hip
    dev = torch.device("cuda:0")
    M, N, K, S, G, L = 2, 1024, 2048, 4, 128, 256
    rng = np.random.default_rng(5)
    bvr, idx, cache = _rand_enc(rng, K, N, S, G, L, oracle)
    x = rng.standard_normal((M, K)).astype(np.float16)
    t = lambda a: torch.from_numpy(a).to(dev)
    dx, db, di, dc = t(x), t(bvr), t(idx), t(cache)
    out = torch.empty((M, N), dtype=torch.float16, device=dev)
    lib = hip._load()
    vp = ctypes.c_void_p
    rc = lib.sbvr_hip_row_deq_mm_T(vp(dx.data_ptr()), vp(db.data_ptr()), vp(di.data_ptr()), 1, vp(dc.data_ptr()), None,
                                   vp(out.data_ptr()), M, N, K, S, G, L, vp(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    want = oracle.C.row_deq_mm_T(x, bvr, idx, cache, G, None).astype(np.float64)
    assert np.abs(out.float().cpu().numpy() - want).max() <= 2.0 ** -9 * max(np.abs(want).max(), 1.0)
    none = torch.zeros(0, dtype=torch.float16, device=dev)
    first = sbvr._sbvr_row_deq_mm_T(dx, db, di, dc, none, 0, bvr_len=G)
    assert np.abs(first.float().cpu().numpy() - want).max() <= 2.0 ** -9 * max(np.abs(want).max(), 1.0)
    for _ in range(4):
        assert torch.equal(first, sbvr._sbvr_row_deq_mm_T(dx, db, di, dc, none, 0, bvr_len=G))


def test_row_deq_golden(oracle, golden):
    import sbvr
    dev = torch.device("cuda:0")
    g = golden("trans_s2")
    K, N = g["decoded"].shape
    x = torch.randn((2, K), generator=torch.Generator().manual_seed(3)).to(torch.float16)
    t = lambda a: torch.from_numpy(a).to(dev)
    y = sbvr._sbvr_row_deq_mm_T(x.to(dev), t(g["bvr"]), t(g["coeff_idx"]), t(g["coeff_cache"]),
                                torch.zeros(0, dtype=torch.float16, device=dev), 0)
    want = x.numpy().astype(np.float64) @ g["decoded"].astype(np.float64)
    assert np.abs(y.float().cpu().numpy() - want).max() <= 1e-2 * np.abs(want).max()


def test_sbvr_linear_module(oracle, golden):
    """SBVRLinear on a reference encoding: leading dims, padding of K, bias, > 16 rows."""
    import sbvr
    dev = torch.device("cuda:0")
    g = golden("pad_s2")                       # weight (3, 300) padded to 512
    enc = sbvr.sbvr.from_parts(*(torch.from_numpy(g[k]).to(dev) for k in ("bvr", "coeff_idx", "coeff_cache")), 256,
                               original_shape=(3, 300))
    lin = sbvr.SBVRLinear.from_sbvr(enc)
    x = torch.randn((2, 5, 300), generator=torch.Generator().manual_seed(4)).to(torch.float16)
    y = lin(x.to(dev))
    assert y.shape == (2, 5, 3)
    want = x.numpy().astype(np.float64) @ g["decoded"].astype(np.float64).T
    assert np.abs(y.float().cpu().numpy() - want).max() <= 1e-2 * np.abs(want).max()
    from sbvr import synth
    bvr, idx, cache = (t.to(dev) for t in synth.random_encoding(128, 256, 4, 128, 64, seed=2))
    bias = torch.randn(128, generator=torch.Generator().manual_seed(5)).to(torch.float16)
    lin2 = sbvr.SBVRLinear(256, 128, bvr, idx, cache, 128, bias.to(dev))
    x2 = torch.randn((40, 256), generator=torch.Generator().manual_seed(6)).to(torch.float16)
    y2 = lin2(x2.to(dev))
    yref, _ = oracle.C.linear_f16(x2.numpy(), bvr.cpu().numpy(), idx.cpu().numpy(), cache.cpu().numpy(), 128, bias.numpy())
    d = np.abs(y2.float().cpu().numpy().astype(np.float64) - yref.astype(np.float64))
    assert d.max() <= 1e-2 * np.abs(yref.astype(np.float64)).max()      # 40 rows: the prefill kernel's rounding
    # q | k | v as one layer: the parts' outputs side by side
    encs = []
    for i, rows in enumerate((256, 64, 64)):
        b, ix, c = (t.to(dev) for t in synth.random_encoding(rows, 512, 4, 128, 200, seed=20 + i))
        encs.append(sbvr.sbvr.from_parts(b, ix, c, 128, original_shape=(rows, 512)))
    fused = sbvr.SBVRLinear.fused(encs)
    assert fused.coeff_idx.dtype == torch.uint16 and fused.coeff_cache.shape[0] == 600
    x3 = torch.randn((3, 512), generator=torch.Generator().manual_seed(7)).to(torch.float16)
    y3 = fused(x3.to(dev))
    assert y3.shape == (3, 384)
    at = 0
    for e in encs:
        _, yd = oracle.C.linear_f16(x3.numpy(), e.bvr.cpu().numpy(), e.coeff_idx.cpu().numpy(), e.coeff_cache.cpu().numpy(), 128)
        rows = e.original_data_shape[0]
        _close(y3[:, at:at + rows], yd)
        at += rows


def test_hip_init_and_bad_arguments():
    import sbvr
    dev = torch.device("cuda:0")
    sbvr._sbvr_hip_init(dev)
    from sbvr import synth
    bvr, idx, cache = (t.to(dev) for t in synth.random_encoding(32, 256, 4, 128, 16))
    x = torch.zeros((1, 256), dtype=torch.float16, device=dev)
    with pytest.raises(TypeError):
        sbvr._sbvr_linear_f16(x.float(), bvr, idx, cache, None, 128)
    with pytest.raises(ValueError):
        sbvr._sbvr_linear_f16(x[:, :128], bvr, idx, cache, None, 128)
    with pytest.raises(ValueError):
        sbvr._sbvr_linear_f16(torch.zeros((2, 512), dtype=torch.float16, device=dev)[:, ::2],
                              bvr, idx, cache, None, 128)                                  # not contiguous
    with pytest.raises(TypeError):
        sbvr._sbvr_linear_f16(x, bvr, idx.to(torch.uint16), cache, None, 128)          # 16 lines want uint8


def test_torch_extension_equals_ctypes_binding(oracle):
    """Both bindings call the same entry points: identical bits, on the caller's stream."""
    import sbvr
    from sbvr import _sbvr_hip_ops as ops, synth
    dev = torch.device("cuda:0")
    ops._sbvr_hip_init()
    none = torch.zeros(0, dtype=torch.float16, device=dev)
    for (M, N, K, S, L) in [(1, 4096, 4096, 4, 256), (3, 1000, 1024, 3, 300), (48, 512, 1024, 4, 64)]:
        bvr, idx, cache = (t.to(dev) for t in synth.random_encoding(N, K, S, 128, L, seed=N))
        x = torch.randn((M, K), generator=torch.Generator().manual_seed(K)).to(torch.float16).to(dev)
        bias = torch.randn((N,), generator=torch.Generator().manual_seed(1)).to(torch.float16).to(dev)
        assert torch.equal(ops._sbvr_linear_f16(x, bvr, idx, cache), sbvr._sbvr_linear_f16(x, bvr, idx, cache))
        assert torch.equal(ops._sbvr_linear_f16(x, bvr, idx, cache, bias, 128),
                           sbvr._sbvr_linear_f16(x, bvr, idx, cache, bias, 128))
    # the reference's two operator forms, reference argument lists
    lb, li, lc = (t.to(dev) for t in synth.random_encoding(2, 1024, 4, 128, 16, seed=3))
    rb, ri, rc = (t.to(dev) for t in synth.random_encoding(640, 1024, 4, 128, 256, seed=4))
    assert torch.equal(ops._sbvr_mm_T(lb, li, lc, rb, ri, rc, none), sbvr._sbvr_mm_T(lb, li, lc, rb, ri, rc, none))
    tb, ti, tc = (t.to(dev) for t in synth.random_encoding(1024, 640, 4, 128, 256, seed=5))      # W^T: (K, N)
    x = torch.randn((2, 1024), generator=torch.Generator().manual_seed(6)).to(torch.float16).to(dev)
    assert torch.equal(ops._sbvr_row_deq_mm_T(x, tb, ti, tc, none, 0), sbvr._sbvr_row_deq_mm_T(x, tb, ti, tc, none, 0))
    # one-row variants
    bvr, idx, cache = (t.to(dev) for t in synth.random_encoding(512, 1024, 4, 128, 256, seed=7))
    gu = torch.randn((1, 2048), generator=torch.Generator().manual_seed(8)).to(torch.float16).to(dev)
    assert torch.equal(ops._sbvr_linear_f16_swiglu(gu, bvr, idx, cache), sbvr._sbvr_linear_f16_swiglu(gu, bvr, idx, cache))
    x1, d1 = x[:1].contiguous(), x[1:].contiguous()
    w = torch.ones(1024, dtype=torch.float16, device=dev)
    xo1, xo2 = torch.empty_like(x1), torch.empty_like(x1)
    a = ops._sbvr_linear_f16_add_rmsnorm(x1, d1, w, 1e-5, xo1, bvr, idx, cache)
    b = sbvr._sbvr_linear_f16_add_rmsnorm(x1, d1, w, 1e-5, xo2, bvr, idx, cache)
    assert torch.equal(a, b) and torch.equal(xo1, xo2)
    # on a side stream the extension launches there too
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        y = ops._sbvr_linear_f16(x, bvr, idx, cache)
    side.synchronize()
    assert torch.equal(y, sbvr._sbvr_linear_f16(x, bvr, idx, cache))
