"""The encoder run on the GPU, as the reference runs it (sbvr(data, device=cuda),
core.py:205-215, 655-813): the arrays it leaves on the device decode to the
nearest points of their lines, meet the error band the reference logs, and
drive the HIP operator directly."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _nearest_point_invariant(w, dec, idx, cache, G, oracle_decode_all):
    """Every element carries the point of its group's line that is nearest to it
    (core.py:492-494).  `oracle_decode_all(line)` -> the 2^S sums of a line."""
    N, K = w.shape
    for g in range(K // G):
        for n in range(N):
            pts = oracle_decode_all(cache[int(idx[g, n])])
            seg_w = w[n, g * G:(g + 1) * G].astype(np.float64)
            seg_d = dec[n, g * G:(g + 1) * G].astype(np.float64)
            best = np.abs(seg_w[:, None] - pts[None, :]).min(axis=1)
            # the search runs in fp16: allow one fp16 step of the data's magnitude
            assert np.all(np.abs(seg_w - seg_d) <= best + 2.0 ** -10 * np.maximum(np.abs(seg_w), 2.0 ** -6))


@pytest.mark.parametrize("S,G,band", [(4, 256, 0.03), (4, 128, 0.03), (2, 256, 0.30), (3, 256, 0.09)])
def test_encode_on_gpu_and_use(oracle, S, G, band):
    import sbvr
    dev = torch.device("cuda:0")
    N, K = 48, 512
    w = (torch.randn((N, K), generator=torch.Generator().manual_seed(S * 1000 + G)) * 0.02).to(torch.float16)
    enc = sbvr.sbvr(w.to(dev), encoder_config={"num_sums": S, "bvr_len": G}, device=dev, verbose_level=0)
    assert enc.bvr.data.device.type == "cuda" and enc.bvr.shape == (K // 32, N, S) and enc.bvr.dtype == torch.uint32
    assert enc.coeff_idx.shape == (K // G, N) and enc.coeff_cache.shape[1] == S

    bvr, idx, cache = (t.cpu().numpy() for t in (enc.bvr.data, enc.coeff_idx.data, enc.coeff_cache.data))
    dec = enc.decode().cpu().numpy()
    # decode() on the device agrees bit for bit with the CPU restatement of the reference's decode
    assert np.array_equal(dec.view(np.uint16), oracle.C.decode(bvr, idx, cache, G).view(np.uint16))
    # error band of the reference's own log (test.txt:30-69: S=2 0.24, S=3 6.5e-2, S=4 1.7e-2 of the variance)
    wf = w.numpy().astype(np.float64)
    rel = ((dec.astype(np.float64) - wf) ** 2).mean() / wf.var()
    assert rel < band, rel

    def all_sums(line):            # the 2^S points of a line: exact sums rounded once to fp16 (core.py:365-366)
        c = line.astype(np.float64)
        pts = [sum(c[j] for j in range(S) if (sel >> j) & 1) for sel in range(1 << S)]
        return np.array(pts, dtype=np.float64).astype(np.float16).astype(np.float64)
    _nearest_point_invariant(w.numpy(), dec, idx, cache, G, all_sums)

    # and the arrays, where they lie, are operands of the HIP operator
    lin = sbvr.SBVRLinear.from_sbvr(enc)
    x = torch.randn((3, K), generator=torch.Generator().manual_seed(9)).to(torch.float16)
    y = lin(x.to(dev)).float().cpu().numpy().astype(np.float64)
    want = x.numpy().astype(np.float64) @ dec.astype(np.float64).T
    assert np.abs(y - want).max() <= 1e-2 * np.abs(want).max()


def test_gpu_and_cpu_encodings_are_of_equal_quality():
    """The search makes the same torch calls on either device; the results may differ in
    the last bit of a reduction, so the comparison is of the error, not of the arrays."""
    import sbvr
    dev = torch.device("cuda:0")
    w = (torch.randn((16, 512), generator=torch.Generator().manual_seed(77)) * 0.02).to(torch.float16)
    conf = {"num_sums": 4, "bvr_len": 128}
    on_gpu = sbvr.sbvr(w.to(dev), encoder_config=conf, device=dev, verbose_level=0).decode().float().cpu()
    on_cpu = sbvr.sbvr(w, encoder_config=conf, device=torch.device("cpu"), verbose_level=0).decode().float()
    e_gpu = (on_gpu - w.float()).pow(2).mean().item()
    e_cpu = (on_cpu - w.float()).pow(2).mean().item()
    assert abs(e_gpu - e_cpu) <= 0.05 * e_cpu


@pytest.mark.parametrize("S,G", [(2, 256), (4, 128), (4, 256), (6, 128)])
def test_search_kernel_is_the_search_expression(S, G):
    """The HIP search kernel against the reference's expression (core.py:485-495) step by step in numpy:
    fp16 difference, fp16 square, minimum over the 2^S points, fp32 sum over the group in element order,
    divided by G -- bit for bit; and against the same expression in torch on the device to 2e-5."""
    from sbvr import hip
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(S * 100 + G)
    B, n, P = 7, 333, 1 << S
    data = (rng.standard_normal((B, G)) * 0.02).astype(np.float16)
    data[2, 5] = 3.0                                   # an outlier, and a group of zeros
    data[4] = 0
    pts = (rng.standard_normal((n, P)) * 0.03).astype(np.float16)
    got = hip.encoder_group_mse(torch.from_numpy(data).to(dev), torch.from_numpy(pts).to(dev)).cpu().numpy()
    diff = (data[:, None, :, None] - pts[None, :, None, :]).astype(np.float16)
    best = (diff * diff).astype(np.float16).min(-1).astype(np.float32)
    want = np.cumsum(best, axis=-1, dtype=np.float32)[..., -1] / np.float32(G)
    assert np.array_equal(got, want)
    d, p = torch.from_numpy(data).to(dev), torch.from_numpy(pts).to(dev)
    t = ((d.view(B, 1, G, 1) - p.view(1, n, 1, P)) ** 2).min(-1)[0].float().mean(-1).cpu().numpy()
    assert np.allclose(got, t, rtol=2e-5, atol=0)          # (torch sums the group in another order)


@pytest.mark.parametrize("case", ["random", "v1_s2", "weights_s4_n64"])
def test_block_lookup_equals_one_group_loop(golden, case):
    """Table look-ups for 512 (or 7) groups at a time give the arrays of the one-group loop: the policy's
    order (hits, the error history, the hit rate that widens the search) is kept."""
    import sbvr
    dev = torch.device("cuda:0")
    if case == "random":
        w = (torch.randn((256, 1024), generator=torch.Generator().manual_seed(1)) * 0.02).to(torch.float16)
        conf = {"num_sums": 4, "bvr_len": 128}
    else:
        g = golden(case)
        w = torch.from_numpy(g["data"])
        conf = {"num_sums": int(g["num_sums"]), "bvr_len": int(g["bvr_len"])}
    made = {}
    for block in (1, 7, 512):
        made[block] = sbvr.sbvr(w.to(dev), encoder_config=dict(conf, group_block=block), device=dev, verbose_level=0)
    for block in (7, 512):
        for part in ("bvr", "coeff_idx", "coeff_cache"):
            assert torch.equal(getattr(made[1], part).data, getattr(made[block], part).data), (block, part)
        assert made[1].encoder_stats == made[block].encoder_stats
    assert made[1].encoder_stats["cache_hits"] > 0


def test_real_4096_encoding_and_config1(oracle, golden):
    """A real (searched, not synthetic) encoding of a 4096 x 4096 weight, 4 planes, groups of 128, made on
    the GPU in seconds: the same arrays as tests/golden/make_encoded_4096.py stored (slice and SHA-256 of
    each array), and the single-row linear of the first benchmark configuration on it against the oracle
    and against the dense product."""
    import sys, os
    sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))
    import make_encoded_4096 as made
    import sbvr
    from sbvr import hip
    dev = torch.device("cuda:0")
    g = golden("encoded_4096_s4_g128")
    enc, seconds = made.encode(dev)
    assert seconds < 60.0, f"encoding took {seconds:.1f} s"
    bvr, idx, cache = (t.cpu().numpy() for t in (enc.bvr.data, enc.coeff_idx.data, enc.coeff_cache.data))
    assert bvr.shape == (made.K // 32, made.N, made.S) and idx.shape == (made.K // made.G, made.N)
    assert np.array_equal(cache, g["coeff_cache"])
    assert np.array_equal(bvr[:, :made.ROWS, :], g["bvr_rows"]) and np.array_equal(idx[:, :made.ROWS], g["coeff_idx_rows"])
    assert made.digest(bvr) == str(g["sha256_bvr"]) and made.digest(idx) == str(g["sha256_coeff_idx"])
    assert enc.encoder_stats["lines"] == int(g["lines"]) and enc.encoder_stats["cache_hits"] == int(g["cache_hits"])
    # config 1: one row through the decode kernel on the real encoding
    x = torch.randn((1, made.K), generator=torch.Generator().manual_seed(5)).to(torch.float16)
    y = sbvr._sbvr_linear_f16(x.to(dev), enc.bvr.data, enc.coeff_idx.data, enc.coeff_cache.data, None, bvr_len=made.G)
    assert hip.last_kernel() == 2
    _, yd = oracle.C.linear_f16(x.numpy(), bvr, idx, cache, made.G)
    got = y.float().cpu().numpy().astype(np.float64)
    rms = float(np.sqrt(np.mean(yd ** 2)))
    assert (np.abs(got - yd) / np.maximum(np.abs(yd), 1e-2 * rms)).max() <= 1e-2
    assert (np.abs(got - yd) / (np.maximum(np.abs(yd), rms) * 2.0 ** -10)).max() <= 2.0
    # the encoding stands for the weight: 4 planes leave under 1 % of the variance (the reference's log: 1.7e-2)
    w = made.weight().numpy().astype(np.float64)
    dense = x.numpy().astype(np.float64) @ w.T
    assert np.mean((got - dense) ** 2) < 0.02 * np.mean(dense ** 2)


@pytest.mark.parametrize("S,G,scale,shift", [(2, 128, 0.02, 0.0), (3, 256, 0.02, 0.001), (4, 128, 0.02, 0.0), (4, 256, 1.0, 0.1),
                                             (5, 64, 0.3, 0.0), (6, 128, 0.02, 0.0), (4, 4, 0.02, 0.0), (4, 128, 1.0, 3.0)])
@pytest.mark.parametrize("extended", [False, True])
def test_fused_candidates_equal_the_general_search(S, G, scale, shift, extended):
    """The search of new lines with the candidates formed in the launch against the one over candidate_lines(): the
    same best error, line and selectors, bit for bit; the last case has a mean that the launch leaves to the other."""
    from sbvr.encoder import EncoderConfig, GroupEncoder
    dev = torch.device("cuda:0")
    conf = EncoderConfig(num_sums=S, bvr_len=G, search_batch_size=1 << 24)
    enc = GroupEncoder(conf, torch.float16, dev, max_lines=16)
    gen = torch.Generator().manual_seed(S * 1000 + G)
    taken = 0
    for i in range(12):
        data = (torch.randn(G, generator=gen) * scale * (1 + i % 3) + shift).to(torch.float16).to(dev)
        found = enc._search_new_fused(data, extended)
        if found is None:
            continue
        taken += 1
        lines = enc.candidate_lines(data, extended)[0]
        mse, at, sel = enc.search(lines, data, conf.acceptable_mse)
        assert found[0] == mse, f"group {i}: error {found[0]} beside {mse}"
        assert torch.equal(found[1], lines[at]), f"group {i}: line {found[1].tolist()} beside {lines[at].tolist()}"
        assert torch.equal(found[2], sel), f"group {i}: selectors"
    assert taken == (0 if shift >= 3 else 12)


def _encode_both_ways(w, conf):
    import sbvr
    made = [sbvr.sbvr(w, encoder_config=dict(conf, **more), device=w.device, verbose_level=0) for more in ({}, {"group_block": 512})]
    for part in ("bvr", "coeff_idx", "coeff_cache"):
        assert torch.equal(getattr(made[0], part).data, getattr(made[1], part).data), part
    assert made[0].encoder_stats == made[1].encoder_stats
    return made[0].encoder_stats


@pytest.mark.parametrize("shape,S,G,scale,more", [
    ((64, 512), 2, 256, 0.02, {}),
    ((100, 768), 3, 128, 0.02, {}),
    ((192, 1024), 4, 128, 0.02, {}),
    ((33, 512), 4, 64, 1.0, {}),                                     # distances out of fp16's subnormals
    ((16, 256), 5, 32, 0.3, {}),
    ((12, 256), 6, 64, 0.02, {}),
    ((5, 20), 4, 32, 0.02, {}),                                      # padded groups
    ((40, 512), 4, 128, 0.02, {"cache_warmup_num": 3, "mse_window_size": 2, "s_search_num": 17, "extend_ratio": 1.3}),
    ((64, 512), 4, 128, 1e-4, {}),                                   # values whose squares vanish: ties everywhere
])
def test_the_policy_on_the_device_equals_the_block_loop(shape, S, G, scale, more):
    """The rounds of search and settle launches leave the arrays and the counts of the loop over blocks, bit for bit."""
    dev = torch.device("cuda:0")
    w = (torch.randn(shape, generator=torch.Generator().manual_seed(S + G)) * scale).to(torch.float16).to(dev)
    stats = _encode_both_ways(w, dict(num_sums=S, bvr_len=G, **more))
    assert stats["groups"] == w.shape[0] * -(-w.shape[1] // G)


@pytest.mark.parametrize("kind", ["mean", "zeros", "outliers", "repeats", "constant"])
def test_groups_that_the_device_leaves_to_the_host(kind):
    """Groups beside a mean that moves the offsets, of zeros or of one value between ordinary ones, and groups that
    repeat, whose lines the table has already."""
    dev = torch.device("cuda:0")
    w = torch.randn((48, 512), generator=torch.Generator().manual_seed(5)) * 0.02
    if kind == "mean":
        w[::3] += 2.0
    elif kind == "zeros":
        w[::5] = 0
    elif kind == "outliers":
        w[::4, 7] = 3.0
    elif kind == "constant":
        w[::4] = 0.25
    else:
        w[24:] = w[:24]
    _encode_both_ways(w.to(torch.float16).to(dev), dict(num_sums=4, bvr_len=128))


@pytest.mark.parametrize("block", [None, 512])
def test_values_that_are_not_numbers_are_refused_as_before(block):
    import sbvr
    w = torch.randn((8, 256), generator=torch.Generator().manual_seed(8)).to(torch.float16)
    w[5, 3] = float("nan")
    with pytest.raises(RuntimeError, match="step must be nonzero"):
        sbvr.sbvr(w.cuda(), encoder_config=dict(num_sums=4, bvr_len=128, group_block=block), device="cuda:0", verbose_level=0)


def test_the_device_policy_over_several_chunks():
    """Chunks of groups that begin with a table of lines and a history of errors."""
    from sbvr import encoder
    dev = torch.device("cuda:0")
    w = (torch.randn((96, 512), generator=torch.Generator().manual_seed(6)) * 0.02).to(torch.float16).to(dev)
    flat, out = w.reshape(-1), []
    for parts in ([384], [5, 30, 349], [100, 284]):
        conf = encoder.EncoderConfig(num_sums=3, bvr_len=128, search_batch_size=1 << 24)
        enc = encoder.GroupEncoder(conf, torch.float16, dev)
        line_of, sel = torch.zeros(384, dtype=torch.int32, device=dev), torch.zeros(flat.numel(), dtype=torch.int32, device=dev)
        at = 0
        for n in parts:
            enc.encode_all(flat[at * 128:(at + n) * 128], line_of[at:at + n], sel[at * 128:(at + n) * 128])
            at += n
        out.append((line_of, sel, enc.table[:conf.num_coeff_cache_lines].clone(), conf.mse_history, conf.cache_hits, conf.group_idx))
    for other in out[1:]:
        assert all(torch.equal(a, b) for a, b in zip(out[0][:3], other[:3])) and out[0][3:] == other[3:]


def test_a_round_leaves_the_slot_it_reads(monkeypatch):
    """A group whose candidates the search does not form: the round says so in the slot it writes, and leaves the one that
    all of its workgroups read as it is."""
    import sys
    import sbvr
    from sbvr import hip
    real, seen = hip.encoder_rounds, []

    def rounds(run, S, lines, slot, many, device):
        if not seen:
            state = sys._getframe(1).f_locals["state"]
            before = state.clone()
            real(run, S, lines, 0, 1, device)
            seen.append((before.tolist(), state.tolist()))
            state.copy_(before)
        real(run, S, lines, slot, many, device)

    monkeypatch.setattr(hip, "encoder_rounds", rounds)
    w = torch.randn((8, 512), generator=torch.Generator().manual_seed(5)) * 0.02
    w[0, :128] += 2.0                                            # (a mean that moves the offsets)
    _encode_both_ways(w.to(torch.float16).to("cuda:0"), dict(num_sums=4, bvr_len=128))
    (before, after), = seen
    assert after[:8] == before[:8] and after[8:13] == before[:3] + [1, before[4]]


@pytest.mark.parametrize("S,covered,more", [
    (3, True, {"s_search_num": 131}), (3, False, {"s_search_num": 134}), (3, False, {"s_search_num": 200}),      # 160 scales at most, 1.2 times as many when wide
    (2, False, {"r_search_num": 1200, "b_search_num": 1200, "s_search_num": 1}),      # too many families for a launch's candidate numbers
    (3, False, {"search_batch_size": 9000, "r_search_num": 16, "b_search_num": 8, "s_search_num": 8}),
])
def test_the_rounds_take_what_their_launches_take(S, covered, more):
    """What the rounds' launches refuse, or could leave to the host group after group, goes through the block loop; the last
    case by a table that may grow beyond a batch of the look-up's scan."""
    from sbvr.encoder import EncoderConfig, GroupEncoder
    dev = torch.device("cuda:0")
    conf = dict(num_sums=S, bvr_len=64, **dict({"search_batch_size": 1 << 24}, **more))
    enc = GroupEncoder(EncoderConfig(**conf), torch.float16, dev)
    flat = torch.zeros(64 * (10000 if "search_batch_size" in more else 40), dtype=torch.float16, device=dev)
    assert (enc._covered_on_device(flat) is not None) == covered
    if "search_batch_size" in more:
        assert enc._covered_on_device(flat[:64 * 9000]) is not None
    w = (torch.randn((5, 512), generator=torch.Generator().manual_seed(S)) * 0.02).to(torch.float16).to(dev)
    _encode_both_ways(w, conf)


def test_few_rounds_are_queued_behind_a_group_for_the_host(monkeypatch):
    """Groups left to the host one after the other: two launches at a time are queued behind such a group, not dozens."""
    from sbvr import hip
    real, queued = hip.encoder_rounds, []

    def rounds(run, S, lines, slot, many, device):
        queued.append(many)
        real(run, S, lines, slot, many, device)

    monkeypatch.setattr(hip, "encoder_rounds", rounds)
    w = torch.randn((48, 512), generator=torch.Generator().manual_seed(5)) * 0.02
    w[::2] += 2.0
    stats = _encode_both_ways(w.to(torch.float16).to("cuda:0"), dict(num_sums=4, bvr_len=128))
    misses = stats["groups"] - stats["cache_hits"]
    assert sum(queued) <= 16 + 4 * misses


@pytest.mark.parametrize("more", [
    {"cache_warmup_num": 3.0}, {"cache_warmup_num": 2.5}, {"cache_warmup_num": np.int64(3)}, {"cache_warmup_num": 10 ** 10}, {"cache_warmup_num": float("inf")},
    {"mse_window_size": np.int64(2)}, {"mse_window_size": 10 ** 10}, {"acceptable_mse": 0},
])
def test_search_options_of_any_kind_of_number(more):
    """Options that are no plain ints, or larger than 32 bits, on the device as in the block loop."""
    from sbvr.encoder import EncoderConfig, GroupEncoder
    dev = torch.device("cuda:0")
    conf = dict(num_sums=3, bvr_len=64, **more)
    w = (torch.randn((6, 512), generator=torch.Generator().manual_seed(9)) * 0.02).to(torch.float16).to(dev)
    enc = GroupEncoder(EncoderConfig(search_batch_size=1 << 24, **conf), torch.float16, dev)
    assert enc._covered_on_device(w.reshape(-1)) is not None
    _encode_both_ways(w, conf)
