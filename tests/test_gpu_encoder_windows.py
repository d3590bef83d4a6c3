"""The encoder's policy on the device where groups meet the table in windows of 2048: the loop over blocks, bit for bit, with
groups, misses and groups left to the host on both sides of a window's end."""
import pytest
import torch

from test_gpu_encoder import _encode_both_ways

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups,S,odd", [
    (2048, 2, ()),                              # one window exactly
    (2049, 3, (2048,)),                         # a last window of one group, and that one left to the host
    (4100, 2, (0, 2047, 2048, 2049, 4095, 4096)),
    (6145, 2, (2046, 2047, 4095)),
])
def test_windows(groups, S, odd):
    G = 32
    w = torch.randn((groups, G), generator=torch.Generator().manual_seed(groups)) * 0.02
    for g in odd:
        w[g] += 2.0                             # (a mean that moves the offsets)
    w[::97] *= 30.0                             # (groups that the table does not serve, also far behind)
    stats = _encode_both_ways(w.to(torch.float16).to("cuda:0"), dict(num_sums=S, bvr_len=G, s_search_num=8, r_search_num=16, b_search_num=8))
    assert stats["groups"] == groups


@pytest.mark.parametrize("groups", [300, 2500])
def test_state_of_two_slots_all_groups_met(groups, monkeypatch):
    """The state is two slots; one whose sixth word is 0 says that best and line are over all lines for all groups, as an empty
    table's are, and is taken on from there without windows: the same arrays."""
    import sys
    from sbvr import hip
    assert hip.encoder_state_words() == 16
    real, started = hip.encoder_rounds, []

    def rounds(run, S, lines, slot, many, device):
        if not started:
            state = sys._getframe(1).f_locals["state"]
            assert state.tolist()[:5] == [0] * 5
            state[5], state[13] = 0, 0
            started.append(groups)
        real(run, S, lines, slot, many, device)

    monkeypatch.setattr(hip, "encoder_rounds", rounds)
    w = torch.randn((groups, 32), generator=torch.Generator().manual_seed(groups)) * 0.02
    w[5], w[::97] = w[5] + 2.0, w[::97] * 30.0
    _encode_both_ways(w.to(torch.float16).to("cuda:0"), dict(num_sums=2, bvr_len=32, s_search_num=8, r_search_num=16, b_search_num=8))
    assert started == [groups]


def test_searches_of_more_than_2_24_lines():
    """The plainer search has less than 2^24 candidate lines, whose numbers are taken apart by products, the wider one more."""
    from sbvr.encoder import EncoderConfig, GroupEncoder
    dev = torch.device("cuda:0")
    conf = dict(num_sums=3, bvr_len=32, r_search_num=280, b_search_num=200, s_search_num=110, cache_warmup_num=2, search_batch_size=1 << 27)
    enc = GroupEncoder(EncoderConfig(**conf), torch.float16, dev)
    w = (torch.randn((6, 64), generator=torch.Generator().manual_seed(3)) * 0.02).to(torch.float16).to(dev)
    _, lines = enc._covered_on_device(w.reshape(-1))
    assert lines[0] < 1 << 24 < lines[1]
    stats = _encode_both_ways(w, conf)
    assert stats["groups"] - stats["cache_hits"] > 2
