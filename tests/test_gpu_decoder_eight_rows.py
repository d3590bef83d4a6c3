"""A prompt eight tokens at a time: two row tiles over the same plane words where the one-row launch shape has them, two launches
where not; new keys and values of eight tokens across blocks of the caches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,S,G,prompt,capture", [
    (dict(hidden=512, layers=1, heads=4, kv_heads=1, ffn=768, vocab=1000), 4, 128, 9, False),      # one pass and one step
    (dict(hidden=1024, layers=2, heads=8, kv_heads=2, ffn=2048, vocab=1000), 6, 256, 41, True),    # positions 24 to 39 in two passes
    (dict(hidden=4096, layers=1, heads=32, kv_heads=8, ffn=14336, vocab=4000), 4, 128, 62, True),  # windows of 7 tiles
    (dict(hidden=4096, layers=1, heads=32, kv_heads=8, ffn=14336, vocab=1000), 2, 128, 21, True),
    (dict(hidden=4096, layers=1, heads=32, kv_heads=8, ffn=14336, vocab=1000), 8, 256, 29, False),  # no room for two tiles there
    # (hidden sizes with the one-launch head, which is what fills `logits`)
    (dict(hidden=2048, layers=2, heads=16, kv_heads=4, ffn=5632, vocab=1000), 3, 128, 90, True),
])
def test_eight_prompt_rows_leave_what_single_steps_leave(shape, S, G, prompt, capture, monkeypatch):
    """The caches bit for bit, the tokens and the logits of the prompt fed token by token."""
    from sbvr import hip
    from sbvr.decoder import LlamaShape, SbvrLlamaDecoder
    made, passes = [], []
    # (a wrapper around the module's function: one around the decoder's own method would make a reference cycle of it, whose
    # recorded graphs the garbage collector might then end in the middle of the next decoder's recording, which aborts)
    advance = hip.dec_rows_advance
    monkeypatch.setattr(hip, "dec_rows_advance", lambda pos, rows, *rest: (passes.append(rows), advance(pos, rows, *rest)))
    tokens = torch.randint(0, shape["vocab"], (prompt,), generator=torch.Generator().manual_seed(prompt))
    for rows in (True, False):
        dec = SbvrLlamaDecoder(LlamaShape(**shape), "cuda:0", num_sums=S, bvr_len=G, max_seq=128, seed=5)
        assert dec.attention_o and dec.prompt_rows
        passes.clear()
        if not rows:
            dec.prompt_rows = 0
        if capture:
            dec.capture()
        out, _ = dec.generate(tokens, 4)
        assert (8 in passes) == rows
        made.append((out, dec.logits.clone(), [t.clone() for layer in dec.layers for t in (layer["k"], layer["v"])]))
    assert all(torch.equal(x, y) for x, y in zip(made[0][2], made[1][2])), "caches differ"
    assert torch.equal(made[0][1], made[1][1]) and torch.equal(made[0][0], made[1][0])
