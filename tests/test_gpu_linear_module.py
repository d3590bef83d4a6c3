"""SBVRLinear.forward: what it does to its input in front of the operator, and where it takes its arrays from."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
K, N, G = 256, 96, 128


def _linear(oracle, bias=True, out_features=N, in_features=K, cls=None, seed=3):
    import sbvr
    from sbvr import synth
    bvr, idx, cache = synth.random_encoding(N, K, 4, G, 16, seed=seed)
    b = torch.randn(N, generator=torch.Generator().manual_seed(seed)).to(torch.float16) if bias else None
    lin = (cls or sbvr.SBVRLinear)(in_features, out_features, bvr.to(DEV), idx.to(DEV), cache.to(DEV), G, None if b is None else b.to(DEV))

    def want(x):
        x2 = torch.nn.functional.pad(x.reshape(-1, x.shape[-1]).to(torch.float16), (0, K - x.shape[-1]))
        _, yd = oracle.C.linear_f16(x2.numpy(), bvr.numpy(), idx.numpy(), cache.numpy(), G)
        if b is not None:
            yd = yd + b.numpy().astype(np.float64)
        return yd[:, :out_features].reshape(*x.shape[:-1], out_features)
    return lin, want, b


def _close(y, want):
    assert y.dtype == torch.float16 and tuple(y.shape) == want.shape
    rms = float(np.sqrt(np.mean(want ** 2)))
    # (one rounding to fp16 of the sum and one of the sum with the bias: 2 ulps; weights rounded once beyond 8 rows)
    assert np.abs(y.float().cpu().numpy() - want).max() <= 4 * 2.0 ** -10 * max(np.abs(want).max(), rms)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(K,), (1, K), (2, 3, K), (3, 1, 1, K), (40, K)])
def test_input_types_and_leading_dimensions(oracle, dtype, shape):
    lin, want, _ = _linear(oracle)
    x = torch.randn(shape, generator=torch.Generator().manual_seed(len(shape))).to(dtype)
    _close(lin(x.to(DEV)), want(x))
    # not contiguous, and at an address of its own
    _close(lin(x.to(DEV).unsqueeze(-1).expand(*shape, 2).contiguous()[..., 1]), want(x))


def test_fewer_outputs_than_rows_and_padded_inputs(oracle):
    """out_features below the rows of the encoding: the output is cut; in_features below its columns: x is padded."""
    lin, want, _ = _linear(oracle, out_features=N - 7, in_features=K - 30)
    x = torch.randn((2, 4, K - 30), generator=torch.Generator().manual_seed(1)).to(torch.float16)
    y = lin(x.to(DEV))
    _close(y, want(x))
    _close(lin(x[0, 0].to(DEV)), want(x[0, 0]))


def test_arrays_that_are_no_buffers(oracle):
    """A bias assigned as a parameter, a plain attribute, a parametrized array, a subclass's property, functional_call."""
    import sbvr
    x = torch.randn((3, K), generator=torch.Generator().manual_seed(2)).to(torch.float16)
    lin, want, b = _linear(oracle)
    first = lin(x.to(DEV))
    _close(first, want(x))
    del lin.bias
    lin.bias = torch.nn.Parameter(b.to(DEV), requires_grad=True)
    assert "bias" not in lin._buffers and torch.equal(lin(x.to(DEV)), first)
    cache = lin.coeff_cache
    del lin.coeff_cache
    lin.coeff_cache = cache.clone()                # (an attribute like any other)
    assert "coeff_cache" not in lin._buffers and torch.equal(lin(x.to(DEV)), first)

    class Double(torch.nn.Module):
        def forward(self, t):
            return t * 2

    lin, want, b = _linear(oracle, bias=False)
    plain = lin(x.to(DEV))
    torch.nn.utils.parametrize.register_parametrization(lin, "coeff_cache", Double())
    assert torch.equal(lin(x.to(DEV)), plain * 2)  # (a power of two: exact)

    class Biased(sbvr.SBVRLinear):
        @property
        def bias(self):
            return torch.ones(N, dtype=torch.float16, device=DEV)

    made, want, b = _linear(oracle, bias=False)
    plain = made(x.to(DEV))
    made.__class__ = Biased
    assert torch.equal(made(x.to(DEV)), (plain.float() + 1).to(torch.float16))

    lin, want, b = _linear(oracle)
    other = torch.zeros(N, dtype=torch.float16, device=DEV)
    assert torch.equal(torch.func.functional_call(lin, {"bias": other}, (x.to(DEV),)), plain)
    lin.bias = None
    assert torch.equal(lin(x.to(DEV)), plain)


def test_inputs_that_are_refused(oracle):
    lin, _, _ = _linear(oracle)
    with pytest.raises(RuntimeError):
        lin(torch.zeros((1, K), dtype=torch.float16))            # not on a GPU
    with pytest.raises(RuntimeError):
        lin(torch.zeros((0, K), dtype=torch.float16, device=DEV))
    with pytest.raises(TypeError):
        lin(None)
    lin.coeff_idx = lin.coeff_idx.to(torch.int32).to(torch.uint16)
    with pytest.raises(RuntimeError):
        lin(torch.zeros((1, K), dtype=torch.float16, device=DEV))  # 16 lines want uint8 indices


@pytest.mark.parametrize("M,N,K,S,G,bias", [(371, 890, 6144, 4, 256, True), (33, 1, 1152, 3, 128, False), (64, 515, 1216, 8, 64, True)])
def test_prefill_parts_in_memory_of_their_own(M, N, K, S, G, bias):
    """SBVRLinear keeps a prefill's partial results outside the shared workspace: the same bits as the function whose
    partial results lie in it, twice, with other work on the stream in between."""
    import sbvr
    from sbvr import hip, synth
    dev = torch.device("cuda:0")
    bvr, idx, cache = (t.to(dev) for t in synth.random_encoding(N, K, S, G, 256, seed=4))
    b = torch.randn(N, generator=torch.Generator().manual_seed(5)).to(torch.float16).to(dev) if bias else None
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(6)).to(torch.float16).to(dev)
    assert hip._load().sbvr_hip_linear_f16_parts(M, N, K, S, G) > 0 and hip._load().sbvr_hip_linear_f16_parts(4, N, K, S, G) == 0
    layer = sbvr.SBVRLinear(K, N, bvr, idx, cache, G, b)
    want = sbvr._sbvr_linear_f16(x, bvr, idx, cache, b, bvr_len=G)
    assert hip.last_kernel() == 5                      # K split
    first = layer(x)
    torch.full((1 << 20,), float("nan"), device=dev)
    assert torch.equal(first, want) and torch.equal(layer(x), want)
