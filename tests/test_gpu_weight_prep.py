"""Conversion of layers on the GPU in one pass (csrc/duq_weight.hip) against the torch statements it stands for, which are
those of the reference: rows inside and beyond the register cache, constant and zero rows, infinities and NaNs, codes
outside the int4 range, and the way of large codes through the pinned buffers."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(3, 24), (5, 32), (64, 512), (7, 2056), (16, 16384), (4, 16392), (3, 28672), (2300, 4096)]


def _weight(dev, N, K, dtype):
    g = torch.Generator(device=dev).manual_seed(N * K)
    w = (torch.randn(N, K, generator=g, device=dev) * 0.02).to(dtype)
    w[0] = 0
    w[1] = -0.25
    if N > 4:
        w[2, 7] = float("inf")
        w[3, 12] = float("nan")
        w[4] *= 1e-3
    return w


@pytest.mark.parametrize("N,K", SHAPES)
def test_one_pass_weight_preparation(dev, monkeypatch, N, K):
    from duqlinear4bitcuda_amd import _HIP as ops
    from duqlinear4bitcuda_amd import nn as qnn
    print("weight preparation", N, K, flush=True)
    lin = torch.nn.Linear(K, N, bias=True, device="meta")
    for dtype, classes in ((torch.float16, ("Linear4bitASQ", "LinearQuant4bitDUASQ", "LinearQuant4bitDUASQRowSum")),
                           (torch.float32, ("LinearQuant8bitASQ",))):
        lin.weight = torch.nn.Parameter(_weight(dev, N, K, dtype), requires_grad=False)
        lin.bias = torch.nn.Parameter(torch.randn(N, device=dev).to(dtype), requires_grad=False)
        assert ops.weight_takes_one_pass(lin.weight.data, dtype)
        for name in classes:
            one = getattr(qnn, name).from_linear(lin).state_dict()
            with monkeypatch.context() as m:
                m.setattr(ops, "weight_takes_one_pass", lambda *a: False)
                steps = getattr(qnn, name).from_linear(lin).state_dict()
            assert one.keys() == steps.keys()
            for k, want in steps.items():
                assert one[k].device == want.device and one[k].dtype == want.dtype and one[k].shape == want.shape
                assert torch.equal(one[k].nan_to_num(nan=3.25) if want.is_floating_point() else one[k],
                                   want.nan_to_num(nan=3.25) if want.is_floating_point() else want), (name, k)


@pytest.mark.parametrize("N,K", SHAPES)
def test_one_pass_symmetric_codes(dev, monkeypatch, N, K):
    from duqlinear4bitcuda_amd import _HIP as ops
    from duqlinear4bitcuda_amd import nn as qnn
    lin = torch.nn.Linear(K, N, bias=False, device="meta")
    w = _weight(dev, N, K, torch.float16)
    w[0, 3] = 0.001
    lin.weight = torch.nn.Parameter(w, requires_grad=False)
    finite = w.nan_to_num(0, 0, 0).abs()
    one, two = finite.amax(1, keepdim=True) / 7 + 1e-4, (finite[:, :10].amax(1, keepdim=True) / 7 + 1e-4, finite[:, 10:].amax(1, keepdim=True) / 7 + 1e-4)
    make = (lambda: qnn.Linear4bitSQ.from_float(lin, one), lambda: qnn.Linear4bitDUSQ.from_float(lin, *two))
    for f in make:
        got = f().weight
        with monkeypatch.context() as m:
            m.setattr(ops, "weight_takes_one_pass", lambda *a: False)
            assert torch.equal(got, f().weight)
    w[N - 1, K - 1] = 9.0 * float(two[1][N - 1])
    for f in make:
        with pytest.raises(AssertionError, match="int4 range"):
            f()
