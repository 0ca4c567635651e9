"""Which matrix path a layer with enable_fp6() runs: one rule, written in Python (_fp6_pays) and in native code, on both sides of
its lines; the same bits either way."""
import pytest
import torch


@pytest.mark.parametrize("rows,K,N,wanted", [(64, 512, 65536, False), (65, 512, 4096, True), (65, 512, 3840, False),    # 32 tiles of 64 x 256,
                                             (257, 960, 1024, True), (257, 960, 768, False), (256, 960, 1024, False),  # 20 above 256 rows
                                             (1024, 1024, 40 * 256, True), (1024, 1024, 39 * 256, False),              # 640 of them
                                             (1024, 1984, 39 * 256, False), (1024, 2048, 20 * 256, True), (1024, 2048, 19 * 256, False),  # 320
                                             (65, 4096, 160 * 256, True), (65, 4096, 159 * 256, False),
                                             (1024, 8192, 16 * 256, True), (1024, 8192, 15 * 256, False),              # 256
                                             (1025, 2048, 512, True)])
def test_rule(monkeypatch, rows, K, N, wanted):
    from duqlinear4bitcuda_amd.nn import Linear4bitASQ
    layer = Linear4bitASQ.__new__(Linear4bitASQ)
    torch.nn.Module.__init__(layer)
    layer.in_features, layer.out_features = K, N
    monkeypatch.setattr(Linear4bitASQ, "_fp6_ready", lambda self: True)
    assert layer._fp6_pays(rows) == wanted


@pytest.mark.parametrize("rows,K,N,least,wanted", [(65, 4096, 256, 1, True), (65, 4096, 256, 2, True), (65, 4096, 256, 3, False),
                                                   (64, 4096, 4096, 1, False), (65, 1024, 31 * 128, 31, True), (65, 1024, 30 * 128, 31, False),
                                                   (257, 4096, 1024, 31, True), (257, 4096, 768, 31, False),     # 5/8 of it above 256 rows
                                                   (65, 4096, 16 * 256, 32, False), (65, 4096, 16 * 256, 31, True),
                                                   (65, 4096, 176 * 256, 33, True), (65, 4096, 164 * 256, 33, False)])
def test_setting_below_the_default(monkeypatch, rows, K, N, least, wanted):
    """A caller who asks for the 6-bit float path from fewer tiles on than the default gets it there for rows of any origin."""
    from duqlinear4bitcuda_amd.nn import Linear4bitASQ
    layer = Linear4bitASQ.__new__(Linear4bitASQ)
    torch.nn.Module.__init__(layer)
    layer.in_features, layer.out_features, layer.fp6_min_tiles = K, N, least
    monkeypatch.setattr(Linear4bitASQ, "_fp6_ready", lambda self: True)
    assert layer._fp6_pays(rows) == wanted
    assert least > 31 or layer._fp6_wanted(rows) == wanted


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(70, 1024, 512), (300, 512, 1024), (1000, 1152, 4096), (1024, 2048, 5120), (1024, 2048, 4864), (1024, 1024, 10240),
                                   (1030, 1024, 512), (300, 2048, 1024)])
def test_native_code_agrees(dev, M, K, N):
    from duqlinear4bitcuda_amd import nn as qnn
    print("fp6 routes", M, K, N, flush=True)
    torch.manual_seed(M + K)
    lin = torch.nn.Linear(K, N, bias=True).half().to(dev).requires_grad_(False)
    x = torch.rand(M, K, device=dev).half() * 6
    for layer in (qnn.Linear4bitASQ.from_linear(lin).to(dev), qnn.LinearQuant4bitDUASQRowSum.from_linear(lin)):
        want = layer(x)
        layer.enable_fp6()
        for tiles in (32, 31, 1, 10 ** 6):
            layer.fp6_min_tiles = tiles
            got = layer(x)
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (type(layer).__name__, tiles)
            native = layer._decode.native if layer._decode is not None else None
            if native is not None:
                y = native.take_rows(layer._buffers, x, tiles)
                assert (y is None) == (M > 1024 or layer._fp6_pays(M)), (type(layer).__name__, tiles)
    s = (lin.weight.abs().amax(1, keepdim=True) / 7).half()
    layer, q = qnn.Linear4bitSQ.from_float(lin, s).to(dev), qnn.SymQuantizer()
    want = layer(q(x))
    layer.enable_fp6()
    for shadow in (False, True, "only"):
        got = layer(qnn.SymQuantizer(shadow=shadow)(x))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), shadow
