"""Prefill of packed codes without shadows, where both are made in the call (csrc/duq_bf6.hip, shadows_kernel): rows, columns and k that
end inside a tile, a pair of weight tiles and a step, output rows and parameters at any alignment, every epilogue; against the oracle on
some of the rows and the integer kernels (which a call as a batch of one runs) on all."""
import numpy as np
import pytest
import torch

from oracle import duq_oracle as orc


def _room(mode, M, N, K):
    from duqlinear4bitcuda_amd import _lib
    return _lib.load().duq_linear4bit_room_bytes(mode, M, N, K)


def test_rule():
    assert _room(0, 4096, 28672, 8192) and _room(4, 1999, 11008, 4096) and _room(1, 1999, 11003, 4160)
    # up to 1024 rows, short rows, few columns, the epilogue with packed heads, what the GEMM refuses
    for mode, M, N, K in ((0, 1024, 28672, 8192), (0, 4096, 4096, 448), (0, 4096, 256, 4096), (5, 4096, 28672, 8192),
                          (0, 4096, 28672, 8200), (0, (1 << 24) + 1, 28672, 8192), (0, 0, 4096, 4096), (0, 4096, 0, 4096),
                          (0, 4096, 4096, 0), (0, 4096, (1 << 22) + 1, 8192)):
        assert _room(mode, M, N, K) == 0, (mode, M, N, K)


def test_errors():
    from duqlinear4bitcuda_amd import _lib
    call, P = _lib.load().duq_linear4bit_forward_room, 4096
    args = lambda mode=0, xq=P, zeros=None, K=8192, room=P, n=1 << 31: (mode, xq, P, zeros, None, P, P, None, None, None, None, None,
                                                                        4096, 28672, K, P, room, n, None)
    assert call(*args(mode=5)) == -4 and call(*args(xq=None)) == -1 and call(*args(mode=1)) == -1 and call(*args(mode=4, zeros=P)) == -1
    assert call(*args(K=8200)) == -3 and call(*args(xq=P + 8)) == call(*args(room=P + 8)) != 0 and call(*args(n=1 << 20)) != 0


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1999, 11003, 4096), (2049, 11015, 4160), (1553, 8561, 7936), (3073, 4097, 4032), (1712, 25720, 2880),
                                   (2100, 12000, 1088), (2401, 8208, 8256), (1025, 30000, 8192), (1323, 16400, 2112)])
def test_against_integer_kernels(dev, M, N, K):
    from duqlinear4bitcuda_amd import _HIP as hip
    print("prefill with shadows made in the call", M, N, K, flush=True)
    assert _room(0, M, N, K)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a, b = (torch.randint(0, 256, (n, K // 2), dtype=torch.uint8, device=dev, generator=g) for n in (M, N))
    a[0], b[-1] = 0x88, 0x88   # the largest products there are
    h = lambda n: (torch.rand(n, device=dev, generator=g) * 4 - 1).half() / 64
    i = lambda n: torch.randint(-5000, 5000, (n,), device=dev, generator=g).int()
    sr, zr, rr, s1, s2, bias, r1 = h(M), (h(M) * 64).round(), i(M), h(N), h(N), h(N), i(N)
    z1, z2 = (h(N) * 64).round(), (h(N) * 64).round()
    place = lambda t: torch.cat([t.flatten()[:1], t.flatten()])[1:]   # parameters at an odd address
    rows = [0, 1, 31, 128, M // 2, M - 2, M - 1]
    acc = orc.matmul_s4(a[rows].cpu().numpy(), b.cpu().numpy())
    n = lambda t, r=None: (t if r is None else t[r]).cpu().numpy().reshape(-1, 1)
    for mode, r, c, want in (
            (hip.EPI_SYM, (sr, None), (s1, None, None, None), lambda: orc.sym_dequant(acc, n(sr, rows), n(s1))),
            (hip.EPI_ASYM, (sr, zr), (s1, z1, None, None), lambda: orc.asym_dequant(acc, n(sr, rows), n(zr, rows), n(s1), n(z1))),
            (hip.EPI_SYM_DUAL, (sr, None), (s1, None, s2, None), lambda: orc.sym_dual_dequant(acc, n(sr, rows), n(s1), n(s2))),
            (hip.EPI_ASYM_DUAL, (sr, zr), (s1, z1, s2, z2),
             lambda: orc.asym_dual_dequant(acc, n(sr, rows), n(zr, rows), n(s1), n(z1), n(s2), n(z2)))):
        for off in (lambda t: t, place):
            got = hip.linear4bit_forward(mode, a, *r, b, *(t if t is None else off(t) for t in c))
            assert np.array_equal(got[rows].cpu().numpy().view(np.uint16), np.asarray(want()).view(np.uint16)), mode
            with_bias = hip.linear4bit_forward(mode, a, *r, b, *(t if t is None else off(t) for t in c), bias=off(bias))
            integer = hip.batch_linear4bit_forward(mode, a[None], *(t if t is None else t[None] for t in r), b[None],
                                                   *(t if t is None else t[None] for t in c))[0]
            assert torch.equal(got.view(torch.int16), integer.view(torch.int16)), mode
            assert torch.equal(with_bias.view(torch.int16), (integer + bias).view(torch.int16)), mode
    got = hip.linear4bit_forward_rowsum(a, sr, zr, rr, b, s1, z1, r1, bias)
    want = hip.asym_rowsum_dequant(hip.matmul(a, b), sr, zr, rr, s1, z1, r1, bias)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.gpu
def test_in_a_recording(dev):
    """Room and shadows of several layers in one graph, replayed with eager work in between."""
    from duqlinear4bitcuda_amd import nn as qnn
    from duqlinear4bitcuda_amd.tools.graphs import GraphedForward
    M, K = 3072, 4096
    assert _room(0, M, K, K)
    g = torch.Generator(device=dev).manual_seed(5)
    mods = []
    for _ in range(3):
        lin = torch.nn.Linear(K, K, device=dev, dtype=torch.float16).requires_grad_(False)
        mods += [qnn.SymQuantizer(), qnn.Linear4bitSQ.from_float(lin, lin.weight.abs().amax(1, keepdim=True) / 7).to(dev)]
    model = torch.nn.Sequential(*mods)
    x = torch.randn(M, K, device=dev, generator=g).half()
    graphed = GraphedForward(model, x)
    for k in range(4):
        x = torch.randn(M, K, device=dev, generator=g).half()
        want = model(x)
        assert torch.equal(graphed(x), want), k
        del want
        torch.cuda.synchronize()


@pytest.mark.gpu
def test_short_of_memory(dev):
    """Where the device has no room left the integer kernel runs, and torch's allocator, which gives all of its cached blocks back
    before it says so, is asked once and not on every call."""
    import gc

    from duqlinear4bitcuda_amd import _HIP as hip
    from duqlinear4bitcuda_amd import _lib
    M, N, K = 4096, 4096, 28672
    need, out = _room(0, M, N, K), 2 * M * N
    assert need > 3 * out
    g = torch.Generator(device=dev).manual_seed(1)
    a, b = (torch.randint(0, 256, (n, K // 2), dtype=torch.uint8, device=dev, generator=g) for n in (M, N))
    s, t = (torch.rand(n, device=dev, generator=g).half() / 64 for n in (M, N))
    run = lambda m=M: hip.linear4bit_forward(hip.EPI_SYM, a[:m], s[:m], None, b, t)

    def took():
        """Bytes beyond what is in use that a call took, its output aside."""
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        del_me = run()
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - before - del_me.nbytes

    _lib.host().forget_refused_rooms()
    want = run()
    assert took() >= need
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.empty_cache()
    # (what earlier tests left in use can keep a segment whose free part is as large as the room: those parts are taken first)
    held = [torch.empty(block["size"], dtype=torch.uint8, device=dev) for segment in torch.cuda.memory_snapshot()
            for block in segment["blocks"] if block["state"] == "inactive" and block["size"] >= out]
    free = out + need // 2   # an output, and half a room
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + free) / torch.cuda.mem_get_info(dev)[1])
        before = torch.cuda.memory_stats()
        for _ in range(5):
            got = None
            got = run()
            torch.cuda.synchronize()
        after = torch.cuda.memory_stats()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    for counter in ("num_ooms", "num_alloc_retries"):
        assert after[counter] - before[counter] == 1, counter
    assert took() < need // 2            # (still the answer)
    small = _room(0, 2048, N, K)         # less than what was refused is asked for
    assert 0 < small < need
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    y = run(2048)
    assert torch.cuda.max_memory_allocated() - before >= small + y.nbytes
    _lib.host().forget_refused_rooms()
    assert took() >= need


@pytest.mark.gpu
@pytest.mark.parametrize("cls", ["Linear4bitSQ", "Linear4bitDUSQ", "Linear4bitASQ", "LinearQuant4bitDUASQ", "Linear4bitASQRowSum"])
def test_a_layer_takes_no_more_than_it_may(dev, cls):
    from duqlinear4bitcuda_amd import _lib
    from duqlinear4bitcuda_amd import nn as qnn
    M, N, K = 3072, 4096, 4096
    need = _room(0, M, N, K)
    assert need
    lin = torch.nn.Linear(K, N, bias=True, device=dev, dtype=torch.float16).requires_grad_(False)
    x = torch.randn(M, K, device=dev, generator=torch.Generator(device=dev).manual_seed(3)).half()
    s = lin.weight.abs().amax(1, keepdim=True) / 7
    if cls in ("Linear4bitSQ", "Linear4bitDUSQ"):
        layer = getattr(qnn, cls).from_float(lin, *((s,) if cls == "Linear4bitSQ" else (s, s))).to(dev)
        x = qnn.SymQuantizer()(x)
    else:
        layer = getattr(qnn, cls).from_linear(lin, False).to(dev)
        x = qnn.AsymQuantizer(shifted=cls.endswith("RowSum"))(x)
    assert layer.prefill_room_bytes == 2 << 30
    _lib.host().forget_refused_rooms()
    want = None
    for most, takes in ((2 << 30, True), (need, True), (need - 1, False), (0, False)):
        layer.prefill_room_bytes = most
        layer(x)
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        y = layer(x)
        torch.cuda.synchronize()
        took = torch.cuda.max_memory_allocated() - before - y.nbytes
        assert (took >= need) == takes and (takes or took == 0), (most, took)
        want = y if want is None else want
        assert torch.equal(y.view(torch.int16), want.view(torch.int16)), most


def _pays(mode, M, N, K):
    from duqlinear4bitcuda_amd import _lib
    return _lib.load().duq_linear4bit_room_pays(mode, M, N, K)


def test_where_it_pays():
    """Short rows and weights beyond the last-level cache have to be ahead by more."""
    for shape in ((4096, 28672, 8192), (1999, 11008, 4096), (3072, 4096, 4096), (3679, 3712, 10240), (1663, 10675, 1728), (5652, 14176, 1664),
                  (3882, 21744, 14784), (1553, 8561, 7936)):
        assert _pays(0, *shape) == _pays(4, *shape) == 1, shape
    for shape in ((3285, 5068, 1152), (2671, 3584, 1664), (2304, 14616, 640), (2238, 21032, 576), (2100, 12000, 1088), (1489, 25479, 11840),
                  (1253, 23636, 16448), (1025, 30000, 8192)):
        assert _room(0, *shape) and _pays(0, *shape) == 0, shape
    assert _pays(5, 4096, 28672, 8192) == _pays(0, 1024, 28672, 8192) == _pays(0, 4096, 28672, 8200) == _pays(0, 0, 4096, 4096) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2100, 12000, 1088), (1323, 16400, 2112), (1025, 30000, 8192), (1651, 3566, 1152), (1712, 25720, 2880)])
def test_room_that_the_caller_brings(dev, M, N, K):
    """Whether it pays or not: the shadows' bits where the room is given."""
    from duqlinear4bitcuda_amd import _HIP as hip
    from duqlinear4bitcuda_amd import _lib
    lib = _lib.load()
    need = _room(0, M, N, K)
    assert need
    g = torch.Generator(device=dev).manual_seed(M)
    a, b = (torch.randint(0, 256, (n, K // 2), dtype=torch.uint8, device=dev, generator=g) for n in (M, N))
    s, t = (torch.rand(n, device=dev, generator=g).half() / 64 for n in (M, N))
    room = torch.full((need,), 0xA5, dtype=torch.uint8, device=dev)
    y = torch.empty(M, N, dtype=torch.float16, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    assert lib.duq_linear4bit_forward_room(0, a.data_ptr(), s.data_ptr(), None, None, b.data_ptr(), t.data_ptr(), None, None, None, None, None,
                                           M, N, K, y.data_ptr(), room.data_ptr(), need, st) == 0
    want = hip.linear4bit_forward(hip.EPI_SYM, a, s, None, b, t, room_bytes=0)
    torch.cuda.synchronize()
    assert not bool((room == 0xA5).all()) and torch.equal(y.view(torch.int16), want.view(torch.int16))
