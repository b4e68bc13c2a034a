"""GEMV operands of any size and address: rows that are no whole 16-byte pieces in both weight orders, and the I_X_W kernel at
the edges of its blocks, row groups and slices.  Reference: the float64 product.  Tolerance per output: half an ulp of fp16
(2^-11 of the value, 2^-25 below the normal range) for the one rounding, and (in + 1) * 2^-24 times the sum of the products'
magnitudes for any order of fp32 sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def at_offset(t, off):
    """The same values at an address `off` halves behind a 16-byte boundary."""
    buf = torch.zeros(t.numel() + off + 8, dtype=torch.float16, device=DEV)
    v = buf[off:off + t.numel()].view(t.shape)
    v.copy_(t)
    return v


def call(order, W, x, b, in_w, out_w, ld, relu, off_y=0):
    from pimaicompiler_amd import _lib as L
    lib = L.load()
    y = torch.full((out_w + off_y + 1,), float("nan"), dtype=torch.float16, device=DEV)
    rc = lib.pimhip_execute_gemv(y[off_y:].data_ptr(), x.data_ptr(), W.data_ptr(), b.data_ptr() if b is not None else None, in_w, out_w, ld,
                                 L.PIMHIP_ACT_RELU if relu else L.PIMHIP_ACT_NONE, order, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.pimhip_last_error()
    assert bool(torch.isnan(y[off_y + out_w:]).all()) and bool(torch.isnan(y[:off_y]).all())   # nothing behind or in front of it
    return y[off_y:off_y + out_w]


def check(y, w_out_in, x, b, relu):
    w, xd = w_out_in.double(), x.double()
    want = w @ xd + (b.double() if b is not None else 0)
    size = w.abs() @ xd.abs() + (b.double().abs() if b is not None else 0)
    want = want.relu() if relu else want
    tol = want.abs() * 2.0 ** -11 + 2.0 ** -25 + (w.size(1) + 1) * 2.0 ** -24 * size
    assert bool(((y.double() - want).abs() <= tol).all())


@pytest.mark.parametrize("out_w,in_w,off_w,off_x,pitch", [
    (1, 1, 1, 1, 0), (3, 5, 0, 0, 0), (9, 7, 3, 5, 2), (5, 8, 1, 0, 0), (4, 15, 0, 0, 1), (130, 513, 0, 1, 0), (1023, 2049, 7, 0, 0),
    (1024, 1023, 0, 3, 5), (1025, 1029, 2, 2, 0), (1024, 1024, 1, 0, 0), (1024, 1024, 0, 1, 0), (40, 4103, 0, 0, 0),
    (1030, 127, 0, 0, 0), (5, 128, 1, 0, 0), (1027, 129, 0, 0, 3), (4099, 257, 3, 1, 0), (1, 505, 0, 0, 0), (1025, 511, 0, 0, 0),
    (7, 512, 0, 1, 0), (1024, 513, 0, 0, 0),
    (2049, 4099, 5, 1, 0), (1500, 6151, 0, 0, 0)])   # the last two exceed 16 MB or 4096 columns: other launch shapes and loads
def test_rows_of_any_length_at_any_address(ops, out_w, in_w, off_w, off_x, pitch):
    from pimaicompiler_amd import _lib as L
    g = torch.Generator().manual_seed(out_w + in_w)
    ld = in_w + pitch
    W = at_offset((0.1 * torch.randn(out_w, ld, generator=g)).half(), off_w)
    x = at_offset(torch.randn(in_w, generator=g).half(), off_x)
    b = torch.randn(out_w, generator=g).half().to(DEV)
    for bias, relu in ((b, True), (None, False)):
        check(call(L.PIMHIP_W_X_I, W, x, bias, in_w, out_w, ld, relu, off_w), W[:, :in_w], x, bias, relu)


@pytest.mark.parametrize("in_w,out_w,off,pitch", [
    (1, 8, 0, 0), (128, 257, 0, 0), (129, 257, 0, 0), (127, 64, 3, 0), (128, 1032, 0, 5), (17, 4001, 0, 0), (600, 7, 0, 0), (600, 8, 0, 0), (600, 9, 1, 0), (513, 63, 0, 0), (512, 64, 0, 0), (513, 64, 0, 3), (513, 65, 0, 0),
    (520, 71, 3, 0), (700, 128, 0, 8), (2305, 129, 0, 0), (8, 4096, 0, 0), (31, 4097, 0, 0), (1025, 1031, 5, 0), (12896, 84, 0, 0),
    (1500, 2000, 0, 0), (1000, 17000, 0, 0), (3001, 3001, 0, 0), (4101, 2056, 1, 0)])   # the last three: more than 16 MB
def test_i_x_w_at_the_edges_of_blocks_row_groups_and_slices(ops, in_w, out_w, off, pitch):
    from pimaicompiler_amd import _lib as L
    g = torch.Generator().manual_seed(in_w * 3 + out_w)
    ld = out_w + pitch
    A = at_offset((0.1 * torch.randn(in_w, ld, generator=g)).half(), off)
    x = at_offset(torch.randn(in_w, generator=g).half(), off)
    b = torch.randn(out_w, generator=g).half().to(DEV)
    w = A[:, :out_w].t()
    y = call(L.PIMHIP_I_X_W, A, x, b, in_w, out_w, ld, True, off)
    check(y, w, x, b, True)
    for _ in range(3):                                     # a fixed order of sums: the same bits in every launch
        assert torch.equal(call(L.PIMHIP_I_X_W, A, x, b, in_w, out_w, ld, True, off), y)
    # reducing blocks that do not wait make the missing sums themselves, with the producers' bits
    torch.cuda.synchronize()
    ops.set_gemv_spin_limit(0)
    try:
        alone = call(L.PIMHIP_I_X_W, A, x, b, in_w, out_w, ld, True, off)
        torch.cuda.synchronize()
    finally:
        ops.set_gemv_spin_limit(1 << 22)
    assert torch.equal(alone, y)
    assert torch.equal(call(L.PIMHIP_I_X_W, A, x, b, in_w, out_w, ld, True, off), y)   # (puts the workspace back in order)
    torch.cuda.synchronize()


PER_THREAD_STREAM = 2   # hipStreamPerThread


@pytest.mark.parametrize("in_w,out_w,off,pitch", [
    (520, 9, 0, 0), (1024, 64, 0, 0), (8192, 8, 0, 0), (1000, 33, 1, 0), (1500, 2001, 0, 0), (4951, 1301, 3, 0), (12896, 84, 0, 0), (16384, 257, 0, 5),
    (2048, 1024, 0, 4), (2100, 4001, 0, 0), (9000, 2001, 0, 7)])   # the last two: more than 16 MB, and one of them in several slices
def test_small_and_odd_products_have_the_same_bits_wherever_they_run(ops, in_w, out_w, off, pitch):
    """Products that need no workspace: the same sums in the same order on a stream with a region, on one without, inside a capture on
    a stream that has never run one, in every replay beside other work of the capture stream, and through the static entry point."""
    from pimaicompiler_amd import _lib as L
    lib = L.load()
    g = torch.Generator().manual_seed(in_w + out_w)
    ld = out_w + pitch
    A = at_offset((0.1 * torch.randn(in_w, ld, generator=g)).half(), off)
    x = at_offset(torch.randn(in_w, generator=g).half(), off)
    b = torch.randn(out_w, generator=g).half().to(DEV)
    eager = call(L.PIMHIP_I_X_W, A, x, b, in_w, out_w, ld, True, off)
    check(eager, A[:, :out_w].t(), x, b, True)
    y = torch.empty(out_w, dtype=torch.float16, device=DEV)

    def launch(fn, stream):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        assert fn(y.data_ptr(), x.data_ptr(), A.data_ptr(), b.data_ptr(), in_w, out_w, ld, L.PIMHIP_ACT_RELU, L.PIMHIP_I_X_W, stream) == 0
        torch.cuda.synchronize()
        return y
    main = torch.cuda.current_stream()
    assert torch.equal(launch(lib.pimhip_execute_gemv_static, main.cuda_stream), eager)
    assert torch.equal(launch(lib.pimhip_execute_gemv, PER_THREAD_STREAM), eager)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    side.wait_stream(main)
    with torch.cuda.graph(graph, stream=side):
        assert lib.pimhip_execute_gemv(y.data_ptr(), x.data_ptr(), A.data_ptr(), b.data_ptr(), in_w, out_w, ld, L.PIMHIP_ACT_RELU, L.PIMHIP_I_X_W,
                                       torch.cuda.current_stream().cuda_stream) == 0
    others = [torch.empty(out_w, dtype=torch.float16, device=DEV) for _ in range(8)]
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        for o in others:                                   # on the capture stream, while the graph is replayed on another one
            assert lib.pimhip_execute_gemv(o.data_ptr(), x.data_ptr(), A.data_ptr(), b.data_ptr(), in_w, out_w, ld, L.PIMHIP_ACT_RELU,
                                           L.PIMHIP_I_X_W, side.cuda_stream) == 0
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager) and all(torch.equal(o, eager) for o in others)


def test_a_product_with_one_odd_destination_needs_no_workspace(ops):
    """Several destinations: one that is not 16-byte aligned is enough."""
    g = torch.Generator().manual_seed(6)
    k, n = 2048, 512
    A, x = (0.1 * torch.randn(1, k, n, generator=g)).half().to(DEV), torch.randn(1, 1, k, generator=g).half().to(DEV)
    buf = torch.zeros(2, n + 8, dtype=torch.float16, device=DEV)
    outs = [buf[0, :n], buf[1, 1:n + 1]]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):            # (refused if it needed the stream's workspace)
        ops.aten_bmm(x, A, outs=outs)
    for _ in range(3):
        buf.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for o in outs:
            check(o, A[0].t(), x.view(-1), None, False)
        assert bool((buf[0, n:] == 0).all()) and float(buf[1, 0]) == 0


def test_a_recorded_product_outlives_a_larger_one_on_its_stream(ops):
    """A graph that holds a sliced product stays valid when products that exchange more partial sums run on its stream later."""
    from pimaicompiler_amd import _lib as L
    lib = L.load()
    side = torch.cuda.Stream()
    g = torch.Generator().manual_seed(5)

    def operands(k, n):
        return (0.1 * torch.randn(k, n, generator=g)).half().to(DEV), torch.randn(k, generator=g).half().to(DEV), torch.empty(n, dtype=torch.float16, device=DEV)

    def launch(A, x, y):
        return lib.pimhip_execute_gemv(y.data_ptr(), x.data_ptr(), A.data_ptr(), None, A.size(0), A.size(1), 0, L.PIMHIP_ACT_NONE, L.PIMHIP_I_X_W,
                                       torch.cuda.current_stream().cuda_stream)
    small, large = operands(2048, 256), operands(16384, 2048)
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        assert launch(*small) == 0
        with torch.cuda.graph(graph, stream=side):
            assert launch(*small) == 0
        for _ in range(3):
            assert launch(*large) == 0
            small[2].fill_(float("nan"))
            graph.replay()
            side.synchronize()
            check(small[2], small[0].t(), small[1], None, False)
            check(large[2], large[0].t(), large[1], None, False)
