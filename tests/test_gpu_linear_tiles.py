"""linear_f16w on split rows copied memory-to-LDS (linear_tile_kernel): every tile shape at its
edges against the oracle, the same bits beside other outputs where the tiles sum alike, and calls
that find no room for the split rows."""
import numpy as np
import pytest

import eyebrowse_amd as eb
import oracle
from tests._gpu import assert_bitwise, assert_close, note, upload

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return eb.Device.new(0)


def _run(dev, x, ws, m, in_f):
    """One launch for all of ws; the outputs start as NaN, so an element left out shows."""
    xt = upload(dev, x)
    wts = [eb.Tensor.from_f16_packed(dev, w.shape, w) for w in ws]
    cs = [upload(dev, np.full((m, w.shape[0]), np.nan, np.float32)) for w in ws]
    rec = eb.Recorder(dev)
    eb.linear_f16w_multi(rec, xt, wts, cs, [w.shape[0] for w in ws], m, in_f)
    rec.submit()
    return [c.to_f32().reshape(m, -1) for c in cs]


# (rows, contraction, features of each output): which shape runs follows the cost model; the
# sizes put the rows and features on, below and above its 32 .. 256 edges.
CASES = [
    (9, 128, (1,)), (31, 256, (33, 32)), (32, 1024, (4096,)), (33, 128, (31, 65, 64)),   # 32 x 32
    (65, 4096, (1000, 513)), (96, 1024, (4095,)),                                          # 32 x 64
    (255, 1024, (4100, 63)), (256, 128, (20000,)),                                         # 64 x 64
    (9, 64, (40,)), (40, 192, (129,)), (257, 64, (64, 1)), (319, 1024, (1001,)),           # one sum
    (513, 128, (2049, 100)), (700, 1024, (4095,)), (1025, 2048, (1025,)),
    (1000, 4096, (4095, 1)), (2049, 64, (4097,)), (2000, 1024, (4096, 250)), (4095, 1024, (4090,)),
    (300, 8256, (300,)),                                                                   # rows read twice
]


@pytest.mark.parametrize("m,in_f,outs", CASES)
def test_tiles_match_oracle(dev, m, in_f, outs):
    note(f"linear tiles m={m} in={in_f} outs={outs}")
    x = oracle.randn((m, in_f), 1)
    x[::3] *= np.float32(1e-6)   # rows of their own scale
    ws = [oracle.randn((o, in_f), 2 + i) * np.float32(in_f ** -0.5) for i, o in enumerate(outs)]
    got = _run(dev, x, ws, m, in_f)
    rows = sorted({r for r in (0, 1, 31, 32, 63, 64, 127, 128, 255, 256, m // 2, m - 2, m - 1)
                   if 0 <= r < m})
    for g, w in zip(got, ws):
        assert np.isfinite(g).all()
        want = oracle.linear_f16w(x[rows], oracle.f16_bits(w), len(rows), in_f, w.shape[0],
                                  threads=16)
        scale = np.abs(x[rows]).max(1, keepdims=True)
        assert_close(g[rows] / scale, want / scale, what=f"{w.shape[0]} features")


@pytest.mark.parametrize("m", [40, 256, 257, 700])
def test_bits_do_not_depend_on_the_launch(dev, m):
    """An output's sums are the same whether it is launched alone or beside others, where the tiles
    of both launches sum alike: all of those for up to 256 rows, and the smaller three beyond (other
    widths of row and feature; the two largest sum in one chain, so a fused and a separate
    projection may differ in their last bits on long prompts)."""
    note(f"linear tiles alone and together m={m}")
    in_f, outs = 1024, (2048, 100, 3000)
    x = oracle.randn((m, in_f), 5)
    ws = [oracle.randn((o, in_f), 6 + i) * np.float32(0.03) for i, o in enumerate(outs)]
    together = _run(dev, x, ws, m, in_f)
    for t, w in zip(together, ws):
        assert_bitwise(_run(dev, x, [w], m, in_f)[0], t, f"{w.shape[0]} features")


def test_extreme_rows(dev):
    """Row scales from 1e-38 to 1e30, zeros, infinities and NaN, as on the other path."""
    note("linear tiles extreme rows")
    m, in_f, out_f = 40, 256, 96
    x = oracle.randn((m, in_f), 7)
    for i in range(30):
        x[i] *= np.float32(10.0 ** (-37 + 2.3 * i))
    x[30] = 0.0
    x[31, 5], x[32, 9] = np.inf, np.nan
    w = oracle.randn((out_f, in_f), 8) * np.float32(0.05)
    got = _run(dev, x, [w], m, in_f)[0]
    want = oracle.linear_f16w(x, oracle.f16_bits(w), m, in_f, out_f, threads=16)
    for i in list(range(30)) + list(range(33, 40)):
        scale = float(np.max(np.abs(want[i])))
        assert_close(got[i] / scale, want[i] / scale, what=f"row {i}")
    assert np.array_equal(got[30], np.zeros(out_f, np.float32))
    assert not np.isfinite(got[31:33]).any()


def test_capture_without_room_for_the_split_rows():
    """A capture that can use the workspace as it is, but not grow it, still records the product;
    replays give its result."""
    note("linear tiles capture without room")
    dev = eb.Device.new(0)
    m, in_f, out_f = 12, 256, 80
    xs = oracle.randn((16, 40), 1)
    rec = eb.Recorder(dev)
    c0 = eb.Tensor.empty(dev, (16, 8))
    eb.linear_f16w(rec, upload(dev, xs), eb.Tensor.from_f16_packed(dev, (8, 40), oracle.randn((8, 40), 2)),
                   c0, 16, 40, 8)   # leaves a workspace of 16 floats
    rec.submit()
    x = oracle.randn((m, in_f), 3)
    w = oracle.randn((out_f, in_f), 4) * np.float32(0.05)
    xt, wt = upload(dev, x), eb.Tensor.from_f16_packed(dev, w.shape, w)
    ct = upload(dev, np.full((m, out_f), np.nan, np.float32))
    dev.begin_capture()
    rec = eb.Recorder(dev)
    eb.linear_f16w(rec, xt, wt, ct, m, in_f, out_f)
    rec.submit()
    g = dev.end_capture()
    want = oracle.linear_f16w(x, oracle.f16_bits(w), m, in_f, out_f, threads=16)
    for _ in range(3):
        ct.write(np.full((m, out_f), np.nan, np.float32))
        g.launch()
        dev.synchronize()
        assert_close(ct.to_f32().reshape(m, out_f), want, what="replay")
    g.release()


def _cold_device():
    """A device whose workspace holds 2048 floats: row exponents, but no split rows."""
    dev = eb.Device.new(0)
    rec = eb.Recorder(dev)
    eb.linear_f16w(rec, upload(dev, oracle.randn((2048, 8), 1)),
                   eb.Tensor.from_f16_packed(dev, (8, 8), oracle.randn((8, 8), 2)),
                   eb.Tensor.empty(dev, (2048, 8)), 2048, 8, 8)
    rec.submit()
    return dev


def test_a_capture_records_what_an_eager_call_does(dev):
    """A captured product is the same bits as an eager one, whatever the workspace held when it was
    captured: several products in one capture, replays between eager work, a recapture."""
    note("linear tiles capture bits")
    cold = _cold_device()
    shapes = [(300, 1024, 100), (12, 256, 80), (700, 2048, 1000)]  # the second within the first's room
    data = [(oracle.randn((m, k), 3 + i), oracle.randn((n, k), 13 + i) * np.float32(k ** -0.5))
            for i, (m, k, n) in enumerate(shapes)]
    want = [_run(dev, x, [w], *x.shape)[0] for x, w in data]
    xts = [upload(cold, x) for x, _ in data]
    wts = [eb.Tensor.from_f16_packed(cold, w.shape, w) for _, w in data]
    cts = [eb.Tensor.empty(cold, (m, n)) for m, _, n in shapes]

    def capture(graph=None):
        cold.begin_capture()
        try:
            rec = eb.Recorder(cold)
            for xt, wt, ct, (m, k, n) in zip(xts, wts, cts, shapes):
                eb.linear_f16w(rec, xt, wt, ct, m, k, n)
            rec.submit()
        finally:
            g = cold.end_capture(graph) if graph else cold.end_capture()
        return g

    graph = capture()
    other = (oracle.randn((900, 1024), 31), oracle.randn((64, 1024), 32) * np.float32(0.03))
    for rep in range(4):
        if rep == 3:
            graph = capture(graph)
        for ct, (m, _, n) in zip(cts, shapes):
            ct.write(np.full((m, n), np.nan, np.float32))
        graph.launch()
        for ct, w in zip(cts, want):
            assert_bitwise(ct.to_f32(), w, f"replay {rep}")
        # eager work between the replays, which grows the workspace and takes pooled buffers
        got = _run(cold, other[0], [other[1]], 900, 1024)[0]
        assert_bitwise(got, _run(dev, other[0], [other[1]], 900, 1024)[0], "eager")
    graph.release()


def test_a_deferred_recorder_does_what_an_eager_call_does(dev):
    note("linear tiles deferred bits")
    m, in_f, out_f = 12, 256, 80
    x, w = oracle.randn((m, in_f), 5), oracle.randn((out_f, in_f), 6) * np.float32(0.03)
    want = _run(dev, x, [w], m, in_f)[0]
    cold = _cold_device()
    xt, wt, ct = upload(cold, x), eb.Tensor.from_f16_packed(cold, w.shape, w), eb.Tensor.empty(cold, (m, out_f))
    for _ in range(2):
        ct.write(np.full((m, out_f), np.nan, np.float32))
        rec = eb.Recorder(cold, deferred=True)
        eb.linear_f16w(rec, xt, wt, ct, m, in_f, out_f)
        rec.submit()
        assert_bitwise(ct.to_f32(), want, "deferred")


def test_raw_launch_with_room_for_the_split_rows(dev):
    """A raw launch given m exponents (to whole 64 floats) and the split rows takes the same path
    as the recorder."""
    note("linear tiles raw")
    m, in_f, out_f = 50, 1024, 320
    x = oracle.randn((m, in_f), 20)
    w = oracle.randn((out_f, in_f), 21) * np.float32(0.05)
    xt, wt = upload(dev, x), eb.Tensor.from_f16_packed(dev, w.shape, w)
    ct = eb.Tensor.empty(dev, (m, out_f))
    n = 64 + m * in_f
    ws = upload(dev, np.full(n, np.nan, np.float32))
    eb.launch_linear_f16w(dev.stream, xt.data_ptr, xt.numel(), wt.data_ptr, 2 * wt.numel(),
                          ct.data_ptr, ct.numel(), m, in_f, out_f, ws.data_ptr, n)
    dev.synchronize()
    assert_bitwise(ct.to_f32(), _run(dev, x, [w], m, in_f)[0], "raw against recorder")


@pytest.mark.parametrize("m,in_f,limit", [(300, 1024, 2.5e-7), (1000, 1024, 2.5e-7), (300, 4096, 4.9e-7)])
def test_sums_are_cut_in_two(dev, m, in_f, limit):
    """Rows past the few that several waves share: the error against 64 bits is that of two chains
    of sums, not of one. Each chain's roundings are half as many, of half the size, so one chain
    is sqrt(2) further off (measured: 2.1e-7 and 2.9e-7 at 1024, 4.1e-7 and 5.8e-7 at 4096, each
    within 1 % over sizes and inputs); the limit lies half way."""
    note(f"linear tiles precision m={m} in={in_f}")
    x = oracle.randn((m, in_f), 30)
    w = (oracle.randn((1024, in_f), 31) * np.float32(in_f ** -0.5)).astype(np.float16)
    got = _run(dev, x, [w.astype(np.float32)], m, in_f)[0].astype(np.float64)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= limit, err


def test_a_refused_call_leaves_the_workspace():
    """A call whose sizes do not fit its tensors is refused before the workspace grows for it. A
    capture shows the workspace: it takes a call whose row exponents have room, and no other."""
    note("linear refused call")
    dev = eb.Device.new(0)
    x, wt = upload(dev, oracle.randn((16, 40), 1)), eb.Tensor.from_f16_packed(dev, (8, 40), oracle.randn((8, 40), 2))
    ct = eb.Tensor.empty(dev, (16, 8))
    rec = eb.Recorder(dev)
    with pytest.raises(eb.ShapeMismatch):
        eb.linear_f16w(rec, x, wt, ct, 64, 64, 8)
    rec.submit()
    dev.begin_capture()
    rec = eb.Recorder(dev)
    with pytest.raises(eb.EyebrowseError, match="would have to grow"):
        eb.linear_f16w(rec, x, wt, ct, 16, 40, 8)
    rec.release()
    dev.end_capture().release()


def test_rows_that_are_not_split_take_no_room_for_it():
    """No outputs: nothing to launch, so no room for split rows."""
    note("linear no outputs")
    dev = eb.Device.new(0)
    x = upload(dev, oracle.randn((16, 64), 1))
    rec = eb.Recorder(dev)
    eb.linear_f16w(rec, x, eb.Tensor.empty(dev, (0, 64), eb.DType.F16), eb.Tensor.empty(dev, (16, 0)), 16, 64, 0)
    rec.submit()
    wt, ct = eb.Tensor.from_f16_packed(dev, (8, 40), oracle.randn((8, 40), 2)), eb.Tensor.empty(dev, (17, 8))
    xt = upload(dev, oracle.randn((17, 40), 3))
    dev.begin_capture()
    rec = eb.Recorder(dev)
    with pytest.raises(eb.EyebrowseError, match="would have to grow"):
        eb.linear_f16w(rec, xt, wt, ct, 17, 40, 8)
    rec.release()
    dev.end_capture().release()
