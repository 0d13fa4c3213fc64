"""Calls captured into a HIP graph and replayed between the program's own eager calls."""
import multiprocessing

import numpy as np
import pytest

from deers_amd import rocm, synth
from forms import rows_128, takes_32_rows
from hipgraph import Graph

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def same_xcd():
    rocm.init(0)
    yield
    rocm.set_handover_mode(-1)


def grow_the_workspace():
    """A backward whose scaled queries need 126 MB of workspace, more than anything else here."""
    B, H, T, D = 40, 12, 2048, 64
    zeros = [rocm.DeviceBuffer((B, H, T, D), np.float16, zeros=True) for _ in range(3)]
    lse = rocm.DeviceBuffer((B, H, T), np.float32, zeros=True)
    q, k, dq = zeros
    rocm.attn_bwd_raw(np.float16, q.ptr, q.ptr, q.ptr, q.ptr, lse.ptr, q.ptr, dq.ptr, k.ptr, k.ptr, B, H, T, D, 0.125)
    rocm.sync()


def fill_free_memory():
    """Allocates and fills blocks of the sizes a freed workspace may be handed out again as."""
    blocks = [rocm.DeviceBuffer((mb << 20,), np.float16) for mb in (1, 1, 2, 4, 16)]
    for b in blocks:
        rocm.fill_raw(np.float16, b.ptr, b.shape[0], float("nan"))
    rocm.sync()
    return blocks


@pytest.mark.parametrize("B,H,L,D", [(1, 7, 1500, 64), (12, 11, 1100, 64)])
def test_a_captured_decode_with_splits_replays_when_the_workspace_has_grown(B, H, L, D):
    x = synth.attention_inputs(f"cap-dec-{B}-{H}-{L}-{D}", B, H, 1, D, np.float16, base_seed=43, kv_len=L,
                               names=("q", "k", "v"))
    q, k, v = (rocm.DeviceBuffer.from_numpy(x[n]) for n in ("q", "k", "v"))
    o = rocm.DeviceBuffer((B, H, D), np.float16)

    def decode(call=rocm.attn_decode_raw):
        call(np.float16, q.ptr, k.ptr, v.ptr, o.ptr, B, H, L, D, rocm.default_scale(D))

    decode()
    want = o.numpy()
    graph = Graph(decode)
    noalloc = Graph(lambda: decode(rocm.attn_decode_noalloc_raw))
    held = []
    try:
        for between in (lambda: None, decode, grow_the_workspace, rocm.empty_cache,
                        lambda: held.extend(fill_free_memory()), decode):
            between()
            for g in (graph, noalloc):
                rocm.fill_raw(np.float16, o.ptr, B * H * D, float("nan"))
                g.launch()
                np.testing.assert_array_equal(o.numpy(), want)
    finally:
        graph.close()
        noalloc.close()


def test_a_captured_few_rows_product_and_lookup_replay():
    """K split over workgroups (3072 in four) and an index kernel; index 99 is out of range and reported by the
    eager call that raises the flag, not by the replays of a graph without it."""
    m, n, k = 5, 768, 3072
    rng = np.random.default_rng(47)
    x = rocm.DeviceBuffer.from_numpy(rng.standard_normal((m, k)).astype(np.float16))
    w = rocm.DeviceBuffer.from_numpy((rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float16))
    y = rocm.DeviceBuffer((m, n), np.float16)
    table = rocm.DeviceBuffer.from_numpy(rng.standard_normal((50, 64)).astype(np.float16))
    good, bad = (rocm.DeviceBuffer.from_numpy(np.array(i, np.int64)) for i in ([3, 49, 0], [3, 99, 0]))
    rows = rocm.DeviceBuffer((3, 64), np.float16)

    def calls():
        rocm.decode_linear_raw(np.float16, "plain", 0.0, x.ptr, k, w.ptr, n, y.ptr, False, m, n, k)
        rocm.index_select_raw(np.float16, table.ptr, good.ptr, rows.ptr, 50, 3, 64)

    graph = Graph(calls)
    try:
        calls()
        want = y.numpy(), rows.numpy()
        np.testing.assert_array_equal(want[1], table.numpy()[[3, 49, 0]])
        for _ in range(3):
            rocm.fill_raw(np.float16, y.ptr, m * n, float("nan"))
            graph.launch()
            np.testing.assert_array_equal(y.numpy(), want[0])
            np.testing.assert_array_equal(rows.numpy(), want[1])
            rocm.index_select_raw(np.float16, table.ptr, bad.ptr, rows.ptr, 50, 3, 64)
            with pytest.raises(rocm.RocmError, match="out of bounds"):
                rocm.sync()
            calls()
            np.testing.assert_array_equal(y.numpy(), want[0])
    finally:
        graph.close()


@pytest.mark.parametrize("B,H,T,D,rows", [(7, 12, 300, 64, 128), (4, 11, 257, 128, 128), (2, 3, 300, 64, 32)])
def test_a_captured_f16_backward_replays(B, H, T, D, rows):
    """The 128-row kernels hand statistics over: captured, they are two launches without flags (a replay could be given
    no fresh epoch).  Eager backwards of the same and of another geometry between the replays move the epochs on."""
    with rows_128(rows == 128):
        assert takes_32_rows("bwd", np.float16, B * H, T, D) == (rows == 32)
        captured_backward(B, H, T, D)


def captured_backward(B, H, T, D):
    dtype = np.float16
    x = synth.attention_inputs(f"cap-bwd-{B}-{H}-{T}-{D}", B, H, T, D, dtype, base_seed=45)
    want = rocm.attn_fwd_bwd(x["q"], x["k"], x["v"], x["do"])
    ins = [rocm.DeviceBuffer.from_numpy(a) for a in (x["q"], x["k"], x["v"], want[0], want[1], x["do"])]
    grads = [rocm.DeviceBuffer((B, H, T, D), dtype) for _ in range(3)]

    def backward():
        rocm.attn_bwd_raw(dtype, *(b.ptr for b in ins + grads), B, H, T, D, rocm.default_scale(D))

    graph = Graph(backward)
    try:
        for between in (lambda: None, backward, grow_the_workspace, backward):
            between()
            for g in grads:
                rocm.fill_raw(dtype, g.ptr, B * H * T * D, float("nan"))
            graph.launch()
            for got, ref in zip(grads, want[2:]):
                np.testing.assert_array_equal(got.numpy(), ref)
    finally:
        graph.close()


def test_a_captured_f16_backward_without_workspace_or_flags():
    """12000 heads need more flags than any other call of these tests: captured first, the launch takes the form
    without them.  Then eagerly, which grows both, and with the graph's replays in between: each the same bits as
    before, one head against the oracle."""
    import oracle
    B, H, T, D = 60, 200, 40, 32
    rng = np.random.default_rng(49)
    x = {n: rng.standard_normal((B, H, T, D), np.float32).astype(np.float16) for n in ("q", "k", "v", "do")}
    o, lse = rocm.attn_fwd(x["q"], x["k"], x["v"])
    ins = [rocm.DeviceBuffer.from_numpy(a) for a in (x["q"], x["k"], x["v"], o, lse, x["do"])]
    grads = [rocm.DeviceBuffer((B, H, T, D), np.float16) for _ in range(3)]

    def backward():
        rocm.attn_bwd_raw(np.float16, *(b.ptr for b in ins + grads), B, H, T, D, rocm.default_scale(D))

    def clear():
        for g in grads:
            rocm.fill_raw(np.float16, g.ptr, B * H * T * D, float("nan"))

    one = (slice(B - 1, B), slice(H - 1, H))
    refs = oracle.attn_bwd(*(x[n][one] for n in ("q", "k", "v", "do")))
    graph = Graph(backward)
    results = {"graph": [], "eager": []}
    try:
        for kind in ("graph", "graph", "eager", "graph", "eager"):
            clear()
            graph.launch() if kind == "graph" else backward()
            results[kind].append([g.numpy() for g in grads])
            for got, ref in zip(results[kind][-1], refs):
                assert np.max(np.abs(got[one].astype(np.float64) - ref)) <= 5e-3
    finally:
        graph.close()
    for runs in results.values():
        for run in runs[1:]:
            for a, b in zip(run, runs[0]):
                np.testing.assert_array_equal(a, b)


# BH, T, D, waves: launches of the 128-row kernel, in the form that needs neither its workspace nor its flags
FIRST_CAPTURED = [(300, 256, 128, 1), (60, 1024, 64, 2), (70, 700, 32, 2), (30, 1300, 128, 2), (200, 600, 64, 1)]


def capture_first():
    """In a process that has run no backward before, so that every capture finds neither."""
    import oracle
    rocm.init(0)
    for BH, T, D, waves in FIRST_CAPTURED:
        print(f"captured first: {BH} x {T} x {D}", flush=True)
        assert not takes_32_rows("bwd", np.float16, BH, T, D)
        x = synth.attention_inputs(f"cap-first-{BH}-{T}-{D}", 1, BH, T, D, np.float16, base_seed=46)
        o, lse = rocm.attn_fwd(x["q"], x["k"], x["v"])
        ins = [rocm.DeviceBuffer.from_numpy(a) for a in (x["q"], x["k"], x["v"], o, lse, x["do"])]
        grads = [rocm.DeviceBuffer((1, BH, T, D), np.float16) for _ in range(3)]
        graph = Graph(lambda: rocm.attn_bwd_raw(np.float16, *(b.ptr for b in ins + grads), 1, BH, T, D, rocm.default_scale(D)))
        assert graph.threads() == [64 * waves], (graph.threads(), waves)
        one = (slice(0, 1), slice(BH - 1, BH))
        refs = oracle.attn_bwd(*(x[n][one] for n in ("q", "k", "v", "do")))
        for _ in range(2):
            for g in grads:
                rocm.fill_raw(np.float16, g.ptr, BH * T * D, float("nan"))
            graph.launch()
            for got, ref in zip(grads, refs):
                assert np.max(np.abs(got.numpy()[one].astype(np.float64) - ref)) <= 5e-3
        graph.close()


def test_a_backward_that_is_captured_first_has_as_many_waves_as_its_size_asks_for():
    """One where many workgroups of short walks cover the device, two for longer ones."""
    child = multiprocessing.get_context("spawn").Process(target=capture_first)
    child.start()
    child.join(100)
    if child.is_alive():
        child.kill()
    assert child.exitcode == 0
