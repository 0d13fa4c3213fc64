"""The memory that the f32 attention backward keeps dS in: its limit, its return, and the form without it."""
import ctypes

import numpy as np
import pytest

import oracle
from deers_amd import rocm, synth
from hipgraph import Graph

pytestmark = pytest.mark.gpu

MB = 1 << 20
B, H, T, D = 2, 20, 1024, 32  # 40 heads, 2.16 MB of dS each


@pytest.fixture(autouse=True)
def default_limit():
    rocm.init(0)
    yield
    rocm.sync()
    rocm.set_bwd_workspace_limit(-1)


def free_bytes():
    rocm.sync()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


class Backward:
    """Operands of one backward on the device; run() enqueues it, grads() reads the three gradients back."""

    def __init__(self, name, shape=(B, H, T, D)):
        self.shape = shape
        x = synth.attention_inputs(name, *shape, np.float32, base_seed=41)
        o, lse = rocm.attn_fwd(x["q"], x["k"], x["v"])
        self.x = x
        self.inputs = [rocm.DeviceBuffer.from_numpy(a) for a in (x["q"], x["k"], x["v"], o, lse, x["do"])]
        self.outputs = [rocm.DeviceBuffer.from_numpy(np.full(shape, np.nan, np.float32)) for _ in range(3)]

    def run(self):
        rocm.attn_bwd_raw(np.float32, *(b.ptr for b in self.inputs + self.outputs), *self.shape,
                          rocm.default_scale(self.shape[3]))

    def poison(self):
        for b in self.outputs:
            rocm.fill_raw(np.float32, b.ptr, int(np.prod(self.shape)), float("nan"))

    def grads(self):
        self.poison()
        self.run()
        return self.read()

    def read(self):
        return [b.numpy() for b in self.outputs]

    def kernels(self):
        rocm.profile_enable(True)
        self.run()
        names = rocm.profile_collect()
        rocm.profile_enable(False)
        return {n: calls for n, (calls, _) in names.items()}


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def test_the_memory_is_taken_on_use_and_given_back():
    p = Backward("ws-return")
    rocm.set_bwd_workspace_limit(0)
    rocm.empty_cache()
    without = free_bytes()
    rocm.set_bwd_workspace_limit(-1)
    want = p.grads()
    assert without - free_bytes() >= 80 * MB      # 40 heads x 2.16 MB
    rocm.empty_cache()
    assert without - free_bytes() <= 16 * MB      # the blocks read() has used apart
    assert same(p.grads(), want)
    rocm.set_bwd_workspace_limit(80 * MB)         # lower than what is held
    assert without - free_bytes() <= 16 * MB


def test_a_limit_means_some_heads_at_a_time_and_then_the_form_without_memory():
    p = Backward("ws-limit")
    want = p.grads()
    assert p.kernels() == {"attn_bwd_prep": 1, "attn_bwd_dkdv": 1, "attn_bwd_dq": 1}
    rocm.set_bwd_workspace_limit(50 * MB)         # 24 heads fit: two shares of 20, each fills the device
    assert p.kernels() == {"attn_bwd_prep": 1, "attn_bwd_dkdv": 2, "attn_bwd_dq": 2}
    assert same(p.grads(), want)
    for limit in (40 * MB, 2 * MB, 0):            # shares of 14 heads, which do not; no head fits; none
        rocm.set_bwd_workspace_limit(limit)
        assert p.kernels() == {"attn_bwd_f32": 1}, limit
    got = p.grads()
    assert not same(got, want)                    # sums in another order
    heads = (slice(1, 2), slice(7, 8))
    refs = oracle.attn_bwd(*(p.x[n][heads] for n in ("q", "k", "v", "do")))
    for a, b, r in zip(got, want, refs):
        assert np.max(np.abs(a.astype(np.float64) - b)) <= 1e-4
        assert np.max(np.abs(a[heads].astype(np.float64) - r)) <= 1e-4


def test_a_captured_backward_keeps_the_memory_it_was_captured_with():
    """Replayed between eager backwards of a larger geometry, which take other memory, and after the
    calls that give memory back."""
    p, larger = Backward("ws-graph"), Backward("ws-graph-larger", (3, 20, T, D))
    want = p.grads()
    want_larger = larger.grads()
    rocm.empty_cache()
    p.grads()
    graph = Graph(p.run)
    try:
        for between in (lambda: None, rocm.empty_cache, lambda: rocm.set_bwd_workspace_limit(0),
                        lambda: rocm.set_bwd_workspace_limit(-1), larger.run, rocm.empty_cache, larger.run):
            between()
            p.poison()
            graph.launch()
            assert same(p.read(), want)
        assert same(larger.grads(), want_larger)
    finally:
        graph.close()


def test_a_capture_without_the_memory_computes_ds_twice():
    p = Backward("ws-graph-none")
    rocm.set_bwd_workspace_limit(0)
    want = p.grads()
    rocm.set_bwd_workspace_limit(-1)
    rocm.empty_cache()
    larger = Backward("ws-graph-none-larger", (8, 20, T, D))
    graph = Graph(larger.run)                         # 346 MB: more than a graph of another test may have kept
    rocm.set_bwd_workspace_limit(0)
    want_larger = larger.grads()
    rocm.set_bwd_workspace_limit(-1)
    try:
        for _ in range(3):
            larger.poison()
            graph.launch()
            assert same(larger.read(), want_larger)
            assert not same(p.grads(), want)          # eager: with the memory
    finally:
        graph.close()
