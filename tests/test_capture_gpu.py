"""Calls captured into a HIP graph and replayed between the program's own eager calls."""
import numpy as np
import pytest

from deers_amd import rocm, synth
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
