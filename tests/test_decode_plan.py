"""Decode attention: which heads stay whole, which are split, and the streams at the edges of a tile."""
import ctypes

import numpy as np
import pytest

import oracle
from deers_amd import rocm, synth

TILE = {32: 256, 64: 128, 128: 64}  # cache rows of a workgroup's tile


@pytest.fixture
def gpu():
    if not rocm.available():
        pytest.fail("no gfx950 device")
    rocm.init(0)
    yield
    rocm.set_handover_mode(-1)


def plan(heads, L, D):
    pick = rocm.load()["_ZN5deers17decode_pick_wholeElllPiS0_"]
    splits, chunk = ctypes.c_int(), ctypes.c_int()
    i64 = ctypes.c_int64
    whole = pick(i64(heads), i64(L), i64(D), ctypes.byref(splits), ctypes.byref(chunk))
    return whole, splits.value, chunk.value


def test_every_row_belongs_to_one_workgroup_and_the_partials_fit():
    """On the host: whole heads only where they fill the 32 CUs of an XCD, splits that cover the cache once and are
    never empty, no more of them than the merge holds (32) and the static memory takes."""
    for D in (32, 64, 128):
        for L in (1, 16, TILE[D], 2 * TILE[D], 2 * TILE[D] + 1, 4 * TILE[D] + 1, 5 * TILE[D] + 1, 1024, 4111, 65536):
            for heads in list(range(1, 300)) + [320, 384, 391, 393, 512, 520, 640, 65535]:
                whole, splits, chunk = plan(heads, L, D)
                per_xcd = (heads + 7) // 8
                assert 1 <= splits <= 32 and whole % 32 == 0 and whole < per_xcd, (D, L, heads)
                assert splits * chunk >= L > (splits - 1) * chunk, (D, L, heads)
                assert whole == 0 or (splits > 1 and (per_xcd - whole) * splits <= 32), (D, L, heads)
                assert splits == 1 or (heads - 8 * whole) * splits * (D + 2) * 4 <= 512 * 1024, (D, L, heads)
                if L <= 2 * TILE[D]:
                    assert splits == 1, (D, L, heads)


def bound(x):
    """One rounding to f16, and weights off by the error of D f32 products and sums under them, at most
    D * 2^-24 * sum |q k| * scale for normal inputs: 2^-10 with room."""
    return (2.0 ** -11 + 2.0 ** -10) * np.max(np.abs(x["v"].astype(np.float64)))


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,L,D", [(1, 3, 256, 64), (1, 3, 257, 64), (1, 3, 512, 32), (2, 4, 1537, 32), (1, 5, 129, 128),
                                     (1, 2, 2049, 64), (1, 1, 16385, 128), (1, 9, 8200, 32),
                                     (3, 87, 130, 128), (8, 33, 300, 64), (2, 131, 1031, 32), (5, 53, 385, 64),
                                     (8, 48, 700, 64), (8, 49, 700, 64), (67, 8, 601, 128), (65, 8, 257, 64)])
def test_decode_at_the_edges_of_the_plan(gpu, B, H, L, D):
    """Caches of two tiles and one row more, up to 32 splits (two batches of a merge), 33 heads of an XCD and up with
    fewer on some XCDs; merged in the launch, after it, and in the static memory: the same bits."""
    x = synth.attention_inputs(f"plan-{B}-{H}-{L}-{D}", B, H, 1, D, np.float16, base_seed=23, kv_len=L,
                               names=("q", "k", "v"))
    q, k, v = (rocm.DeviceBuffer.from_numpy(x[n]) for n in ("q", "k", "v"))
    outs = []
    for mode in (rocm.HANDOVER_SAME_XCD, rocm.HANDOVER_STREAM_ORDER, rocm.HANDOVER_SAME_XCD):
        rocm.set_handover_mode(mode)
        for call in (rocm.attn_decode_raw, rocm.attn_decode_noalloc_raw):
            o = rocm.DeviceBuffer.from_numpy(np.full((B, H, D), np.nan, np.float16))
            call(np.float16, q.ptr, k.ptr, v.ptr, o.ptr, B, H, L, D, rocm.default_scale(D))
            outs.append(o.numpy())
    want = oracle.attn_fwd(x["q"], x["k"], x["v"])[:, :, 0]
    assert np.max(np.abs(outs[0].astype(np.float64) - want)) <= bound(x)
    for other in outs[1:]:
        np.testing.assert_array_equal(outs[0], other)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,D,pos", [(1, 2, 64, 0), (33, 8, 64, 0), (1, 3, 64, 128), (1, 2, 32, 513), (3, 89, 64, 300),
                                       (8, 40, 128, 129)])
def test_an_appending_decode_at_the_edges_of_the_plan(gpu, B, H, D, pos):
    """From an empty cache on: the last split, or the whole head, attends over the new row as well.  No rotation
    (cos 1, sin 0), so that the plain attention over pos + 1 rows is the result."""
    x = synth.attention_inputs(f"plan-app-{B}-{H}-{pos}-{D}", B, H, 1, D, np.float16, base_seed=29, kv_len=pos + 1,
                               names=("q", "k", "v"))
    cap = pos + 3
    caches, rows = [], []
    for n in ("k", "v"):
        c = np.full((B, H, cap, D), np.nan, np.float16)
        c[:, :, :pos] = x[n][:, :, :pos]
        caches.append(rocm.DeviceBuffer.from_numpy(c))
        rows.append(rocm.DeviceBuffer.from_numpy(np.ascontiguousarray(x[n][:, :, pos])))
    q = rocm.DeviceBuffer.from_numpy(np.ascontiguousarray(x["q"][:, :, 0]))
    cos, sin = (rocm.DeviceBuffer.from_numpy(np.full(D // 2, c, np.float16)) for c in (1, 0))
    o = rocm.DeviceBuffer.from_numpy(np.full((B, H, D), np.nan, np.float16))
    rocm.attn_decode_append_raw(np.float16, q.ptr, rows[0].ptr, rows[1].ptr, (H * D, D), cos.ptr, sin.ptr, caches[0].ptr,
                                caches[1].ptr, (H * cap * D, cap * D, D), o.ptr, pos, cap, B, H, D, rocm.default_scale(D))
    want = oracle.attn_fwd(x["q"], x["k"], x["v"])[:, :, 0]
    assert np.max(np.abs(o.numpy().astype(np.float64) - want)) <= bound(x)
    for c, n in zip(caches, ("k", "v")):
        np.testing.assert_array_equal(c.numpy()[:, :, pos], x[n][:, :, pos])
        assert np.isnan(c.numpy()[:, :, pos + 1:]).all()
