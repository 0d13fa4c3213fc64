"""The f16 attention kernels that give a workgroup 32 rows: every form at the sizes where it can go wrong (a walk of one
block, of as many blocks as waves and one more, rows past the end of the last block), and the rule that chooses them."""
import numpy as np
import pytest

import oracle
from deers_amd import rocm, synth
from forms import takes_32_rows
from hipgraph import Graph

# relative 2-norm error of a result against the f32 oracle on the same f16 inputs: three roundings to f16 on the way
# (scores' operand or probability, score gradient, result), each 2^-12 / sqrt(3) in the root mean square, and the
# same again for what they do to small sums
REL = 2 * 3 ** 0.5 * 2.0 ** -12 / 3 ** 0.5


def takes(direction, heads, T, D):
    return takes_32_rows(direction, np.float16, heads, T, D)


def test_what_the_backward_takes_the_forward_takes_too():
    """Both then form their scores from Q itself; otherwise a probability would be recomputed from another score than
    the one it was normalised with."""
    for D in (32, 64, 128):
        for T in [32 * nb for nb in range(1, 140)] + [8192, 9000]:
            for BH in sorted({*range(1, 140), *range(140, 3000, 37), *(int(1.15 ** i) for i in range(70))}):
                assert not takes("bwd", BH, T, D) or takes("fwd", BH, T, D), (BH, T, D)


def test_the_f32_forward_leaves_the_32_row_form_at_one_size():
    """Up to a number of heads, and not again beyond it."""
    for D in (32, 64, 128):
        for T in [32 * nb for nb in range(1, 140)]:
            took = [takes_32_rows("fwd", np.float32, heads, T, D) for heads in range(1, 400)]
            assert took == sorted(took, reverse=True), (T, D)


def test_the_f16_lines_follow_the_lengths_around_them():
    """Walks of up to 11 blocks leave the 32-row form at one size, and the backward's line does not drop by more than a
    tenth between longer walks and others a few blocks longer."""
    for D in (32, 64, 128):
        for nb in range(1, 12):
            for direction in ("fwd", "bwd"):
                took = [takes(direction, heads, 32 * nb, D) for heads in range(1, 1500)]
                assert took == sorted(took, reverse=True), (direction, nb, D)
        line = [max(heads for heads in range(1, 200) if takes("bwd", heads, 32 * nb, D)) * nb for nb in range(17, 30)]
        for i in range(len(line) - 6):  # a head is up to 29 workgroups
            assert line[i] + 29 >= 0.9 * max(line[i:i + 7]), (D, 17 + i, line)


def rel(got, want):
    return float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want))


# BH, T: forms by waves (4 with K and V twice in LDS, 4, 2, 1), remainders of T / 32 and of the blocks by the waves
@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("BH,T", [(3, 1), (2, 31), (5, 33), (4, 97), (3, 129), (2, 160), (9, 417), (30, 255), (61, 250),
                                  (130, 200), (300, 65), (500, 100)])
def test_every_form_matches_the_oracle(BH, T, D):
    assert takes("fwd", BH, T, D)
    x = synth.attention_inputs(f"split-{BH}-{T}-{D}", 1, BH, T, D, np.float16, base_seed=61)
    print(f"{BH} x {T} x {D}", flush=True)
    got = rocm.attn_fwd_bwd(x["q"], x["k"], x["v"], x["do"])
    again = rocm.attn_fwd_bwd(x["q"], x["k"], x["v"], x["do"])
    for a, b in zip(got, again):
        np.testing.assert_array_equal(a, b)
    few = (slice(None), sorted({0, BH // 2, BH - 1}))
    o, lse = oracle.attn_fwd(x["q"][few], x["k"][few], x["v"][few], return_lse=True)
    refs = (o, lse, *oracle.attn_bwd(x["q"][few], x["k"][few], x["v"][few], x["do"][few]))
    for name, g, want in zip(("o", "lse", "dq", "dk", "dv"), got, refs):
        if name == "dq" and T == 1:  # one key: exactly zero but for the rounding of dO . (O - V)
            assert np.max(np.abs(g[few])) <= 2.0 ** -8
        elif name == "dk" and T == 1:
            assert np.max(np.abs(g[few])) <= 2.0 ** -8
        else:
            assert rel(g[few], want) <= REL, name


@pytest.mark.gpu
@pytest.mark.parametrize("BH,T,waves", [(100, 54, 2), (150, 54, 1), (50, 86, 4), (150, 86, 2), (300, 86, 1), (90, 118, 4),
                                        (200, 150, 2), (90, 246, 4), (250, 246, 1)])
def test_short_walks_at_head_width_32_have_the_waves_that_are_fastest(BH, T, waves):
    """Read from the captured launch; its result like any other's."""
    x = synth.attention_inputs(f"split-waves-{BH}-{T}", 1, BH, T, 32, np.float16, base_seed=64, names=("q", "k", "v"))
    q, k, v = (rocm.DeviceBuffer.from_numpy(x[n]) for n in ("q", "k", "v"))
    o, lse = rocm.DeviceBuffer((1, BH, T, 32), np.float16), rocm.DeviceBuffer((1, BH, T), np.float32)
    graph = Graph(lambda: rocm.attn_fwd_raw(np.float16, q.ptr, k.ptr, v.ptr, o.ptr, lse.ptr, 1, BH, T, 32, rocm.default_scale(32)))
    try:
        assert graph.threads() == [64 * waves]
        for _ in range(2):
            rocm.fill_raw(np.float16, o.ptr, BH * T * 32, float("nan"))
            graph.launch()
            few = (slice(None), sorted({0, BH // 2, BH - 1}))
            assert rel(o.numpy()[few], oracle.attn_fwd(x["q"][few], x["k"][few], x["v"][few])) <= REL
    finally:
        graph.close()


@pytest.mark.gpu
@pytest.mark.parametrize("T,D,stride", [(3, 64, 1 << 20), (40, 128, 1 << 14), (70, 32, 1 << 13)])
def test_rows_far_apart_give_the_same_bits(T, D, stride):
    """Row strides at which 32 rows reach past what a block's rows span; between the rows NaN."""
    H = 2
    x = synth.attention_inputs(f"split-far-{T}-{D}", 1, H, T, D, np.float16, base_seed=62)
    want = rocm.attn_fwd_bwd(x["q"], x["k"], x["v"], x["do"])
    st = (T * stride, D, stride, 1)

    def spread(a):
        buf = np.full((T, stride), np.nan, np.float16)
        for h in range(H):
            buf[:, h * D:h * D + D] = a[0, h]
        return rocm.DeviceBuffer.from_numpy(buf)

    bufs = {n: spread(x[n]) for n in ("q", "k", "v", "do")}
    outs = {n: rocm.DeviceBuffer((T, stride), np.float16) for n in ("o", "dq", "dk", "dv")}
    lse = rocm.DeviceBuffer((1, H, T), np.float32)
    scale = rocm.default_scale(D)
    rocm.attn_fwd_raw(np.float16, bufs["q"].ptr, bufs["k"].ptr, bufs["v"].ptr, outs["o"].ptr, lse.ptr, 1, H, T, D, scale,
                      q_strides=st, k_strides=st, v_strides=st, o_strides=st)
    rocm.attn_bwd_raw(np.float16, bufs["q"].ptr, bufs["k"].ptr, bufs["v"].ptr, outs["o"].ptr, lse.ptr, bufs["do"].ptr,
                      outs["dq"].ptr, outs["dk"].ptr, outs["dv"].ptr, 1, H, T, D, scale,
                      strides={n: st for n in ("q", "k", "v", "o", "do", "dq", "dk", "dv")})
    for name, ref in zip(("o", "dq", "dk", "dv"), (want[0], *want[2:])):
        got = outs[name].numpy()
        for h in range(H):
            np.testing.assert_array_equal(got[:, h * D:h * D + D], ref[0, h], err_msg=name)
    np.testing.assert_array_equal(lse.numpy(), want[1])
