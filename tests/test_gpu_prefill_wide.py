"""GPU parity of the wide-tile prefill kernel (csrc/q4_prefill_wide.hip) against the CPU oracle, at the edges of
its tiles and of the rule that picks it: ragged last token and weight tiles, one to an odd number of 128-column
steps (K = 128 .. 2304), outputs of every form, K split with a short last part, fp16 overflow.

Bar: max |gpu - oracle| <= 1e-2 * RMS(oracle) on f32 outputs; bf16 outputs are the RNE of a value within
1e-3 * RMS of the oracle.
"""
import numpy as np
import pytest
import torch

import oracle as O
from _util import assert_bf16_rounded_close, assert_rms_close, dev_bf16, host_bits, q4_dev, rms

pytestmark = pytest.mark.gpu


def synth():
    from kriya_q4 import synth as s
    return s


def case(msg):
    print(f"[case] {msg}", flush=True)


# 128 x 256 tiles (192 of them), 64 x 256 (192) and 64 x 128 (192), each with ragged edges
@pytest.mark.parametrize("m,n,k", [(129, 24573, 128), (257, 16376, 384), (65, 24568, 640), (64, 24571, 128),
                                   (191, 16384, 256)])
def test_plain_tiles(kq, m, n, k):
    case(f"wide prefill linear m={m} n={n} k={k}")
    s = synth()
    wq, x = s.q4_weight(n, k, 5000 + m), s.bf16_normal((m, k), 5001 + m)
    want = O.q4_matmul(O.Q4Planar(*wq), x)
    w, xd = q4_dev(kq, wq), dev_bf16(x)
    assert_rms_close(kq.q4_linear(w, xd, out_dtype=kq.DTYPE_F32).cpu().numpy(), want, what="f32")
    r0 = s.bf16_normal((m, n), 5002 + m)
    r = dev_bf16(r0).clone()
    kq.q4_linear(w, xd, y=r, accumulate=True)
    assert_bf16_rounded_close(host_bits(r), O.bf16_to_f32(r0) + want, rms(want), what="bf16 accumulate")


def test_qkv_bias_tiles(kq):
    """Three problems in one launch: tiles of each, biases, q_out whose row count ends inside a tile."""
    case("wide prefill qkv m=130")
    s = synth()
    m, k, ns = 130, 256, (20000, 1000, 4100)
    x = s.bf16_normal((m, k), 5100)
    ws = [s.q4_weight(n, k, 5101 + i) for i, n in enumerate(ns)]
    bs = [s.bf16_normal((1, n), 5110 + i)[0] for i, n in enumerate(ns)]
    outs = kq.qkv(*[q4_dev(kq, w) for w in ws], dev_bf16(x), *[dev_bf16(b) for b in bs], out_dtype=kq.DTYPE_F32)
    for i, n in enumerate(ns):
        want = O.q4_matmul(O.Q4Planar(*ws[i]), x) + O.bf16_to_f32(bs[i])[None, :]
        assert_rms_close(outs[i].cpu().numpy(), want, what=f"problem {i}")


@pytest.mark.parametrize("activation", [0, 1, 2])
@pytest.mark.parametrize("m,n,k", [(129, 24573, 256), (385, 12288, 128)])
def test_gate_up_tiles(kq, m, n, k, activation):
    case(f"wide prefill gate_up m={m} n={n} k={k} activation={activation}")
    s = synth()
    g, u, x = s.q4_weight(n, k, 5200), s.q4_weight(n, k, 5201), s.bf16_normal((m, k), 5202 + m)
    want = O.q4_gate_up_act(O.Q4Planar(*g), O.Q4Planar(*u), x, activation)
    got = kq.gate_up_act(q4_dev(kq, g), q4_dev(kq, u), dev_bf16(x), activation=activation)
    assert_rms_close(got.cpu().numpy(), want, what="f32")


@pytest.mark.parametrize("m,hidden,inter", [(385, 256, 12288), (641, 1024, 8256)])
def test_mlp_operands(kq, m, hidden, inter):
    """The MLP: x and the activation as fp16 operands converted once (inter 8256 = 129 groups: an odd count, whose
    down projection stays on the 64-column kernel)."""
    case(f"wide prefill mlp m={m} hidden={hidden} inter={inter}")
    s = synth()
    g, u, d = s.q4_weight(inter, hidden, 5301), s.q4_weight(inter, hidden, 5302), s.q4_weight(hidden, inter, 5303)
    x = s.bf16_normal((m, hidden), 5304)
    h = torch.zeros((m, hidden), dtype=torch.float32, device="cuda")
    kq.mlp(q4_dev(kq, g), q4_dev(kq, u), q4_dev(kq, d), h, x=dev_bf16(x))
    want = O.q4_mlp(O.Q4Planar(*g), O.Q4Planar(*u), O.Q4Planar(*d), x)
    for i in range(0, m, 16):
        assert_rms_close(h.cpu().numpy()[i], want[i], what=f"row {i}")


@pytest.mark.parametrize("m,n,k", [(385, 5112, 2304), (385, 5117, 2304), (300, 7168, 2048)])
def test_split_k(kq, m, n, k):
    """kr_q4_linear_ws: K split over blocks (36 groups in parts of 10, 10, 10 and 6), the same bits twice."""
    case(f"wide prefill split K m={m} n={n} k={k}")
    s = synth()
    wq, x = s.q4_weight(n, k, 5400), s.bf16_normal((m, k), 5401)
    want = O.q4_matmul(O.Q4Planar(*wq), x)
    w, xd, ws = q4_dev(kq, wq), dev_bf16(x), kq.linear_workspace(m, n, k)
    y = kq.q4_linear(w, xd, out_dtype=kq.DTYPE_F32, workspace=ws).cpu().numpy()
    assert_rms_close(y, want, what="f32")
    again = kq.q4_linear(w, xd, out_dtype=kq.DTYPE_F32, workspace=ws).cpu().numpy()
    assert np.array_equal(y.view(np.uint32), again.view(np.uint32))


def test_fp16_overflow_rows_exact(kq):
    """A row beyond fp16's range sends its blocks to the f32 tile; every row meets the bar by itself."""
    case("wide prefill fp16 overflow m=129 n=24576 k=256")
    s = synth()
    m, n, k = 129, 24576, 256
    wq = s.q4_weight(n, k, 5500)
    big = O.bf16_to_f32(s.bf16_normal((m, k), 5501)).copy()
    big[5] *= 1e5
    big[128] *= 1e5
    x = O.f32_to_bf16(big)
    want = O.q4_matmul(O.Q4Planar(*wq), x)
    got = kq.q4_linear(q4_dev(kq, wq), dev_bf16(x), out_dtype=kq.DTYPE_F32).cpu().numpy()
    for i in range(m):
        assert_rms_close(got[i], want[i], what=f"row {i}")


@pytest.mark.parametrize("m,n,k", [(129, 24573, 128), (65, 24568, 640), (64, 65521, 128)])
def test_overflow_leaves_other_outputs(kq, m, n, k):
    """Only outputs that are not finite are computed again: rows beside one beyond fp16's range keep their bits, and
    infinities and NaNs come out as the oracle has them."""
    case(f"wide prefill, rows beside an overflowing one m={m} n={n} k={k}")
    s = synth()
    wq, x = s.q4_weight(n, k, 5600 + m), s.bf16_normal((m, k), 5601 + m)
    w = q4_dev(kq, wq)
    plain = kq.q4_linear(w, dev_bf16(x), out_dtype=kq.DTYPE_F32).cpu().numpy()
    big = O.bf16_to_f32(x).copy()
    big[7, 3], big[40, 100], big[m - 1, k - 1], big[12, 0] = 1e5, np.inf, -np.inf, np.nan
    rows = [7, 40, m - 1, 12]
    xb = O.f32_to_bf16(big)
    got = kq.q4_linear(w, dev_bf16(xb), out_dtype=kq.DTYPE_F32).cpu().numpy()
    others = np.setdiff1d(np.arange(m), rows)
    assert np.array_equal(got[others].view(np.uint32), plain[others].view(np.uint32))
    want = O.q4_matmul(O.Q4Planar(*wq), xb[rows])
    assert_rms_close(got[7], want[0], what="row 7")
    assert np.array_equal(np.isnan(got[rows]), np.isnan(want)) and np.isnan(want[3]).all()
    inf = np.isinf(want)
    assert inf.any() and np.array_equal(np.isinf(got[rows]), inf) and np.array_equal(got[rows][inf], want[inf])


# m, n, k and the launch (test_launch_rules.py holds the rule to it): 128 x 256 tiles at one to five steps with ragged
# edges, and with K split by kr_q4_linear_ws, the last part shorter
PLAIN_42 = [((257, 20477, 256), (42, 1)), ((257, 20480, 640), (42, 1))]
SPLIT_42 = [((641, 1021, 4224), (42, 8)), ((1025, 1024, 4224), (42, 4)), ((1025, 2045, 6272), (42, 2))]
# m, hidden, inter and the launch of kr_q4_mlp's down projection, which reads the converted operand
MLP_DOWN = [((1025, 2048, 1024), (42, 1)), ((1025, 2048, 2176), (42, 2)), ((641, 2048, 4224), (42, 4)),
            ((769, 1024, 8320), (42, 8))]


def some_rows(m):
    return np.unique(np.r_[0, 1, 31, 32, 63, 64, 127, 128, m // 2, m - 2, m - 1])


@pytest.mark.parametrize("shape,launch", PLAIN_42)
def test_wide_tiles(kq, shape, launch):
    m, n, k = shape
    case(f"wide prefill 128 x 256 tiles m={m} n={n} k={k}")
    s = synth()
    wq, x = s.q4_weight(n, k, 5700 + k), s.bf16_normal((m, k), 5701)
    big = O.bf16_to_f32(x).copy()
    big[130, 5] = -3e5
    x = O.f32_to_bf16(big)
    rows = np.union1d(some_rows(m), [129, 130, 131])
    got = kq.q4_linear(q4_dev(kq, wq), dev_bf16(x), out_dtype=kq.DTYPE_F32).cpu().numpy()
    want = O.q4_matmul(O.Q4Planar(*wq), x[rows])
    for i, r in enumerate(rows):
        assert_rms_close(got[r], want[i], what=f"row {r}")
    assert np.isfinite(got).all()


@pytest.mark.parametrize("shape,launch", SPLIT_42)
def test_wide_split_k(kq, shape, launch):
    m, n, k = shape
    case(f"wide prefill split K {launch[1]} m={m} n={n} k={k}")
    s = synth()
    wq, x = s.q4_weight(n, k, 5800 + m), s.bf16_normal((m, k), 5801)
    big = O.bf16_to_f32(x).copy()
    big[33, [1, k - 1]] = 1e5, -2e5   # overflows in the first and the last part
    big[64, 70] = np.inf
    x = O.f32_to_bf16(big)
    w, xd, ws = q4_dev(kq, wq), dev_bf16(x), kq.linear_workspace(m, n, k)
    got = kq.q4_linear(w, xd, out_dtype=kq.DTYPE_F32, workspace=ws).cpu().numpy()
    rows = np.setdiff1d(np.union1d(some_rows(m), [33]), [64])
    want = O.q4_matmul(O.Q4Planar(*wq), x[rows])
    for i, r in enumerate(rows):
        assert_rms_close(got[r], want[i], what=f"row {r}")
    inf = O.q4_matmul(O.Q4Planar(*wq), x[64:65])[0]
    assert np.array_equal(np.isnan(got[64]), np.isnan(inf)) and np.array_equal(got[64][np.isinf(inf)], inf[np.isinf(inf)])
    y0 = s.bf16_normal((m, n), 5802)
    y = dev_bf16(y0).clone()
    kq.q4_linear(w, xd, y=y, accumulate=True, workspace=ws)
    for i, r in enumerate(rows):
        full = O.bf16_to_f32(y0[r]) + want[i]
        assert_bf16_rounded_close(host_bits(y)[r:r + 1], full[None], rms(want[i]), what=f"bf16 accumulate row {r}")


@pytest.mark.parametrize("shape,launch", MLP_DOWN)
def test_mlp_down_operand(kq, shape, launch):
    """The down projection on the wide kernel with the activation as its fp16 operand: rows against the oracle (one whose
    activations leave fp16 among them), and the same bits with the operand converted in the blocks
    (KR_OPT_PREFILL_OPERANDS = 0) and with the other tile order (KR_OPT_PREFILL_XCD_SPLIT = 0)."""
    m, hidden, inter = shape
    case(f"wide prefill mlp m={m} hidden={hidden} inter={inter}")
    s = synth()
    g, u, d = s.q4_weight(inter, hidden, 5901), s.q4_weight(inter, hidden, 5902), s.q4_weight(hidden, inter, 5903)
    big = O.bf16_to_f32(s.bf16_normal((m, hidden), 5904)).copy()
    big[40] *= 1e3
    x = O.f32_to_bf16(big)
    G, U, D, xd = q4_dev(kq, g), q4_dev(kq, u), q4_dev(kq, d), dev_bf16(x)
    ws = kq.mlp_workspace(m, hidden, inter)

    def run():
        h = torch.zeros((m, hidden), dtype=torch.float32, device="cuda")
        kq.mlp(G, U, D, h, x=xd, workspace=ws)
        return h.cpu().numpy()

    y = run()
    rows = np.union1d(some_rows(m), [40])
    want = O.q4_mlp(O.Q4Planar(*g), O.Q4Planar(*u), O.Q4Planar(*d), x[rows])
    act = O.q4_gate_up_act(O.Q4Planar(*g), O.Q4Planar(*u), x[40:41], 0)
    assert np.abs(act).max() > 65504
    for i, r in enumerate(rows):
        assert_rms_close(y[r], want[i], what=f"row {r}")
    for option in (kq.OPT_PREFILL_OPERANDS, kq.OPT_PREFILL_XCD_SPLIT):
        kq.set_option(option, 0)
        try:
            z = run()
        finally:
            kq.set_option(option, 1)
        assert np.array_equal(y.view(np.uint32), z.view(np.uint32)), option


def test_scale_planes_two_byte_aligned(kq):
    """Scale and bias planes need 2-byte alignment only: the same bits from planes that start two bytes further on."""
    case("wide prefill, scale planes on odd 2-byte boundaries")
    s = synth()
    m, n, k = 65, 12281, 384
    wq, xd = s.q4_weight(n, k, 5950), dev_bf16(s.bf16_normal((m, k), 5951))
    w = q4_dev(kq, wq)

    def shifted(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        buf[1:].copy_(t.view(-1))
        return buf[1:].view(t.shape)

    w2 = kq.Q4Matrix(w.qw, shifted(w.scales), shifted(w.biases))
    assert w2.scales.data_ptr() % 4 == 2 or w.scales.data_ptr() % 4 == 2
    a = kq.q4_linear(w, xd, out_dtype=kq.DTYPE_F32).cpu().numpy()
    b = kq.q4_linear(w2, xd, out_dtype=kq.DTYPE_F32).cpu().numpy()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
