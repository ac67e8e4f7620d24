"""GPU parity of the few-token kernel's slab loop (K of several 2048-column slabs, no workspace) against the CPU
oracle: one to many tiles per block (more than it sums at a time), odd 64-group counts, a short last slab, one to
four groups of 16 token rows, both group widths, and q/k/v tiles that cross a problem inside a block's run.

Bar: max |gpu - oracle| <= 1e-2 * RMS(oracle); the loop's sums are f32 of exact products, so also
2e-5 * RMS(oracle) on f32 outputs (the oracle adds up to 19000 products one after the other in f32: about
2^-24 sqrt(19000 / 3), times 4.5 for the largest of 1e5).
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


@pytest.mark.parametrize("m,n,k", [(17, 77, 2112), (27, 2048, 4160), (32, 40, 8192), (33, 130, 4096), (63, 300, 6208),
                                   (48, 33, 2176), (2, 50, 16448), (5, 100, 18944), (16, 65, 16512)])
def test_linear(kq, m, n, k):
    case(f"slab loop linear m={m} n={n} k={k}")
    s = synth()
    wq, x = s.q4_weight(n, k, 7000 + m), s.bf16_normal((m, k), 7001 + m)
    want = O.q4_matmul(O.Q4Planar(*wq), x)
    w, xd = q4_dev(kq, wq), dev_bf16(x)
    assert_rms_close(kq.q4_linear(w, xd, out_dtype=kq.DTYPE_F32).cpu().numpy(), want, rel=2e-5, what="f32")
    r0 = s.bf16_normal((m, n), 7002 + m)
    r = dev_bf16(r0).clone()
    kq.q4_linear(w, xd, y=r, accumulate=True)
    assert_bf16_rounded_close(host_bits(r), O.bf16_to_f32(r0) + want, rms(want), what="bf16 accumulate")
    y = torch.zeros((m, n), dtype=torch.float32, device="cuda") + 1.0
    kq.q4_linear(w, xd, y=y, accumulate=True)
    assert_rms_close(y.cpu().numpy(), want + 1.0, rel=2e-5, what="f32 accumulate")


@pytest.mark.parametrize("m,n,k,act", [(2, 35, 2112, 0), (4, 300, 4096, 1), (16, 33000, 2176, 0), (17, 129, 4160, 2),
                                       (32, 1000, 6144, 0)])
def test_gate_up(kq, m, n, k, act):
    case(f"slab loop gate_up m={m} n={n} k={k} activation={act}")
    s = synth()
    g, u, x = s.q4_weight(n, k, 7100), s.q4_weight(n, k, 7101), s.bf16_normal((m, k), 7102)
    want = O.q4_gate_up_act(O.Q4Planar(*g), O.Q4Planar(*u), x, act)
    got = kq.gate_up_act(q4_dev(kq, g), q4_dev(kq, u), dev_bf16(x), activation=act)
    assert_rms_close(got.cpu().numpy(), want, what="f32")


@pytest.mark.parametrize("m,k", [(2, 3584), (16, 2112), (31, 4160)])
def test_qkv(kq, m, k):
    case(f"slab loop qkv m={m} k={k}")
    s = synth()
    ns = (4500, 40, 300)  # about 300 tiles: runs of two that cross from one problem into the next
    x = s.bf16_normal((m, k), 7200)
    ws = [s.q4_weight(n, k, 7201 + i) for i, n in enumerate(ns)]
    bs = [s.bf16_normal((1, n), 7210 + i)[0] for i, n in enumerate(ns)]
    outs = kq.qkv(*[q4_dev(kq, w) for w in ws], dev_bf16(x), *[dev_bf16(b) for b in bs], out_dtype=kq.DTYPE_F32)
    for i in range(3):
        want = O.q4_matmul(O.Q4Planar(*ws[i]), x) + O.bf16_to_f32(bs[i])[None, :]
        assert_rms_close(outs[i].cpu().numpy(), want, rel=2e-5, what=f"problem {i}")


@pytest.mark.parametrize("m,n,k", [(27, 2048, 4160), (63, 3000, 2176), (8, 500, 16448)])
def test_options_keep_the_bits(kq, m, n, k):
    """KR_OPT_SKINNY_GROUPS and KR_OPT_SKINNY_MAX_BLOCKS choose row groups and grid, not the route or the sums."""
    case(f"slab loop options m={m} n={n} k={k}")
    s = synth()
    wq, x = s.q4_weight(n, k, 7250 + m), dev_bf16(s.bf16_normal((m, k), 7251 + m))
    w = q4_dev(kq, wq)
    groups, blocks = kq.get_option(15), kq.get_option(6)
    got = {}
    try:
        for o in ((2, 256), (1, 256), (2, 64), (1, 40), (2, 1000)):
            kq.set_option(15, o[0])
            kq.set_option(6, o[1])
            got[o] = kq.q4_linear(w, x, out_dtype=kq.DTYPE_F32).cpu().numpy().view(np.uint32)
    finally:
        kq.set_option(15, groups)
        kq.set_option(6, blocks)
    for o, y in got.items():
        assert np.array_equal(y, got[2, 256]), o


def beyond_range(x):
    """Rows 1 .. 5 of x get an infinity of either sign, a NaN, one column and three columns of 3e37 (31 times that
    overflows f32, times a weight of about 0.1 it does not)."""
    big = O.bf16_to_f32(x).copy()
    big[1, 70], big[2, -1], big[3, 5] = np.inf, -np.inf, np.nan
    big[4, 2050] = 3e37
    big[5, [0, 100, 2100]] = 3e37, -3e37, 2e37
    return O.f32_to_bf16(big)


def assert_beyond_range(got, want, rel, what):
    """Infinities and NaNs where the oracle has them; finite rows at the bar, each against its own RMS."""
    assert np.array_equal(np.isnan(got), np.isnan(want)), what
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf]), what
    for i in np.nonzero(np.isfinite(want).all(axis=1))[0]:
        assert_rms_close(got[i], want[i], rel=rel, what=f"{what} row {i}")


@pytest.mark.parametrize("m,n,k", [(27, 300, 4160), (63, 33, 2176), (8, 50, 16448)])
def test_linear_beyond_range(kq, m, n, k):
    """s D + (b - 16 s) S overflows, or adds opposite infinities, where the product itself does not."""
    case(f"slab loop linear, infinite and near-maximal x m={m} n={n} k={k}")
    s = synth()
    wq, x = s.q4_weight(n, k, 7300 + m), beyond_range(s.bf16_normal((m, k), 7301 + m))
    want = O.q4_matmul(O.Q4Planar(*wq), x)
    assert np.isinf(want[1:3]).any() and np.isfinite(want[4:6]).all()
    got = kq.q4_linear(q4_dev(kq, wq), dev_bf16(x), out_dtype=kq.DTYPE_F32).cpu().numpy()
    assert_beyond_range(got, want, 2e-5, "f32")


@pytest.mark.parametrize("m,n,k,act", [(16, 35, 2112, 2), (27, 300, 4096, 0)])
def test_gate_up_beyond_range(kq, m, n, k, act):
    case(f"slab loop gate_up, infinite and near-maximal x m={m} n={n} k={k} activation={act}")
    s = synth()
    g, u, x = s.q4_weight(n, k, 7400), s.q4_weight(n, k, 7401), beyond_range(s.bf16_normal((m, k), 7402))
    x[4:6] = s.bf16_normal((2, k), 7403)  # gate times up of such rows leaves f32's range
    want = O.q4_gate_up_act(O.Q4Planar(*g), O.Q4Planar(*u), x, act)
    got = kq.gate_up_act(q4_dev(kq, g), q4_dev(kq, u), dev_bf16(x), activation=act).cpu().numpy()
    assert_beyond_range(got, want, 1e-2, "f32")


def test_qkv_beyond_range(kq):
    case("slab loop qkv, infinite and near-maximal x m=16 k=2112")
    s = synth()
    m, k, ns = 16, 2112, (500, 40, 300)
    x = beyond_range(s.bf16_normal((m, k), 7500))
    ws = [s.q4_weight(n, k, 7501 + i) for i, n in enumerate(ns)]
    bs = [s.bf16_normal((1, n), 7510 + i)[0] for i, n in enumerate(ns)]
    outs = kq.qkv(*[q4_dev(kq, w) for w in ws], dev_bf16(x), *[dev_bf16(b) for b in bs], out_dtype=kq.DTYPE_F32)
    for i in range(3):
        want = O.q4_matmul(O.Q4Planar(*ws[i]), x) + O.bf16_to_f32(bs[i])[None, :]
        assert_beyond_range(outs[i].cpu().numpy(), want, 2e-5, f"problem {i}")
