"""The decode GEMV at rows whose 32-weight chunks do not fill a wave's segments
(K not a multiple of 2048), with epilogues and bf16 outputs, and the streaming
form of the gated epilogue: parity with the oracle, and a row's bits the same
for every number of rows in the bucket."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_ffi as O
from r9v_amd import ffi, synth
from tol import check_close

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _weight(scheme, seed, n, k):
    wire = synth.quant_weights(scheme, seed, n, k)
    d = torch.from_numpy(wire.reshape(-1)).cuda()
    return (wire, d, None) if scheme in (O.Q4_K, O.IQ4_XS) else (wire, *ffi.repack(d, scheme, n, k))


def _x(seed, m, k):
    x = synth.normal_bf16(seed, (m, k))
    return x, torch.from_numpy(x.view(np.int16)).cuda().view(torch.bfloat16)


@pytest.mark.parametrize("scheme", [O.Q4_K, O.IQ4_XS, O.Q6_K, O.Q8_0, O.IQ3_S])
@pytest.mark.parametrize("n,k", [(1, 768), (70, 1280), (333, 1792), (200, 2304), (129, 3840), (67, 6400)])
def test_ragged_rows(scheme, n, k):
    wire, w, sc = _weight(scheme, 9900 + k, n, k)
    x, xd = _x(9901 + k, 8, k)
    bias = np.linspace(-2, 2, n, dtype=np.float32)
    alone = None
    for m in (1, 2, 4, 5, 8):
        y = ffi.matmul(w, scheme, n, k, xd[:m], w_scales=sc, m_bucket=8)
        check_close(y.cpu().numpy(), O.matmul(scheme, wire, n, k, x[:m], O.BF16), f"{scheme} m={m} k={k}")
        alone = y[0] if alone is None else alone
        assert torch.equal(y[0], alone), f"row bits, m={m}"
        yb = ffi.matmul(w, scheme, n, k, xd[:m], w_scales=sc, m_bucket=8, bias=torch.from_numpy(bias).cuda())
        assert torch.equal(yb, y + torch.from_numpy(bias).cuda()), f"bias, m={m}"
        y16 = ffi.matmul(w, scheme, n, k, xd[:m], w_scales=sc, m_bucket=8, out_dtype=ffi.BF16)
        assert torch.equal(y16, y.to(torch.bfloat16)), f"bf16 output, m={m}"


@pytest.mark.parametrize("scheme", [O.Q4_K, O.IQ4_XS])
@pytest.mark.parametrize("n,k", [(65, 1280), (77, 3328), (40, 5376)])
def test_ragged_rows_f32_activations(scheme, n, k):
    wire, w, _ = _weight(scheme, 9930 + k, n, k)
    x = synth.normal_f32(9931 + k, (3, k))
    xd = torch.from_numpy(x).cuda()
    y = ffi.matmul(w, scheme, n, k, xd)
    check_close(y.cpu().numpy(), O.matmul(scheme, wire, n, k, x, O.F32), f"{scheme} f32 k={k}")
    assert torch.equal(ffi.matmul(w, scheme, n, k, xd[:1])[0], y[0])


@pytest.mark.parametrize("scheme", [O.Q4_K, O.Q6_K, O.IQ3_S])
@pytest.mark.parametrize("n,k", [(8209, 1280), (8192, 2048), (9001, 3840)])
def test_gated_streaming_form_has_the_one_shot_forms_bits(scheme, n, k):
    """n of 8 rows a SIMD and more streams; the same rows in a weight of fewer
    take the one-shot kernel."""
    wire, w, sc = _weight(scheme, 9950, 2 * n, k)
    _, xd = _x(9951, 4, k)
    few = 300
    gate, up = torch.arange(few, device="cuda"), torch.arange(n, n + few, device="cuda")
    rows = torch.cat([gate, up])
    ws = w.view(2 * n, -1).index_select(0, rows).contiguous().view(-1)
    ss = sc.view(2 * n, -1).index_select(0, rows).contiguous().view(-1) if sc is not None else None
    for m in (1, 3, 4):
        y = ffi.matmul(w, scheme, n, k, xd[:m], w_scales=sc, swiglu=True)
        part = ffi.matmul(ws, scheme, few, k, xd[:m], w_scales=ss, swiglu=True)
        assert torch.equal(y[:, :few], part), f"m={m}"
        y16 = ffi.matmul(w, scheme, n, k, xd[:m], w_scales=sc, swiglu=True, out_dtype=ffi.BF16)
        assert torch.equal(y16, y.to(torch.bfloat16))
        assert torch.equal(ffi.matmul(w, scheme, n, k, xd[m - 1:m], w_scales=sc, swiglu=True)[0], y[m - 1])


def _last_block_infinite(scheme, wire, n, k):
    """The last block of every row of `wire`, made of positive weights under an infinite scale."""
    w = wire.reshape(n, k // ffi.BLOCK_LEN[scheme], -1)
    last = w[:, -1]
    if scheme == O.Q8_0:  # quants 1
        last[:, 2:] = 1
    elif scheme == O.IQ4_XS:  # sub-block scales 63 - 32, the codebook's largest value
        last[:, 2:] = 0xFF
    elif scheme == O.Q6_K:  # quants 63 - 32, sub-block scales 1
        last[:, :192], last[:, 192:208] = 0xFF, 1
    else:  # IQ3_S: no signs (the codebook's values are positive)
        last[:, 74:106] = 0
    at = 208 if scheme == O.Q6_K else 0
    last[:, at:at + 2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    return w.reshape(wire.shape)


# n, K, m, gated: one and several segments, one and two chunks a lane, the streaming forms, full rows
INFINITE = [(5, 768, 1, False), (70, 2304, 3, False), (70, 2304, 8, False), (33, 6400, 5, False), (33, 2816, 2, True),
            (20, 4352, 6, True), (8200, 1280, 3, True), (12300, 1280, 1, False), (5, 2048, 1, False)]


@pytest.mark.parametrize("scheme,n,k,m,swiglu,x_f32",
                         [(s, *c, False) for s in (O.IQ4_XS, O.Q6_K, O.Q8_0, O.IQ3_S) for c in INFINITE]
                         + [(O.IQ4_XS, 40, 3840, 2, False, True), (O.IQ4_XS, 9, 768, 1, False, True)])
def test_infinite_last_block_is_not_nan(scheme, n, k, m, swiglu, x_f32):
    """Lanes past a ragged row's end read its last block again: its infinite
    scale must stay the row's infinity, as in rows that fill their segments."""
    rows = 2 * n if swiglu else n
    wire = _last_block_infinite(scheme, synth.quant_weights(scheme, 9970 + k, rows, k).copy(), rows, k)
    w = torch.from_numpy(wire.reshape(-1)).cuda()
    w, sc = (w, None) if scheme == O.IQ4_XS else ffi.repack(w, scheme, rows, k)
    x = torch.ones((m, k), dtype=torch.float32 if x_f32 else torch.bfloat16, device="cuda")
    y = ffi.matmul(w, scheme, n, k, x, w_scales=sc, swiglu=swiglu)
    assert bool((y == float("inf")).all())


@pytest.mark.parametrize("scheme", [O.Q4_K, O.IQ3_S])
@pytest.mark.parametrize("n,k,swiglu", [(16384, 2304, False), (16391, 2816, False), (32768, 768, False),
                                        (5120, 2304, True), (5133, 4352, True), (10240, 1280, True)])
def test_many_ragged_rows_take_fewer_lanes(scheme, n, k, swiglu):
    """From the lines where a row's idle lanes cost more than their latency: the
    oracle's values at sampled rows, and the same bits in every bucket."""
    rows = 2 * n if swiglu else n
    wire, w, sc = _weight(scheme, 9990 + k, rows, k)
    x, xd = _x(9991 + k, 8, k)
    cols = np.r_[0:9, n // 2 - 5:n // 2 + 5, n - 9:n]
    some = np.ascontiguousarray(wire.reshape(rows, -1)[np.r_[cols, cols + n] if swiglu else cols])
    want = O.matmul(scheme, some, len(some), k, x, O.BF16)
    if swiglu:
        g, u = want[:, :len(cols)].astype(np.float64), want[:, len(cols):].astype(np.float64)
        with np.errstate(over="ignore"):  # exp(-g) past 1e308: g / inf is the 0 that it stands for
            want = (g / (1.0 + np.exp(-g)) * u).astype(np.float32)
    whole = ffi.matmul(w, scheme, n, k, xd, w_scales=sc, swiglu=swiglu)
    check_close(whole.cpu().numpy()[:, cols], want, f"{scheme} n={n} k={k}")
    for m in (1, 2, 4, 5):
        assert torch.equal(ffi.matmul(w, scheme, n, k, xd[:m], w_scales=sc, swiglu=swiglu), whole[:m]), f"m={m}"
