"""Every prefill kernel by name (r9vx_probe_matmul_tiles_launch), so that what is
covered does not hang on the size rule's constants: each thin shape at the edges
of its tiles, and the 256 x 256 tiles' row-chunk plans, for all five schemes.
All of them give an output the same bits; the oracle's values pin them."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_ffi as O
from r9v_amd import ffi, synth
from tol import check_close

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SCHEMES = [O.Q4_K, O.IQ4_XS, O.Q6_K, O.Q8_0, O.IQ3_S]
THIN = [(1, 1), (2, 1), (4, 1), (1, 2), (2, 2), (4, 2), (8, 2)]


def _weight(scheme, seed, n, k):
    wire = synth.quant_weights(scheme, seed, n, k)
    d = torch.from_numpy(wire.reshape(-1)).cuda()
    return (wire, d, None) if scheme in (O.Q4_K, O.IQ4_XS) else (wire, *ffi.repack(d, scheme, n, k))


def _x(seed, m, k):
    x = synth.normal_bf16(seed, (m, k))
    return x, torch.from_numpy(x.view(np.int16)).cuda().view(torch.bfloat16)


def _randn(seed, *shape):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def _same(a, b):
    return torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("nr,nc", THIN)
@pytest.mark.parametrize("scheme", SCHEMES)
def test_thin_shape(scheme, nr, nc):
    """Row tiles: all of a workgroup's, one more row, one tile of a second
    workgroup but for a row; columns: one, whole tiles, ragged (n % 4 too); K of
    one super-block and of counts with every remainder of the loops' three."""
    tile = 32 * nr
    for i, (m, n, k) in enumerate([(tile, 64 * nc, 256), (tile + 1, 32 * nc + 5, 768), (2 * tile - 1, 1, 1280),
                                   (tile + 33, 32 * nc * 3 + 2, 2048), (9, 100, 1024)]):
        wire, w, sc = _weight(scheme, 9100 + i, n, k)
        x, xd = _x(9110 + i, m, k)
        y = ffi.probe_matmul_tiles(w, scheme, n, k, xd, nr, nc, w_scales=sc)
        check_close(y.cpu().numpy(), O.matmul(scheme, wire, n, k, x, O.BF16), f"{scheme} ({nr}, {nc}) {m}x{n}x{k}")
        assert _same(y, ffi.probe_matmul_tiles(w, scheme, n, k, xd, 0, 0, w_scales=sc)), (m, n, k)
        assert _same(y, ffi.matmul(w, scheme, n, k, xd, w_scales=sc, m_bucket=max(m, 16))), (m, n, k)


# one weight block; one 32-row tile a chunk; uniform chunks in the XCD band order;
# two chunk counts across blocks; several rounds; a ragged last block with rows of
# whole 16 bytes and without (element stores)
PLANS = [(9, 256), (700, 2560), (2048, 4096), (1100, 5376), (2600, 14336), (600, 2504), (600, 1001)]


@pytest.mark.parametrize("m,n", PLANS)
@pytest.mark.parametrize("scheme", SCHEMES)
def test_256_column_plans(scheme, m, n):
    """The 256 x 256 tiles' plans with every epilogue and both outputs: sampled
    rows and columns against the oracle, every output's bits against thin tiles."""
    k = 512
    wire, w, sc = _weight(scheme, 9200 + n, n, k)
    x, xd = _x(9201 + m, m, k)
    bias, res = _randn(9202, n), _randn(9203, m, n)
    rows = np.unique(np.r_[np.arange(0, m, 97), 0, m - 1])
    cols = np.unique(np.r_[np.arange(0, n, 61), n - 1])
    some = np.ascontiguousarray(wire.reshape(n, -1)[cols])
    want = O.matmul(scheme, some, len(cols), k, np.ascontiguousarray(x[rows]), O.BF16)
    y = ffi.probe_matmul_tiles(w, scheme, n, k, xd, 0, 0, w_scales=sc)
    check_close(y.cpu().numpy()[np.ix_(rows, cols)], want, f"{scheme} {m}x{n}")
    assert _same(y, ffi.probe_matmul_tiles(w, scheme, n, k, xd, 8, 2, w_scales=sc))
    for kw in (dict(bias=bias), dict(residual=res), dict(out_dtype=ffi.BF16), dict(residual=res, out_dtype=ffi.BF16)):
        got = ffi.probe_matmul_tiles(w, scheme, n, k, xd, 0, 0, w_scales=sc, **kw)
        assert _same(got, ffi.probe_matmul_tiles(w, scheme, n, k, xd, 4, 1, w_scales=sc, **kw)), kw
        # bias and residual are f32 adds of the plain launch's values, bf16 its last rounding
        plain = y + kw["bias"] if "bias" in kw else y + kw["residual"] if "residual" in kw else y
        assert _same(got, plain.to(torch.bfloat16) if "out_dtype" in kw else plain), kw
