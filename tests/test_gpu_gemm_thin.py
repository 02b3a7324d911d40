"""The thin tiles of the prefill GEMM (r9v_amd/csrc/gemm_thin.hip) where the size
rule takes them: buckets above the decode GEMV's whose rows do not fill 256-row
tiles.  Their outputs have the bits of the 256-row kernel's, and lie within the
matmul tolerance of the oracle at the edges of the tiles.  (Every shape of tiles
by name: test_gpu_prefill_tiles.py.)"""
from __future__ import annotations

import numpy as np
import pytest

import oracle_ffi as O
from r9v_amd import ffi, synth
from tol import check_close

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SCHEMES = [O.Q4_K, O.IQ4_XS, O.Q6_K, O.Q8_0, O.IQ3_S]


def _weight(scheme, seed, n, k):
    """(wire blocks, device tensor, scales) of a seeded [n, k] weight."""
    wire = synth.quant_weights(scheme, seed, n, k)
    d = torch.from_numpy(wire.reshape(-1)).cuda()
    if scheme in (O.Q4_K, O.IQ4_XS):
        return wire, d, None
    return (wire, *ffi.repack(d, scheme, n, k))


def _x(seed, m, k):
    x = synth.normal_bf16(seed, (m, k))
    return x, torch.from_numpy(x.view(np.int16)).cuda().view(torch.bfloat16)


@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("m,n,k", [(9, 1, 256), (32, 33, 512), (33, 95, 768), (64, 64, 1024), (65, 130, 1280),
                                   (100, 31, 1792), (129, 257, 2048)])
def test_thin_tiles_parity(scheme, m, n, k):
    """One row tile by one column tile a workgroup, up to five row tiles."""
    wire, w, sc = _weight(scheme, 9500 + n, n, k)
    x, xd = _x(9600 + m, m, k)
    y = ffi.matmul(w, scheme, n, k, xd, w_scales=sc)
    check_close(y.cpu().numpy(), O.matmul(scheme, wire, n, k, x, O.BF16), f"thin {scheme} {m}x{n}x{k}")


@pytest.mark.parametrize("scheme", SCHEMES)
def test_thin_tiles_have_the_256_row_kernels_bits(scheme):
    """Rows alone in launches of 9 to 300 rows (two column tiles by one, two and
    four row tiles) against the same rows among 3000 (the 256-row kernel), f32
    and bf16 outputs, with a bias."""
    n, k = 8481, 768
    _, w, sc = _weight(scheme, 9700, n, k)
    _, x = _x(9701, 3000, k)
    bias = torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(9702), device="cuda")
    for out in (ffi.F32, ffi.BF16):
        whole = ffi.matmul(w, scheme, n, k, x, out_dtype=out, bias=bias, w_scales=sc)
        for m in (9, 32, 40, 64, 96, 128, 300):
            part = ffi.matmul(w, scheme, n, k, x[:m], out_dtype=out, bias=bias, w_scales=sc)
            assert torch.equal(part.view(torch.uint8), whole[:m].view(torch.uint8)), f"m={m} out={out}"


@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("m,k", [(577, 768), (777, 256), (1024, 512)])
def test_eight_chain_tiles(scheme, m, k):
    """Prompt chunks whose workgroups run eight row tiles, the last of them three
    (m = 577), one (777) and all of it (1024), ragged n: sampled columns against
    the oracle, and the bits of the kernel that the sizes choose and of the same
    rows in a launch of one and of ten row tiles."""
    n = 4099
    wire, w, sc = _weight(scheme, 9850, n, k)
    x, xd = _x(9851 + m, m, k)
    y = ffi.probe_matmul_tiles(w, scheme, n, k, xd, 8, 2, w_scales=sc)
    assert torch.equal(ffi.matmul(w, scheme, n, k, xd, w_scales=sc), y)
    cols = np.r_[0:33, 2017:2051, n - 35:n]
    rows = wire.reshape(n, -1)[cols]
    check_close(y.cpu().numpy()[:, cols], O.matmul(scheme, np.ascontiguousarray(rows), len(cols), k, x, O.BF16), f"eight {scheme} {m}")
    for part in (21, 300):
        assert torch.equal(ffi.matmul(w, scheme, n, k, xd[:part], w_scales=sc), y[:part]), part


def test_thin_tiles_under_a_captured_graph():
    """Replays of a captured launch, eager work between them, against the
    eager result, with a residual."""
    m, n, k = 37, 300, 1024
    _, w, _ = _weight(O.Q4_K, 9800, n, k)
    _, x = _x(9801, m, k)
    res = torch.randn((m, n), device="cuda")
    want = ffi.matmul(w, O.Q4_K, n, k, x, residual=res)
    y = torch.zeros_like(want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ffi.matmul(w, O.Q4_K, n, k, x, residual=res, y=y)
    for _ in range(4):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


def test_thin_rows_past_one_launch():
    """More rows than one launch takes (2^20): the rows beside the cut and the
    last ones have the bits of a launch of their own, bias and residual."""
    m, n, k = (1 << 20) + 45, 40, 256
    _, w, _ = _weight(O.Q4_K, 9870, n, k)
    x = torch.randn((m, k), generator=torch.Generator(device="cuda").manual_seed(9871), device="cuda", dtype=torch.bfloat16)
    res = torch.randn((m, n), generator=torch.Generator(device="cuda").manual_seed(9872), device="cuda")
    y = ffi.probe_matmul_tiles(w, O.Q4_K, n, k, x, 8, 2, residual=res)
    for rows in (slice(0, 64), slice((1 << 20) - 40, (1 << 20) + 40), slice(m - 33, m)):
        alone = ffi.matmul(w, O.Q4_K, n, k, x[rows].contiguous(), residual=res[rows].contiguous())
        assert torch.equal(y[rows], alone), rows
