"""The one-launch router at 9 to 128 rows (six checking waves): bit-exact with
the oracle at the edges of its rows per checking wave and per bucket, and a
refused batch writes nothing wherever its bad row is."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_ffi as O
from r9v_amd import ffi, synth

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("t", [9, 24, 25, 31, 48, 49, 127, 128, 129])
@pytest.mark.parametrize("e,k", [(64, 6), (100, 7), (512, 10), (1024, 32)])
def test_route_mid_bit_exact(t, e, k):
    z = synth.normal_f32(9300 + t + e, (t, e))
    ids, w = ffi.moe_route(torch.from_numpy(z).cuda(), k)
    ids_o, w_o = O.moe_route(z, k)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), ids_o)
    assert np.array_equal(w.cpu().numpy().view(np.uint32), w_o.view(np.uint32))


@pytest.mark.parametrize("t", [9, 25, 128])
def test_route_mid_refuses_before_writing(t):
    for bad in {0, 7, 8, t // 2, t - 1}:
        z = synth.normal_f32(9400 + bad, (t, 64))
        z[bad, 63] = np.inf
        ids = torch.full((t, 4), -7, dtype=torch.int32, device="cuda")
        w = torch.full((t, 4), -7.0, device="cuda")
        status = torch.zeros(1, dtype=torch.int32, device="cuda")
        ffi.moe_route(torch.from_numpy(z).cuda(), 4, ids=ids, weights=w, status=status)
        assert ffi.status_read(status) == ffi.STATUS_NONFINITE, f"bad row {bad}"
        assert bool((ids == -7).all()) and bool((w == -7.0).all())


@pytest.mark.parametrize("scoring,e,line", [(ffi.SCORING_SIGMOID, 128, 48), (ffi.SCORING_SIGMOID, 256, 32),
                                            (ffi.SCORING_SIGMOID, 512, 24), (ffi.SCORING_SIGMOID, 1024, 16),
                                            (ffi.SCORING_SOFTMAX, 300, 96)])
def test_route_mid_lines_with_a_bias(scoring, e, line):
    """Both sides of the row count up to which one launch routes."""
    bias = synth.normal_f32(9350 + e, (e,))
    for t in (line, line + 1):
        z = synth.normal_f32(9360 + t + e, (t, e))
        ids, w = ffi.moe_route(torch.from_numpy(z).cuda(), 6, bias=torch.from_numpy(bias).cuda(), scoring=scoring)
        ids_o, w_o = O.moe_route(z, 6, bias=bias, scoring=scoring)
        assert np.array_equal(ids.cpu().numpy().view(np.uint32), ids_o)
        assert np.array_equal(w.cpu().numpy().view(np.uint32), w_o.view(np.uint32))
