"""Which kernels the library launches for a call, and with what grids, recorded
on the CPU (tests/launch_record.py): the dispatch rules' lines, and HIP's limits
on a launch."""
from __future__ import annotations

import shutil

import pytest

import launch_record
from r9v_amd import ffi

pytestmark = pytest.mark.skipif(not launch_record.LIB.exists() or shutil.which("gcc") is None,
                                reason="needs the built libr9vx.so and gcc")


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return launch_record.build(tmp_path_factory.mktemp("hip"))


def kernels(runtime, calls):
    out = launch_record.record(runtime, calls)
    assert all(rc == 0 for rc, _, _ in out), out
    return [[k for k, _, _ in launches] for _, _, launches in out]


# experts, scores, the most rows that one launch routes: past them checking every
# row in every workgroup costs more than the launches that it saves
ROUTE_LINES = [(64, ffi.SCORING_SOFTMAX, 128), (256, ffi.SCORING_SOFTMAX, 128), (300, ffi.SCORING_SOFTMAX, 96),
               (512, ffi.SCORING_SOFTMAX, 96), (768, ffi.SCORING_SOFTMAX, 64), (1024, ffi.SCORING_SOFTMAX, 48),
               (64, ffi.SCORING_SIGMOID, 48), (128, ffi.SCORING_SIGMOID, 48), (256, ffi.SCORING_SIGMOID, 32),
               (512, ffi.SCORING_SIGMOID, 24), (768, ffi.SCORING_SIGMOID, 16), (1024, ffi.SCORING_SIGMOID, 16)]


@pytest.mark.parametrize("e,scoring,line", ROUTE_LINES)
def test_router_launches(runtime, e, scoring, line):
    last, past = kernels(runtime, [("route", dict(t=t, e=e, k=8, scoring=scoring)) for t in (line, line + 1)])
    assert len(last) == 1 and last[0].startswith("route_small_kernel")
    assert [k.split("<")[0] for k in past] == ["clear_status_kernel", "route_check_kernel", "route_kernel"]


@pytest.mark.parametrize("m,n,k", [((1 << 24) + 7, 64, 256), (1 << 24, 1, 256), ((1 << 20) + 1, 33, 512), (1 << 20, 64, 256)])
def test_prefill_rows_within_the_launch_limits(runtime, m, n, k):
    """Row counts past 2^32 / 256: launches that HIP accepts, and on the thin
    tiles every row converted once and in a tile."""
    call = dict(scheme=ffi.Q4_K, m=m, n=n, k=k)
    (rc, msg, _), (thin_rc, thin_msg, launches) = launch_record.record(
        runtime, [("matmul", call), ("matmul", dict(call, tiles=(8, 2)))])
    assert rc == 0, msg
    assert thin_rc == 0, thin_msg
    thin = [(name, g) for name, g, _ in launches if name.startswith("gemm_thin_kernel")]
    assert len(thin) == -(-m // (1 << 20)) and len(launches) == 2 * len(thin)
    assert sum(g[0] for name, g, _ in launches if "x_to_f16_thin" in name) == m
    tiles = [32 * int(name.split("<")[1].split(",")[1]) * g[1] for name, g in thin]
    assert tiles[:-1] == [1 << 20] * (len(thin) - 1) and 0 <= sum(tiles) - m < 256


THIN_SHAPES = [(1, 1), (2, 1), (4, 1), (1, 2), (2, 2), (4, 2), (8, 2)]


@pytest.mark.parametrize("scheme", [ffi.Q4_K, ffi.IQ4_XS, ffi.Q6_K, ffi.Q8_0, ffi.IQ3_S])
def test_thin_shapes_launch_or_are_refused(runtime, scheme):
    """Every pair of row and column tiles runs its kernel or is an error: none
    returns 0 with nothing launched."""
    pairs = [(nr, nc) for nr in (1, 2, 3, 4, 6, 8, 16) for nc in (1, 2, 4)] + [(0, 1), (2, 0)]
    out = launch_record.record(runtime, [("matmul", dict(scheme=scheme, m=300, n=500, k=512, tiles=p)) for p in pairs])
    for (nr, nc), (rc, _, launches) in zip(pairs, out):
        ran = [k for k, _, _ in launches if k.startswith("gemm")]
        assert ran == ([f"gemm_thin_kernel<{scheme}, {nr}, {nc}>"] if (nr, nc) in THIN_SHAPES else []), (nr, nc)
        assert (rc == 0) == bool(ran), (nr, nc, rc)
    # and the decode bucket and f32 activations have none
    for kw in (dict(m=8), dict(m=300, x_f32=True), dict(m=300, scheme=ffi.Q4_K, x_f32=True)):
        call = dict(dict(scheme=scheme, n=500, k=512, tiles=(1, 1)), **kw)
        assert launch_record.record(runtime, [("matmul", call)])[0][0] < 0


# sizes beside the line between the two prefill kernels (256 compute units), each
# with the kernel that was measured the faster there (gemm.hip, gemm3_cost)
PREFILL_SIDES = [(ffi.Q4_K, 32, 14336, 4096, "thin"), (ffi.Q4_K, 777, 4096, 4096, "thin"),
                 (ffi.Q4_K, 2048, 2048, 4096, "thin"), (ffi.Q4_K, 2600, 2048, 4096, "gemm3"),
                 (ffi.Q4_K, 4096, 2048, 4096, "gemm3"), (ffi.Q4_K, 1600, 3072, 4096, "gemm3"),
                 (ffi.Q8_0, 4096, 2048, 14336, "gemm3"), (ffi.Q4_K, 4096, 512, 4096, "gemm3"),
                 (ffi.IQ3_S, 2048, 4096, 4096, "thin"), (ffi.Q6_K, 1600, 3072, 256, "gemm3"),
                 (ffi.Q4_K, 2048, 14336, 4096, "gemm3"), (ffi.Q6_K, 57, 4096, 14336, "thin")]


@pytest.mark.parametrize("scheme,m,n,k,kernel", PREFILL_SIDES)
def test_prefill_kernel_by_size(runtime, scheme, m, n, k, kernel):
    (names,) = kernels(runtime, [("matmul", dict(scheme=scheme, m=m, n=n, k=k))])
    assert names[-1].startswith({"thin": "gemm_thin_kernel", "gemm3": "gemm3_kernel"}[kernel]), names


# n, K, gated: the first sizes at which a ragged row is read by fewer than 64 lanes
FEWER_LANES = [(16384, 2304, False), (16384, 6400, False), (32768, 768, False), (5120, 2304, True), (10240, 1280, True),
               (24576, 768, True)]


@pytest.mark.parametrize("n,k,swiglu", FEWER_LANES)
@pytest.mark.parametrize("m", [1, 3, 8])
def test_lanes_of_many_ragged_rows(runtime, n, k, swiglu, m):
    """A wave takes several rows from the line on (fewer waves, or the kernel
    of any number of lanes), for every m alike; 1024 SIMDs."""
    def launch(rows):
        (out,) = launch_record.record(runtime, [("matmul", dict(scheme=ffi.Q4_K, m=m, n=rows, k=k, m_bucket=8,
                                                                epilogue=3 if swiglu else 0))])
        (name, g, b), = out[2]
        return name, g[0] * b[0] // 64
    (name, waves), (below, waves_below) = launch(n), launch(n - 1)
    assert name != below or waves < 0.9 * waves_below


@pytest.mark.parametrize("scheme,k,streams", [(ffi.Q4_K, 2048, ()), (ffi.IQ4_XS, 2048, (4,)), (ffi.Q6_K, 2048, (2, 4)),
                                              (ffi.Q8_0, 2048, (3, 4)), (ffi.IQ3_S, 2048, (2, 3, 4)),
                                              (ffi.Q4_K, 4096, (1, 2, 3, 4)), (ffi.IQ4_XS, 4096, (2, 3, 4)),
                                              (ffi.Q6_K, 4096, (1, 2, 3, 4)), (ffi.Q8_0, 4096, (2, 3, 4)),
                                              (ffi.IQ3_S, 4096, (1, 2, 3, 4))])
def test_gated_streaming_where_it_is_faster(runtime, scheme, k, streams):
    """n = 14336, the gated epilogue: the streaming kernel for the row counts at
    which it was measured the faster, the one-shot kernel elsewhere (the same bits)."""
    names = kernels(runtime, [("matmul", dict(scheme=scheme, m=m, n=14336, k=k, epilogue=3)) for m in (1, 2, 3, 4, 5)])
    for m, (name,) in zip((1, 2, 3, 4, 5), names):
        assert name.startswith("gemv_gated_stream_kernel" if m in streams else "gemv_gated_kernel"), (m, name)


def test_gated_iq3s_workgroups(runtime):
    """IQ3_S: four waves share the codebook's table where there are two waves a
    SIMD, one wave a workgroup below (1024 SIMDs); other schemes one from m = 3."""
    calls = [(ffi.IQ3_S, 2047), (ffi.IQ3_S, 2048), (ffi.Q6_K, 2048)]
    out = launch_record.record(runtime, [("matmul", dict(scheme=s, m=8, n=n, k=2048, epilogue=3)) for s, n in calls])
    blocks = [(g[0], b[0]) for _, _, launches in out for _, g, b in launches]
    assert blocks == [(2047, 64), (512, 256), (2048, 64)]


# kernels that the GPU tests' texts name for their sizes, all schemes
NAMED = [(3000, 8481, 768, "gemm3_kernel"), (300, 8481, 768, "gemm_thin_kernel 4, 2"), (64, 8481, 768, "gemm_thin_kernel 2, 2"),
         (9, 8481, 768, "gemm_thin_kernel 1, 2"), (1024, 4096, 4096, "gemm_thin_kernel 8, 2"),
         (129, 257, 2048, "gemm_thin_kernel 1, 1"), (2600, 14336, 512, "gemm3_kernel"), (520, 32768, 256, "gemm3_kernel"),
         (600, 28000, 256, "gemm3_kernel"), (600, 1001, 256, "gemm_thin_kernel 4, 1")]


@pytest.mark.parametrize("scheme", [ffi.Q4_K, ffi.IQ4_XS, ffi.Q6_K, ffi.Q8_0, ffi.IQ3_S])
def test_kernels_named_by_the_gpu_tests(runtime, scheme):
    names = kernels(runtime, [("matmul", dict(scheme=scheme, m=m, n=n, k=k)) for m, n, k, _ in NAMED])
    for (m, n, k, want), ran in zip(NAMED, names):
        kernel, _, shape = want.partition(" ")
        assert ran[-1] == f"{kernel}<{scheme}{', ' + shape if shape else ''}>", (m, n, k)
