"""bench.py's attribution of Newton-Schulz launches: the kernel a launch runs and the MFMA work it executes."""
from types import SimpleNamespace

import pytest

import bench
from monarch_muon_amd import _abi


def group(rows, cols, nblocks, ns_dtype, param_dtype=_abi.BF16):
    return SimpleNamespace(rows=rows, cols=cols, nblocks=nblocks, transposed=rows > cols,
                           struct=SimpleNamespace(ns_dtype=ns_dtype, param_dtype=param_dtype),
                           ws=SimpleNamespace(layout=_abi.ns_layout(rows, cols, ns_dtype, nblocks)))


@pytest.mark.parametrize("shape,edge", [((1024, 1024), ""), ((2752, 1024), ""), ((384, 384), "edge_")])
def test_partial_tiles_have_their_own_kernels(shape, edge):
    gl = group(*shape, 8, _abi.BF16)
    assert bench.kernel_symbol("syrk", gl, 0) == f"ns_sym_{edge}bf16<0>"
    assert bench.kernel_symbol("px_apply", gl, 0) == \
        f"ns_px_{edge}bf16<3, {'true' if shape[0] > shape[1] else 'false'}, BF16T>"


def test_a_partial_long_side_is_an_edge_for_px_only():
    gl = group(512, 1376, 8, _abi.BF16)
    assert gl.ws.layout.np_ == 1408
    assert bench.kernel_symbol("poly", gl, 0) == "ns_sym_bf16<1>"
    assert bench.kernel_symbol("px", gl, 0) == "ns_px_edge_bf16<2, false, BF16T>"


def test_executed_work_of_bf16_tiles():
    """1024: 6 whole tiles and 36/64 of 4; 384: one whole tile is diagonal (36/64), one is 256 x 128 and the last,
    128 x 128 of one, holds 10 of its 16 MFMA tiles."""
    assert bench.stage_exec_flops("poly", group(1024, 1024, 1, _abi.BF16)) == 2 * 1024 * (6 + 4 * 36 / 64) * 65536
    assert bench.stage_exec_flops("poly", group(384, 384, 1, _abi.BF16)) == 2 * 384 * (36 * 1024 + 256 * 128 + 10 * 1024)
    gl = group(512, 1376, 3, _abi.BF16)   # the last 32 of 1408 columns lie in a window that holds valid ones
    assert bench.stage_exec_flops("px", gl) == 3 * 2 * 512 * 512 * 1408
    assert bench.stage_exec_flops("syrk", gl) == 3 * 2 * 1376 * (65536 + 2 * 36 * 1024)
    assert bench.stage_exec_flops("pack", gl) == 0


def test_executed_work_of_fp32_tiles():
    """64-wide tiles below 256 128-wide ones: 10 of the 16 of a 256 x 256 product; tiles in the padding left out."""
    gl = group(256, 256, 44, _abi.F32, _abi.F32)
    assert bench.kernel_symbol("syrk", gl, 0) == "ns_f32<0, F32T, 1>"
    assert bench.stage_exec_flops("syrk", gl) == 44 * 2 * 256 * 10 * 64 * 64
    gl = group(512, 512, 176, _abi.F32, _abi.F32)
    assert bench.kernel_symbol("px", gl, 0) == "ns_f32<2, F32T, 2>"
    assert bench.stage_exec_flops("poly", gl) == 176 * 2 * 512 * 10 * 128 * 128
    gl = group(150, 200, 3, _abi.F32, _abi.F32)
    assert bench.stage_exec_flops("px", gl) == 3 * 2 * 160 * 3 * 4 * 64 * 64


@pytest.mark.parametrize("kind,want", [("syrk", 4 * (512 * 1376 + 512 * 512)), ("poly", 8 * 512 * 512),
                                       ("px", 4 * (512 * 512 + 2 * 512 * 1408)),
                                       ("px_apply", 4 * (512 * 512 + 512 * 1408) + 8 * 512 * 1376)])
def test_fp32_stage_bytes(kind, want):
    import bench_studies
    assert bench_studies.stage_bytes(kind, group(512, 1376, 2, _abi.F32, _abi.F32)) == 2 * want
