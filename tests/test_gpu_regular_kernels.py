"""The 256 x 256 GEMM tiles and the regular flash kernels at the edges of
their tiles.  The built-in plan gives launches this small to the smaller tiles
and the small-launch flash kernels; the tests of the kernels that serve the
large ones run here again under a forced plan (PHX_GEMM_SPLIT,
PHX_FLASH_SPLIT): unsplit, in three chunks, and in the chunks the rule names."""
import os

import numpy as np
import pytest

import oracle
from test_gpu_flash import (test_flash16_bh_any_grid, test_flash16_rows_past_nq_untouched,
                            test_flash_bh_equals_per_head_bit_exact,
                            test_flash_block_sum_over_limit_without_raise,
                            test_flash_large_scores_and_single_block, test_flash_one_head_full)
from test_gpu_gemm import (test_gemm_fp16_full_small, test_gemm_fp16tc_full_small,
                           test_gemm_fp16tc_rounds_f32_inputs_to_f16,
                           test_gemm_fp32_beta_zero_and_alpha, test_gemm_fp32_full_small,
                           test_gemm_integer_fixture_exact)
from test_gpu_gemm_tiles import SHAPES, _Case
from test_gpu_gemm_tiles import _check as _check_bound
from test_gpu_ragged import (test_flash_bh_ragged_equals_per_head,
                             test_flash_negative_and_zero_scale,
                             test_flash_partial_block_with_very_negative_scores,
                             test_flash_ragged, test_gemm_fp16_ragged, test_gemm_fp16tc_ragged,
                             test_gemm_fp32_ragged, test_gemm_partial_k_step_reads_nothing_past_k,
                             test_masking_example_exact_at_its_own_shape)
from test_gpu_shapes import GEMM_SHAPES, TOL, _check, _flash_inputs, _flash_rel, _gemm, _upload

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, params=["1", "3"])
def forced(request, monkeypatch):
    """Every launch of the module runs the regular kernels in this many chunks."""
    monkeypatch.setenv("PHX_GEMM_SPLIT", request.param)
    monkeypatch.setenv("PHX_FLASH_SPLIT", request.param)
    return int(request.param)


@pytest.mark.parametrize("kern_name", ["GEMM_FP32", "GEMM_FP16TC_FP32ACC", "GEMM_FP16"])
@pytest.mark.parametrize("M,N,K", GEMM_SHAPES + [(769, 1032, 200)])
def test_gemms_in_the_rules_chunks(px_gpu, stream, monkeypatch, forced, kern_name, M, N, K):
    # with the forced count, and (in its place) the count the built-in rule names
    px = px_gpu
    kern = getattr(px, kern_name)
    counts = [forced]
    if forced == 1:
        monkeypatch.delenv("PHX_GEMM_SPLIT")
        counts.append(px.split_plan(kern, [M, N, K])[0])
    A = oracle.normal_f32(21, M * K, 1 / np.sqrt(K)).reshape(M, K)
    B = oracle.normal_f32(22, K * N, 1 / np.sqrt(K)).reshape(K, N)
    C = oracle.normal_f32(23, M * N).reshape(M, N)
    r16 = kern_name != "GEMM_FP32"
    if r16:
        A, B, C = oracle.f16_round(A), oracle.f16_round(B), oracle.f16_round(C)
    want = oracle.gemm_full(A, B, C, 0.5, 0.25, round16=r16)
    for sp in counts:
        monkeypatch.setenv("PHX_GEMM_SPLIT", str(sp))
        _check(kern_name, _gemm(px, stream, kern, A, B, C, 0.5, 0.25), want)


@pytest.mark.parametrize("bits", [16, 32])
@pytest.mark.parametrize("BH,Nq,Nk,scale", [(1, 1000, 4133, 0.125), (1, 300, 2048, -0.2),
                                            (3, 529, 700, 0.125)])
def test_flash_in_the_rules_chunks(px_gpu, stream, monkeypatch, forced, bits, BH, Nq, Nk, scale):
    px, D = px_gpu, 64
    kern = px.FLASH_FP16_BH if bits == 16 else px.FLASH_FP32_BH
    counts = [forced]
    if forced == 1:
        monkeypatch.delenv("PHX_FLASH_SPLIT")
        counts.append(px.split_plan(kern, [BH, Nq, Nk, D])[0])
    q, k, v = _flash_inputs(BH, Nq, Nk, bits, 41)
    dq, dk, dv = (_upload(px, t, bits) for t in (q, k, v))
    rows = np.unique(np.linspace(0, Nq - 1, 32).astype(np.int64))
    want = [oracle.flash_rows(rows, q[h], k[h], v[h], scale) for h in range(BH)]
    for sp in counts:
        monkeypatch.setenv("PHX_FLASH_SPLIT", str(sp))
        do = px.DeviceBuffer(BH * Nq * D * bits // 8)
        px.launch_flash_bh(stream, kern, dq.ptr, dk.ptr, dv.ptr, do.ptr, BH, Nq, Nk, D, scale)
        stream.synchronize()
        got = (oracle.f16_to_f32(do.download(np.uint16, BH * Nq * D)) if bits == 16
               else do.download(np.float32, BH * Nq * D)).reshape(BH, Nq, D)
        for h in range(BH):
            assert _flash_rel(got[h][rows], want[h]) < TOL[bits], (sp, h)


@pytest.mark.parametrize("pad", [0, 8])
@pytest.mark.parametrize("M,N,K", SHAPES + [(513, 260, 300)])
def test_the_leafs_256_tile(px_gpu, stream, M, N, K, pad):
    # the cluster step leaf's own entry, launched by itself (no plan names it)
    px = px_gpu
    case = _Case(px, px.MATMUL, M, N, K, pad)
    with open(os.path.join(px.LIB_DIR, "matmul_cluster_fp32.hsaco"), "rb") as f:
        mod = px.module_load_data(f.read())
    fn = px.module_get_function(mod, "matmul")
    tiles = -(-M // 256) * -(-N // 256)
    outs = [case.launch(stream, fn, grid, 256, 0.75, 0.0) for grid in (tiles, max(1, tiles // 2))]
    _check_bound(case, outs[0], 0.75, 1.0)
    assert np.array_equal(*outs)
    px.module_unload(mod)
