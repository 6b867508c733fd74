"""The C-ABI library loads and exports every symbol include/folx_hip.h declares; argument
checks reject bad calls before anything is launched (no GPU needed: nothing computes)."""

import ctypes
import os

import pytest

import __graft_entry__ as entry
from folx_amd import _lib


@pytest.fixture(scope='module')
def lib():
    if not os.path.exists(_lib.LIBPATH):
        from folx_amd import build

        build.build(verbose=False)
    return _lib.load()


def test_exports_every_declared_symbol(lib):
    declared = entry.declared_symbols()
    assert len(declared) >= 12
    assert set(declared) == set(_lib.SIGNATURES)
    for name in declared:
        assert getattr(lib, name) is not None


def test_gemm_mode_switch(lib):
    """The mode is a host-side flag: setting and reading it needs no GPU."""
    if 'FOLX_AMD_GEMM' not in os.environ:
        assert lib.folx_hip_get_gemm_mode() == _lib.GEMM_MODE['f32']  # the default
    before = lib.folx_hip_get_gemm_mode()
    assert lib.folx_hip_set_gemm_mode(_lib.GEMM_MODE['bf16x3']) == _lib.OK
    assert lib.folx_hip_get_gemm_mode() == _lib.GEMM_MODE['bf16x3']
    assert lib.folx_hip_set_gemm_mode(7) == _lib.EINVAL
    assert lib.folx_hip_get_gemm_mode() == _lib.GEMM_MODE['bf16x3']  # unchanged by the refused call
    assert lib.folx_hip_set_gemm_mode(_lib.GEMM_MODE['f32']) == _lib.OK
    assert lib.folx_hip_get_gemm_mode() == _lib.GEMM_MODE['f32']
    assert lib.folx_hip_set_gemm_mode(before) == _lib.OK


def test_version_and_strerror(lib):
    assert lib.folx_hip_version() >= 100
    assert lib.folx_hip_strerror(0) == b'ok'
    for code in (-1, -2, -3, -99):
        assert len(lib.folx_hip_strerror(code)) > 0


def test_argument_checks_return_error_codes(lib):
    null = ctypes.c_void_p(None)
    # negative sizes / null pointers -> EINVAL, nothing launched
    assert lib.folx_hip_dense_fwdlap(*([null] * 12), 4, 1, 8, 8) == _lib.EINVAL
    assert lib.folx_hip_dense_fwdlap(*([null] * 12), -1, 1, 8, 8) == _lib.EINVAL
    assert lib.folx_hip_elementwise_fwdlap(null, 99, 0.0, null, null, null, null, null, null, 4, 1) == _lib.EINVAL
    assert lib.folx_hip_elementwise_fwdlap(null, 0, 0.0, null, null, null, null, null, null, 4, 1) == _lib.EINVAL
    assert lib.folx_hip_binary_fwdlap(null, 0, null, null, null, null, null, null, null, null, null, null, 1, 1, 1) == _lib.EINVAL
    assert lib.folx_hip_rows_affine(null, null, null, 1, 1, null, null, 1.0, 1.0, null) == _lib.EINVAL
    assert lib.folx_hip_reduce_sum(null, null, null, 1, 1, -1, 1, 1.0) == _lib.EINVAL
    assert lib.folx_hip_slogdet_fwdlap(null, null, null, null, null, null, null, null, 4, 0, 1) == _lib.EINVAL
    assert lib.folx_hip_layernorm_fwdlap(*([null] * 9), 4, 8, 1, 1e-5) == _lib.EINVAL
    assert lib.folx_hip_mhsa_fwdlap(*([null] * 15), 1, 8, 1, 8, 1) == _lib.EINVAL
    assert lib.folx_hip_mhsea_fwdlap(*([null] * 18), 1, 8, 1, 8, 1) == _lib.EINVAL
    assert lib.folx_hip_dense_act_fwdlap(null, 0, 0.0, *([null] * 11), 4, 1, 8, 8, null, 0) == _lib.EINVAL
    assert lib.folx_hip_dense_act_workspace_bytes(-1, 1, 8, 8) == _lib.EINVAL
    assert lib.folx_hip_mhsa_sparse_fwdlap(*([null] * 14), 1, 8, 1, 8, 3) == _lib.EINVAL
    assert lib.folx_hip_mul_sparse_fwdlap(*([null] * 11), 8, 4, 2, 1) == _lib.EINVAL
    assert lib.folx_hip_mul_sparse_fwdlap(*([null] * 11), 9, 4, 2, 1) == _lib.EINVAL       # S not a multiple of S_w
    assert lib.folx_hip_exp_envelope_fwdlap(*([null] * 9), 4, 2, 8, 1) == _lib.EINVAL
    assert lib.folx_hip_slogdet_scaled_fwdlap(*([null] * 12), 1, 1, 4, 1, 16, 0, 4, 16, 16, 1) == _lib.EINVAL
    assert lib.folx_hip_dense_rows_fwdlap(*([null] * 12), 4, 1, 8, 8, 1, 1) == _lib.EINVAL
    assert lib.folx_hip_dot_two_fwdlap(*([null] * 10), 1, 1, 4, 4, 4, 1, null) == _lib.EINVAL
    assert lib.folx_hip_reduce_max(null, null, null, 2, 3, 4) == _lib.EINVAL
    assert lib.folx_hip_reduce_max(null, null, null, -2, 3, 4) == _lib.EINVAL
    assert lib.folx_hip_gather_reduce_rows(null, null, null, null, 2, 2, 1, 1, 4, 4, 1, 1, 1.0) == _lib.EINVAL
    assert lib.folx_hip_gather_cols(null, null, null, null, 2, 4, 4, 1, 1) == _lib.EINVAL
    assert lib.folx_hip_gather_cols(null, null, null, null, -2, 4, 4, 1, 1) == _lib.EINVAL
    assert lib.folx_hip_scatter_add_rows(null, null, null, null, 2, 4, 1, 4, 1) == _lib.EINVAL
    assert lib.folx_hip_slogdet_strided_fwdlap(*([null] * 8), 1, 1, 4, 1, 16, 16, 4, 16) == _lib.EINVAL
    assert lib.folx_hip_sparse_slogdet_fwdlap(*([null] * 11), 1, 4, 1, 1, 1, 1, 0) == _lib.EINVAL
    assert lib.folx_hip_inv_values(null, null, null, null, null, 1, 4) == _lib.EINVAL
    assert lib.folx_hip_trace_pair(null, null, null, null, 1, 4) == _lib.EINVAL
    assert lib.folx_hip_trace_pair(null, null, null, null, -1, 4) == _lib.EINVAL
    assert lib.folx_hip_inv_fwdlap(*([null] * 7), 1, 4, 1) == _lib.EINVAL
    assert lib.folx_hip_inv_fwdlap(*([null] * 7), -1, 4, 1) == _lib.EINVAL
    assert lib.folx_hip_solve_fwdlap(*([null] * 10), 1, 4, 1, 1) == _lib.EINVAL
    assert lib.folx_hip_solve_fwdlap(*([null] * 10), 1, 0, 1, 1) == _lib.EINVAL
    # empty problems are fine and launch nothing
    assert lib.folx_hip_dense_fwdlap(*([null] * 12), 0, 1, 8, 8) == _lib.OK
    assert lib.folx_hip_elementwise_fwdlap(null, 0, 0.0, null, null, null, null, null, null, 0, 1) == _lib.OK
    assert lib.folx_hip_gather_rows(null, null, null, null, 1, 0, 1, 4, 4, 4) == _lib.OK


def test_unsupported_sizes(lib):
    one = ctypes.c_void_p(16)  # non-null, never dereferenced: the size check comes first
    assert lib.folx_hip_slogdet_fwdlap(None, one, one, one, one, one, one, one, 4, 33, 1) == _lib.ENOTSUP
    assert lib.folx_hip_mhsa_fwdlap(None, *([one] * 9), None, None, one, one, one, 1, 65, 1, 8, 1) == _lib.ENOTSUP
    assert lib.folx_hip_mhsa_fwdlap(None, *([one] * 9), None, None, one, one, one, 1, 8, 1, 6, 1) == _lib.ENOTSUP
    assert lib.folx_hip_layernorm_fwdlap(None, one, one, one, None, None, one, one, one, 4, 6, 1, 1e-5) == _lib.ENOTSUP
    assert lib.folx_hip_layernorm_fwdlap(None, one, one, one, None, None, one, one, one, 4, 2048, 1, 1e-5) == _lib.ENOTSUP
    # fused / structure-aware entry points outside the sizes they are built for: the caller takes
    # the general rules instead
    assert lib.folx_hip_dense_act_fwdlap(None, 0, 0.0, *([one] * 5), None, None, None, *([one] * 3), 4, 1, 6, 8, None, 0) == _lib.ENOTSUP     # K % 4
    assert lib.folx_hip_dense_act_fwdlap(None, 0, 0.0, *([one] * 5), None, None, None, *([one] * 3), 4, 1, 256, 8, None, 0) == _lib.ENOTSUP   # K > 128
    assert lib.folx_hip_dense_act_fwdlap(None, 3, 0.0, *([one] * 5), None, None, None, *([one] * 3), 4, 1, 8, 8, None, 0) == _lib.ENOTSUP     # log: not fused
    assert lib.folx_hip_dense_act_workspace_bytes(64, 4, 8, 200) == _lib.ENOTSUP
    assert lib.folx_hip_dense_act_workspace_bytes(1 << 20, 4, 100, 100) == 0                                  # no split
    assert lib.folx_hip_dense_act_workspace_bytes(64, 64, 256, 256) == 2 * 64 * 256 * 4     # wide: 2 groups of 32 rows
    assert lib.folx_hip_dense_act_workspace_bytes(64, 33, 256, 256) == 3 * 64 * 256 * 4     # wide: 3 groups of 16 rows
    assert lib.folx_hip_dense_act_workspace_bytes(60, 33, 256, 256) == 2 * 60 * 256 * 4     # rows % 8: groups of 32
    assert lib.folx_hip_dense_act_workspace_bytes(63, 33, 256, 256) == _lib.ENOTSUP         # wide: rows % 4
    assert lib.folx_hip_dense_act_workspace_bytes(64, 33, 200, 256) == _lib.ENOTSUP         # wide: K % 16
    assert lib.folx_hip_dense_act_fwdlap(None, 0, 0.0, *([one] * 5), None, None, None, *([one] * 3), 64, 33, 256, 256, None, 0) == _lib.EINVAL  # no workspace
    assert lib.folx_hip_dense_act_fwdlap(None, 0, 0.0, *([one] * 11), 64, 33, 256, 256, one, 1 << 30) == _lib.ENOTSUP  # skip connection on a wide layer
    assert lib.folx_hip_dense_act_fwdlap(None, 0, 0.0, *([one] * 5), one, None, None, *([one] * 3), 4, 1, 8, 8, None, 0) == _lib.EINVAL    # part of a residual
    assert lib.folx_hip_reduce_sum_window(None, one, one, 2, 3, 8, 5, 9, 4, 1.0) == _lib.EINVAL   # window past the axis
    assert lib.folx_hip_reduce_sum_window(None, one, one, 2, 3, 8, 5, 4, 4, 1.0) == _lib.EINVAL   # hi < lo
    # Jacobian operand in parts: host arrays of pointers, widths and broadcast flags
    ptrs, wd, bc = (ctypes.c_void_p * 2)(16, 32), (ctypes.c_int32 * 2)(16, 32), (ctypes.c_int32 * 2)(0, 1)
    parts = lambda wd_, R, group, ws, nb: lib.folx_hip_dense_act_parts_fwdlap(
        None, 0, 0.0, one, one, 2, ptrs, wd_, bc, group, one, one, None, None, None, None, None, None, one, one, one, R, 33,
        256, ws, nb)
    assert parts(wd, 64, 4, None, 0) == _lib.EINVAL                                  # no workspace
    assert parts((ctypes.c_int32 * 2)(16, 24), 64, 4, one, 1 << 30) == _lib.ENOTSUP  # width % 16
    assert parts(wd, 64, 5, one, 1 << 30) == _lib.ENOTSUP                            # rows % group
    assert parts(wd, 64, 0, one, 1 << 30) == _lib.EINVAL
    assert lib.folx_hip_dense_act_parts_fwdlap(None, 0, 0.0, one, one, 2, ptrs, wd, bc, 4, one, one, one, None, None,
                                               None, None, None, one, one, one, 64, 33, 256, one, 1 << 30) == _lib.EINVAL  # part of a residual
    assert lib.folx_hip_dense_act_parts_fwdlap(None, 0, 0.0, one, one, 2, ptrs, wd, bc, 4, one, one, None, None, None,
                                               one, one, None, one, one, one, 64, 33, 256, one, 1 << 30) == _lib.EINVAL  # part of a pre-activation term
    # LayerNorm + dense (+ activation): act = -1 means none
    assert lib.folx_hip_norm_dense_workspace_bytes(64, 33, 256, 256, -1) > 2 * 64 * 256 * 4
    assert lib.folx_hip_norm_dense_workspace_bytes(64, 33, 256, 256, 0) > lib.folx_hip_norm_dense_workspace_bytes(64, 33, 256, 256, -1)
    assert lib.folx_hip_norm_dense_workspace_bytes(64, 33, 1024, 256, -1) == _lib.ENOTSUP    # K > 512
    assert lib.folx_hip_norm_dense_workspace_bytes(64, 33, 256, 128, -1) == _lib.ENOTSUP     # narrow layer
    assert lib.folx_hip_norm_dense_workspace_bytes(64, 33, 256, 256, 3) == _lib.ENOTSUP      # log: not fused
    assert lib.folx_hip_norm_dense_workspace_bytes(-1, 33, 256, 256, -1) == _lib.EINVAL
    nd = lambda act, R, K, N, ws, nb: lib.folx_hip_norm_dense_fwdlap(None, act, 0.0, one, one, one, one, one, 1e-5, one,
                                                                    one, one, one, one, R, 33, K, N, ws, nb)
    assert nd(-1, 64, 256, 256, None, 0) == _lib.EINVAL        # no workspace
    assert nd(-1, 62, 256, 256, one, 1 << 30) == _lib.ENOTSUP  # rows % 4
    assert nd(3, 64, 256, 256, one, 1 << 30) == _lib.ENOTSUP   # log: not fused
    # the same rule on the library's own scratch array: size checks come before any GPU call
    nds = lambda act, R, K, N: lib.folx_hip_norm_dense_static_fwdlap(None, act, 0.0, one, one, one, one, one, 1e-5, one,
                                                                     one, one, one, one, R, 33, K, N)
    assert nds(-1, 62, 256, 256) == _lib.ENOTSUP      # rows % 4
    assert nds(3, 64, 256, 256) == _lib.ENOTSUP       # log: not fused
    assert nds(-1, -4, 256, 256) == _lib.EINVAL
    assert lib.folx_hip_norm_dense_workspace_bytes(1 << 17, 33, 256, 256, 0) > _lib.STATIC_SCRATCH_BYTES
    assert nds(0, 1 << 17, 256, 256) == _lib.ESCRATCH  # beyond the 64 MiB array: refused, nothing launched
    assert b'scratch' in lib.folx_hip_strerror(_lib.ESCRATCH)
    assert lib.folx_hip_dense_act_workspace_bytes(2000, 400, 100, 100) > 0                                    # rows split
    assert lib.folx_hip_mhsa_sparse_fwdlap(None, *([one] * 13), 1, 65, 1, 8, 3) == _lib.ENOTSUP
    assert lib.folx_hip_mhsa_sparse_fwdlap(None, *([one] * 13), 1, 8, 1, 6, 3) == _lib.ENOTSUP
    assert lib.folx_hip_mul_sparse_fwdlap(None, *([one] * 10), 8, 4, 2, 9) == _lib.ENOTSUP
    assert lib.folx_hip_exp_envelope_fwdlap(None, *([one] * 8), 4, 9, 8, 1) == _lib.ENOTSUP
    assert lib.folx_hip_exp_envelope_fwdlap(None, *([one] * 8), 4, 2, 6, 1) == _lib.ENOTSUP
    assert lib.folx_hip_slogdet_scaled_fwdlap(None, *([one] * 11), 1, 1, 32, 1, 1024, 0, 32, 1024, 1024, 1) == _lib.ENOTSUP
    assert lib.folx_hip_slogdet_scaled_fwdlap(None, *([one] * 11), 1, 1, 8, 1, 64, 0, 8, 64, 64, 5) == _lib.ENOTSUP


def test_product_fails_loudly_without_gpu():
    import numpy as np
    import torch

    import folx_amd
    from folx_amd import numpy as fnp

    if torch.cuda.is_available():
        pytest.skip('GPU present')
    with pytest.raises(_lib.FolxHipError):
        folx_amd.forward_laplacian(lambda x: fnp.tanh(x), 0)(np.zeros(3, np.float32))


# us (plain product + activation, groups of 8, 16, 32) of a dense + activation layer, measured in both product modes: a form whose
# estimate is not well ahead must not displace the faster one
MEASURED_LAYERS = [
    # mode, R, P, K, N, times, Jacobian rows of a group, whether the fused rule is the faster one
    ('f32', 5376, 8, 512, 256, (152, 176, 237, 419), None, 0),
    ('f32', 1788, 21, 64, 300, (45, 65, 63, 61), None, 0),
    ('f32', 6000, 117, 64, 256, (518, 329, 319, 297), 32, 1),
    ('f32', 3584, 39, 256, 256, (230, 209, 231, 263), 8, 1),
    ('f32', 5376, 24, 512, 256, (380, 321, 441, 436), 8, 1),
    ('bf16x3', 5376, 21, 512, 256, (218, 244, 304, 294), None, 0),
    ('bf16x3', 3584, 8, 256, 256, (55, 65, 76, 112), None, 0),
    ('bf16x3', 6000, 117, 64, 256, (453, 310, 286, 261), 32, 1),
    ('bf16x3', 1968, 87, 16, 256, (104, 71, 57, 50), 32, 1),
]


@pytest.mark.parametrize('mode,R,P,K,N,times,group,faster', MEASURED_LAYERS)
def test_wide_dense_act_takes_the_form_that_was_measured_faster(lib, mode, R, P, K, N, times, group, faster):
    before = lib.folx_hip_get_gemm_mode()
    lib.folx_hip_set_gemm_mode(_lib.GEMM_MODE[mode])
    try:
        assert lib.folx_hip_dense_act_faster(R, P, K, N, K) == faster
        if group is not None:
            assert lib.folx_hip_dense_act_form(R, P, K, N, 0) == group
            assert dict(zip((8, 16, 32), times[1:]))[group] <= 1.05 * min(times)
        else:
            assert times[0] == min(times)
        # read in parts, the fused rule contracts 320 of 832 features
        assert lib.folx_hip_dense_act_faster(3584, 21, 320, 256, 832) == 1
    finally:
        lib.folx_hip_set_gemm_mode(before)


# narrow layers without a skip connection: time of the few-rows kernel over the general one's
@pytest.mark.parametrize('R,P,K,N,ratio', [
    (2000, 4, 100, 100, 0.63), (6000, 6, 128, 128, 1.14), (6000, 4, 128, 128, 1.07), (4091, 6, 128, 128, 0.71), (6000, 6, 4, 128, 0.92),
    (5115, 3, 64, 64, 0.67), (60000, 1, 20, 48, 0.85), (60000, 6, 64, 48, 1.07), (60000, 6, 4, 48, 1.16), (60000, 4, 128, 100, 1.06),
    (32763, 6, 8, 96, 1.26), (28795, 2, 8, 96, 1.08), (140795, 6, 32, 48, 1.20), (60000, 4, 128, 48, 0.64), (187472, 0, 128, 48, 0.52),
    (195179, 5, 20, 42, 1.67), (21110, 4, 24, 87, 1.56), (74292, 1, 16, 43, 1.37), (27965, 6, 124, 41, 0.84), (68104, 1, 80, 85, 0.77),
    (105354, 0, 44, 11, 0.50), (49595, 3, 124, 11, 0.46), (3299, 1, 20, 78, 0.79),
])
def test_narrow_dense_act_takes_the_kernel_that_was_measured_faster(lib, R, P, K, N, ratio):
    assert lib.folx_hip_dense_act_form(R, P, K, N, 0) == (2 if ratio < 1 else 1)
    assert lib.folx_hip_dense_act_form(R, P, K, N, 1) == 2


# chains of narrow layers: time in one launch over that of the layers one by one
@pytest.mark.parametrize('R,P,widths,ratio', [
    (2000, 4, (4, *[100] * 10, 1), 0.5), (25600, 4, (4, *[100] * 10, 1), 0.77), (100000, 6, (128,) * 7, 0.82),
    (400, 1, (128, 4, 128), 0.54), (4000, 1, (128, 4, 128), 0.68), (40000, 1, (128, 4, 128), 1.26), (200000, 3, (128, 4, 128), 1.26),
    (200000, 1, (128, 8, 8, 128), 1.72), (4000, 6, (128, 8, 8, 128), 0.64), (180793, 3, (128, 8, 4), 2.70), (37974, 6, (100, 4, 1), 1.83),
    (123571, 2, (100, 8, 100), 1.67), (191836, 1, (48, 48, 4, 128), 1.50), (169064, 3, (128, 8, 16, 12, 16, 20, 128), 1.39),
    (200000, 6, (4,) * 9, 0.61), (200000, 6, (16,) * 9, 0.39), (200000, 6, (32, 128, 32), 0.77),
    (200000, 3, (3, 64, 64, 1), 0.48), (200000, 1, (5, 127, 3, 127, 1), 0.37),
])
def test_a_chain_is_taken_where_it_was_measured_faster(lib, R, P, widths, ratio):
    act = (ctypes.c_int32 * (len(widths) - 1))(*[-1 if n == 1 else _lib.ACT['tanh'] for n in widths[1:]])
    got = lib.folx_hip_dense_chain_faster(len(widths) - 1, act, (ctypes.c_int32 * len(widths))(*widths), R, P)
    assert got == (1 if ratio < 1 else 0)


def test_one_workspace_serves_both_product_modes(lib):
    before = lib.folx_hip_get_gemm_mode()
    forms, sizes = [], []
    for mode in _lib.GEMM_MODE.values():
        lib.folx_hip_set_gemm_mode(mode)
        forms.append(lib.folx_hip_dense_act_form(2060, 21, 80, 256, 0))
        sizes.append(lib.folx_hip_dense_act_workspace_bytes(2060, 21, 80, 256))
    lib.folx_hip_set_gemm_mode(before)
    assert forms == [8, 32] and sizes == [3 * 2060 * 256 * 4] * 2


def test_questions_about_a_shape(lib):
    form, faster = lib.folx_hip_dense_act_form, lib.folx_hip_dense_act_faster
    assert form(2000, 4, 100, 100, 0) == 2 and form(1 << 20, 4, 100, 100, 0) == 1 and form(1 << 20, 4, 100, 100, 1) == 2
    assert faster(2000, 4, 100, 100, 100) == 1
    assert form(64, 33, 200, 256, 0) == faster(64, 33, 200, 256, 200) == _lib.ENOTSUP   # K % 16
    assert form(64, 0, 256, 256, 0) == faster(64, 0, 256, 256, 256) == _lib.ENOTSUP     # no Jacobian row
    tile = lib.folx_hip_dense_form
    # R, P, K, N of tests/test_kernel_edges_gpu.py::test_dense_small_tiles, then the line between the two
    for shape in ((1, 1, 16, 68), (63, 2, 48, 100), (64, 3, 32, 128), (65, 9, 256, 132), (130, 7, 64, 300), (400, 30, 256, 256), (1280, 62, 256, 256)):
        assert tile(*shape) == 64
    assert tile(1550, 100, 256, 256) == 128 and tile(3000, 98, 512, 100) == 128
    assert tile(64, 3, 32, 64) == tile(64, 3, 40, 128) == tile(64, 3, 32, 130) == _lib.ENOTSUP
    assert form(-1, 4, 100, 100, 0) == faster(64, 33, 256, 256, 0) == _lib.EINVAL


def test_lds_permission_is_asked_for_once_per_device(tmp_path):
    """The helper on the host, with the two runtime calls it makes replaced: a second device of the process asks for itself."""
    import subprocess

    from folx_amd import build

    (tmp_path / 'grant.hip').write_text(r'''
#include "common.h"
static int device = 0, asked = 0;
static hipError_t answer = hipSuccess;
extern "C" hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { ++asked; return answer; }
int main() {
  FolxLdsGrant g;
  answer = hipErrorInvalidValue;
  if (g.ask(&g, 1) || asked != 1) return 1;                                  // refused: asked again
  answer = hipSuccess;
  if (!g.ask(&g, 1) || !g.ask(&g, 1) || asked != 2) return 2;
  device = 3;
  if (!g.ask(&g, 1) || !g.ask(&g, 1) || asked != 3) return 3;
  device = 0;
  if (!g.ask(&g, 1) || asked != 3) return 4;
  device = 64;                                                               // beyond the mask: every time
  if (!g.ask(&g, 1) || !g.ask(&g, 1) || asked != 5) return 5;
  return 0;
}
''')
    exe = str(tmp_path / 'grant')
    subprocess.run([build._hipcc(), '--offload-arch=gfx950', '-I', build.CSRC, '-x', 'hip', str(tmp_path / 'grant.hip'), '-o', exe],
                   check=True, capture_output=True)
    assert subprocess.run([exe]).returncode == 0
