"""The sizes at which a kernel's own launch or 32-bit arithmetic ends, on the CPU:
the rules that leave such calls to another route (no GPU needed)."""
import ctypes

import pytest

import ane_amd


def rule(mangled, restype, *argtypes):
    f = getattr(ane_amd.lib(), mangled)
    f.restype, f.argtypes = restype, argtypes
    return f


@pytest.mark.parametrize("N,nb,T,fits", [
    (4096, 128, 512, True), (1, 1, 5, True),
    # weights of 2 GiB and more, and N + 64 past 2^32
    (61_680_000, 1, 64, True), (63_161_284, 1, 64, False), ((1 << 32) - 64, 1, 5, False), ((1 << 32) - 1, 1, 5, False),
    # 512 threads per 64 rows x 64 tokens (x 32 up to 32 tokens): 2^32 work items
    (1 << 20, 1, 32704, True), (1 << 20, 1, 32768, False), ((1 << 20) + 64, 1, 32768, False),
    (1 << 11, 1, 16_700_000, True), (1 << 12, 1, 16_700_000, False),
])
def test_prompt_kernel(N, nb, T, fits):
    """ane::prompt_eligible (q8_0_prompt.hip)."""
    f = rule("_ZN3ane15prompt_eligibleEjjjPKv", ctypes.c_bool, *[ctypes.c_uint32] * 3, ctypes.c_void_p)
    assert f(N, nb, T, 0) == fits


@pytest.mark.parametrize("n,blocks", [(1, 1), (4, 2), (2048, 2), (2052, 3), (1 << 30, (1 << 19) + 1),
                                      (((1 << 24) - 2) * 2048, (1 << 24) - 1), (((1 << 24) - 2) * 2048 + 4, 0),
                                      (1 << 35, 0), (1 << 40, 0)])
def test_flat_elementwise(n, blocks):
    """ane::flat_ew_blocks (ggml_backend.hip): 256 threads a workgroup, 2^24
    workgroups are one too many."""
    f = rule("_ZN3ane14flat_ew_blocksEm", ctypes.c_uint64, ctypes.c_uint64)
    assert f(n) == blocks


@pytest.mark.parametrize("N,T,fits", [(1, 2, True), (4096, 512, True), (119_000_000, 32, True),
                                      (1 << 20, (1 << 15) - 64, True), (1 << 20, (1 << 15) - 63, False),
                                      (1 << 15, 1 << 20, False), (119_000_000, 16_000_000, False)])
def test_handlers_product(N, T, fits):
    """ane::rmode_launch_fits (rmode_mul_mat.hip): 512 threads per 64 x 64 outputs
    above 32 tokens."""
    f = rule("_ZN3ane17rmode_launch_fitsEjj", ctypes.c_bool, *[ctypes.c_uint32] * 2)
    assert f(N, T) == fits


@pytest.mark.parametrize("rows,pairs,step", [(1, 64, 1), (4096, 64, 4096), (5000, 64, 4096), (40000, 64, 5000),
                                             (1 << 29, 64, (1 << 26) - 4), (1 << 29, 1, 1 << 26), (7, 1 << 30, 3),
                                             (2, (1 << 31) - 1, 1), (1 << 36, 1, (1 << 32) - 256)])
def test_rope_sweep(rows, pairs, step):
    """ane::rope_node_step (decode_ref.hip): a sweep stays below 2^32 threads."""
    f = rule("_ZN3ane14rope_node_stepEmj", ctypes.c_uint64, ctypes.c_uint64, ctypes.c_uint32)
    assert f(rows, pairs) == step
    assert -(-step * pairs // 256) * 256 < 1 << 32
