"""CPU-only checks of the boundary: the C-ABI library loads without a GPU and exports every symbol
the header declares; the host layer rejects what it must without touching the device."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, 'include', 'quest_hip.h')).read()
    text = re.sub(r'/\*.*?\*/', '', text, flags=re.S)
    return sorted(set(re.findall(r'\b(quest_[a-z0-9_]+)\s*\(', text)))


def test_header_declares_the_expected_entry_points():
    names = declared_symbols()
    for n in ['quest_version', 'quest_status_string', 'quest_find_scale_int4', 'quest_quantize_int4',
              'quest_add_mul_vv', 'quest_matmul_int4_int4t_int32', 'quest_fused_matmul_dequantize_int4_int4t', 'quest_fused_matmul_dequantize_swiglu_int4_int4t',
              'quest_hadamard128', 'quest_hadamard_quantize_int4', 'quest_hadamard_quantize_int4_rule',
              'quest_rmsnorm_hadamard_quantize_int4', 'quest_add_rmsnorm_hadamard_quantize_int4', 'quest_silu_mul_hadamard_quantize_int4', 'quest_rope_interleaved']:
        assert n in names


def test_library_exports_every_declared_symbol():
    from quest_amd import _lib
    lib = _lib.load()
    for name in declared_symbols():
        assert hasattr(lib, name), name
        assert name in _lib.SIGNATURES, f'{name} has no ctypes signature'
    assert set(_lib.SIGNATURES) == set(declared_symbols())
    assert lib.quest_version() >= 100
    assert lib.quest_status_string(0) == b'ok'
    assert b'NULL' in lib.quest_status_string(-1)


def test_argument_errors_need_no_gpu():
    from quest_amd import _lib
    lib = _lib.load()
    null = ctypes.c_void_p(0)
    fake = ctypes.c_void_p(0x1000)
    assert lib.quest_find_scale_int4(null, fake, 128, 1, 0, null) == -1
    assert lib.quest_find_scale_int4(fake, fake, 12, 1, 0, null) == -2
    assert lib.quest_find_scale_int4(fake, fake, 128, 1, 5, null) == -3
    assert lib.quest_find_scale_int4(fake, ctypes.c_void_p(0x1004), 128, 1, 0, null) == -4
    assert lib.quest_quantize_int4(fake, null, null, null, null, 128, 1, 0, 0, null) == -1
    assert lib.quest_hadamard128(fake, fake, 64, 1, 0.1, 0, null) == -2
    assert lib.quest_hadamard_quantize_int4(fake, fake, null, null, null, 128 * 1024, 1, 0.1, 0, null) == -5
    assert lib.quest_matmul_int4_int4t_int32(fake, fake, fake, 0, 128, 4, null) == -2
    assert lib.quest_matmul_int4_int4t_int32(fake, fake, fake, 4, 100, 4, null) == -2
    assert lib.quest_matmul_int4_int4t_int32(fake, fake, fake, 4, 1 << 18, 4, null) == -5
    assert lib.quest_fused_matmul_dequantize_int4_int4t(fake, fake, fake, null, fake, fake, fake, 4, 128, 4, 0, null) == -1
    assert lib.quest_add_mul_vv(fake, fake, fake, fake, fake, fake, 4, 4, 2, null) == -3


def test_host_layer_refuses_cpu_tensors_and_foreign_backends():
    import quest
    import quest_amd
    from quest_amd import harness
    assert quest.find_scale_int4 is quest_amd.find_scale_int4
    x = torch.zeros(4, 128, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match='GPU only'):
        quest_amd.find_scale_int4(x)
    with pytest.raises(AssertionError):
        quest_amd.find_scale_int4(x.float())
    with pytest.raises(NotImplementedError):
        harness.find_scale_int4(x, backend='pytorch')
    with pytest.raises(NotImplementedError):
        harness.preprocess_weight(x, use_sparse=True)
    with pytest.raises(NotImplementedError):
        quest_amd.generate_random_meta48_int4(4, 64)


def test_unpack_int4_host_helper_matches_oracle():
    from oracle import quest_oracle as qo
    from quest_amd import harness
    b = torch.arange(256, dtype=torch.int32).to(torch.uint8).view(2, 128)
    assert torch.equal(harness.unpack_int4(b), qo.unpack_int4(b))


def test_e2m3_plan_names_the_kernel_that_runs():
    """(tile rows, tile channels, k per slot) on 256 compute units for the sizes that the GPU tests of the tile shapes use: 64 k = K
    split over the waves, 128 k = the waves share the tile; 256 x 256 tiles otherwise."""
    from quest_amd import _lib
    lib = _lib.load()
    expected = {(32, 32, 64): [(1, 128, 8), (257, 2560, 77), (97, 640, 264)], (32, 64, 64): [(33, 1024, 4100), (257, 128, 1500)],
                (64, 64, 64): [(100, 512, 4104), (333, 128, 2056), (2100, 384, 203), (257, 4096, 3104)], (128, 64, 64): [(257, 4096, 4100), (65, 4096, 11000)],
                (64, 64, 128): [(200, 128, 11000), (1000, 128, 2051)], (64, 128, 128): [(257, 384, 6008), (257, 2560, 10999)],
                (128, 64, 128): [(200, 384, 4104), (1000, 2560, 1031)], (128, 128, 128): [(130, 512, 10999), (1400, 1024, 2056)],
                (128, 192, 128): [(333, 1024, 11000), (3000, 512, 1501)], (256, 128, 128): [(2100, 128, 3099), (3000, 384, 2056)],
                (256, 256, 64): [(4098, 256, 2104), (4096, 4096, 11008)]}
    plan = (ctypes.c_int * 8)()
    for (rows, channels, k), sizes in expected.items():
        for m, size_k, n in sizes:
            assert lib.quest_e2m3_gemm_plan(m, size_k, n, 256, plan) == 0
            assert (plan[4], plan[5], plan[7]) == (rows, channels, k), (m, size_k, n, list(plan))
            tiles = -(-m // rows) * -(-n // channels)
            assert plan[6] >= 3 and (rows == 256 == channels or tiles <= plan[0] < tiles + 8)
    assert lib.quest_e2m3_gemm_plan(200, 100, 64, 256, plan) == -2


def test_e2m3_short_rows_take_the_resident_kernel_where_it_is_the_faster_one():
    """Rows of 512 to 1664 elements on 256 compute units: 256 x 256 tiles where the kernel that keeps a channel tile in LDS would leave
    workgroups idle or fetch all weights eight times for few tokens (measured 3 to 19 % slower there)."""
    from quest_amd import _lib, harness
    lib = _lib.load()
    plan = (ctypes.c_int * 8)()
    large = [(512, 1408, 16640), (700, 1664, 16640), (658, 1408, 16832), (700, 1664, 19584), (2048, 1024, 16640), (2048, 1536, 18112),
             (3000, 1536, 16640), (3000, 640, 18112), (4000, 1024, 18112), (3913, 1536, 17712), (4827, 1280, 17536),
             (3769, 1664, 2096), (4061, 1536, 2104), (4650, 1280, 10416)]
    resident = [(563, 1024, 22016), (1022, 1024, 22016), (3000, 1024, 22016), (5000, 1536, 16640), (8192, 1024, 18112), (1000, 1536, 11264), (6000, 1024, 13824),
                (4227, 1536, 3192), (4542, 1664, 1808), (5003, 1024, 10448)]
    for sizes, rows in ((large, 256), (resident, 64)):
        for m, k, n in sizes:
            assert lib.quest_e2m3_gemm_plan(m, k, n, 256, plan) == 0 and plan[4] == rows, (m, k, n, list(plan))
    # a fused block goes back to the INT8 kernels with it
    assert not harness.block_prefers_e2m3(4200, 1024, 17536) and harness.block_prefers_e2m3(5000, 1024, 17536) and harness.block_prefers_e2m3(4200, 1024, 11264)


def test_e2m3_few_channel_tiles_are_128_wide():
    """128 x 96 tiles only where the XCDs do not read the tokens more often for them: eight 128-channel tiles and more, or as many of
    either width (measured up to 1.28 times slower elsewhere)."""
    from quest_amd import _lib
    lib = _lib.load()
    plan = (ctypes.c_int * 8)()
    sizes = {128: [(4000, 6272, 768), (8613, 6272, 224), (7460, 1792, 320), (4386, 9472, 640), (5084, 2048, 512), (6929, 3712, 384), (3118, 2048, 896),
                   (28978, 2560, 67), (20148, 3072, 83)],
             96: [(3072, 5120, 897), (2560, 8192, 1024), (15669, 3456, 138), (16201, 1536, 192), (7191, 9600, 257), (200, 4096, 11008), (1000, 2560, 2560)]}
    for channels, shapes in sizes.items():
        for m, k, n in shapes:
            assert lib.quest_e2m3_gemm_plan(m, k, n, 256, plan) == 0 and list(plan[4:6]) == [128, channels], (m, k, n, list(plan))
