"""Which form of a linear a call takes (csrc/gemm_rows.hip: gemm_rows_form, csrc/skinny.hip: skinny_form), asked of the library on the host: K slices never need more scratch than
the caller brings."""
import pytest
import torch

ROWS = [(20, 4096, 11008), (139, 12288, 4096), (139, 4096, 11008), (250, 4096, 11008), (300, 4096, 4096), (512, 4096, 11008), (1087, 4096, 11008)]
BATCH = [(2, 1088, 11008), (16, 640, 13824), (32, 2048, 13824), (32, 4032, 13824), (32, 4096, 11008), (32, 5120, 13824)]


@pytest.mark.parametrize("M,N,K", ROWS)
def test_slices_fit_the_scratch(M, N, K):
    from llava_mi355x import ops
    full = ops.gemm_form(torch.bfloat16, M, N, K)
    assert full[3] > 1
    for s in range(1, full[3] + 1):
        for short in (0, 1):                            # room for s slices, and one byte less
            room = s * (M if full[0] else -(-M // 256) * 256) * (N if full[0] else -(-N // 256) * 256) * 4
            form = ops.gemm_form(torch.bfloat16, M, N, K, scratch_bytes=room - short)
            if form[0] == full[0]:
                assert form[3] <= max(1, s - short)
            assert form[3] == 1 or form[3] * M * N * 4 <= room
    assert ops.gemm_form(torch.bfloat16, M, N, K, scratch_bytes=0)[3] == 1


@pytest.mark.parametrize("M,N,K", BATCH)
def test_slices_of_a_decode_batch_fit_the_scratch(M, N, K):
    from llava_mi355x import ops
    _, rt, ct, ks = ops.gemm_form(torch.bfloat16, M, N, K, batch=True)
    need = -(-N // (16 * rt)) * ks * rt * ct * 1024
    assert need <= 64 << 20
    if ks > 1:
        assert ops.gemm_form(torch.bfloat16, M, N, K, batch=True, scratch_bytes=need) == (0, rt, ct, ks)
        assert ops.gemm_form(torch.bfloat16, M, N, K, batch=True, scratch_bytes=need - 1) != (0, rt, ct, ks)
    assert ops.gemm_form(torch.bfloat16, M, N, K, batch=True, scratch_bytes=0)[3] == 1


# rows, weights, K: where a row-tile form measured at least a twentieth slower / faster than the other kernels
OTHERS = [(257, 3072, 2048, 0), (300, 3072, 3072, 0), (128, 4096, 2048, 0), (256, 8192, 1536, 0), (96, 6656, 4096, 0), (257, 2560, 5120, 0), (258, 9792, 7296, 0), (183, 18176, 7744, 0), (2048, 4096, 2048, 0), (2308, 3072, 1024, 0), (33, 10240, 2048, 0)]
ROW_TILES = [(20, 4096, 11008, 0), (64, 3072, 2048, 0), (139, 12288, 4096, 0), (139, 22016, 4096, 3), (251, 11456, 2304, 0), (257, 4096, 4096, 0), (384, 5120, 13824, 0), (250, 27648, 5120, 3), (257, 6208, 2048, 0), (600, 4096, 4096, 0), (2308, 1024, 4096, 0), (25, 26816, 1216, 0), (11, 18048, 4224, 0)]


# past 256 rows and 640 tiles of 64 x 64, where the four-wave tiles measured faster than both: mb, nb, K slices
FOUR_WAVES = {(484, 14720, 2816, 0): (6, 6, 1), (512, 16384, 3072, 3): (5, 8, 1), (500, 12288, 4096, 0): (5, 6, 1), (500, 15360, 5120, 0): (6, 6, 1), (1087, 4096, 2048, 0): (5, 4, 1),
              (2048, 3072, 2048, 0): (5, 6, 1), (1087, 4096, 11008, 0): (7, 8, 3), (258, 9792, 7296, 0): (5, 8, 3)}


@pytest.mark.parametrize("case", OTHERS + ROW_TILES)
def test_the_faster_kernel(case):
    from llava_mi355x import ops
    M, N, K, act = case
    assert (ops.gemm_form(torch.bfloat16, M, N, K, act=act)[0] == 1) == (case in ROW_TILES)


@pytest.mark.parametrize("case", list(FOUR_WAVES))
def test_four_wave_tiles(case):
    from llava_mi355x import ops
    M, N, K, act = case
    assert ops.gemm_form(torch.bfloat16, M, N, K, act=act) == (2,) + FOUR_WAVES[case]


@pytest.mark.parametrize("M,N", [(256, 12288), (257, 12288), (257, 8192), (257, 8256)])
def test_the_line_of_the_four_wave_tiles(M, N):
    """256 rows, 640 tiles of 64 x 64: on the line another kernel, past it the four-wave tiles."""
    from llava_mi355x import ops
    assert (ops.gemm_form(torch.float16, M, N, 2048)[0] == 2) == ((M, N) in ((257, 12288), (257, 8256)))


# products past that line that the four-wave tiles make in a tenth more time than another form, or half as much again (a short K, an activation behind a K of up to some 2000), and the
# same products with a longer K or without the activation; three that one round of small tiles makes in less time than the row tiles
SHORT = [(1087, 12288, 192, 1), (2693, 2048, 128, 0), (3303, 13824, 576, 1), (722, 8824, 512, 2), (1152, 5120, 1024, 2), (1348, 21056, 448, 3), (1620, 20648, 448, 2)]
LONG = [(1087, 12288, 4096, 1), (2693, 2048, 1024, 0), (3303, 13824, 4096, 1), (722, 8824, 4096, 2), (1152, 5120, 8192, 0), (1348, 21056, 1024, 3), (1620, 20648, 1024, 0),
        (2304, 4096, 1024, 2), (2308, 4096, 1024, 1), (2200, 1280, 2048, 0), (680, 4096, 4096, 0), (520, 4640, 3072, 0)]


@pytest.mark.parametrize("case", SHORT + LONG)
def test_products_that_the_four_wave_tiles_leave(case):
    from llava_mi355x import ops
    M, N, K, act = case
    assert (ops.gemm_form(torch.bfloat16, M, N, K, act=act)[0] == 2) == (case in LONG)


@pytest.mark.parametrize("M,N,K,act,rt", [(2, 15360, 5120, 0, 1), (8, 12288, 4096, 0, 1), (8, 32000, 4096, 0, 1), (9, 12288, 4096, 0, 4), (32, 15360, 5120, 0, 4), (8, 22016, 4096, 3, 2),
                                          (8, 27648, 5120, 3, 4), (16, 6208, 4096, 0, 2), (32, 6208, 4096, 0, 2)])
def test_tiles_of_a_decode_batch(M, N, K, act, rt):
    """The measured best at widths where the forms are a twentieth and more apart."""
    from llava_mi355x import ops
    assert ops.gemm_form(torch.bfloat16, M, N, K, act=act, batch=True)[1] == rt


@pytest.mark.parametrize("dt,N,K,ldx,ldw,words", [(torch.bfloat16, 256, 128, 132, 128, "16-byte row alignment"), (torch.float16, 256, 128, 128, 129, "16-byte row alignment"),
                                                  (torch.bfloat16, 250, 128, 128, 128, "multiple of 8"), (torch.bfloat16, 256, 96, 96, 96, "multiple of 64"), (torch.float32, 256, 128, 128, 128, "16-bit dtypes")])
@pytest.mark.parametrize("variant", [1101, 2201])
def test_a_form_by_number_checks_what_the_choice_checks(dt, N, K, ldx, ldw, words, variant):
    """Refused on the host, before anything is allocated or launched (the pointers are not memory)."""
    import ctypes
    from llava_mi355x import _C
    any_ = ctypes.c_void_p(4096)
    assert _C.lib.lmx_op_gemm(_C.torch_dtype_code(dt), any_, any_, any_, None, None, 64, N, K, ldx, ldw, N, 0, 0, variant, None) != 0
    assert words in _C.last_error()


@pytest.mark.parametrize("dt,K,ldx,ldw,words", [(torch.bfloat16, 256, 260, 256, "16-byte row alignment"), (torch.float16, 256, 256, 257, "16-byte row alignment"), (torch.bfloat16, 96, 96, 96, "multiple of 64"),
                                                (torch.float32, 256, 256, 256, "16-bit dtypes")])
@pytest.mark.parametrize("variant", [881, 882, 443])
def test_a_four_wave_form_by_number_checks_what_the_choice_checks(dt, K, ldx, ldw, words, variant):
    import ctypes
    from llava_mi355x import _C
    any_ = ctypes.c_void_p(4096)
    assert _C.lib.lmx_op_gemm(_C.torch_dtype_code(dt), any_, any_, any_, None, None, 64, 256, K, ldx, ldw, 256, 0, 0, variant, None) != 0
    assert words in _C.last_error()


@pytest.mark.parametrize("variant", [100, 102, 109, 331, 492, 802, 803, 902])
def test_a_four_wave_tile_that_is_not_there(variant):
    """No tile of 0 blocks, none outside the table: an error before anything is computed from its sizes."""
    import ctypes
    from llava_mi355x import _C
    any_ = ctypes.c_void_p(4096)
    assert _C.lib.lmx_op_gemm(_C.torch_dtype_code(torch.bfloat16), any_, any_, any_, None, None, 64, 256, 256, 256, 256, 256, 0, 0, variant, None) != 0
    assert "no such tile" in _C.last_error()


@pytest.mark.parametrize("M,N,K,tiles", [(385, 2048, 8192, True), (384, 2048, 8192, False), (385, 1472, 8192, True), (385, 1408, 8192, False), (1100, 1024, 5120, True), (1100, 896, 5120, False),
                                         (1024, 1024, 5120, False), (1100, 1024, 5056, False)])
def test_a_long_k_moves_the_line(M, N, K, tiles):
    """Past 384 rows more than 160 tiles of 64 x 64 from a K of 8192 on, more than 256 (and 1024 weights) from 5120 on."""
    from llava_mi355x import ops
    assert (ops.gemm_form(torch.bfloat16, M, N, K)[0] == 2) == tiles
