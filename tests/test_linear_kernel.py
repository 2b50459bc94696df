"""Which kernel a linear layer or grouped projection runs, by its sizes
(kvp_linear_kernel, host code): the rules' edges."""

import pytest

FP32, BF16 = 0, 1
ANY, SHORT = 0, 1


def _kernel(lib, in_dtype, rows, K, N, groups=1, out_dtype=None, acc=False):
    out_dtype = in_dtype if out_dtype is None else out_dtype
    return lib.kvp_linear_kernel(in_dtype, out_dtype, rows, K, N, groups, int(acc))


@pytest.mark.parametrize("rows,K,N,want", [
    (12480, 16, 1536, SHORT), (1560, 16, 1536, SHORT), (64, 16, 256, SHORT),
    (63, 16, 1536, ANY), (1, 4, 1536, ANY),
    # rows of few features, alone or as the rest of a column block
    (12480, 16, 4, ANY), (12480, 16, 124, ANY), (12480, 16, 128, SHORT),
    (12480, 12, 60, ANY), (12480, 12, 64, SHORT), (12480, 8, 64, SHORT), (12480, 4, 4, SHORT),
    (1560, 16, 260, ANY), (16383, 8, 300, ANY), (16384, 8, 300, SHORT), (1560, 8, 320, SHORT),
    (5461, 16, 772, ANY), (5462, 16, 772, SHORT),
    # other inner dimensions, features not in fours
    (12480, 20, 256, ANY), (12480, 15, 256, ANY), (12480, 16, 258, ANY),
])
def test_short_inner_fp32(lib, rows, K, N, want):
    assert _kernel(lib, FP32, rows, K, N) == want
    assert _kernel(lib, FP32, rows, K, N, acc=True) == want
    assert _kernel(lib, BF16, rows, K, N) == ANY


@pytest.mark.parametrize("rows,K,N,groups,out_dtype,acc,want", [
    (12480, 1536, 1536, 3, BF16, False, 4), (12480, 1536, 1536, 1, FP32, True, 4),
    (3120, 1536, 1536, 3, BF16, False, 3), (1560, 1536, 1536, 3, BF16, False, 2),
    # few chunks of K
    (12480, 128, 4608, 1, BF16, False, 2), (12480, 192, 1536, 3, BF16, False, 2),
    (12480, 256, 1536, 3, BF16, False, 4), (12480, 704, 3072, 1, FP32, True, 2),
    (12480, 768, 3072, 1, FP32, True, 4), (12480, 704, 3072, 1, FP32, False, 4),
    # not tiled: K not a multiple of 64, N of 128
    (12480, 1568, 1536, 1, BF16, False, ANY), (12480, 1536, 1500, 1, BF16, False, ANY),
])
def test_bf16_tiles(lib, rows, K, N, groups, out_dtype, acc, want):
    assert _kernel(lib, BF16, rows, K, N, groups, out_dtype, acc) == want


def test_fp32_tiles_are_128_by_128(lib):
    assert _kernel(lib, FP32, 12480, 1536, 1536, 3) == 2
    assert _kernel(lib, FP32, 1, 32, 128, acc=True) == 2
    assert _kernel(lib, FP32, 12480, 48, 1536) == ANY


@pytest.mark.parametrize("args", [
    (FP32, BF16, 8, 64, 128, 1, 0), (2, 0, 8, 64, 128, 1, 0), (BF16, BF16, 8, 64, 128, 1, 1),
    (FP32, FP32, 0, 64, 128, 1, 0), (FP32, FP32, 8, 0, 128, 1, 0), (FP32, FP32, 8, 64, 128, 4, 0),
])
def test_refused(lib, args):
    assert lib.kvp_linear_kernel(*args) == -1
