"""The launch plans (csrc/plans.h) over sizes that no device is needed for."""
import plans
import pytest


@pytest.fixture(scope="module")
def lib():
    return plans.load()


# wan_qkv_proj_sumsq accepts row strides of x below 2^23 elements; a tile's rows are copied from 32-bit
# byte offsets (row * stride * 2, and up to 128 bytes of k).  320 rows: 319 * 2 * 6731920 + 128 = 2^32 - 2208
@pytest.mark.parametrize("ldx,tall", [(3072, True), (6731920, True), (6731928, False), (7000000, False),
                                      ((1 << 23) - 8, False)])
def test_gemm_tiles_end_within_their_offsets(lib, ldx, tall):
    assert (plans.gemm(lib, 2160, 9216, 3072, ldx)[0] == 320) == tall


@pytest.mark.parametrize("ldx", [6731920, 6731928, 7500000, (1 << 23) - 8])
def test_gemm_offsets_fit_at_every_size(lib, ldx):
    for scratch in (0, 1 << 30):
        for M in [1, 2, 255, 256, 257, 319, 320, 321] + list(range(400, 16000, 117)):
            for N, K in ((9216, 3072), (3072, 14336), (3072, 3072), (512, 64)):
                rows = plans.gemm(lib, M, N, K, ldx, scratch=scratch)[0]
                assert rows in (128, 192, 256, 320)
                assert (min(rows, M) - 1) * ldx * 2 + 128 <= 1 << 32, (M, N, K, rows)


def test_gemm_plan_is_the_same_with_ordinary_strides(lib, W):
    """... and its scratch is what wan_qkv_proj_workspace asks for (256 CUs without a device)."""
    ws = W._native.lib().wan_qkv_proj_workspace
    for M in range(1, 9000, 61):
        for N, K in ((9216, 3072), (3072, 14336), (3072, 3072)):
            p = plans.gemm(lib, M, N, K, scratch=1 << 40)
            assert p == plans.gemm(lib, M, N, K, 3 * K, scratch=1 << 40) and p[4] == ws(M, N, K)


@pytest.mark.parametrize("waves", [1, 2, 3, 4, 6, 8])
def test_row_grid(lib, waves):
    """Workgroups for every row, fewer than 2^32 threads along x (what a launch takes) at any row count,
    one line where they fit, and at most a line's end too many."""
    threads = lib.threads(waves)
    assert threads == (256 if waves == 1 else 64 * waves)
    line = (2 ** 32 - 1) // threads
    for blocks in (1, 2, 15708, line - 1, line, line + 1, 22 * 10 ** 6, 33 * 10 ** 6, 3 * line + 7, 2 ** 31 - 1, 2 ** 32 - 1):
        x, y = plans.rows(lib, blocks, threads)
        assert x * threads < 2 ** 32 and y < 2 ** 16
        assert blocks <= x * y < blocks + y
        assert y == 1 or blocks > line


def test_attention_splits_with_the_scratch_of_all_keys(lib, W):
    """A call over the first `keys` of the tensor's keys is given the scratch of all of them (256 CUs
    without a device): it splits as far as that goes wherever a call without a limit would."""
    ws = W._native.lib().wan_flash_attn_workspace
    assert plans.attention(lib, 1, 32, 256, 4100)[2] == 6 and plans.attention(lib, 1, 32, 256, 4096)[2] == 8
    assert plans.attention(lib, 1, 32, 256, 4096, scratch=ws(1, 32, 256, 4100))[2] == 6
    for blocks in (1, 8, 32, 33, 48, 120, 128, 200, 256 + 32, 816):
        for keys in range(1025, 9000, 37):
            whole = plans.attention(lib, 1, 1, 256 * blocks, keys)
            assert whole[3] == ws(1, 1, 256 * blocks, keys)
            for fewer in (keys - 1, keys - 64, keys - 300):
                free = plans.attention(lib, 1, 1, 256 * blocks, fewer)
                p = plans.attention(lib, 1, 1, 256 * blocks, fewer, scratch=whole[3])
                assert p[3] <= whole[3] and p[2] <= free[2]
                assert (p[2] > 1) == (free[2] > 1 and whole[2] > 1), (blocks, keys, fewer)
