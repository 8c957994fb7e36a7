"""The projection GEMM's split over k (wan_qkv_proj_sumsq_ws, gemm_merge_kernel): the scratch it
asks for (CPU), and its results where parts, tiles and rows end, against float64 (GPU)."""
import pytest
import torch

DEV = torch.device("cuda:0")

# (M, N, K), all with scratch: one tile in parts of four k-tiles; parts of unequal length and a
# second block of one row; the longest product; every tile height; whole rounds before the split tiles
SIZES = [(1, 256, 1024), (129, 256, 2112), (80, 3072, 14336), (321, 512, 4096), (1640, 3072, 14336),
         (1000, 3072, 14336), (2113, 3072, 14336), (2280, 9216, 3072), (2500, 9216, 3072)]


def test_scratch_sizes(W):
    """256 CUs (also assumed without a device): never more parts than CUs, of 320 rows at most;
    none where the tiles fill more than half of the CUs, or the product is short."""
    ws = W._native.lib().wan_qkv_proj_workspace
    for size in SIZES:
        assert ws(*size) > 0, size
    assert ws(2160, 3072, 14336) == 84 * 3 * 320 * 256 * 4
    assert ws(80, 9216, 3072) % (36 * 128 * 256 * 4) == 0
    for size in ((2160, 9216, 3072), (1, 256, 512), (0, 256, 1024), (80, 255, 512), (80, 256, 500), (-1, 256, 512),
                 (80, 0, 512), (80, 256, 0)):
        assert ws(*size) == 0, size
    for m in range(1, 16000, 37):
        for n, k in ((3072, 3072), (9216, 3072), (3072, 14336)):
            assert ws(m, n, k) <= 256 * 320 * 256 * 4


def test_misaligned_scratch_is_refused(W):
    N = W._native
    rc = N.lib().wan_qkv_proj_sumsq_ws(256, 256, 256, 256, 256, 80, 256, 512, 512, 512, 256, 0, 128, 1 << 20, None)
    assert rc == 1 and "workspace" in N.last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N_,K", SIZES)
@pytest.mark.parametrize("scratch", ["all", "half"])
def test_split(W, M, N_, K, scratch):
    lib, ab = W._native.lib(), W._native
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x, w = (torch.randn(n, K, generator=g, device=DEV).bfloat16() for n in (M, N_))
    b = torch.randn(N_, generator=g, device=DEV).bfloat16()
    C = N_ // 2                                       # columns with sums of squares
    out = torch.full((M + 8, N_ + 8), 7.0, dtype=torch.bfloat16, device=DEV)     # a margin that stays as it is
    sums = torch.full((C // 64 * M + 64,), 7.0, device=DEV)
    n = lib.wan_qkv_proj_workspace(M, N_, K) // (1 if scratch == "all" else 2)
    part = torch.full((n // 4 + 64,), float("nan"), device=DEV)
    ab.check("gemm", lib.wan_qkv_proj_sumsq_ws(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), sums.data_ptr(),
                                               M, N_, K, K, K, N_ + 8, C, part.data_ptr(), n,
                                               torch.cuda.current_stream().cuda_stream))
    if scratch == "all":
        assert not part[:n // 4].isnan().any()
    assert part[n // 4:].isnan().all()
    assert (out[M:] == 7).all() and (out[:, N_:] == 7).all() and (sums[C // 64 * M:] == 7).all()
    got = out[:M, :N_].double()
    want = x.double() @ w.double().t() + b.double()
    # one bf16 rounding (2^-9 relative) of an fp32 sum (K 2^-24 of the sum of magnitudes at most)
    room = want.abs() * 2 ** -8 + (x.double().abs() @ w.double().abs().t() + b.double().abs()) * (K + 1) * 2 ** -24
    assert ((got - want).abs() <= room).all()
    squares = got[:, :C].reshape(M, C // 64, 64).square().sum(-1).t()
    # 64 positive fp32 terms
    assert ((sums[:C // 64 * M].view(C // 64, M) - squares).abs() <= squares * 65 * 2 ** -24).all()


@pytest.mark.gpu
@pytest.mark.parametrize("k,n,tokens", [(14336, 3072, 80), (14336, 3072, 2160), (14336, 3072, 2600), (14336, 3072, 2848),
                                        (3072, 3072, 5504), (3072, 3072, 5502),
                                        (3072, 18432, 12), (3072, 18432, 42)])
def test_projection_route(W, k, n, tokens):
    """A projection by either GEMM: bf16 roundings of the same sums."""
    lin = torch.nn.Linear(k, n, device=DEV, dtype=torch.bfloat16).requires_grad_(False)
    x = torch.randn(2, tokens // 2, k, device=DEV, generator=torch.Generator(device=DEV).manual_seed(tokens)).bfloat16()
    got, want = W.fast_dit._linear_own(x, lin).double(), x.double() @ lin.weight.double().t() + lin.bias.double()
    room = want.abs() * 2 ** -8 + (x.double().abs() @ lin.weight.double().abs().t() + 1) * (k + 1) * 2 ** -24
    assert got.shape == want.shape and ((got - want).abs() <= room).all()


def test_projection_route_without_library_conditions(W):
    """Rows outside the ranges, other widths, a missing bias or another type stay torch's."""
    for lin, rows in ((torch.nn.Linear(3072, 3072, dtype=torch.bfloat16), 4), (torch.nn.Linear(64, 32), 8),
                      (torch.nn.Linear(14336, 3072, bias=False), 2), (torch.nn.Linear(14336, 3072), 2)):
        x = torch.randn(1, rows, lin.in_features, dtype=lin.weight.dtype)
        assert torch.equal(W.fast_dit._linear_own(x, lin), torch.nn.functional.linear(x, lin.weight, lin.bias))
