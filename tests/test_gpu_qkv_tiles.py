"""GPU: wan_qkv_proj_sumsq at the edges of its tile heights (128, 192, 256 and 320 rows of x),
against float64.  With N = 9216 (36 column tiles) and 256 CUs the launcher takes 128 rows up to
M 896, 192 up to 1344, 256 up to 1792 and 320 up to 2240."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("M,K", [
    (1, 64), (127, 128), (128, 192), (129, 256), (896, 64),      # 128 rows: 1 to 4 tiles of k in 3 slots
    (897, 64), (1152, 128), (1153, 192),                         # 192
    (1345, 64), (1536, 128), (1537, 320),                        # 256
    (1793, 64), (1920, 128), (1921, 192), (2240, 3072),          # 320
])
def test_tile_heights(W, M, K):
    N_, C = 9216, 6144
    lib, ab = W._native.lib(), W._native
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x, w = (torch.randn(n, K, generator=g, device=DEV).bfloat16() for n in (M, N_))
    b = torch.randn(N_, generator=g, device=DEV).bfloat16()
    out = torch.full((M + 8, N_ + 8), 7.0, dtype=torch.bfloat16, device=DEV)     # a margin that stays as it is
    sums = torch.full((C // 64 * M + 64,), 7.0, device=DEV)
    ab.check("gemm", lib.wan_qkv_proj_sumsq(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), sums.data_ptr(),
                                            M, N_, K, K, K, N_ + 8, C, torch.cuda.current_stream().cuda_stream))
    assert (out[M:] == 7).all() and (out[:, N_:] == 7).all() and (sums[C // 64 * M:] == 7).all()
    got = out[:M, :N_].double()
    want = x.double() @ w.double().t() + b.double()
    # one bf16 rounding (2^-9 relative) of an fp32 sum (K 2^-24 of the sum of magnitudes at most)
    room = want.abs() * 2 ** -8 + (x.double().abs() @ w.double().abs().t() + b.double().abs()) * (K + 1) * 2 ** -24
    assert ((got - want).abs() <= room).all()
    squares = got[:, :C].reshape(M, C // 64, 64).square().sum(-1).t()
    # 64 positive fp32 terms
    assert ((sums[:C // 64 * M].view(C // 64, M) - squares).abs() <= squares * 65 * 2 ** -24).all()
