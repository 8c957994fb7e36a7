"""GPU: wan_qkv_proj_sumsq at the edges of its tile heights (128, 192, 256 and 320 rows of x),
against float64.  With N = 9216 (36 column tiles), K = 1024 and 256 CUs the launcher takes 128 rows
from M 193, 192 from 897, 256 from 1345 and 320 from 1793; shorter products choose differently."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("M,K", [
    (769, 192), (896, 192), (577, 256), (193, 1024), (896, 1024),       # 128 rows: 3, 4 and 16 tiles of k in 3 slots
    (1, 64), (192, 128), (897, 1024), (1153, 1024), (1344, 1024),       # 192
    (193, 64), (1345, 1024), (1537, 1024), (1792, 1024),                # 256
    (577, 64), (1537, 128), (1793, 1024), (1921, 1024), (2240, 3072),   # 320
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
