"""GPU: the forms of the token-row kernels (waves a row, chunks of 8 channels a lane) at the row
counts and channel counts where the launchers change between them and where a lane's chunks end.

The forms sum a row's squares in different orders, which moves a bf16 value of the normalised
row across a rounding boundary now and then."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
D = 128


def _bf(shape, seed, std=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def _inv64(x, eps):
    return (x.double().flatten(2).square().mean(-1) + eps).rsqrt()


@pytest.mark.parametrize("H", [1, 4, 5, 8, 9, 16, 24, 25, 32, 33, 64])     # 64 W NCH = H*16 and one head past it
@pytest.mark.parametrize("rows", [1, 1024, 1025])
def test_statistics(W, H, rows):
    x = _bf((1, rows, H, D), H * rows, 2.0)
    inv = W.ops.rms_inv(x, 1e-6)
    want = _inv64(x, 1e-6)
    # H*128 squares in fp32, any order: their sum is off by (H*128) 2^-24 relative at most
    assert ((inv.double() - want).abs() <= want * (H * D + 8) * 2 ** -24).all()


@pytest.mark.parametrize("H,rows", [(24, 1024), (24, 1025), (5, 3), (5, 1025), (33, 1025), (24, 10922), (24, 10923)])
@pytest.mark.parametrize("rotate", [False, True])
def test_normalised_rows(W, H, rows, rotate):
    """Strided rows (a view of a wider projection); 1024 rows is where the form changes and
    10923 (128 MB read and written) where the stores become plain ones."""
    x = _bf((1, rows, 2 * H * D), rows, 2.0)[..., H * D:].view(1, rows, H, D)
    g = 1 + _bf((H * D,), 7).abs()
    ang = torch.rand(rows, 64, device=DEV) * 6
    cos, sin = (ang.cos(), ang.sin()) if rotate else (None, None)
    got = W.ops.rms_norm(x, g, 1e-6, cos, sin).double()
    n = (x.double() * _inv64(x, 1e-6)[..., None, None]).to(torch.bfloat16)
    u = (n * g.view(H, D)).double()
    if rotate:
        re, im = u[..., 0::2], u[..., 1::2]
        c, s = cos.double()[None, :, None], sin.double()[None, :, None]
        u = torch.stack((re * c - im * s, re * s + im * c), -1).flatten(-2)
        size = u.unflatten(-1, (64, 2)).norm(dim=-1).repeat_interleave(2, -1)
    else:
        size = u.abs()
    # where the fp32 sum moves the norm across a rounding boundary it changes by one ulp (2^-7 of a
    # value at the foot of its binade), its rounded product with gamma by up to one more; the rotated
    # pair is rounded once more, by 2^-9 of its length and 2^-8 at most
    assert ((got - u).abs() <= size * (2 ** -6 + 2 ** -8)).all()
    assert float(((got - u).abs() > size * (2 ** -8 if rotate else 0)).double().mean()) < 1e-2


@pytest.mark.parametrize("C", [8, 512, 520, 1024, 1032, 2048, 2056, 3072, 3080, 4096, 4104, 8192])
@pytest.mark.parametrize("rows", [1, 6])
def test_adaln_channels(W, C, rows):
    """Gated residual, LayerNorm and modulation where a lane's chunks or a row's waves end."""
    x, y, e = _bf((1, rows, C), C), _bf((1, rows, C), C + 1), _bf((1, 6, C), C + 2, 0.5)
    r, h = W.ops.adaln(x, y, e, 1, gate_idx=2, shift_idx=0, scale_idx=1)
    assert torch.equal(r, x + y * e[:, 2])
    d = r.double()
    n = (d - d.mean(-1, keepdim=True)) * (d.var(-1, unbiased=False, keepdim=True) + 1e-6).rsqrt()
    s1, sh = (1 + e[:, 1]).double(), e[:, 0].double()
    # roundings of the norm (2^-9 and the sums' order), of its product (2^-9) and of the result
    size = (n * s1).abs()
    assert ((h.double() - (n * s1 + sh)).abs() <= size * (2 ** -7 + 2 ** -9) + (size + sh.abs()) * 2 ** -8 + 1e-6).all()


# 2 H partial sums a token; four rows to a block up to 4 heads (8 from 1025 rows of both tasks on),
# where a block of the q side, 256 tokens, is not its waves times 64
@pytest.mark.parametrize("H", [1, 4, 5, 8, 9, 24, 32])
@pytest.mark.parametrize("tokens", [1, 63, 65, 255, 257, 512, 513, 769])
def test_statistics_from_sums(W, H, tokens):
    """wan_rms_norm_qk_sumsq: q's inverse RMS of every token, and k normalised by its own sums."""
    N, s = W._native, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=DEV).manual_seed(H * tokens)
    sums = torch.rand(4 * H, tokens, generator=g, device=DEV) * 128
    k = _bf((1, tokens, H, D), H + tokens)
    gamma = 1 + _bf((H * D,), 7).abs()
    ones, zeros = torch.ones(tokens, 64, device=DEV), torch.zeros(tokens, 64, device=DEV)
    khat = torch.full((tokens + 1, H, D), 7.0, dtype=torch.bfloat16, device=DEV)      # margins that stay as they are
    inv = torch.full((tokens + 64,), 7.0, device=DEV)
    N.check("sums", N.lib().wan_rms_norm_qk_sumsq(N.tensor4(k), khat.data_ptr(), 1, tokens, H, D, gamma.data_ptr(), 1e-6,
                                                  ones.data_ptr(), zeros.data_ptr(), sums.data_ptr(), inv.data_ptr(), s))
    want = (sums.double().unflatten(0, (2, 2 * H)).sum(1) / (H * D) + 1e-6).rsqrt()      # q's, k's
    # 2 H positive fp32 terms in any order, the division, the square root and the reciprocal
    assert ((inv[:tokens].double() - want[0]).abs() <= want[0] * (H + 3) * 2 ** -24).all()
    assert (inv[tokens:] == 7).all() and (khat[tokens:] == 7).all()
    n = (k[0].double() * want[1][:, None, None]).to(torch.bfloat16)
    u = (n * gamma.view(H, D)).double()
    # an ulp of the norm where the sums' order flips it, and its product's (as test_normalised_rows)
    assert ((khat[:tokens].double() - u).abs() <= u.abs() * 2 ** -6).all()
    assert float((khat[:tokens].double() != u).double().mean()) < 1e-2 or u.numel() < 1e4


@pytest.mark.parametrize("H", [1, 7, 8, 24, 32])
def test_statistics_from_sums_keep_small_terms(W, H):
    """One partial sum of 1 before 2 H - 1 of just under half its last place: a chain of additions
    loses every one of them, sums in a tree of 8 levels lose 8 roundings."""
    N, s, tokens = W._native, torch.cuda.current_stream().cuda_stream, 300
    sums = torch.full((4 * H, tokens), 2.0 ** -24 * 0.99, device=DEV)
    sums[0] = sums[2 * H] = 1.0
    k, gamma = _bf((1, tokens, H, D), H), torch.ones(H * D, dtype=torch.bfloat16, device=DEV)
    ones, zeros = torch.ones(tokens, 64, device=DEV), torch.zeros(tokens, 64, device=DEV)
    khat, inv = torch.empty_like(k), torch.empty(tokens, device=DEV)
    N.check("sums", N.lib().wan_rms_norm_qk_sumsq(N.tensor4(k), khat.data_ptr(), 1, tokens, H, D, gamma.data_ptr(), 0.0,
                                                  ones.data_ptr(), zeros.data_ptr(), sums.data_ptr(), inv.data_ptr(), s))
    want = (sums[:2 * H].double().sum(0) / (H * D)).rsqrt()
    # half of 8 roundings of the sum, the division's, the square root's and the reciprocal's
    assert ((inv.double() - want).abs() <= want * (4 + 2.5) * 2 ** -24).all()


def test_more_rows_than_a_line_of_the_grid(W):
    """2^32 / 128 rows of 1152 channels (two waves a row) and one batch entry more, and 2^32 / 64 rows of 8
    (one wave): the launch goes on along y."""
    x = _bf((1, 1024, 9, D), 3)
    inv = W.ops.rms_inv(x.expand(32769, -1, -1, -1), 1e-6)
    assert (inv == W.ops.rms_inv(x.expand(2, -1, -1, -1), 1e-6)[0]).all()      # (2048 rows: the same form)
    del inv
    x = _bf((1, 1024, 8), 4)
    _, h = W.ops.adaln(x.expand(65537, -1, -1).contiguous())
    assert (h == W.ops.adaln(x)[1]).all()
