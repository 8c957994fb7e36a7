"""GPU: both forms of the token-row kernels (a row per wave, a row per block) at the row counts
and channel counts where the launchers change between them and where a lane's chunks end.

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
@pytest.mark.parametrize("rows", [1, 2047, 2048, 2049])
def test_statistics(W, H, rows):
    x = _bf((1, rows, H, D), H * rows, 2.0)
    inv = W.ops.rms_inv(x, 1e-6)
    want = _inv64(x, 1e-6)
    # H*128 squares in fp32, any order: their sum is off by (H*128) 2^-24 relative at most
    assert ((inv.double() - want).abs() <= want * (H * D + 8) * 2 ** -24).all()


@pytest.mark.parametrize("H,rows", [(24, 4095), (24, 4096), (24, 4097), (5, 3), (33, 4097), (24, 10923), (24, 10924)])
@pytest.mark.parametrize("rotate", [False, True])
def test_normalised_rows(W, H, rows, rotate):
    """Strided rows (a view of a wider projection); 4096 rows is where the form changes and
    10923 (128 MB read and written) where the loads become non-temporal."""
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
