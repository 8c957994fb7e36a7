"""The key split of the attention's last round of workgroups (wan_*_ws, flash_merge_kernel):
the scratch it asks for (CPU), and its results against the unsplit launch of the same call and
a float64 softmax (GPU).

Both launches round the same bf16 probabilities and differ in the reference point of the
exponentials and the order of fp32 sums only, so the split's error against 64 bits may be a
few per cent off the unsplit one's either way, and not more."""
import pytest
import torch

D = 128
SCALE = D ** -0.5
DEV = torch.device("cuda:0")
PART = 8 * (64 * 64 + 128) * 4      # bytes of one part: 256 rows of O, m and l in fp32


def test_scratch_sizes(W):
    """256 CUs (also assumed without a device): 17 blocks per head at 4114 tokens leave 48 of
    816 for a fourth round, five parts each; nothing where the last round is more than half
    full, where there are no whole tiles to save, or where a call has up to 1024 keys."""
    ws = W._native.lib().wan_flash_attn_workspace
    assert ws(2, 24, 4114, 4114) == 48 * 5 * PART
    assert ws(2, 24, 2048, 2048) == 128 * 2 * PART
    assert ws(1, 1, 1, 1025) == 6 * PART
    for args in ((2, 24, 7854, 7854), (2, 24, 1080, 1080), (2, 24, 7854, 1024), (1, 24, 2049, 2049),
                 (2, 16, 2048, 4096), (0, 24, 4114, 4114), (2, 24, 0, 4114)):
        assert ws(*args) == 0, args
    for blocks in range(1, 600):    # never more parts than CUs
        assert ws(1, 1, 256 * blocks, 8192) <= 256 * PART


def test_fused_scratch_is_optional(W):
    """The fused call asks for the split's scratch too, and needs only what it needed before."""
    N = W._native
    lib = N.lib()
    rows = 2 * 4114
    need = -(-rows * 4 // 256) * 256 + rows * 24 * D * 2
    assert lib.wan_self_attn_fused_workspace(2, 24, 4114) == need + 48 * 5 * PART
    t = N.WanTensor(256, 4114 * 24 * D, 24 * D, D)
    rc = lib.wan_self_attn_fused(t, t, t, t, 2, 24, 4114, D, 256, 256, 1e-6, 256, 256, 0.1, 256, need - 1, None)
    assert rc == 3 and str(need) in N.last_error()


def _bf(shape, seed, std=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def _softmax64(q, k, v, lens):
    """float64 attention on the device, a length of 0 giving zeros."""
    out = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    for b, n in enumerate(lens):
        for h in range(q.shape[2] if n else 0):
            s = q[b, :, h].double() @ k[b, :n, h].double().t().contiguous() * SCALE
            out[b, :, h] = torch.softmax(s, -1) @ v[b, :n, h].double()
    return out


def _unsplit(W, q, k, v, lens_dev, actual=0):
    N = W._native
    lib, out = N.lib(), torch.empty_like(q)
    B, Lq, H, _ = q.shape
    args = (N.tensor4(q), N.tensor4(k), N.tensor4(v), N.tensor4(out), B, H, Lq, k.shape[1], D, SCALE)
    s = torch.cuda.current_stream().cuda_stream
    if lens_dev is None:
        N.check("unsplit", lib.wan_flash_self_attn(*args, actual, s))
    else:
        N.check("unsplit", lib.wan_cross_attn(*args, lens_dev.data_ptr(), s))
    return out


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Lq,Lk,actual", [
    (1, 1, 1, 1025, 0),         # the smallest: one row, six parts of two or three tiles
    (2, 3, 257, 1500, 0),       # a second block of one row, a partial last tile
    (1, 5, 300, 4000, 1100),    # fewer keys than the tensor holds: NaN and large keys past them
    (1, 24, 1025, 2000, 0),     # 120 blocks, two parts each
    (2, 24, 1500, 1500, 0),     # a whole round of 256 blocks, then 32 split
])
def test_split_against_unsplit(W, B, H, Lq, Lk, actual):
    assert W._native.lib().wan_flash_attn_workspace(B, H, Lq, Lk) > 0
    q, k, v = _bf((B, Lq, H, D), Lq), _bf((B, Lk, H, D), Lq + 1), _bf((B, Lk, H, D), Lq + 2)
    n = actual or Lk
    k[:, n:] = 1e4
    v[:, n:] = float("nan")
    out = W.ops.flash_self_attn(q, k, v, SCALE, actual)
    whole = _unsplit(W, q, k, v, None, actual)
    want = _softmax64(q, k, v, [n] * B)
    e, e0 = _rel(out, want), _rel(whole, want)
    print(f"B={B} H={H} Lq={Lq} Lk={n}: split {e:.3e}, unsplit {e0:.3e}")
    assert e <= 1.05 * e0 + 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("std", [1.0, 12.0])
def test_split_per_sample_lengths(W, std):
    """Lengths from none to all in one batch: parts without a tile, zeros for the length 0; with
    large logits the parts' reference points lie hundreds apart."""
    B, H, Lq, Lk = 5, 3, 300, 2048
    lens = [1, 130, 2000, 0, 2048]
    q, k, v = _bf((B, Lq, H, D), 1, std), _bf((B, Lk, H, D), 2, std), _bf((B, Lk, H, D), 3)
    want = _softmax64(q, k, v, lens)
    for b, n in enumerate(lens):
        k[b, n:] = 1e4
        v[b, n:] = float("nan")
    sk = torch.tensor(lens, dtype=torch.int32, device=DEV)
    assert W._native.lib().wan_flash_attn_workspace(B, H, Lq, Lk) > 0
    out, whole = W.ops.cross_attn(q, k, v, sk, SCALE), _unsplit(W, q, k, v, sk)
    assert torch.count_nonzero(out[3]) == 0
    for b in (0, 1, 2, 4):
        e, e0 = _rel(out[b], want[b]), _rel(whole[b], want[b])
        print(f"std {std} len {lens[b]}: split {e:.3e}, unsplit {e0:.3e}")
        assert e <= 1.05 * e0 + 1e-5


@pytest.mark.gpu
def test_split_fused_under_capture(W):
    """The fused call at a size that splits (norm and rotation in the kernel), eager, with the
    scratch of an unsplit call, and captured and replayed on new inputs."""
    N, g = W._native, (5, 12, 20)
    B, H, L = 2, 4, 1200
    q, k, v = (_bf((B, L, H, D), i) for i in (1, 2, 3))
    gq, gk = (1 + _bf((H * D,), i).abs() for i in (4, 5))
    cos, sin = (t.to(DEV) for t in W.rope.rope_tables(W.rope.wan_freqs(D), g, D))
    call = lambda: W.ops.self_attn_fused(q, k, v, gq, gk, 1e-6, cos, sin, SCALE)  # noqa: E731
    eager = call()
    lib, out = N.lib(), torch.empty_like(q)
    need = lib.wan_self_attn_fused_workspace(B, H, L) - lib.wan_flash_attn_workspace(B, H, L, L)
    assert need < lib.wan_self_attn_fused_workspace(B, H, L)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    N.check("fused", lib.wan_self_attn_fused(
        N.tensor4(q), N.tensor4(k), N.tensor4(v), N.tensor4(out), B, H, L, D, gq.data_ptr(), gk.data_ptr(), 1e-6,
        cos.data_ptr(), sin.data_ptr(), SCALE, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream))
    # two bf16 results of one value differ by one rounding at most (2^-8 relative) where they differ at all
    assert _rel(eager, out.double()) <= 2 ** -8
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        call()
        with torch.cuda.graph(graph, stream=s):
            captured = call()
    torch.cuda.current_stream().wait_stream(s)
    for i in range(3):
        q.copy_(_bf(q.shape, 50 + i))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, call())


@pytest.mark.gpu
def test_split_of_fewer_keys_than_the_scratch_was_sized_for(W):
    """65 tiles in the tensor (32 blocks: six parts), 64 of them attended to (eight parts, were there room)."""
    N, lib = W._native, W._native.lib()
    H, Lq, Lk, n = 32, 256, 4100, 4096
    q, k, v = _bf((1, Lq, H, D), 1), _bf((1, Lk, H, D), 2), _bf((1, Lk, H, D), 3)
    k[:, n:], v[:, n:] = 1e4, float("nan")
    size = lib.wan_flash_attn_workspace(1, H, Lq, Lk)
    part, out = torch.full((size // 4 + 64,), float("nan"), device=DEV), torch.empty_like(q)
    N.check("split", lib.wan_flash_self_attn_ws(N.tensor4(q), N.tensor4(k), N.tensor4(v), N.tensor4(out), 1, H, Lq, Lk, D,
                                                SCALE, n, part.data_ptr(), size, torch.cuda.current_stream().cuda_stream))
    assert not part[:size // 4].isnan().any() and part[size // 4:].isnan().all()     # it was split, within its scratch
    want = _softmax64(q, k, v, [n])
    e, e0 = _rel(out, want), _rel(_unsplit(W, q, k, v, None, n), want)
    assert e <= 1.05 * e0 + 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("low", [float("-inf"), -3e38])
@pytest.mark.parametrize("first,last", [(64, 1500), (200, 1500), (700, 1300), (0, 700)])
def test_split_with_scores_of_minus_infinity(W, low, first, last):
    """Keys whose scores are -inf weigh nothing, also where a part's first tile, or all of a part, has no
    others; a first tile without others gives NaN, split or not."""
    B, H, Lq, Lk = 2, 3, 257, 1500
    assert W._native.lib().wan_flash_attn_workspace(B, H, Lq, Lk) > 0
    q, k, v = _bf((B, Lq, H, D), 1).abs() + 1, _bf((B, Lk, H, D), 2), _bf((B, Lk, H, D), 3)
    k[:, first:last] = low
    out, whole = W.ops.flash_self_attn(q, k, v, SCALE, 0), _unsplit(W, q, k, v, None)
    if first == 0:
        assert out.isnan().all() and whole.isnan().all()
        return
    keep = torch.cat([torch.arange(first), torch.arange(last, Lk)]).to(DEV)
    want = _softmax64(q, k[:, keep], v[:, keep], [len(keep)] * B)
    e, e0 = _rel(out, want), _rel(whole, want)
    print(f"{low} at {first}..{last}: split {e:.3e}, unsplit {e0:.3e}")
    assert e <= 1.05 * e0 + 1e-5
