"""Tracing of a whole WanAttentionBlock (torch.compile with fullgraph, plain fake tensors), on fake
device tensors: no kernel runs and no device is needed."""
import collections
import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode


def _block(W, tokens, frames, dtype=torch.bfloat16):
    """A full-width block with the "hip" backends and its inputs, in the active fake mode."""
    cfg = W.model.WanConfig()
    default = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        with torch.device("cuda"):
            blk = W.model.WanAttentionBlock(cfg.dim, cfg.ffn_dim, cfg.num_heads)
    finally:
        torch.set_default_dtype(default)
    L, C = tokens // 2, cfg.dim
    args = [torch.empty(s, dtype=d, device="cuda") for s, d in (
        ((2, L, C), dtype), ((1, frames, 6, C), dtype), ((L, 64), torch.float32), ((L, 64), torch.float32),
        ((2, 512, cfg.num_heads, 128), dtype), ((2, 512, cfg.num_heads, 128), dtype))]
    return W.fast_dit._FastBlock(blk, frames, "hip", "hip", "hip"), args


# tokens of both samples: all projections by hipBLASLt (15708), some (720) or nearly all (2160) by the
# library's own GEMM when they are run
@pytest.mark.parametrize("tokens,frames", [(720, 3), (2160, 6), (15708, 21)])
@pytest.mark.parametrize("dynamic", [False, True])
def test_block_is_one_graph(W, tokens, frames, dynamic):
    graphs = []

    def backend(gm, inputs):
        graphs.append(gm)
        return gm

    torch._dynamo.reset()
    with FakeTensorMode(), torch.no_grad():
        fb, args = _block(W, tokens, frames)
        traced = torch.compile(lambda *a: fb(*a), backend=backend, fullgraph=True)
        for n in (tokens, tokens + 2 * frames) if dynamic else (tokens,):
            a = [t.new_empty((t.shape[0], n // 2, *t.shape[2:])) if i == 0 else t.new_empty((n // 2, 64)) if i in (2, 3) else t
                 for i, t in enumerate(args)]
            if dynamic:
                torch._dynamo.mark_dynamic(a[0], 1)
                torch._dynamo.mark_dynamic(a[2], 0)
                torch._dynamo.mark_dynamic(a[3], 0)
            out = traced(*a)
            assert out.shape == a[0].shape and out.dtype == torch.bfloat16
    assert len(graphs) == 1            # the token count of a dynamic graph may change
    torch._dynamo.reset()


@pytest.mark.parametrize("tokens,frames", [(720, 3), (2160, 6)])
def test_block_on_fake_tensors(W, tokens, frames):
    """Without a tracer too: no look at a data pointer, which fake tensors do not have."""
    with FakeTensorMode(), torch.no_grad(), warnings.catch_warnings():
        warnings.simplefilter("error")
        fb, args = _block(W, tokens, frames)
        assert fb(*args).shape == args[0].shape


class _Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.count = collections.Counter()

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.count[str(func)] += 1
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("impl,pointwise", [("sdpa", "eager"), ("hip", "hip")])
def test_torch_side_runs_torch_alone(W, impl, pointwise, monkeypatch):
    """With attention "sdpa" and pointwise "eager" nothing of this library runs on the device, in the
    blocks or around them (2160 tokens, where the other side takes its own kernels throughout)."""
    cfg, grid = W.model.WanConfig(), (6, 12, 15)
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda t: t)      # fake tensors have no pinned form
    monkeypatch.setattr(W.fast_dit, "_sdpa", lambda q, *rest: torch.empty_like(q))      # asks for a device
    torch.set_default_dtype(torch.bfloat16)
    try:
        with FakeTensorMode(), torch.no_grad():
            with torch.device("cuda"):
                m = W.model.WanModel(cfg, num_layers=1)
            fast = W.fast_dit.FastWanDiT.__new__(W.fast_dit.FastWanDiT)
            fast.model, fast.grid, fast.num_frames, fast.device = m, grid, grid[0], torch.device("cuda")
            fb = W.fast_dit._FastBlock(m.blocks[0], grid[0], impl, impl, pointwise)
            _, args = _block(W, 2160, grid[0])
            with _Names() as seen:
                fast.time_rows(500)
                before = {n for n in seen.count if n.startswith("wan_hip.")}
                fb(*args)
    finally:
        torch.set_default_dtype(torch.float32)
    assert not before
    own = {n for n in seen.count if n.startswith("wan_hip.")}
    assert bool(own) == (impl == "hip"), own


# the ends of the ranges in which a projection is this library's: (tokens of both samples, q/k/v, the
# 3072-wide ones, FFN-down); odd counts do not occur with guidance
@pytest.mark.parametrize("tokens,qkv,wide,down", [
    (2, 0, 0, 0), (64, 0, 0, 0), (66, 0, 0, 1), (1080, 0, 0, 1), (1792, 0, 0, 1), (1794, 0, 0, 0), (1822, 0, 0, 0),
    (1824, 1, 0, 0), (2110, 1, 0, 0), (2160, 1, 0, 1), (2240, 1, 0, 1), (2242, 0, 0, 1), (2306, 0, 0, 0),
    (5470, 0, 0, 0), (5504, 1, 1, 1), (5888, 1, 1, 1), (6656, 0, 1, 0), (6658, 0, 0, 0), (8704, 1, 0, 1),
    (12288, 1, 0, 0), (14336, 0, 0, 1), (14338, 0, 0, 0), (15708, 0, 0, 0)])
def test_projection_routes(W, tokens, qkv, wide, down):
    with FakeTensorMode(), torch.no_grad():
        fb, args = _block(W, tokens, 1)
        with _Names() as seen:
            fb(*args)
        assert seen.count["wan_hip.qkv_proj_sumsq.default"] == qkv
        assert seen.count["wan_hip.self_attn_fused_sumsq.default"] == qkv
        assert seen.count["wan_hip.linear.default"] == 3 * wide + down
        for impl, calls in (("hipblaslt", 0), ("hip", 1)):      # chosen by name: at every size
            fb.qkv_impl = impl
            with _Names() as seen:
                fb._self_attention(args[0], args[2], args[3])
            assert seen.count["wan_hip.qkv_proj_sumsq.default"] == calls
