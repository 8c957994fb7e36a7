"""Tracing of a whole WanAttentionBlock (torch.compile with fullgraph, plain fake tensors), on fake
device tensors: no kernel runs and no device is needed."""
import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


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
