"""Row movement at the edges of its kernels: the permuted rows are x's rows
bit for bit, whichever direction of the layout moves them."""
from __future__ import annotations

import dataclasses

import pytest
import torch

import expert_mlp as mlp

pytestmark = pytest.mark.gpu


def _routing(tokens, experts, top_k, masked, dev, seed=0, dtype=torch.int64):
    gen = torch.Generator().manual_seed(seed)
    idx = torch.topk(torch.randn(tokens, experts, generator=gen), top_k, dim=1)[1]
    idx[torch.rand(idx.shape, generator=gen) < masked] = -1
    return idx.to(dtype).to(dev)


@pytest.mark.parametrize("tokens,experts,top_k,hidden,pad,masked", [
    (1, 4, 2, 8, 0, 0.0),          # one token, one chunk
    (37, 5, 3, 2048, 8, 0.3),      # one whole block of chunks, strided x, masked slots
    (129, 16, 4, 2056, 0, 0.1),    # one chunk past a block
    (64, 8, 2, 1028, 4, 0.2),      # rows of x not 16-byte multiples: the gather
    (100, 8, 1, 512, 0, 0.2),      # one slot a token: the gather
    (50, 8, 6, 64, 0, 1.0),        # every slot masked
    (4096, 64, 8, 2056, 0, 0.01),  # past the last-level cache: non-temporal stores
])
def test_permute_rows(cuda_device, tokens, experts, top_k, hidden, pad, masked):
    lay = mlp.dispatch_layout(_routing(tokens, experts, top_k, masked, cuda_device), experts)
    x = torch.randn(tokens + 3, hidden + pad, device=cuda_device).to(torch.bfloat16)[:, :hidden]
    n = int(lay.offsets[-1])
    want = x[lay.token_index[:n].long()]
    assert torch.equal(mlp.permute_tokens(x, lay)[:n], want)
    # A layout that holds one direction only goes by token_index.
    one_way = dataclasses.replace(lay, slot_position=None)
    assert torch.equal(mlp.permute_tokens(x, one_way)[:n], want)


@pytest.mark.parametrize("tokens,top_k,experts", [
    (1, 1, 1), (512, 2, 16), (128, 8, 1024),  # one chunk: counted in place
    (513, 2, 3), (1025, 1, 64),               # two chunks: the table's sums in eight parts
    (2048, 8, 257), (900, 8, 512), (900, 8, 513), (2048, 8, 1024),  # three, two and one part
    (20000, 4, 300),                          # past the table: bases from the scan pass
])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_dispatch_layout_paths(cuda_device, tokens, top_k, experts, dtype):
    gen = torch.Generator().manual_seed(tokens)
    idx = torch.randint(-1, experts + 1, (tokens, top_k), generator=gen)  # both ends masked
    lay = mlp.dispatch_layout(idx.to(dtype).to(cuda_device), experts)
    flat = idx.flatten()
    valid = (flat >= 0) & (flat < experts)
    order = torch.argsort(torch.where(valid, flat, experts), stable=True)[: int(valid.sum())]
    pos = torch.full_like(flat, -1)
    pos[order] = torch.arange(order.numel())
    counts = torch.bincount(flat[valid], minlength=experts)
    n = order.numel()
    assert torch.equal(lay.counts.cpu().long(), counts)
    assert torch.equal(lay.offsets.cpu().long(), torch.cat([counts.new_zeros(1), counts.cumsum(0)]))
    assert torch.equal(lay.slot_position.cpu().long(), pos)
    assert torch.equal(lay.row_assignment[:n].cpu().long(), order)
    assert torch.equal(lay.token_index[:n].cpu().long(), order // top_k)
