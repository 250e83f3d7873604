"""Row movement at the edges of its kernels: the permuted rows are x's rows
bit for bit, whichever direction of the layout moves them."""
from __future__ import annotations

import dataclasses

import pytest
import torch

import expert_mlp as mlp
import mgg_native as nat

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


@pytest.mark.parametrize("tokens,top_k,hidden", [(50, 3, 2056), (130, 8, 64), (7, 64, 16), (9, 65, 16)])
def test_permute_rows_follows_token_index(cuda_device, tokens, top_k, hidden):
    """A layout whose arrays were changed one without the other: the rows are
    those of token_index up to offsets[E], whatever slot_position holds, and
    rows past offsets[E] stay as they were."""
    gen = torch.Generator().manual_seed(top_k)
    lay = mlp.dispatch_layout(_routing(tokens, 2 * top_k, top_k, 0.2, cuda_device), 2 * top_k)
    n, total = int(lay.offsets[-1]), lay.max_rows
    x = torch.randn(tokens + 5, hidden, device=cuda_device).to(torch.float16)
    slots = lay.slot_position
    fewer = lay.offsets.clone()
    fewer[-1] = n // 2
    moved = lay.token_index.clone()  # other tokens' rows, among them rows past the layout's tokens
    moved[:n] = torch.randint(0, tokens + 5, (n,), generator=gen).to(moved)
    some = torch.where(torch.rand(total, generator=gen).to(cuda_device) < 0.3, -1, slots).to(torch.int32)
    junk = torch.randint(-3, total + 3, (total,), generator=gen, dtype=torch.int32).to(cuda_device)
    for what, changed in (("fewer rows", dict(offsets=fewer)), ("tokens moved", dict(token_index=moved)),
                          ("slots dropped", dict(slot_position=some)), ("slots junk", dict(slot_position=junk)),
                          ("both", dict(token_index=moved, slot_position=junk))):
        changed = dataclasses.replace(lay, **changed)
        rows = int(changed.offsets[-1])
        want = x[changed.token_index[:rows].long()]
        out = torch.full((total, hidden), 7.0, device=cuda_device, dtype=x.dtype)
        nat.check(nat.lib().mgg_permute_rows(
            nat.MGG_DTYPE_FP16, x.data_ptr(), hidden, changed.slot_position.data_ptr(),
            changed.token_index.data_ptr(), changed.offsets[-1:].data_ptr(), tokens, top_k, hidden,
            out.data_ptr(), hidden, torch.cuda.current_stream().cuda_stream))
        assert torch.equal(mlp.permute_tokens(x, changed)[:rows], want), what
        assert torch.equal(out[:rows], want) and bool((out[rows:] == 7.0).all()), what


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
