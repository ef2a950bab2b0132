"""Expert MLPs at the row counts where their kernels change path."""

import pytest
import torch

from gpu_util import announce, bf16_randn
from qmoe import ops

pytestmark = pytest.mark.gpu


def _route(dev, counts, E, tile_m):
    """k = 1 dispatch giving expert e ``counts[e]`` tokens, in shuffled order."""
    ids = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(counts)])
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(len(ids)))]
    return ids, ops.moe_permute(ids.view(-1, 1).to(dev), E, tile_m)


def _check(dev, counts, H, I, tile_m, fn, rel):
    E = len(counts)
    g = torch.Generator(device=dev).manual_seed(H + I + sum(counts))
    w13 = bf16_randn((E, 2 * I, H), g, dev, std=0.02)
    w2 = bf16_randn((E, I // 8, H, 8), g, dev, std=0.02)
    ids, route = _route(dev, counts, E, tile_m)
    x = bf16_randn((len(ids), H), g, dev)
    y = fn(x, w13, w2, route)
    again = fn(x, w13, w2, route)
    torch.cuda.synchronize()
    assert torch.equal(y, again)
    for e, c in enumerate(counts):
        if c == 0:
            continue
        s = int(route.offsets[e])
        xe = x[route.slot_token[s : s + c].long()].double()
        gu = w13[e].double().view(I // 32, 2, 32, H)
        act = torch.nn.functional.silu(xe @ gu[:, 0].reshape(I, H).t()) * (xe @ gu[:, 1].reshape(I, H).t())
        ref = act @ w2[e].double().permute(0, 2, 1).reshape(I, H)
        row = (y[s : s + c].double() - ref).norm(dim=1) / ref.norm(dim=1)
        assert float(row.max()) <= rel, f"expert {e} ({c} rows): {float(row.max()):.2e}"


# both sides of the 64- and 128-row pipelines and of the 256-row tile, with
# remainder tiles of each size behind a full one, and experts without rows
@pytest.mark.parametrize("H,I", [(2048, 768), (512, 192), (1024, 96)])
@pytest.mark.parametrize("tile_m", [256, 224])
def test_grouped_tile_sizes(dev, H, I, tile_m):
    announce(f"grouped tile sizes H={H} I={I} tile_m={tile_m}")
    counts = [1, 0, 32, 33, 64, 65, 0, 96, 97, 127, 128, 129, 255, 256, 257, 320, 321, 384, 390, 513, 2, 0]
    # act and y are bf16: two roundings of 2^-9 relative each, far above the fp32 sums
    _check(dev, counts, H, I, tile_m, ops.moe_experts_grouped, 2.0 ** -7)


# every remainder of the 4-token chunks, one to sixteen chunks, every H
@pytest.mark.parametrize("H", [512, 1024, 2048, 4096])
@pytest.mark.parametrize("counts", [[1, 0, 2, 3, 4, 5, 6, 7, 8], [9, 0, 17, 29], [0, 64]])
def test_gemv_token_chunks(dev, H, counts):
    announce(f"gemv token chunks H={H} counts={counts}")
    # fp32 activations as bf16 hi + lo parts (2^-16) and fp32 sums over H and I terms
    _check(dev, counts, H, 96, 128, ops.moe_experts_gemv, 1e-4)
