"""Host-side routing of the attention layer: which entry points a decode step
of 9 to 64 rows calls, by the alignment of its operands.  The ops are replaced
by recorders, so no GPU is touched."""

import pytest
import torch

from qmoe import ops
from qmoe.attention import FUSED_DECODE_MAX_ROWS, Attention, KVCache

HQ, HKV, D, CAP = 4, 2, 128, 64


def _bf16(*shape, offset=0):
    """bf16 zeros, ``offset`` bytes past a 16-byte boundary."""
    n = 1
    for s in shape:
        n *= s
    t = torch.zeros(n + 8, dtype=torch.bfloat16)
    first = (-t.data_ptr() % 16 + offset) // 2
    t = t[first:first + n].view(shape)
    assert t.data_ptr() % 16 == offset and t.is_contiguous()
    return t


def _route(monkeypatch, B, H, w_offset=0, x_offset=0):
    calls = []

    def record(name, result):
        def fn(*args, **kw):
            calls.append(name)
            return result(*args, **kw) if callable(result) else result
        monkeypatch.setattr(ops, name, fn)

    rows = torch.zeros(B, HQ * D, dtype=torch.bfloat16)
    record("gemm", None)
    record("gemm_workspace", None)
    record("qkv_norm_rope", rows.view(B, HQ, D))
    record("attn_decode", rows)
    record("attn_decode_fused", rows)
    record("attn_decode_workspace", None)
    nw = torch.ones(D, dtype=torch.bfloat16)
    a = Attention(_bf16((HQ + 2 * HKV) * D, H, offset=w_offset), nw, nw, _bf16(H, HQ * D), HQ, HKV, D, 1e-6)
    cache = KVCache(B, HKV, CAP, D, "cpu")
    positions = torch.zeros(B, dtype=torch.int32)
    rope = torch.zeros(CAP, D // 2)
    a.forward(_bf16(B, H, offset=x_offset), torch.zeros(B, H), positions, B, 1, cache, rope, rope)
    return [c for c in calls if "workspace" not in c]


FUSED = ["gemm", "attn_decode_fused", "gemm"]
PLAIN = ["qkv_norm_rope", "attn_decode", "gemm"]


# 9 rows of 4096: the smallest batch whose QKV has no GEMV path
@pytest.mark.parametrize("B,H", [(17, 2048), (20, 512), (64, 1024), (9, 4096), (33, 4096)])
def test_batched_decode_takes_the_raw_projection_when_aligned(monkeypatch, B, H):
    assert _route(monkeypatch, B, H) == FUSED


# The plain projection of more rows than the GEMV's copies both operands by
# 16-byte LDS-DMA for some shapes; qkv_norm_rope loads such operands into
# registers.
@pytest.mark.parametrize("B,H", [(17, 2048), (20, 512), (64, 1024), (9, 4096), (33, 4096)])
@pytest.mark.parametrize("w_offset,x_offset", [(4, 0), (8, 0), (0, 4), (0, 8), (12, 12), (2, 0)])
def test_batched_decode_off_the_dma_alignment_keeps_the_qkv_kernel(monkeypatch, B, H, w_offset, x_offset):
    assert _route(monkeypatch, B, H, w_offset, x_offset) == PLAIN


def test_decode_outside_the_fused_range(monkeypatch):
    assert _route(monkeypatch, FUSED_DECODE_MAX_ROWS + 1, 2048) == PLAIN
    assert _route(monkeypatch, 20, 1536) == PLAIN  # a hidden size that no skinny kernel takes
    # the GEMV's batches stay on it, aligned or not
    assert _route(monkeypatch, 16, 2048) == FUSED
    assert _route(monkeypatch, 16, 2048, 4, 4) == FUSED
