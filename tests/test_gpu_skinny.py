"""Batched-decode sizes (9 to 64 rows): the skinny and sliced GEMMs, the QKV
projection of short prompts, and the fused decode attention layer."""

import pytest
import torch

import oracle
from gpu_util import announce, assert_close_layer, bf16_randn
from qmoe import _lib, ops
from qmoe.attention import Attention, KVCache, rope_tables

pytestmark = pytest.mark.gpu

H, HQ, HKV, D = 2048, 32, 4, 128


def _gen(dev, seed):
    return torch.Generator(device=dev).manual_seed(seed)


# every row-tile count and its edges; every K; column remainders of the 4-, 8-,
# 16- and 20-column workgroups (up to 1024, 2048, 4096 and 5120 columns on 256
# CUs) and of their second round (7181; 4133 at K = 4096)
@pytest.mark.parametrize("M", [9, 16, 17, 24, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(5120, 2048), (2048, 4096), (1111, 512), (4133, 1024), (5129, 1024), (64, 2048),
                                 (1023, 512), (1021, 4096), (1301, 2048), (2051, 1024), (4133, 2048), (4609, 512),
                                 (4133, 4096), (7181, 2048), (7181, 1024)])
def test_skinny_gemm(dev, M, N, K):
    announce(f"skinny gemm M={M} N={N} K={K}")
    g = _gen(dev, M * 7 + N)
    A = bf16_randn((M, K), g, dev)
    B = bf16_randn((N, K), g, dev, std=0.05)
    base = torch.randn(M, N, generator=g, device=dev)
    ref = A.double() @ B.double().t()
    # fp32 sums of K products in any order: K * 2^-24 of the sum of magnitudes
    bound = (A.double().abs() @ B.double().abs().t()).mul_(K * 2.0 ** -24)
    ws = ops.gemm_workspace(M, N, K, dev)
    for w in (None, ws) if ws is not None else (None,):
        c = ops.gemm(A, B, _lib.GEMM_STORE_F32, workspace=w)
        again = ops.gemm(A, B, _lib.GEMM_STORE_F32, workspace=w)
        cb = ops.gemm(A, B, _lib.GEMM_STORE_BF16, workspace=w)
        acc = base.clone()
        ops.gemm(A, B, _lib.GEMM_ADD_F32, out=acc, workspace=w)
        torch.cuda.synchronize()
        assert bool(((c.double() - ref).abs() <= bound).all())
        assert torch.equal(c, again)
        assert torch.equal(cb, c.to(torch.bfloat16))
        assert torch.equal(acc, base + c)


# Shapes at which the 64 x 64 tiles are ahead of the skinny kernel (a second
# round of its workgroups, the wide workgroups and the fourth row tile at a
# short K) or of the vocabulary kernel (its first columns, from 25 rows).  The tiles sum K in one chain, so their rows carry the bits of the
# same rows in a product of more rows than the skinny kernel takes.
@pytest.mark.parametrize("M,N,K", [(17, 5632, 2048), (48, 6144, 2048), (64, 10240, 2048), (33, 5120, 1024),
                                   (64, 9216, 1024), (25, 8192, 4096), (17, 10240, 4096), (25, 10244, 1024),
                                   (64, 12160, 1024), (32, 12160, 2048)])
def test_tiles_keep_their_shapes(dev, M, N, K):
    announce(f"tiles M={M} N={N} K={K}")
    g = _gen(dev, M + N)
    A = bf16_randn((65, K), g, dev)
    B = bf16_randn((N, K), g, dev, std=0.05)
    c = ops.gemm(A[:M].contiguous(), B, _lib.GEMM_STORE_F32)
    ref = ops.gemm(A, B, _lib.GEMM_STORE_F32)[:M]
    torch.cuda.synchronize()
    assert torch.equal(c, ref)


# the slices of the split-K plans of 512 columns (two, four and eight of them) on
# 64-column tiles whose last one is partial, at each row-tile count, against
# 64 bits (the comparison is test_skinny_gemm's), and with the norm in the reduction
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(2000, 4096), (1924, 4096), (4004, 2048), (5004, 1024)])
def test_slice_remainders(dev, M, N, K):
    ws = ops.gemm_workspace(M, N, K, dev)
    assert ws is not None and ws.numel() == K // 512 * M * N and -(-N // 64) * (K // 512) <= 256
    test_skinny_gemm(dev, M, N, K)
    g = _gen(dev, M + N + K)
    A = bf16_randn((M, K), g, dev)
    B = bf16_randn((N, K), g, dev, std=0.05)
    w = bf16_randn((N,), g, dev)
    h = torch.randn(M, N, generator=g, device=dev)
    want = ops.gemm(A, B, _lib.GEMM_ADD_F32, out=h.clone(), workspace=ws)
    x = ops.gemm_add_rmsnorm(A, B, h, w, 1e-6, workspace=ws)
    torch.cuda.synchronize()
    assert torch.equal(h, want)
    assert torch.equal(x, ops.rmsnorm_residual(h, w, 1e-6))


# The sum over K keeps the accuracy of four chains up to 16 rows.  Rounding a
# chain of n of the K / 32 steps after each one walks n (n + 1) / 2 / (K / 32)
# steps of (2^-24)^2 / 3 of the final variance, and adding four chains 2.25 more:
# 7.5e-8 of the norm at K = 512 and 8.9e-8 at 1024 (one and two chains: 1.0e-7
# and 1.06e-7 at least).  The bound leaves a quarter on top
@pytest.mark.parametrize("K,walk", [(512, 7.5e-8), (1024, 8.9e-8)])
@pytest.mark.parametrize("M", [9, 16])
def test_skinny_sum_accuracy(dev, M, K, walk):
    announce(f"skinny sum accuracy M={M} K={K}")
    g = _gen(dev, K + M)
    A = bf16_randn((M, K), g, dev)
    B = bf16_randn((4096, K), g, dev, std=0.05)
    c = ops.gemm(A, B, _lib.GEMM_STORE_F32)
    ref = A.double() @ B.double().t()
    torch.cuda.synchronize()
    assert float((c.double() - ref).norm() / ref.norm()) <= 1.25 * walk


# the vocabulary kernel: row-tile edges, a last tile of one column, one to five
# tiles per workgroup (from the third on the ring's slots are filled again) and
# both K
@pytest.mark.parametrize("M", [2, 8, 9, 16, 17, 24, 33, 48, 64])
@pytest.mark.parametrize("N,K", [(10241, 2048), (12289, 1024), (40001, 2048), (12161, 1024), (40001, 1024),
                                 (20002, 1024), (20003, 2048)])
def test_vocab_gemm(dev, M, N, K):
    test_skinny_gemm(dev, M, N, K)


# every slice count of the partial pass (256, 34, 8), slices longer and shorter
# than a thread's eight values, rows of one value; both sides of the slice
# lengths of one, two, four and eight values a thread (256, 512, 1024)
@pytest.mark.parametrize("rows,n", [(1, 1), (3, 255), (4, 151936), (30, 20011), (64, 151936), (130, 4097), (300, 7),
                                    (4, 65536), (4, 65537), (4, 131072), (4, 131073), (4, 262144), (4, 262145),
                                    (3, 600000)])
def test_argmax_slices(dev, rows, n):
    announce(f"argmax rows={rows} n={n}")
    g = _gen(dev, rows + n)
    x = torch.randn(rows, n, generator=g, device=dev)
    x[0] = float("-inf")
    if rows > 1:
        x[1, :] = 1.5  # all equal: the first wins
    if rows > 2:
        x[2, n - 1] = float("inf")
    got = ops.argmax(x)
    torch.cuda.synchronize()
    best = x.cpu().max(dim=1).values.unsqueeze(1)
    first = (x.cpu() == best).float().argmax(dim=1)
    assert torch.equal(got.cpu(), first)


@pytest.mark.parametrize("B,S", [(1, 17), (1, 33), (2, 32), (1, 65), (5, 40), (1, 255)])
def test_short_prompt_qkv(dev, B, S):
    announce(f"short prompt qkv B={B} S={S}")
    g = _gen(dev, S)
    wqkv = bf16_randn(((HQ + 2 * HKV) * D, H), g, dev, std=0.02)
    qn = (1.0 + 0.1 * torch.randn(D, generator=g, device=dev)).to(torch.bfloat16)
    kn = (1.0 + 0.1 * torch.randn(D, generator=g, device=dev)).to(torch.bfloat16)
    x = bf16_randn((B * S, H), g, dev)
    pos = torch.arange(S, device=dev, dtype=torch.int32).repeat(B)
    cos, sin = rope_tables(D, S, 1.0e6, dev)
    kc = torch.zeros(B, HKV, S + 3, D, dtype=torch.bfloat16, device=dev)
    vc = torch.zeros_like(kc)
    q = ops.qkv_norm_rope(x, wqkv, qn, kn, cos, sin, pos, B, S, HQ, HKV, kc, vc, 1e-6)
    torch.cuda.synchronize()
    wq, wk, wv = wqkv.float().cpu().split([HQ * D, HKV * D, HKV * D])
    rq, rk, rv = oracle.qkv_norm_rope(x.cpu().view(B, S, H), wq, wk, wv, qn.cpu(), kn.cpu(),
                                      pos.cpu().view(B, S).long(), HQ, HKV, D, 1e-6, 1.0e6)
    for a, r, what in ((q.view(B, S, HQ, D).transpose(1, 2), rq, "q"), (kc[:, :, :S], rk, "k"), (vc[:, :, :S], rv, "v")):
        err = (a.float().cpu() - r).abs() - r.abs() * 2 ** -8  # one bf16 rounding
        assert float(err.max()) <= 2e-4, what
    assert int(kc[:, :, S:].abs().sum()) == 0


@pytest.mark.parametrize("B", [9, 17, 40, 64, 65])
def test_batched_decode_layer(dev, B):
    """The attention layer's decode step, on both sides of the fused path's
    limit, at ragged positions (one of them 0) against the same rows run as
    batches of 8."""
    announce(f"batched decode layer B={B}")
    g = _gen(dev, B)
    cap = 700
    wqkv = bf16_randn(((HQ + 2 * HKV) * D, H), g, dev, std=0.02)
    wo = bf16_randn((H, HQ * D), g, dev, std=0.02)
    qn = (1.0 + 0.1 * torch.randn(D, generator=g, device=dev)).to(torch.bfloat16)
    kn = (1.0 + 0.1 * torch.randn(D, generator=g, device=dev)).to(torch.bfloat16)
    cos, sin = rope_tables(D, cap, 1.0e6, dev)
    attn = Attention(wqkv, qn, kn, wo, HQ, HKV, D, 1e-6)
    x = bf16_randn((B, H), g, dev)
    pos = torch.randint(0, cap, (B,), generator=g, device=dev, dtype=torch.int32)
    pos[0] = 0
    cache = KVCache(B, HKV, cap, D, dev)
    cache.k.normal_(0.0, 1.0, generator=g)
    cache.v.normal_(0.0, 1.0, generator=g)
    rows = torch.arange(B, device=dev)
    k0, v0 = cache.k.clone(), cache.v.clone()
    res = torch.randn(B, H, generator=g, device=dev)
    out = attn.forward(x, res.clone(), pos, B, 1, cache, cos, sin)
    for b0 in range(0, B, 8):
        b1 = min(B, b0 + 8)
        part = KVCache.wrap((k0[b0:b1].contiguous(), v0[b0:b1].contiguous()))
        ref = attn.forward(x[b0:b1].contiguous(), res[b0:b1].clone(), pos[b0:b1].contiguous(), b1 - b0, 1, part, cos, sin)
        torch.cuda.synchronize()
        # bf16 q/k/v and attention output: one ulp apart where sums differ in order
        assert_close_layer(out[b0:b1], ref, f"rows {b0}..{b1}", max_abs_tol=1e-2, mean_rel_tol=1e-3)
        r = rows[b0:b1] - b0
        for a, e in ((cache.k[b0:b1], part.k), (cache.v[b0:b1], part.v)):
            new, want = a[r, :, pos[b0:b1].long()].float(), e[r, :, pos[b0:b1].long()].float()
            # one bf16 step of the value, and the fp32 sums' order below it
            assert bool(((new - want).abs() <= want.abs() * 2.0 ** -7 + 1e-5).all())
            a[r, :, pos[b0:b1].long()] = e[r, :, pos[b0:b1].long()]
            assert torch.equal(a, e)


def _off_by_four_bytes(t):
    """The same values as ``t`` in storage that is 4-byte but not 16-byte aligned."""
    buf = torch.empty(t.numel() + 2, dtype=t.dtype, device=t.device)[2:].view(t.shape)
    buf.copy_(t)
    assert buf.is_contiguous() and buf.data_ptr() % 16 == 4
    return buf


def _f64_decode(x, w, cos, sin, pos, cache):
    """The decode step in 64 bits: o_proj's output and the new key and value rows."""
    wqkv, wo, qn, kn = (t.double() for t in w)
    B = x.shape[0]
    qkv = (x.double() @ wqkv.t()).view(B, HQ + 2 * HKV, D)
    c, s = (t[pos.long()].double().unsqueeze(1) for t in (cos, sin))

    def finish(t, nw):
        t = t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6) * nw
        lo, hi = t[..., : D // 2], t[..., D // 2 :]
        return torch.cat([lo * c - hi * s, hi * c + lo * s], dim=-1)

    q, k, v = finish(qkv[:, :HQ], qn), finish(qkv[:, HQ : HQ + HKV], kn), qkv[:, HQ + HKV :]
    o = torch.empty(B, HQ, D, dtype=torch.float64, device=x.device)
    for b, n in enumerate(pos.tolist()):
        kk = torch.cat([cache.k[b, :, :n].double(), k[b].unsqueeze(1)], 1)
        vv = torch.cat([cache.v[b, :, :n].double(), v[b].unsqueeze(1)], 1)
        for j in range(HKV):
            heads = slice(j * (HQ // HKV), (j + 1) * (HQ // HKV))
            o[b, heads] = (q[b, heads] @ kk[j].t() * D ** -0.5).softmax(-1) @ vv[j]
    return o.reshape(B, HQ * D) @ wo.t(), k, v


# both sides of the row counts where the projection changes kernel (16, 64) and
# of its row tiles, the same layer with the QKV weights off the DMA alignment
@pytest.mark.parametrize("B,aligned", [(9, True), (16, True), (17, True), (20, False), (33, True), (48, True),
                                       (64, True), (64, False), (65, True)])
def test_batched_decode_layer_against_64_bits(dev, B, aligned):
    announce(f"batched decode layer in 64 bits B={B} aligned={aligned}")
    g = _gen(dev, 100 + B)
    cap = 700
    w = (bf16_randn(((HQ + 2 * HKV) * D, H), g, dev, std=0.02), bf16_randn((H, HQ * D), g, dev, std=0.02),
         (1.0 + 0.1 * torch.randn(D, generator=g, device=dev)).to(torch.bfloat16),
         (1.0 + 0.1 * torch.randn(D, generator=g, device=dev)).to(torch.bfloat16))
    cos, sin = rope_tables(D, cap, 1.0e6, dev)
    x = bf16_randn((B, H), g, dev)
    pos = torch.randint(0, cap, (B,), generator=g, device=dev, dtype=torch.int32)
    pos[0], pos[1], pos[2], pos[3] = 0, 63, 64, cap - 1
    cache = KVCache(B, HKV, cap, D, dev)
    cache.k.normal_(0.0, 1.0, generator=g)
    cache.v.normal_(0.0, 1.0, generator=g)
    y, k, v = _f64_decode(x, w, cos, sin, pos, cache)
    before = cache.k.clone(), cache.v.clone()
    wqkv = w[0] if aligned else _off_by_four_bytes(w[0])
    attn = Attention(wqkv, w[2], w[3], w[1], HQ, HKV, D, 1e-6)
    out = attn.forward(x, torch.zeros(B, H, device=dev), pos, B, 1, cache, cos, sin)
    torch.cuda.synchronize()
    # the layer's update alone (no residual in front of it).  q, k, v, the
    # probabilities and the heads' outputs are each rounded to bf16: 2^-9 / sqrt(3)
    # of a value at rms, sqrt(5) times that (2.5e-3) of a row together; the bound
    # is three times as much.  A lost 64-key block of 700 would be 0.3 of the row
    row = (out.double() - y).norm(dim=1) / y.norm(dim=1)
    assert float(row.max()) <= 2.0 ** -7, f"{float(row.max()):.2e}"
    rows = torch.arange(B, device=dev)
    for a, b, want in ((cache.k, before[0], k), (cache.v, before[1], v)):
        err = (a[rows, :, pos.long()].double() - want).abs() - want.abs() * 2.0 ** -8
        assert float(err.max()) <= 2e-4  # one bf16 rounding, and the fp32 sums below it
        a[rows, :, pos.long()] = b[rows, :, pos.long()]
        assert torch.equal(a, b)  # no other row of the cache is written


def _off_by(t, nbytes):
    """The same values as ``t``, ``nbytes`` past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)[nbytes // 2 :][: t.numel()].view(t.shape)
    buf.copy_(t)
    assert buf.is_contiguous() and buf.data_ptr() % 16 == nbytes
    return buf


# every GEMM of few rows (packed and 16-row GEMV, tiles, split K), each operand
# off the 16-byte boundary by each whole dword
@pytest.mark.parametrize("M", [1, 2, 8, 9, 16, 17, 64])
@pytest.mark.parametrize("N,K", [(512, 2048), (10304, 2048), (2048, 4096), (2050, 1024)])
def test_gemm_off_the_dma_alignment(dev, M, N, K):
    announce(f"gemm off the DMA alignment M={M} N={N} K={K}")
    g = _gen(dev, M + N)
    A = bf16_randn((M, K), g, dev)
    B = bf16_randn((N, K), g, dev, std=0.05)
    ref = A.double() @ B.double().t()
    # fp32 sums of K products in any order: K * 2^-24 of the sum of magnitudes
    bound = (A.double().abs() @ B.double().abs().t()).mul_(K * 2.0 ** -24)
    ws = ops.gemm_workspace(M, N, K, dev)
    for oa, ob in ((4, 0), (0, 4), (8, 8), (12, 4)):
        a, b = (_off_by(t, o) if o else t for t, o in ((A, oa), (B, ob)))
        for w in (None, ws) if ws is not None else (None,):
            c = ops.gemm(a, b, _lib.GEMM_STORE_F32, workspace=w)
            torch.cuda.synchronize()
            assert bool(((c.double() - ref).abs() <= bound).all()), (oa, ob, w is not None)


def test_operands_off_the_dma_alignment(dev):
    """Rows and weights that are not 16-byte aligned take the register-loading
    kernels: same values to the fp32 sums' order."""
    announce("operands off the DMA alignment")
    g = _gen(dev, 5)
    x = bf16_randn((12, H), g, dev)
    for N in (512, 10304):
        w = bf16_randn((N, H), g, dev, std=0.02)
        a = ops.gemm(x, w, _lib.GEMM_STORE_F32)
        b = ops.gemm(_off_by_four_bytes(x), _off_by_four_bytes(w), _lib.GEMM_STORE_F32)
        torch.cuda.synchronize()
        # two fp32 sums of 2048 products in different orders
        bound = (x.double().abs() @ w.double().abs().t()) * (2 * 2048 * 2.0 ** -24)
        assert bool(((a.double() - b.double()).abs() <= bound).all())
    xs = bf16_randn((20, H), g, dev)
    w13 = bf16_randn((4, 128, H), g, dev, std=0.02)
    w2 = bf16_randn((4, 8, H, 8), g, dev, std=0.02)
    ids = torch.randint(0, 4, (20, 1), generator=g, device=dev, dtype=torch.int32)
    route = ops.moe_permute(ids, 4, 128)
    ya = ops.moe_experts_gemv(xs, w13, w2, route)
    yb = ops.moe_experts_gemv(_off_by_four_bytes(xs), w13, w2, route)
    torch.cuda.synchronize()
    assert torch.equal(ya, yb)
    wqkv = bf16_randn(((HQ + 2 * HKV) * D, H), g, dev, std=0.02)
    nw = torch.ones(D, dtype=torch.bfloat16, device=dev)
    pos = torch.arange(20, device=dev, dtype=torch.int32)
    cos, sin = rope_tables(D, 20, 1.0e6, dev)
    got = []
    for f in (lambda t: t, _off_by_four_bytes):
        kc = torch.zeros(1, HKV, 20, D, dtype=torch.bfloat16, device=dev)
        vc = torch.zeros_like(kc)
        q = ops.qkv_norm_rope(f(xs), f(wqkv), nw, nw, cos, sin, pos, 1, 20, HQ, HKV, kc, vc, 1e-6)
        got.append((q, kc, vc))
    torch.cuda.synchronize()
    for a, b in zip(*got):
        # one bf16 step, and the fp32 sums' order below it
        assert bool(((a.float() - b.float()).abs() <= a.float().abs() * 2.0 ** -7 + 1e-5).all())
