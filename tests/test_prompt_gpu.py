"""The prompt pass's non-matmul kernels (csrc/prompt.hip) against fp64 on the CPU, at the edges of their tiles (32
positions of a wavefront, 64 of a key tile), every head grouping, both output forms."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# prompt_attn: queries and keys are rounded to bf16 (2^-9 each of scores up to ~8, so 2^-5 of a probability) and so are the
# probabilities (2^-9); errors of both signs average out over the positions but not where one dominates. 2^-5 of the
# largest value covers it; the mean error is far below (2^-8 of the root mean square asserted).
ATTN_TOL = 2.0 ** -5


def reference(qkv, qk_w, rope, nkv, scale, eps):
    """fp64: (out [B, T, nh 64], rotated keys, values [B, T, nkv, 64])."""
    B, T, _ = qkv.shape
    nh = qk_w.shape[1] - nkv
    x = qkv.double().view(B, T, nh + 2 * nkv, 64)
    qk, v = x[:, :, :nh + nkv], x[:, :, nh + nkv:]
    n = qk * torch.rsqrt(qk.pow(2).mean(-1, keepdim=True) + eps) * qk_w[0].double()
    cos, sin = rope[:T, 0].double()[:, None], rope[:T, 1].double()[:, None]
    r = n * cos + torch.cat((-n[..., 32:], n[..., :32]), -1) * sin
    q, k = r[:, :, :nh], r[:, :, nh:]
    kr, vr = k.repeat_interleave(nh // nkv, 2), v.repeat_interleave(nh // nkv, 2)
    s = torch.matmul(q.transpose(1, 2), kr.permute(0, 2, 3, 1)) * scale
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool).triu(1), float("-inf"))
    return torch.matmul(torch.softmax(s, -1), vr.transpose(1, 2)).transpose(1, 2).reshape(B, T, -1), k, v


SHAPES = [(1, 1, 8), (2, 31, 40), (1, 33, 256), (3, 64, 64), (1, 65, 72), (2, 129, 256), (1, 500, 512)]
# with 2 kv heads on 256 CUs: more tiles of positions than a round of the work order holds, so rounds of falling order and
# a shorter last one (per G: tiles of 128, 64, 32 and 32 positions)
ROUNDS = [(1, 64, 300, 304), (2, 64, 300, 304), (4, 32, 430, 432), (8, 16, 300, 304)]


@pytest.mark.parametrize("G,B,T,max_len", [(G, *s) for G in (1, 2, 4, 8) for s in SHAPES] + ROUNDS)
def test_prompt_attn(cuda, G, B, T, max_len):
    from lfm2opt.kernels import ext, int8_ext

    print(f"prompt_attn G={G} B={B} T={T} max_len={max_len}", flush=True)
    nkv, eps, scale = 2, 1e-5, 64 ** -0.5
    nh = G * nkv
    g = torch.Generator().manual_seed(T + G)
    qkv = torch.randn(B, T, (nh + 2 * nkv) * 64, generator=g).to(BF)
    w = 1 + 0.2 * torch.randn(nh + nkv, 64, generator=g)
    qk_w = torch.stack((w, torch.cat((-w[:, 32:], w[:, :32]), -1)))
    ang = torch.rand(max_len, 32, generator=g).repeat(1, 2) * 6
    rope = torch.stack((ang.cos(), ang.sin()), 1)
    want, kn, vn = reference(qkv, qk_w, rope, nkv, scale, eps)
    k = torch.full((B, nkv, 64, max_len), 7.0, dtype=BF, device=cuda)
    v = torch.full((B, nkv, max_len, 64), 7.0, dtype=BF, device=cuda)
    out = torch.full((B * T, nh * 64), float("nan"), dtype=BF, device=cuda)  # a tile left out stays NaN
    args = (qk_w.to(cuda), rope.to(cuda))
    ext().prompt_attn(qkv.to(cuda), *args, k, v, out, scale, eps)
    err = (out.cpu().double().view_as(want) - want).abs()
    assert err.max() <= ATTN_TOL * max(1.0, float(want.abs().max())), f"{err.max():.3e}"
    assert err.pow(2).mean() ** 0.5 <= 2.0 ** -8 * want.pow(2).mean() ** 0.5 + 2.0 ** -12
    kc, vc = k.cpu(), v.cpu()
    assert torch.equal(vc[:, :, :T], vn.transpose(1, 2).to(BF))
    assert ((kc[..., :T].double() - kn.permute(0, 2, 3, 1)).abs() <= 2.0 ** -7 * kn.abs().max()).all()
    assert (kc[..., T:] == 7).all() and (vc[:, :, T:] == 7).all()
    # the quantized form is quant_groups of the bf16 form
    q, s = torch.empty(B * T, nh * 64, dtype=torch.int8, device=cuda), torch.full((nh, B * T), float("nan"), device=cuda)
    ext().prompt_attn(qkv.to(cuda), *args, k, v, (q, s), scale, eps)
    q2, s2 = torch.empty_like(q), torch.empty_like(s)
    int8_ext().quant_rows(out, q2, s2)
    assert torch.equal(q, q2) and torch.equal(s, s2)


@pytest.mark.parametrize("B,T,H,L,bias", [(1, 1, 64, 3, False), (2, 2, 64, 3, True), (1, 3, 576, 8, False),
                                          (3, 5, 128, 1, True), (1, 37, 2048, 3, False), (2, 64, 2112, 4, True)])
def test_prompt_conv_equals_the_bf16_ops(cuda, B, T, H, L, bias):
    """Outputs within a bf16 step of the bf16 tensor ops on the CPU (the fp32 sum of at most 8 rounded products differs
    by 2^-22 in another order, a tie apart), the ring equal; the quantized form is quant_groups of the bf16 form."""
    from lfm2opt.kernels import ext, int8_ext

    g = torch.Generator().manual_seed(T + L)
    bcx, wt = torch.randn(B, T, 3 * H, generator=g).to(BF), torch.randn(L, H, generator=g).to(BF)
    b = torch.randn(H, generator=g).to(BF) if bias else None
    ring = torch.full((L, B, H), 7.0, dtype=BF, device=cuda)
    out = torch.empty(B * T, H, dtype=BF, device=cuda)
    args = (bcx.to(cuda), ring, wt.to(cuda), None if b is None else b.to(cuda))
    ext().prompt_conv(*args, out)
    bb, cc, xx = bcx.chunk(3, -1)
    u = torch.cat((torch.zeros(B, L, H, dtype=BF), bb * xx), 1)
    want_ring = torch.stack([u[:, L + T - 1 - (T - 1 - r) % L] for r in range(L)])
    assert torch.equal(ring.cpu(), want_ring)
    prod = torch.stack([u[:, j + 1:j + 1 + T] * wt[j] for j in range(L)])
    y = prod.float().sum(0).to(BF)
    want = (cc * (y if b is None else y + b)).float()
    got = out.cpu().float().view_as(want)
    assert ((got - want).abs() <= 2.0 ** -7 * (cc.float() * prod.float().abs().sum(0)).abs()).all()
    assert (got != want).float().mean() <= 0.01
    q, s = torch.empty(B * T, H, dtype=torch.int8, device=cuda), torch.empty(H // 64, B * T, device=cuda)
    ext().prompt_conv(*args, (q, s))
    q2, s2 = torch.empty_like(q), torch.empty_like(s)
    int8_ext().quant_rows(out, q2, s2)
    assert torch.equal(q, q2) and torch.equal(s, s2)
