"""The decode step's non-matmul kernels (csrc/step.hip) against fp64 on the CPU, at the sizes where they can go wrong:
the edges of a chunk of 256 positions, of a 16-byte run of positions and of the splits, every head grouping."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# attn_step: the output is one bf16 rounding (2^-9 of the value) of fp32 sums over at most 16,384 positions (2^-10 in the
# worst order) of values up to max |v|; q stays fp32, so its own error is the exp2 of an fp32 score (|score| < 2^6: 2^-18).
# 2^-8 of the largest value covers all of it.
ATTN_TOL = 2.0 ** -8


def attention_reference(qkv, qk_w, rope, pos, k, v, scale, eps):
    """fp64: (out, the new key, the new value); k [B, nkv, 64, max_len], v [B, nkv, max_len, 64]."""
    B, nkv, hd, _ = k.shape
    nh = qk_w.shape[1] - nkv
    x = qkv.double().view(B, nh + 2 * nkv, hd)
    qk = x[:, :nh + nkv]
    n = qk * torch.rsqrt(qk.pow(2).mean(-1, keepdim=True) + eps) * qk_w[0].double()
    cos, sin = rope[pos].double()
    rot = torch.cat((-n[..., hd // 2:], n[..., :hd // 2]), -1)
    r = n * cos + rot * sin
    q, kn, vn = r[:, :nh], r[:, nh:].to(torch.bfloat16), x[:, nh + nkv:]
    ks = torch.cat((k[..., :pos].double(), kn.double()[..., None]), -1)
    vs = torch.cat((v[:, :, :pos].double(), vn[:, :, None]), 2)
    p = torch.softmax(torch.matmul(q.view(B, nkv, nh // nkv, hd), ks) * scale, -1)
    return torch.matmul(p, vs).reshape(B, nh * hd), kn, vn.to(torch.bfloat16)


@pytest.mark.parametrize("G", [1, 2, 4, 8])
@pytest.mark.parametrize("B,max_len,positions", [(1, 8, (0, 3, 7)), (2, 256, (0, 31, 255)), (1, 264, (256, 263)),
                                                 (3, 512, (255, 256, 511)), (1, 1032, (767, 768, 1031)),
                                                 (1, 4096, (2047, 4095)), (40, 1280, (0, 300, 1279)),
                                                 # eight heads a workgroup (G = 8); splits of two and four chunks, at and
                                                 # beside their edges; more than 16 and up to 64 splits to combine
                                                 (65, 512, (255, 256, 511)), (16, 4096, (511, 512, 1023, 1024, 1500, 4095)),
                                                 (1, 8192, (4095, 4096, 8191)), (1, 16384, (12288, 16383))])
def test_attn_step(cuda, G, B, max_len, positions):
    from lfm2opt.kernels import ext

    E, nkv, hd, eps, scale = ext(), 2, 64, 1e-5, 64 ** -0.5
    nh = G * nkv
    for pos in positions:
        print(f"attn_step G={G} B={B} max_len={max_len} pos={pos}", flush=True)
        g = torch.Generator().manual_seed(pos + G)
        qkv = torch.randn(B, (nh + 2 * nkv) * hd, generator=g).to(torch.bfloat16)
        w = 1 + 0.2 * torch.randn(nh + nkv, hd, generator=g)
        qk_w = torch.stack((w, torch.cat((-w[:, hd // 2:], w[:, :hd // 2]), -1)))
        ang = torch.rand(max_len, hd // 2, generator=g).repeat(1, 2) * 6
        rope = torch.stack((ang.cos(), ang.sin()), 1)
        k = (torch.randn(B, nkv, hd, max_len, generator=g) * 2).to(torch.bfloat16)
        v = torch.randn(B, nkv, max_len, hd, generator=g).to(torch.bfloat16)
        k[..., pos:] = float("nan")  # unwritten slots are never read
        v[:, :, pos:] = float("nan")
        want, kn, vn = attention_reference(qkv, qk_w, rope, pos, k, v, scale, eps)
        kd, vd = k.to(cuda), v.to(cuda)
        out = torch.empty(B, nh * hd, device=cuda, dtype=torch.bfloat16)
        ctr = torch.tensor([pos, 0], device=cuda)
        E.attn_step(qkv.to(cuda), qk_w.to(cuda), rope.to(cuda), ctr, kd, vd, out, scale, eps,
                    E.attn_step_workspace(B, nh, nkv, max_len, cuda))
        err = (out.cpu().double() - want).abs().max()
        assert err <= ATTN_TOL * max(1.0, float(want.abs().max())), f"pos {pos}: {err:.3e}"
        kc, vc = kd.cpu(), vd.cpu()
        assert torch.equal(vc[:, :, pos], vn)
        assert (kc[..., pos].double() - kn.double()).abs().max() <= 2.0 ** -8 * float(kn.double().abs().max())
        assert torch.equal(kc[..., :pos], k[..., :pos]) and torch.equal(vc[:, :, :pos], v[:, :, :pos])
        assert kc[..., pos + 1:].isnan().all() and vc[:, :, pos + 1:].isnan().all()


@pytest.mark.parametrize("pos,max_len", [(-1, 64), (64, 64), (4096, 4096)])
def test_attn_step_outside_the_cache(cuda, pos, max_len):
    """A position outside the cache gives NaN and leaves the cache alone (one chunk, and several splits)."""
    from lfm2opt.kernels import ext

    E, z = ext(), lambda *s, dt=torch.bfloat16: torch.zeros(*s, dtype=dt, device=cuda)  # noqa: E731
    k, v, out = z(2, 2, 64, max_len), z(2, 2, max_len, 64), z(2, 4 * 64)
    E.attn_step(z(2, 8 * 64) + 1, z(2, 6, 64, dt=torch.float32), z(max_len, 2, 64, dt=torch.float32),
                torch.tensor([pos, 0], device=cuda), k, v, out, 0.1, 1e-5, E.attn_step_workspace(2, 4, 2, max_len, cuda))
    assert out.isnan().all() and not k.any() and not v.any()


def test_attn_step_refuses_other_shapes(cuda):
    from lfm2opt.kernels import ext

    E, bf = ext(), torch.bfloat16

    def call(nh, nkv, hd, max_len):
        z = lambda *s, dt=bf: torch.zeros(*s, dtype=dt, device=cuda)  # noqa: E731
        E.attn_step(z(1, (nh + 2 * nkv) * hd), z(2, nh + nkv, hd, dt=torch.float32),
                    z(max_len, 2, hd, dt=torch.float32), z(2, dt=torch.int64), z(1, nkv, hd, max_len),
                    z(1, nkv, max_len, hd), z(1, nh * hd), 0.1, 1e-5, z(0, dt=torch.float32))

    for args, what in (((4, 2, 32, 64), "head_dim"), ((6, 2, 64, 64), "1, 2, 4 or 8"), ((4, 2, 64, 12), "multiple of 8"),
                       ((4, 2, 64, 4096), "workspace")):
        with pytest.raises(RuntimeError, match=what):
            call(*args)


@pytest.mark.parametrize("B,H,L,bias", [(1, 4, 3, False), (3, 252, 3, True), (1, 260, 1, False), (2, 512, 4, True),
                                        (1, 2048, 8, True), (33, 1028, 2, False)])
def test_conv_step_equals_the_bf16_ops(cuda, B, H, L, bias):
    """L + 2 steps over a ring, the outputs and the ring equal to the bf16 tensor ops on the CPU: the products are
    rounded alike and an fp32 sum of at most 8 of them differs by 2^-22 in another order, a tie apart: at most one
    bf16 step (2^-8) of the sum."""
    from lfm2opt.kernels import ext

    bf = torch.bfloat16
    g = torch.Generator().manual_seed(H + L)
    wt = torch.randn(L, H, generator=g).to(bf)
    b = torch.randn(H, generator=g).to(bf) if bias else None
    ring = torch.randn(L, B, H, generator=g).to(bf)
    dev = ring.to(cuda)
    for pos in range(5, 7 + L):
        bcx = torch.randn(B, 3 * H, generator=g).to(bf)
        out = torch.empty(B, H, dtype=bf, device=cuda)
        ext().conv_step(bcx.to(cuda), dev, wt.to(cuda), None if b is None else b.to(cuda),
                        torch.tensor([pos, 0], device=cuda), out)
        bb, cc, xx = bcx.chunk(3, -1)
        ring[pos % L] = bb * xx
        taps = torch.stack([wt[L - 1 - (pos - s) % L] for s in range(L)])
        prod = ring * taps[:, None]
        y = prod.float().sum(0).to(bf)
        y = y if b is None else y + b
        want = (cc * y).float()
        assert torch.equal(dev.cpu(), ring)
        step = 2.0 ** -7 * (cc.float() * prod.float().abs().sum(0)).abs()
        assert ((out.cpu().float() - want).abs() <= step).all()
        assert (out.cpu().float() != want).float().mean() <= 0.01


@pytest.mark.parametrize("B,V", [(1, 8), (1, 2048), (2, 2056), (9, 4096), (33, 65536), (70, 6000)])
def test_step_tail_equals_the_torch_ops(cuda, B, V):
    """Tokens, output row, counters and the fp32 copy equal copy_ / masked_fill_ / argmax / index_copy_ / add_, with ties
    (within a chunk and across), blocked maxima, NaN, infinities and both zeros; the workspace serves every call."""
    from lfm2opt.kernels import ext

    E, g = ext(), torch.Generator().manual_seed(V)
    ws = E.step_tail_workspace(B, V, cuda)
    block = torch.zeros(V, dtype=torch.bool)
    block[[0, V - 1, V // 2]] = True
    ctr, out = torch.tensor([5, 0], device=cuda), torch.full((3, B), -1, device=cuda)
    tok = torch.zeros(B, dtype=torch.long, device=cuda)
    for row in range(5):
        x = torch.randint(-8, 9, (B, V), generator=g).to(torch.bfloat16)  # many ties
        if row == 1:
            x[:, V // 2] = 100.0  # blocked
        elif row == 2:
            x[0] = float("-inf")
            x[-1, torch.randint(V, (2,), generator=g)] = float("nan")
        elif row == 3:
            x = -x.abs()  # -0 and 0 tie
            x[:, torch.randint(V, (V // 2,), generator=g)] = 0.0
        copy = torch.empty(B, V, device=cuda)
        E.step_tail(x.to(cuda), block.to(cuda), copy, tok, out, ctr, ws, set_pos=9 if row == 4 else -1)
        want = x.float().masked_fill(block, float("-inf")).argmax(-1)
        assert torch.equal(tok.cpu(), want)
        assert torch.equal(copy.cpu().view(torch.int32), x.float().view(torch.int32))
        if row < 3:
            assert torch.equal(out[row].cpu(), want) and (out[row + 1:] == -1).all()
        assert ctr.tolist() == ([9, 1] if row == 4 else [6 + row, 1 + row])
    assert torch.equal(out[0].cpu(), want)  # the call with set_pos wrote row 0, the one at row 3 of 3 nothing


@pytest.mark.parametrize("B,H", [(1, 8), (3, 520), (17, 2048)])
def test_embed_step(cuda, B, H):
    from lfm2opt.kernels import ext

    g = torch.Generator().manual_seed(H)
    table = torch.randn(100, H, generator=g).to(torch.bfloat16)
    tok = torch.randint(100, (B,), generator=g)
    h = torch.empty(B, H, dtype=torch.bfloat16, device=cuda)
    ext().embed_step(table.to(cuda), tok.to(cuda), h)
    assert torch.equal(h.cpu(), table[tok])
    tok[-1] = 100
    ext().embed_step(table.to(cuda), tok.to(cuda), h)
    assert h[-1].isnan().all() and torch.equal(h[:-1].cpu(), table[tok[:-1]])
