"""Extension entry points with the reference's Python surface, backed by the gfx950 library liblfm2q.so.

`ext()` stands in for the JIT-built decode extension and `int8_ext()` for the INT8 GEMM extension of
src/lfm2opt/kernels.py:16-32,66-68. The ops keep their names, argument order and meaning, destination-passing
style (every output is preallocated by the caller, ops return None) and launch on torch's current stream. Argument
errors raise RuntimeError with the reference's TORCH_CHECK wording (kernels/lfm2_decode.cpp:28-150) before any
launch. The reference's attention and convolution ops are not provided under its names; the decode step's and the prompt
pass's have kernels of their own (attn_step, conv_step, prompt_attn, ...). The hot ops' checks and calls are native
(_capi.native()).
"""

import ctypes
import os

import torch

from . import _capi

# The per-stream GEMM workspace (the K split across workgroups): create it on a capture stream before capturing,
# release it when a stream is retired.
prepare_workspace = _capi.prepare_workspace
release_workspace = _capi.release_workspace

_EXT = None


def _check_bf16(t, name):
    if not (t.is_cuda and t.dtype == torch.bfloat16 and t.is_contiguous()):
        raise RuntimeError(f"{name} must be contiguous CUDA bf16")


def _check_t(t, dtype, name):
    if not (t.is_cuda and t.dtype == dtype and t.is_contiguous()):
        raise RuntimeError(f"{name} must be contiguous CUDA {dtype}")


def _same_device(*ts):
    dev = ts[0].device
    for t in ts[1:]:
        if t is not None and t.device != dev:
            raise RuntimeError("all tensors must be on the same device")


class DecodeOps:
    """Decode-path ops (reference: kernels/lfm2_decode.cpp)."""

    def __init__(self):
        self._n = _capi.native()
        self.pdl = True
        self.gemv_impl = 1

    # ---- reference ops ------------------------------------------------------------------------------------
    def gemv(self, W, scale, x, y, rows=0):
        """y [B, N] = x [B, K] @ W^T, W [N, K] bf16 or int8 (then scale [N] fp32 is required); any B >= 1.
        Reference: gemv(), kernels/lfm2_decode.cpp:74-85. rows: output rows per wavefront for B == 1."""
        self._n.gemv(W, scale, x, y, int(rows))

    def gemv_epi(self, epi, W, scale, x, y, state=None, cw=None, cbias=None):
        """epi 0: W = w1|w3 [2S, K] -> y [B, S] = silu(w1 x) * (w3 x), fused into the GEMV.
        Reference: gemv_epi(), kernels/lfm2_decode.cpp:130-150 (batch 1 there; any B >= 1 here). epi 1 (the LFM2
        short-conv step) is not a matmul epilogue and is not provided by this library."""
        if epi != 0:
            if epi == 1:
                raise RuntimeError("gemv_epi: epi 1 (short-conv step) is outside the quantized-matmul library")
            raise RuntimeError("epi 0 (swiglu) or 1 (shortconv)")
        W, scale, B, S, K, wtype = self._epi_args(W, scale, x, y, rows_per_out=2)
        _capi.call("lfm2q_gemv_swiglu", wtype, W.data_ptr(), _capi.ptr(scale), x.data_ptr(), y.data_ptr(), B, S, K,
                   _capi.stream(x))

    def gemv_w4(self, Wp, S, x, y, rows=0, epi=0):
        """INT4 weight-only GEMV in the reference format: Wp uint8 [R, K/2] (two int4 + 8 per byte, weight 2j in the
        low nibble of byte j), S fp32 [R, K/group]; y [B, N] = x [B, K] @ dequant(Wp)^T with R = N.
        Reference: gemv_w4(), kernels/lfm2_decode.cpp:86-98 (batch 1 there; any B >= 1 here). rows is accepted for
        the reference's signature and has no effect. epi (an addition): 0 plain, 1 SwiGLU over Wp = w1|w3
        (R = 2N, y [B, N]), 2 residual add in place into y."""
        self._n.gemv_w4(Wp, S, x, y, epi)

    def gemv_w4z(self, qweight, scales, qzeros, x, y, epi=0):
        """INT4 weight-only GEMV in GPTQ-style storage (an addition): qweight int32 [R, K/8] (nibble i of word w =
        q for k = 8 w + i, q in [0, 15]), scales fp16 [R, K/group], qzeros int32 [R, ceil(K/group/8)] (nibble j of
        word w = zero point of group 8 w + j); w = s (q - z). epi as in gemv_w4."""
        self._n.gemv_w4z(qweight, scales, qzeros, x, y, epi)

    @staticmethod
    def _w4_group(S, R, K):
        if not (S.dim() == 2 and S.size(0) == R and S.size(1) >= 1 and K % S.size(1) == 0):
            raise RuntimeError("S must be [N, K / group]")
        group = K // S.size(1)
        if group <= 0 or group % 32:
            raise RuntimeError("group size must be a multiple of 32")
        return group

    def silu_mul(self, g, y):
        """y = silu(a) * b on g = [a | b]; reference: silu_mul(), kernels/lfm2_decode.cpp:100-103."""
        self._n.silu_mul(g, y)

    def gemv_chain(self, ops):
        """A GemvChain over ops [(epi, W, scale, x, y), ...] (an addition): call it to run all of them in one launch."""
        return GemvChain(ops)

    def set_pdl(self, on):
        """Accepted for compatibility (kernels/lfm2_decode.cpp:165); HIP has no programmatic dependent launch,
        back-to-back kernels on one stream are ordered by the stream and captured into HIP graphs instead."""
        self.pdl = bool(on)

    def set_gemv_impl(self, impl):
        """Accepted for compatibility (kernels/lfm2_decode.cpp:166): there is one GEMV implementation per batch
        size class here, so the choice between shared-memory and direct activation loads has no effect."""
        if impl not in (0, 1):
            raise RuntimeError("GEMV implementation: 0 = x staged in shared memory, 1 = direct x loads")
        self.gemv_impl = int(impl)

    # ---- additions ----------------------------------------------------------------------------------------
    def gemv_rmsnorm(self, W, scale, h, norm_w, eps, y, epi=0):
        """The batch-1 GEMV of RMSNorm(h) (an addition): x = bf16(norm_w * bf16(h * rsqrt(mean(h^2) + eps))) is
        formed inside the GEMV, then y [1, N] = x @ W^T * scale (epi 0) or the SwiGLU of x over W = w1|w3 (epi 1, y
        [1, N] from W [2N, K]). Bit-identical to add_rmsnorm (no residual input) followed by gemv / gemv_epi(0), the
        pair the reference's decode step runs before each of these linears (src/lfm2opt/runtime.py:251-255,
        :276-285). h, norm_w bf16 [K]; W int8 (K in 1024 .. 8192, powers of two, fp32 scale) or bf16 (K in 512 ..
        4096, scale optional)."""
        _check_bf16(h, "h")
        _check_bf16(norm_w, "norm_w")
        _check_bf16(y, "y")
        if epi not in (0, 1):
            raise RuntimeError("gemv_rmsnorm: epi 0 (none) or 1 (swiglu)")
        if not (W.is_cuda and W.is_contiguous() and W.dim() == 2 and W.dtype in (torch.int8, torch.bfloat16)):
            raise RuntimeError("W must be a contiguous CUDA bf16 or int8 matrix")
        int8 = W.dtype == torch.int8
        R, K = W.shape
        N = R // 2 if epi == 1 else R
        if int8 and (scale is None or scale.dtype != torch.float32):
            raise RuntimeError("int8 W needs fp32 scale")
        if scale is not None:
            _check_t(scale, torch.float32, "scale")
            if scale.numel() != R:
                raise RuntimeError("scale must have one value per weight row")
        if (epi == 1 and R % 2) or h.numel() != K or norm_w.numel() != K or y.numel() != N:
            raise RuntimeError("gemv_rmsnorm: h [1, K], norm_w [K], y [1, N] (batch 1)")
        _same_device(W, h, norm_w, y, scale)
        _capi.call("lfm2q_gemv_rmsnorm", 0 if int8 else 1, int(epi), W.data_ptr(), _capi.ptr(scale), h.data_ptr(),
                   norm_w.data_ptr(), float(eps), y.data_ptr(), N, K, _capi.stream(h))

    def gemv_w4_rmsnorm(self, Wp, S, zeros, h, norm_w, eps, y, epi=0):
        """The batch-1 INT4 GEMV of RMSNorm(h) (an addition), as gemv_rmsnorm: Wp, S as in gemv_w4 (zeros None) or
        gemv_w4z; epi 0 or 1 (SwiGLU). Bit-identical to add_rmsnorm (no residual input), then that GEMV. 128 <= K <= 2048."""
        for t, name in ((h, "h"), (norm_w, "norm_w"), (y, "y")):
            _check_bf16(t, name)
        fmt, per = (0, 2) if zeros is None else (1, 8)
        wdt, sdt = (torch.uint8, torch.float32) if fmt == 0 else (torch.int32, torch.float16)
        _check_t(Wp, wdt, "Wp")
        _check_t(S, sdt, "S")
        if epi not in (0, 1) or Wp.dim() != 2:
            raise RuntimeError("gemv_w4_rmsnorm: Wp [R, K / 2] or [R, K / 8], epi 0 (none) or 1 (swiglu)")
        R, K = Wp.size(0), Wp.size(1) * per
        group = self._w4_group(S, R, K)
        if fmt == 1:
            _check_t(zeros, torch.int32, "zeros")
            if tuple(zeros.shape) != (R, (K // group + 7) // 8):
                raise RuntimeError("qzeros: contiguous int32 [N, ceil(K/group/8)]")
        N = R // 2 if epi == 1 else R
        if (epi == 1 and R % 2) or h.numel() != K or norm_w.numel() != K or y.numel() != N:
            raise RuntimeError("gemv_w4_rmsnorm: h [1, K], norm_w [K], y [1, N] (batch 1)")
        _same_device(Wp, S, zeros, h, norm_w, y) if fmt == 1 else _same_device(Wp, S, h, norm_w, y)
        _capi.call("lfm2q_gemv_w4_rmsnorm", fmt, Wp.data_ptr(), S.data_ptr(), _capi.ptr(zeros), h.data_ptr(),
                   norm_w.data_ptr(), float(eps), y.data_ptr(), N, K, group, int(epi), _capi.stream(h))

    def gemv_conv_rmsnorm(self, W, scale, zeros, h, norm_w, eps, ring, wt, bias, ctr, out):
        """The batch-1 projection of a short-conv layer and its conv step in one launch (an addition): the GEMV of
        RMSNorm(h) over W = b | c | x [3 H, K] (INT8 or bf16 with its scale, or INT4 as in gemv_w4_rmsnorm), then conv_step
        of it with ring [3, 1, H]; bit-identical to that pair. Replaces gemv_epi(1, ...), kernels/lfm2_decode.cpp:130-150,
        with the norm before it."""
        for t, name in ((h, "h"), (norm_w, "norm_w"), (ring, "ring"), (wt, "wt"), (out, "out")):
            _check_bf16(t, name)
        _check_t(ctr, torch.int64, "ctr")
        if bias is not None:
            _check_bf16(bias, "bias")
        if not (W.is_cuda and W.is_contiguous() and W.dim() == 2 and ring.dim() == 3):
            raise RuntimeError("gemv_conv_rmsnorm: W [3 H, K] contiguous, ring [L, 1, H]")
        per = {torch.int8: 1, torch.bfloat16: 1, torch.uint8: 2, torch.int32: 8}.get(W.dtype)
        if per is None:
            raise RuntimeError("W must be int8, bf16, uint8 (INT4) or int32 (INT4)")
        R, K = W.size(0), W.size(1) * per
        L, B, H = ring.shape
        if not (R == 3 * H and B == 1 and h.numel() == K and norm_w.numel() == K and tuple(wt.shape) == (L, H)
                and out.numel() == H and ctr.numel() >= 1 and (bias is None or bias.numel() == H)):
            raise RuntimeError("gemv_conv_rmsnorm: W [3 H, K], h [1, K], ring [L, 1, H], wt [L, H], out [1, H] (batch 1)")
        tail = (h.data_ptr(), norm_w.data_ptr(), float(eps), ring.data_ptr(), wt.data_ptr(), _capi.ptr(bias),
                ctr.data_ptr(), out.data_ptr(), H, K)
        if per == 1:
            if W.dtype == torch.int8 and scale is None:
                raise RuntimeError("int8 W needs fp32 scale")
            if scale is not None:
                _check_t(scale, torch.float32, "scale")
                if scale.numel() != R:
                    raise RuntimeError("scale must have one value per weight row")
            _same_device(W, scale, h, norm_w, ring, wt, bias, ctr, out)
            _capi.call("lfm2q_gemv_conv_rmsnorm", 0 if W.dtype == torch.int8 else 1, W.data_ptr(), _capi.ptr(scale), *tail,
                       L, _capi.stream(h))
            return
        fmt = 0 if per == 2 else 1
        _check_t(scale, torch.float32 if fmt == 0 else torch.float16, "S")
        group = self._w4_group(scale, R, K)
        if fmt == 1:
            _check_t(zeros, torch.int32, "zeros")
            if tuple(zeros.shape) != (R, (K // group + 7) // 8):
                raise RuntimeError("qzeros: contiguous int32 [N, ceil(K/group/8)]")
        _same_device(W, scale, zeros, h, norm_w, ring, wt, bias, ctr, out)
        _capi.call("lfm2q_gemv_w4_conv_rmsnorm", fmt, W.data_ptr(), scale.data_ptr(), _capi.ptr(zeros), *tail, group, L,
                   _capi.stream(h))

    def add_rmsnorm(self, h, y, w, x, eps):
        """h += y (optional, in place, bf16-rounded); x = bf16(w * bf16(rmsnorm(h))): add_rmsnorm_q's h and x without the
        INT8 row. Reference: add_rmsnorm(), kernels/lfm2_decode.cpp:33-38."""
        for t, name in ((h, "h"), (w, "w"), (x, "x")):
            _check_bf16(t, name)
        H = h.size(-1)
        if not (w.numel() == H and H % 8 == 0 and 0 < H <= 8192 and h.numel() > 0 and x.numel() == h.numel()):
            raise RuntimeError("add_rmsnorm: h, x [rows, H], w [H] (H % 8 == 0, H <= 8192)")
        if y is not None:
            _check_bf16(y, "y")
            if y.numel() != h.numel():
                raise RuntimeError("y shape")
        _same_device(h, y, w, x)
        _capi.call("lfm2q_add_rmsnorm", h.data_ptr(), _capi.ptr(y), w.data_ptr(), x.data_ptr(), h.numel() // H, H,
                   float(eps), _capi.stream(h))

    def gemv_residual(self, W, scale, x, h):
        """h [B, N] += bf16(x @ W^T * scale) in place, rounded as the reference's residual add
        (kernels/lfm2_decode.cu:108-113): h = bf16(h + bf16(acc * s))."""
        W, scale, B, N, K, wtype = self._epi_args(W, scale, x, h, rows_per_out=1)
        _capi.call("lfm2q_gemv_residual", wtype, W.data_ptr(), _capi.ptr(scale), x.data_ptr(), h.data_ptr(), B, N,
                   K, _capi.stream(x))

    @staticmethod
    def attn_step_workspace(B, n_heads, n_kv, max_len, device):
        """The workspace attn_step needs for this shape (fp32; may be empty). Calls that share one must not overlap."""
        n = _capi.lib().lfm2q_attn_step_workspace_bytes(B, n_heads, n_kv, max_len)
        return torch.empty(n // 4, dtype=torch.float32, device=device)

    def attn_step(self, qkv, qk_w, rope, ctr, k, v, out, scale, eps, ws):
        """One decode step's attention of one layer (an addition): q / k head RMSNorm and rotary embedding of qkv
        [B, (nh + 2 nkv) 64], the new key and value into k [B, nkv, 64, max_len] / v [B, nkv, max_len, 64] at position
        ctr[0], out [B, nh 64] = attention over positions 0 .. ctr[0]. qk_w fp32 [2, nh + nkv, 64], rope fp32 [max_len,
        2, 64], ctr int64 (lfm2q_attn_step). Replaces the step's attention ops, src/lfm2opt/runtime.py:256-271."""
        for t, name in ((qkv, "qkv"), (k, "k"), (v, "v"), (out, "out")):
            _check_bf16(t, name)
        for t, dt, name in ((qk_w, torch.float32, "qk_w"), (rope, torch.float32, "rope"), (ctr, torch.int64, "ctr"),
                            (ws, torch.float32, "ws")):
            _check_t(t, dt, name)
        if not (k.dim() == 4 and v.dim() == 4 and qk_w.dim() == 3):
            raise RuntimeError("attn_step: k [B, nkv, hd, max_len], v [B, nkv, max_len, hd], qk_w [2, nh + nkv, hd]")
        B, nkv, hd, max_len = k.shape
        nh = qk_w.size(1) - nkv
        if not (tuple(v.shape) == (B, nkv, max_len, hd) and qk_w.size(0) == 2 and qk_w.size(2) == hd and nh >= 1
                and qkv.numel() == B * (nh + 2 * nkv) * hd and out.numel() == B * nh * hd
                and rope.numel() >= max_len * 2 * hd and ctr.numel() >= 1):
            raise RuntimeError("attn_step: shapes")
        _same_device(qkv, qk_w, rope, ctr, k, v, out, ws)
        _capi.call("lfm2q_attn_step", qkv.data_ptr(), qk_w.data_ptr(), rope.data_ptr(), ctr.data_ptr(), k.data_ptr(),
                   v.data_ptr(), out.data_ptr(), B, nh, nkv, hd, max_len, float(scale), float(eps), ws.data_ptr(),
                   ws.numel() * 4, _capi.stream(qkv))

    def conv_step(self, bcx, ring, wt, bias, ctr, out):
        """One decode step of a gated short convolution (an addition): bcx [B, 3 H] = b | c | x, b x into row ctr[0] mod L
        of ring [L, B, H], out [B, H] = c (conv of the ring with the taps wt [L, H] + bias), rounded as the bf16 tensor
        ops (lfm2q_conv_step). Replaces the short-conv epilogue of gemv_epi(1, ...), kernels/lfm2_decode.cpp:130-150,
        without its projection."""
        for t, name in ((bcx, "bcx"), (ring, "ring"), (wt, "wt"), (out, "out")):
            _check_bf16(t, name)
        _check_t(ctr, torch.int64, "ctr")
        if bias is not None:
            _check_bf16(bias, "bias")
        if ring.dim() != 3:
            raise RuntimeError("conv_step: ring [L, B, H]")
        L, B, H = ring.shape
        if not (bcx.numel() == 3 * B * H and tuple(wt.shape) == (L, H) and out.numel() == B * H and ctr.numel() >= 1
                and (bias is None or bias.numel() == H)):
            raise RuntimeError("conv_step: bcx [B, 3H], ring [L, B, H], wt [L, H], out [B, H]")
        _same_device(bcx, ring, wt, bias, ctr, out)
        _capi.call("lfm2q_conv_step", bcx.data_ptr(), ring.data_ptr(), wt.data_ptr(), _capi.ptr(bias), ctr.data_ptr(),
                   out.data_ptr(), B, H, L, _capi.stream(bcx))

    def embed_step(self, table, tok, h):
        """h [B, H] = rows tok [B] (int64) of table [V, H], bf16 (an addition; lfm2q_embed_step)."""
        _check_bf16(table, "table")
        _check_bf16(h, "h")
        _check_t(tok, torch.int64, "tok")
        if not (table.dim() == 2 and h.numel() == tok.numel() * table.shape[1]):
            raise RuntimeError("embed_step: table [V, H], tok [B], h [B, H]")
        _same_device(table, tok, h)
        _capi.call("lfm2q_embed_step", table.data_ptr(), tok.data_ptr(), h.data_ptr(), tok.numel(), table.shape[1],
                   table.shape[0], _capi.stream(h))

    @staticmethod
    def step_tail_workspace(B, V, device):
        """A zeroed workspace for step_tail. Calls that share one must not overlap."""
        n = _capi.lib().lfm2q_step_tail_workspace_bytes(B, V)
        return torch.zeros(n // 8, dtype=torch.int64, device=device)

    def step_tail(self, logits, block, copy, tok, out, ctr, ws, set_pos=-1):
        """The end of a greedy decode step (an addition; lfm2q_step_tail): copy [B, V] fp32 (or None) = logits [B, V]
        bf16, tok [B] = argmax of the logits not blocked (block [V] bool), row ctr[1] of out [max_new, B] = tok, ctr +=
        1; with set_pos >= 0 row 0 and ctr = (set_pos, 1)."""
        _check_bf16(logits, "logits")
        _check_t(block, torch.bool, "block")
        for t, name in ((tok, "tok"), (out, "out"), (ctr, "ctr"), (ws, "ws")):
            _check_t(t, torch.int64, name)
        if copy is not None:
            _check_t(copy, torch.float32, "copy")
        if not (logits.dim() == 2 and out.dim() == 2):
            raise RuntimeError("step_tail: logits [B, V], out [max_new, B]")
        B, V = logits.shape
        if not (block.numel() == V and tok.numel() == B and out.shape[1] == B and ctr.numel() == 2
                and (copy is None or copy.numel() == B * V)):
            raise RuntimeError("step_tail: block [V], copy [B, V], tok [B], out [max_new, B], ctr [2]")
        _same_device(logits, block, copy, tok, out, ctr, ws)
        _capi.call("lfm2q_step_tail", logits.data_ptr(), block.data_ptr(), _capi.ptr(copy), tok.data_ptr(),
                   out.data_ptr(), ctr.data_ptr(), B, V, out.shape[0], int(set_pos), ws.data_ptr(), ws.numel() * 8,
                   _capi.stream(logits))

    def prompt_attn(self, qkv, qk_w, rope, k, v, out, scale, eps):
        """Causal attention over a whole prompt (an addition): qkv [B, T, (nh + 2 nkv) 64] normalized and rotated IN
        PLACE, its keys and values into k [B, nkv, 64, max_len] / v [B, nkv, max_len, 64], out = bf16 [B T, nh 64] or
        (int8 [B T, nh 64], scales [nh, B T]), the grouped input of the next W8A8 layer (lfm2q_prompt_attn). Replaces the
        attention of the reference's prefill, src/lfm2opt/runtime.py:335-418."""
        for t, name in ((qkv, "qkv"), (k, "k"), (v, "v")):
            _check_bf16(t, name)
        for t, name in ((qk_w, "qk_w"), (rope, "rope")):
            _check_t(t, torch.float32, name)
        if not (qkv.dim() == 3 and k.dim() == 4 and v.dim() == 4 and qk_w.dim() == 3):
            raise RuntimeError("prompt_attn: qkv [B, T, (nh + 2 nkv) hd], k [B, nkv, hd, max_len], v [B, nkv, max_len, hd]")
        B, T, W = qkv.shape
        nkv, hd, max_len = k.shape[1:]
        nh = qk_w.shape[1] - nkv
        if not (W == (nh + 2 * nkv) * hd and tuple(qk_w.shape) == (2, nh + nkv, hd) and k.shape[0] == B
                and tuple(v.shape) == (B, nkv, max_len, hd) and rope.numel() >= T * 2 * hd and T <= max_len):
            raise RuntimeError("prompt_attn: qkv [B, T, (nh + 2 nkv) hd], qk_w [2, nh + nkv, hd], rope [>= T, 2, hd]")
        y, q, s = self._prompt_out(out, B * T, nh * hd)
        _same_device(qkv, qk_w, rope, k, v, y, q, s)
        n = _capi.lib().lfm2q_prompt_attn_workspace_bytes(B, T, nkv)
        ws = torch.empty(n, dtype=torch.uint8, device=qkv.device)
        _capi.call("lfm2q_prompt_attn", qkv.data_ptr(), qk_w.data_ptr(), rope.data_ptr(), k.data_ptr(), v.data_ptr(),
                   _capi.ptr(y), _capi.ptr(q), _capi.ptr(s), B, T, nh, nkv, hd, max_len, float(scale), float(eps),
                   ws.data_ptr(), n, _capi.stream(qkv))

    def prompt_conv(self, bcx, ring, wt, bias, out):
        """The gated short convolution over a whole prompt (an addition): bcx [B, T, 3 H] = b | c | x, the last L
        positions' b x into ring [L, B, H], out = bf16 [B T, H] or (int8 [B T, H], scales [H / 64, B T])
        (lfm2q_prompt_conv). Replaces the short convolution of the reference's prefill, src/lfm2opt/runtime.py:335-418."""
        for t, name in ((bcx, "bcx"), (ring, "ring"), (wt, "wt")):
            _check_bf16(t, name)
        if bias is not None:
            _check_bf16(bias, "bias")
        if not (bcx.dim() == 3 and ring.dim() == 3):
            raise RuntimeError("prompt_conv: bcx [B, T, 3H], ring [L, B, H]")
        B, T, W = bcx.shape
        L, H = ring.shape[0], ring.shape[2]
        if not (W == 3 * H and ring.shape[1] == B and tuple(wt.shape) == (L, H) and (bias is None or bias.numel() == H)):
            raise RuntimeError("prompt_conv: bcx [B, T, 3H], ring [L, B, H], wt [L, H], bias [H]")
        y, q, s = self._prompt_out(out, B * T, H)
        _same_device(bcx, ring, wt, bias, y, q, s)
        _capi.call("lfm2q_prompt_conv", bcx.data_ptr(), wt.data_ptr(), _capi.ptr(bias), ring.data_ptr(), _capi.ptr(y),
                   _capi.ptr(q), _capi.ptr(s), B, T, H, L, _capi.stream(bcx))

    @staticmethod
    def _prompt_out(out, rows, cols):
        """(bf16 output, int8 output, its scales), the absent ones None."""
        if isinstance(out, tuple):
            q, s = out
            _check_t(q, torch.int8, "q")
            _check_t(s, torch.float32, "s")
            if not (cols % 64 == 0 and q.numel() == rows * cols and tuple(s.shape) == (cols // 64, rows)):
                raise RuntimeError("output: int8 [rows, cols], scales [cols / 64, rows]")
            return None, q, s
        _check_bf16(out, "out")
        if out.numel() != rows * cols:
            raise RuntimeError("output: [rows, cols]")
        return out, None, None

    def _epi_args(self, W, scale, x, y, rows_per_out):
        _check_bf16(x, "x")
        _check_bf16(y, "y")
        if not (W.is_cuda and W.is_contiguous() and W.dim() == 2):
            raise RuntimeError("W must be a contiguous CUDA matrix")
        int8 = W.dtype == torch.int8
        if not (int8 or W.dtype == torch.bfloat16):
            raise RuntimeError("W must be bf16 or int8")
        if int8 and (scale is None or scale.dtype != torch.float32):
            raise RuntimeError("int8 W needs fp32 scale")
        Nw, K = W.shape
        Nout = Nw // rows_per_out
        B = x.numel() // K if K else 0
        if not (Nw == rows_per_out * Nout and B >= 1 and x.numel() == B * K and y.numel() == B * Nout):
            raise RuntimeError("x [B, K], y [B, N]" if rows_per_out == 1 else "x [B, K], W [2S, K], y [B, S]")
        if scale is not None:
            _check_t(scale, torch.float32, "scale")
            if scale.numel() != Nw:
                raise RuntimeError("scale must have one element per row of W")
        _same_device(W, x, y, scale)
        return W, scale, B, Nout, K, 0 if int8 else 1


class GemvChain:
    """A fixed sequence of batch-1 INT8 GEMVs run as one launch (lfm2q_gemv_chain): op j may read anything ops
    0 .. j-1 wrote; every output equals the separate gemv / gemv_epi(0) / gemv_residual call bit for bit.

    ops: (epi, W, scale, x, y) per GEMV -- epi 0 y = x W^T s, 1 SwiGLU over W = w1|w3 (y [1, S]), 2 y += x W^T s in
    place; W int8 [R, K] with K in {1024, 2048, 4096, 8192}, scale fp32 [R], x bf16 [1, K], y bf16 [1, N]. The
    tensors are kept alive and their addresses fixed in the table, so the chain is replayed on the same buffers
    (graph-capturable: one kernel launch, no allocation). The op table is copied to the device and a workspace
    allocated once, here."""

    def __init__(self, ops):
        if not ops:
            raise RuntimeError("gemv_chain: at least one op")
        lib = _capi.lib()
        self._keep, table = [], []
        dev = None
        for j, (epi, W, scale, x, y) in enumerate(ops):
            if epi not in (0, 1, 2):
                raise RuntimeError(f"gemv_chain: op {j}: epi 0 (none), 1 (swiglu) or 2 (residual)")
            _check_t(W, torch.int8, f"op {j}: W")
            _check_t(scale, torch.float32, f"op {j}: scale")
            _check_bf16(x, f"op {j}: x")
            _check_bf16(y, f"op {j}: y")
            R, K = W.shape
            N = R // 2 if epi == 1 else R
            if (epi == 1 and R % 2) or scale.numel() != R or x.numel() != K or y.numel() != N:
                raise RuntimeError(f"gemv_chain: op {j}: x [1, K], W [{'2N' if epi == 1 else 'N'}, K], y [1, N]")
            _same_device(W, scale, x, y)
            if dev is not None and W.device != dev:
                raise RuntimeError("all tensors must be on the same device")
            dev = W.device
            self._keep += [W, scale, x, y]
            table.append(_capi.GemvOp(W.data_ptr(), scale.data_ptr(), x.data_ptr(), y.data_ptr(), N, K, epi, 0))
        self.n = len(table)
        self.host = (_capi.GemvOp * self.n)(*table)
        self.dev = torch.frombuffer(bytearray(bytes(self.host)), dtype=torch.uint8).to(dev)
        self.ws_bytes = lib.lfm2q_gemv_chain_workspace_bytes()
        self.ws = torch.zeros(-(-self.ws_bytes // 4), dtype=torch.int32, device=dev)
        self.device = dev

    def __call__(self):
        with torch.cuda.device(self.device):
            _capi.call("lfm2q_gemv_chain", ctypes.addressof(self.host), self.dev.data_ptr(), self.n,
                       self.ws.data_ptr(), self.ws_bytes, torch.cuda.current_stream(self.device).cuda_stream)

    def wait_expired(self):
        """True if a dependency wait of the last launch on this chain ran out (its outputs are then undefined; the
        launches after it are not affected). Reads the workspace's launch count and error tag on the host
        (synchronizes)."""
        gen, tag = (int(v) for v in self.ws[:2].tolist())
        return gen != 0 and tag == gen


class Int8Ops:
    """INT8 prefill / vision ops (reference: kernels/int8_gemm.cpp): quantizers, fused producers, the W8A8 GEMM with
    per-token or grouped-64 activation scales, its INT8-output form gemm_i8_q, and the W8A16 gemm_w8."""

    def __init__(self):
        self._n = _capi.native()

    def gemm_i8(self, xq, sx, w, sw, bias, y, gelu):
        """W8A8: y [M, N] = bf16(gelu?((xq . w^T) * sx[m] * sw[n] + bias[n])), exact int32 accumulation; with 2-D sx
        [K/64, M] (grouped-64 activation scales) the per-group sums fold into fp32 with their scales first.
        Reference: gemm_i8(), kernels/int8_gemm.cpp:39-50."""
        self._n.gemm_i8(xq, sx, w, sw, bias, y, gelu)

    def gemm_i8_bf16a(self, x, sx, w, sw, bias, y, gelu):
        """The per-token pair quant_rows(x) + gemm_i8 as one call on bf16 activations x [M, K]: sx [M] receives the
        scales quant_rows would write, the GEMM quantizes x inside (no int8 copy of x), and y is bit-identical to
        the pair's. Reference pair: src/lfm2opt/int8.py:45-51 (quantize_rows, then gemm_i8)."""
        _check_bf16(x, "x")
        _check_t(sx, torch.float32, "sx")
        K = x.size(-1)
        M = x.numel() // K if K else 0
        if sx.numel() != M:
            raise RuntimeError("sx shape")
        N = self._check_common(w, sw, bias, y, M, K)
        _same_device(x, sx, w, sw, bias, y)
        _capi.call("lfm2q_gemm_i8_bf16a", x.data_ptr(), sx.data_ptr(), w.data_ptr(), sw.data_ptr(), _capi.ptr(bias),
                   y.data_ptr(), M, N, K, int(bool(gelu)), _capi.stream(x))

    def gemm_i8_fq(self, x, xq, sx, w, sw, bias, y, gelu):
        """The per-token pair quant_rows(x) -> (xq, sx), then gemm_i8, behind one call with the stream's workspace;
        xq, sx and y are bit-identical to the pair's. By default the library runs the pair; with the tuning knob
        LFM2Q_GEMM_FQ = 1 the persistent GEMM's workgroups quantize x first and then run the tiles, in one launch.
        Reference pair: src/lfm2opt/int8.py:45-51 (quantize_rows, then gemm_i8)."""
        _check_bf16(x, "x")
        _check_t(xq, torch.int8, "xq")
        _check_t(sx, torch.float32, "sx")
        K = x.size(-1)
        M = x.numel() // K if K else 0
        if xq.numel() != M * K or xq.size(-1) != K:
            raise RuntimeError("xq shape")
        if sx.numel() != M:
            raise RuntimeError("sx shape")
        N = self._check_common(w, sw, bias, y, M, K)
        _same_device(x, xq, sx, w, sw, bias, y)
        ws = _capi.workspace(x)
        _capi.call("lfm2q_gemm_i8_fq", x.data_ptr(), xq.data_ptr(), sx.data_ptr(), w.data_ptr(), sw.data_ptr(),
                   _capi.ptr(bias), y.data_ptr(), M, N, K, int(bool(gelu)), ws.data_ptr(), ws.numel(),
                   _capi.stream(x))

    def gemm_i8_q(self, xq, sxT, w, sw, bias, yq, ysT, gelu):
        """Grouped W8A8 writing the next W8A8 GEMM's input: (yq [M, N], ysT [N/64, M]) = quant_groups(the bf16 output
        gemm_i8 would write), bit-identical to that pair of calls. Reference: gemm_i8_q(), kernels/int8_gemm.cpp:53-69
        (N % 128 there, N % 64 here)."""
        self._n.gemm_i8_q(xq, sxT, w, sw, bias, yq, ysT, gelu)

    def gemm_w8(self, x, w, sw, bias, y, gelu):
        """W8A16: y [M, N] = bf16(gelu?((x . w^T) * sw[n] + bias[n])), bf16 x, int8 w, fp32 accumulation.
        Reference: gemm_w8(), kernels/int8_gemm.cpp:72-79."""
        self._n.gemm_w8(x, w, sw, bias, y, gelu)

    def gemm_i8_i32(self, xq, w, c):
        """The exact int32 accumulators c [M, N] = xq [M, K] . w [N, K]^T (the torch._int_mm analogue)."""
        _check_t(xq, torch.int8, "xq")
        _check_t(w, torch.int8, "w")
        _check_t(c, torch.int32, "c")
        K = xq.size(-1)
        M = xq.numel() // K if K else 0
        if not (w.dim() == 2 and w.size(1) == K):
            raise RuntimeError("w must be [N, K]")
        N = w.size(0)
        if c.numel() != M * N:
            raise RuntimeError("c shape")
        if K % 16:
            raise RuntimeError("need K % 16 == 0")
        _same_device(xq, w, c)
        _capi.call("lfm2q_gemm_i8_i32", xq.data_ptr(), w.data_ptr(), c.data_ptr(), M, N, K, _capi.stream(xq))

    def quant_rows(self, x, q, s):
        """Symmetric quantization: s = max|x| / 127, q = round(x / s), per row (1-D s [rows]) or per row and group of
        64 columns (2-D s [K/64, rows], transposed as gemm_i8 reads it). Reference: quant_rows(),
        kernels/int8_gemm.cpp:83-96 (K % 128 and, per row, K <= 2048 there; K % 8, grouped K % 64, any K here)."""
        self._n.quant_rows(x, q, s)

    # ---- fused producers (kernels/int8_gemm.cpp:99-141). x (an addition): also write the bf16 row that was
    # quantized; q / s are then exactly quant_rows(x, ...) of it.
    def add_layernorm_q(self, h, y, w, b, q, s, eps, x=None):
        """vision: h += y (optional, in place, bf16-rounded); (q, s) = quant(LayerNorm(h) * w + b).
        Reference: add_layernorm_q(), kernels/int8_gemm.cpp:108-119 (D % 128, D <= 2048 there; D % 8, D <= 8192)."""
        self._n.add_layernorm_q(h, y, w, b, q, s, eps, x)

    def add_rmsnorm_q(self, h, y, w, q, s, eps, x=None):
        """LM prefill: h += y (optional, in place, bf16-rounded); (q, s) = quant(bf16(w * bf16(rmsnorm(h)))).
        Reference: add_rmsnorm_q(), kernels/int8_gemm.cpp:122-132 (H <= 8192 here)."""
        self._n.add_rmsnorm_q(h, y, w, q, s, eps, x)

    def silu_mul_q(self, g, q, s, x=None):
        """LM prefill: g [rows, 2I] = w1 | w3 outputs -> (q, s) = quant(bf16(bf16(silu(g1)) * g3)).
        Reference: silu_mul_q(), kernels/int8_gemm.cpp:135-141 (I % 64, I <= 20000 there; I % 8, I <= 8192)."""
        self._n.silu_mul_q(g, q, s, x)

    @staticmethod
    def _check_common(w, sw, bias, y, M, K):
        """kernels/int8_gemm.cpp:22-36 (N % 8 is not required here)."""
        _check_t(w, torch.int8, "w")
        _check_t(sw, torch.float32, "sw")
        _check_bf16(y, "y")
        if not (w.dim() == 2 and w.size(1) == K):
            raise RuntimeError("w must be [N, K]")
        N = w.size(0)
        if K % 16:
            raise RuntimeError("need K % 16 == 0")
        if not (sw.numel() == N and y.numel() == M * N):
            raise RuntimeError("sw / y shape")
        if bias is not None:
            _check_bf16(bias, "bias")
            if bias.numel() != N:
                raise RuntimeError("bias shape")
        return N


_INT8 = None


def int8_ext():
    """INT8 GEMM ops for prefill and the vision encoder (reference: src/lfm2opt/kernels.py:66-68)."""
    global _INT8
    if _INT8 is None:
        _INT8 = Int8Ops()
    return _INT8


def ext():
    """The decode-op extension (reference: src/lfm2opt/kernels.py:16-32). LFM2_PDL is read like the reference
    does; it has no effect on HIP."""
    global _EXT
    if _EXT is None:
        _EXT = DecodeOps()
        _EXT.set_pdl(os.environ.get("LFM2_PDL", "1") != "0")
    return _EXT
