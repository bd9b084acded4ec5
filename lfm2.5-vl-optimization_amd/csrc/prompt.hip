// The non-matmul ops of a whole-prompt pass of LFM2 on gfx950:
//   prompt_qkv   q / k head RMSNorm and rotary embedding in place, keys and values into the cache, values transposed
//   prompt_attn  causal attention over the prompt on the bf16 matrix cores; bf16 output or the next W8A8 layer's input
//   prompt_conv  the gated short convolution over the prompt and its ring; bf16 output or the next W8A8 layer's input
//
// Reference: the prompt passes of src/lfm2opt/runtime.py:335-418 (transformers' attention and short convolution there).
#include "common.hpp"
#include "quantize.hpp"
#include "status.hpp"

#include <algorithm>

namespace lfm2q {
namespace {

constexpr int HD = 64;         // head_dim
constexpr int DPP_XOR3 = 0x1b;  // quad_perm [3, 2, 1, 0]

// ------------------------------------------------------------------------------------------------ q / k / v
// One workgroup per (32 positions, kv head, batch row): thread t holds dims 8 (t % 8) .. + 7 of position t / 8, so a head
// is 8 lanes (the squares' sum and the rotary partner, dims + 32, are DPP permutations). The group's q heads and the k head
// are normalized, rotated (fp32, rounded once) and written back in place; keys go to the cache transposed and values
// transposed to vt through LDS. vt [B, nkv, 64, Tp]: Tp = T rounded up to 64, zero past T, positions of each 16 in the
// order 0-3, 8-11, 4-7, 12-15: the order in which prompt_attn's lanes hold their probabilities. MI355X, 32
// heads over 8: 7.8 us at 461 positions and 10.2 at 2,048, in place of twelve PyTorch launches (norm, swap, products,
// transposes, cache copies).
constexpr int QP = 32;

__global__ __launch_bounds__(256) void prompt_qkv_kernel(uint16_t *qkv, const float *__restrict__ qkw,
                                                         const float *__restrict__ rope, uint16_t *__restrict__ kc,
                                                         uint16_t *__restrict__ vc, uint16_t *__restrict__ vt, int T,
                                                         int Tp, int nkv, int grp, int max_len, float eps) {
    const int t = threadIdx.x, r = t >> 3, d0 = 8 * (t & 7);
    const int p0 = blockIdx.x * QP, p = p0 + r, kv = blockIdx.y, b = blockIdx.z;
    const int nh = nkv * grp, rows = nh + nkv, ld = (nh + 2 * nkv) * HD;
    const bool in = p < T;
    uint16_t *row = qkv + ((size_t)b * T + (in ? p : T - 1)) * ld + d0;
    __shared__ __attribute__((aligned(16))) uint16_t tile[2][QP][HD + 8];  // keys, values
    {
        const v4i v = in ? ld16(row + (rows + kv) * HD) : v4i{0, 0, 0, 0};
        *reinterpret_cast<v4i *>(&tile[1][r][d0]) = v;
        if (in) *reinterpret_cast<v4i *>(vc + (((size_t)b * nkv + kv) * max_len + p) * HD + d0) = v;
    }
    float c[8], s[8];
    const float *rp = rope + (size_t)(in ? p : T - 1) * 2 * HD + d0;
#pragma unroll
    for (int e = 0; e < 8; ++e) c[e] = rp[e], s[e] = rp[HD + e];
    for (int h = 0; h <= grp; ++h) {  // the q heads, then the k head
        const int head = h < grp ? kv * grp + h : nh + kv;
        const v4i xv = ld16(row + head * HD);
        const float *w = qkw + (size_t)head * HD + d0, *wb = qkw + (size_t)(rows + head) * HD + d0;
        float x[8], ss = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[2 * e] = bf2f_lo((uint32_t)xv[e]), x[2 * e + 1] = bf2f_hi((uint32_t)xv[e]);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(x[e], x[e], ss);
        ss += dpp<DPP_XOR1>(ss);
        ss += dpp<DPP_XOR2>(ss);
        ss += dpp<DPP_HALF_MIRROR>(ss);
        const float rs = 1.f / sqrtf(ss * (1.f / HD) + eps);
        v4i o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float y[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int i = 2 * e + k;
                const float n = x[i] * rs, other = dpp<DPP_XOR3>(dpp<DPP_HALF_MIRROR>(n));  // lane ^ 4
                y[k] = n * (w[i] * c[i]) + other * (wb[i] * s[i]);
            }
            o[e] = (int)pack_bf16x2(y[0], y[1]);
        }
        if (in) *reinterpret_cast<v4i *>(row + head * HD) = o;
        if (h == grp) *reinterpret_cast<v4i *>(&tile[0][r][d0]) = o;
    }
    __syncthreads();
    const int d = t >> 2, q0 = 8 * (t & 3);  // one dim, 8 positions
    v4i kt, vv;
    const int v0 = (q0 & ~15) + ((q0 & 8) ? 4 : 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        kt[e] = (int)((uint32_t)tile[0][q0 + 2 * e][d] | (uint32_t)tile[0][q0 + 2 * e + 1][d] << 16);
        const int pv = v0 + (e < 2 ? 2 * e : 8 + 2 * (e - 2));
        vv[e] = (int)((uint32_t)tile[1][pv][d] | (uint32_t)tile[1][pv + 1][d] << 16);
    }
    *reinterpret_cast<v4i *>(vt + (((size_t)b * nkv + kv) * HD + d) * Tp + p0 + q0) = vv;
    uint16_t *kd = kc + (((size_t)b * nkv + kv) * HD + d) * max_len + p0 + q0;
    if (p0 + q0 + 8 <= T) {
        *reinterpret_cast<v4i *>(kd) = kt;
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (p0 + q0 + e < T) kd[e] = (uint16_t)((uint32_t)kt[e >> 1] >> (16 * (e & 1)));
    }
}

// ------------------------------------------------------------------------------------------------ attention
// One workgroup of 4 wavefronts per (32 x 4 / GW positions, GW = min(grp, 4) query heads of a kv head, batch row); a
// wavefront takes 32 positions of one head against key / value tiles of 64 positions, staged in LDS for all four (two
// buffers; 16-byte chunks XOR-swizzled by row), with an online softmax in fp32.
// S^T = K Q^T (mfma 32x32x16) leaves each lane one query's scores (16 of 32 positions, the other lane half the rest), so
// the row maximum, its correction and the sum stay in the lane, and the probabilities, rounded to bf16, are the next
// product's operand (O^T = V^T P^T) in the registers they are in: vt's order of positions is the lanes'. Bound by the
// softmax's VALU work (an exponential costs 16 cycles a wavefront; 64 dims give each only two short products). MI355X, 32
// heads over 8: 16.0 us at 461 positions and 53.4 at 2,048; the PyTorch ops that this kernel and prompt_qkv replace (norm,
// rotary embedding, masked products, softmax, copies) took about 120 and 560.
template <int GW, bool QUANT>
__global__ __launch_bounds__(256) void prompt_attn_kernel(const uint16_t *__restrict__ qkv,
                                                          const uint16_t *__restrict__ vt, uint16_t *__restrict__ out,
                                                          int8_t *__restrict__ oq, float *__restrict__ os, int T, int Tp,
                                                          int nkv, int grp, int tiles, int round, float scale_log2) {
    constexpr int PW = 32 * 4 / GW;  // positions per workgroup
    constexpr int KT = 64;           // positions per tile
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, half = lane >> 5, col = lane & 31;
    // workgroups of one kv head on one XCD where there are 8; the longest tiles first, then alternately in rising and
    // falling order, so that the workgroups that meet on a CU are about equally long together
    const int parts = grp / GW, kv = blockIdx.x % nkv, part = blockIdx.x / nkv % parts, rank = blockIdx.y, b = blockIdx.z;
    const int rd = rank / round, in_rd = rank % round, len = min(round, tiles - rd * round);
    const int tile = tiles - 1 - (rd * round + ((rd & 1) ? len - 1 - in_rd : in_rd));
    const int head = kv * grp + part * GW + wave % GW;
    const int q0 = tile * PW + 32 * (wave / GW);  // this wavefront's first position
    const int nh = nkv * grp, ld = (nh + 2 * nkv) * HD;
    const int lastq = min(tile * PW + PW, T) - 1, nt = lastq / KT + 1;
    const uint16_t *base = qkv + (size_t)b * T * ld;
    const uint16_t *kb = base + (nh + kv) * HD;
    const uint16_t *vb = vt + ((size_t)b * nkv + kv) * HD * Tp;

    __shared__ __attribute__((aligned(16))) uint16_t lk[2][KT * HD], lv[2][HD * KT];
    const int sr = t >> 2, sc = 2 * (t & 3);  // staging: row, first of two 16-byte chunks
    v4i kr[2], vr[2];
    auto load = [&](int p0) {
        const uint16_t *k = kb + (size_t)min(p0 + sr, T - 1) * ld + sc * 8;
        const uint16_t *v = vb + (size_t)sr * Tp + p0 + sc * 8;
        kr[0] = ld16(k), kr[1] = ld16(k + 8), vr[0] = ld16(v), vr[1] = ld16(v + 8);
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int o = sr * 64 + 8 * ((sc + j) ^ (sr & 7));
            *reinterpret_cast<v4i *>(&lk[buf][o]) = kr[j];
            *reinterpret_cast<v4i *>(&lv[buf][o]) = vr[j];
        }
    };
    auto frag = [&](const uint16_t *l, int row, int chunk) {
        return __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i *>(&l[row * 64 + 8 * (chunk ^ (row & 7))]));
    };
    load(0);
    v8bf qf[4];
    const int q = q0 + col;  // this lane's query position
    {
        const uint16_t *qp = base + (size_t)min(q, T - 1) * ld + head * HD + 8 * half;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qf[ks] = __builtin_bit_cast(v8bf, ld16(qp + 16 * ks));
    }
    store(0);
    typedef float v16f __attribute__((ext_vector_type(16)));
    v16f o[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) o[0][i] = o[1][i] = 0.f;
    float m = -__builtin_inff(), l = 0.f;
    for (int it = 0; it < nt; ++it) {
        const int p0 = it * KT, buf = it & 1;
        __syncthreads();
        if (it + 1 < nt) load(p0 + KT);
        if (p0 <= q0 + 31) {  // uniform in the wavefront; false only past its last position
            v16f s[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int i = 0; i < 16; ++i) s[u][i] = 0.f;
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
                    s[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(lk[buf], 32 * u + col, 2 * ks + half), qf[ks],
                                                                   s[u], 0, 0, 0);
            }
            if (p0 + KT - 1 > q0) {
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (p0 + 32 * u + 8 * (i >> 2) + 4 * half + (i & 3) > q) s[u][i] = -__builtin_inff();
            }
            float mt = m;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < 16; ++i) mt = fmaxf(mt, s[u][i]);
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
            mt = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
            if (__builtin_amdgcn_ballot_w64(mt != m)) {
                const float a = __builtin_amdgcn_exp2f((m - mt) * scale_log2);  // 0 at the first tile
                m = mt;
                l *= a;
#pragma unroll
                for (int i = 0; i < 16; ++i) o[0][i] *= a, o[1][i] *= a;
            }
            const float mc = m * scale_log2;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    float e[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        e[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][8 * cc + i], scale_log2, -mc));
                        l += e[i];
                    }
                    const v4i pk = {(int)pack_bf16x2(e[0], e[1]), (int)pack_bf16x2(e[2], e[3]),
                                    (int)pack_bf16x2(e[4], e[5]), (int)pack_bf16x2(e[6], e[7])};
                    const v8bf pf = __builtin_bit_cast(v8bf, pk);
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt)
                        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            frag(lv[buf], 32 * dt + col, 4 * u + 2 * cc + half), pf, o[dt], 0, 0, 0);
                }
        }
        if (it + 1 < nt) store(buf ^ 1);
    }
    const auto ls = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    const float inv = 1.f / (__uint_as_float(ls[0]) + __uint_as_float(ls[1]));
    // dims 32 dt + 8 j + 4 half + 0..3 of query q
    uint32_t w[2][4][2];
    float am = 0.f;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t v = pack_bf16x2(o[dt][4 * j + 2 * k] * inv, o[dt][4 * j + 2 * k + 1] * inv);
                w[dt][j][k] = v;
                if (QUANT) am = fmaxf(am, fmaxf(fabsf(bf2f_lo(v)), fabsf(bf2f_hi(v))));
            }
    const size_t orow = (size_t)b * T + q;
    if constexpr (QUANT) {  // a head is one group of 64 columns: quant_groups of the bf16 output
        const auto sa = __builtin_amdgcn_permlane32_swap(__float_as_uint(am), __float_as_uint(am), false, false);
        const float scl = scale_of(fmaxf(__uint_as_float(sa[0]), __uint_as_float(sa[1]))), rc = 1.f / scl;
        if (q < T && half == 0) os[(size_t)head * ((size_t)gridDim.z * T) + orow] = scl;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                int lo, hi;
                quant8(v4i{(int)w[dt][j][0], (int)w[dt][j][1], (int)w[dt][j + 1][0], (int)w[dt][j + 1][1]}, scl, rc, lo,
                       hi);
                if (q < T) {
                    int8_t *qp = oq + orow * nh * HD + head * HD + 32 * dt + 8 * j + 4 * half;
                    *reinterpret_cast<int *>(qp) = lo;
                    *reinterpret_cast<int *>(qp + 8) = hi;
                }
            }
    } else {
        if (q < T) {
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *reinterpret_cast<uint2 *>(out + orow * nh * HD + head * HD + 32 * dt + 8 * j + 4 * half) =
                        make_uint2(w[dt][j][0], w[dt][j][1]);
        }
    }
}

// ------------------------------------------------------------------------------------------------ short convolution
// Thread: 8 channels of CP consecutive positions (the L - 1 before them read again, from the cache). bcx [B T, 3 H] = b |
// c | x; with u = b x rounded, y = sum over the taps of rounded products (fp32, newest last as the decode step's taps), the
// bias, times c, each rounded as the bf16 tensor ops round. The last L positions' u become the ring's rows (position p in
// row p mod L; rows of positions before the prompt zero). Bound by memory: 4 H values in and out a position. MI355X,
// 2,048 channels, with the quantized output: 7.8 us at 461 positions and 12.0 at 2,048, in place of ten PyTorch launches
// (41 and 59 us) and the quantizer (3.7 and 5.6).
constexpr int CP = 4;

template <int L, bool QUANT>
__global__ __launch_bounds__(256) void prompt_conv_kernel(const uint16_t *__restrict__ bcx,
                                                          const uint16_t *__restrict__ wt,
                                                          const uint16_t *__restrict__ bias, uint16_t *__restrict__ ring,
                                                          uint16_t *__restrict__ out, int8_t *__restrict__ oq,
                                                          float *__restrict__ os, int T, int H) {
#pragma clang fp contract(off)
    const int c = 8 * (blockIdx.y * 256 + threadIdx.x), p0 = blockIdx.x * CP, b = blockIdx.z, B = gridDim.z;
    if (c >= H) return;  // (with QUANT whole groups of 8 lanes: H % 64 == 0)
    const uint16_t *base = bcx + (size_t)b * T * 3 * H + c;
    v4i vb[L - 1 + CP], vx[L - 1 + CP], vc[CP], wv[L];
#pragma unroll
    for (int i = 0; i < L - 1 + CP; ++i) {
        const int p = p0 - (L - 1) + i;
        const bool ok = p >= 0 && p < T;
        const uint16_t *r = base + (size_t)(ok ? p : 0) * 3 * H;
        vb[i] = ok ? ld16(r) : v4i{0, 0, 0, 0};
        vx[i] = ok ? ld16(r + 2 * H) : v4i{0, 0, 0, 0};
        if (i >= L - 1) vc[i - (L - 1)] = ok ? ld16(r + H) : v4i{0, 0, 0, 0};
    }
#pragma unroll
    for (int j = 0; j < L; ++j) wv[j] = ld16(wt + (size_t)j * H + c);
    const v4i bv = bias ? ld16(bias + c) : v4i{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < L - 1 + CP; ++i) {  // u = bf16(b x), in vb
#pragma unroll
        for (int e = 0; e < 4; ++e)
            vb[i][e] = (int)pack_bf16x2(bf2f_lo((uint32_t)vb[i][e]) * bf2f_lo((uint32_t)vx[i][e]),
                                        bf2f_hi((uint32_t)vb[i][e]) * bf2f_hi((uint32_t)vx[i][e]));
        const int p = p0 - (L - 1) + i;
        const bool first = p < 0 && p0 == 0;  // before the prompt: zero rows, written by the first workgroup
        if ((i >= L - 1 ? p < T : first) && p >= T - L)
            *reinterpret_cast<v4i *>(ring + ((size_t)((p + L) % L) * B + b) * H + c) = vb[i];
    }
#pragma unroll
    for (int i = 0; i < CP; ++i) {
        const int p = p0 + i;
        v4i o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float y[2] = {0.f, 0.f};
#pragma unroll
            for (int j = 0; j < L; ++j) {
                y[0] += rbf(bf2f_lo((uint32_t)vb[i + j][e]) * bf2f_lo((uint32_t)wv[j][e]));
                y[1] += rbf(bf2f_hi((uint32_t)vb[i + j][e]) * bf2f_hi((uint32_t)wv[j][e]));
            }
            y[0] = rbf(y[0]), y[1] = rbf(y[1]);
            if (bias) y[0] = rbf(y[0] + bf2f_lo((uint32_t)bv[e])), y[1] = rbf(y[1] + bf2f_hi((uint32_t)bv[e]));
            o[e] = (int)pack_bf16x2(bf2f_lo((uint32_t)vc[i][e]) * y[0], bf2f_hi((uint32_t)vc[i][e]) * y[1]);
        }
        const size_t row = (size_t)b * T + p;
        if constexpr (QUANT) {
            const float sc = scale_of(max8(absmax8(o, 0.f))), rc = 1.f / sc;
            int lo, hi;
            quant8(o, sc, rc, lo, hi);
            if (p < T) {
                if ((threadIdx.x & 7) == 0) os[(size_t)(c >> 6) * ((size_t)B * T) + row] = sc;
                *reinterpret_cast<int2 *>(oq + row * H + c) = make_int2(lo, hi);
            }
        } else {
            if (p < T) *reinterpret_cast<v4i *>(out + row * H + c) = o;
        }
    }
}

}  // namespace
}  // namespace lfm2q

using namespace lfm2q;

extern "C" size_t lfm2q_prompt_attn_workspace_bytes(int B, int T, int n_kv) {
    if (B < 1 || T < 1 || n_kv < 1) return 0;
    return (size_t)B * n_kv * HD * ((T + 63) / 64 * 64) * 2;
}

extern "C" int lfm2q_prompt_attn(lfm2q_bf16 *qkv, const float *qk_w, const float *rope, lfm2q_bf16 *k, lfm2q_bf16 *v,
                                 lfm2q_bf16 *out, int8_t *oq, float *os, int B, int T, int n_heads, int n_kv,
                                 int head_dim, int max_len, float scale, float eps, void *ws, size_t ws_bytes,
                                 lfm2q_stream_t stream) {
    LFM2Q_REQUIRE(qkv && qk_w && rope && k && v && (out || (oq && os)), LFM2Q_ERR_ARG, "prompt_attn: null pointer");
    LFM2Q_REQUIRE(!out || (!oq && !os), LFM2Q_ERR_ARG, "prompt_attn: out, or oq and os, not both");
    LFM2Q_REQUIRE(head_dim == HD, LFM2Q_ERR_SHAPE, "prompt_attn: head_dim must be %d (%d)", HD, head_dim);
    LFM2Q_REQUIRE(B >= 1 && B <= 65535 && T >= 1 && n_kv >= 1 && n_kv <= 65535 && n_heads >= 1 && n_heads <= 65535 &&
                      n_heads % n_kv == 0,
                  LFM2Q_ERR_SHAPE, "prompt_attn: bad B / T / heads (%d, %d, %d, %d)", B, T, n_heads, n_kv);
    LFM2Q_REQUIRE((int64_t)B * T < (1ll << 31) && T <= 65535 * 32, LFM2Q_ERR_SHAPE, "prompt_attn: B T too large");
    const int grp = n_heads / n_kv;
    LFM2Q_REQUIRE(grp == 1 || grp == 2 || grp == 4 || grp == 8, LFM2Q_ERR_SHAPE,
                  "prompt_attn: query heads per kv head must be 1, 2, 4 or 8 (%d)", grp);
    LFM2Q_REQUIRE(max_len >= T && max_len % 8 == 0, LFM2Q_ERR_SHAPE,
                  "prompt_attn: max_len must be a multiple of 8 and hold the prompt (%d, T=%d)", max_len, T);
    LFM2Q_REQUIRE(scale > 0.f, LFM2Q_ERR_ARG, "prompt_attn: scale must be positive");
    LFM2Q_REQUIRE(aligned16(qkv) && aligned16(k) && aligned16(v) && aligned16(out) && aligned16(oq) && aligned16(ws),
                  LFM2Q_ERR_ALIGN, "prompt_attn: qkv, k, v, outputs and ws must be 16-byte aligned");
    LFM2Q_REQUIRE(ws && ws_bytes >= lfm2q_prompt_attn_workspace_bytes(B, T, n_kv), LFM2Q_ERR_ARG,
                  "prompt_attn: workspace smaller than lfm2q_prompt_attn_workspace_bytes()");
    const hipStream_t st = (hipStream_t)stream;
    uint16_t *vt = static_cast<uint16_t *>(ws);
    const int Tp = (T + 63) / 64 * 64, gw = std::min(grp, 4), pw = 32 * 4 / gw, tiles = (T + pw - 1) / pw;
    prompt_qkv_kernel<<<dim3(Tp / QP, n_kv, B), 256, 0, st>>>(qkv, qk_w, rope, k, v, vt, T, Tp, n_kv, grp, max_len, eps);
    const int heads = n_kv * (grp / gw), round = std::max(1, (int)(device_cus() / ((long)heads * B)));
    const dim3 grid(heads, tiles, B);
    const float sl = scale * 1.44269504088896341f;
#define LFM2Q_PATTN(G_)                                                                                                \
    case G_:                                                                                                           \
        if (out)                                                                                                       \
            prompt_attn_kernel<G_, false><<<grid, 256, 0, st>>>(qkv, vt, out, nullptr, nullptr, T, Tp, n_kv, grp,      \
                                                                tiles, round, sl);                                     \
        else                                                                                                           \
            prompt_attn_kernel<G_, true><<<grid, 256, 0, st>>>(qkv, vt, nullptr, oq, os, T, Tp, n_kv, grp, tiles,      \
                                                               round, sl);                                             \
        break;
    switch (gw) {
        LFM2Q_PATTN(1)
        LFM2Q_PATTN(2)
        LFM2Q_PATTN(4)
    }
#undef LFM2Q_PATTN
    return launch_status("prompt_attn");
}

extern "C" int lfm2q_prompt_conv(const lfm2q_bf16 *bcx, const lfm2q_bf16 *wt, const lfm2q_bf16 *bias, lfm2q_bf16 *ring,
                                 lfm2q_bf16 *out, int8_t *oq, float *os, int B, int T, int H, int L,
                                 lfm2q_stream_t stream) {
    LFM2Q_REQUIRE(bcx && wt && ring && (out || (oq && os)), LFM2Q_ERR_ARG, "prompt_conv: null pointer");
    LFM2Q_REQUIRE(!out || (!oq && !os), LFM2Q_ERR_ARG, "prompt_conv: out, or oq and os, not both");
    LFM2Q_REQUIRE(B >= 1 && B <= 65535 && T >= 1 && (int64_t)B * T < (1ll << 31) && H >= 8 && H % 8 == 0 &&
                      H <= 65535 * 2048 && (out || H % 64 == 0),
                  LFM2Q_ERR_SHAPE, "prompt_conv: bad shape (B=%d T=%d H=%d; H %% 8, quantized H %% 64)", B, T, H);
    LFM2Q_REQUIRE(aligned16(bcx) && aligned16(wt) && aligned16(bias) && aligned16(ring) && aligned16(out) && aligned16(oq),
                  LFM2Q_ERR_ALIGN, "prompt_conv: tensors must be 16-byte aligned");
    const hipStream_t st = (hipStream_t)stream;
    const dim3 grid((T + CP - 1) / CP, (H / 8 + 255) / 256, B);
#define LFM2Q_PCONV(L_)                                                                                          \
    case L_:                                                                                                     \
        if (out)                                                                                                 \
            prompt_conv_kernel<L_, false><<<grid, 256, 0, st>>>(bcx, wt, bias, ring, out, nullptr, nullptr, T, H); \
        else                                                                                                     \
            prompt_conv_kernel<L_, true><<<grid, 256, 0, st>>>(bcx, wt, bias, ring, nullptr, oq, os, T, H);        \
        break;
    switch (L) {
        LFM2Q_PCONV(1)
        LFM2Q_PCONV(2)
        LFM2Q_PCONV(3)
        LFM2Q_PCONV(4)
        LFM2Q_PCONV(5)
        LFM2Q_PCONV(6)
        LFM2Q_PCONV(7)
        LFM2Q_PCONV(8)
    default: return set_error(LFM2Q_ERR_SHAPE, "prompt_conv: need 1 <= L <= 8 (%d)", L);
    }
#undef LFM2Q_PCONV
    return launch_status("prompt_conv");
}
